// ibp_fetch_wide.hip -- the plain fetch of rows of more than 64 elements of 4 or 8 bytes
// (ibp_fetch_wide.h), in every layout.
#include "ibp_fetch_wide.h"
#include "ibp_internal.h"

namespace ibp {

// How a kernel of teams takes its rows: in batches of rows that follow each
// other; with clusters in batches of one row, in whole windows, or the part of
// a window that shares a mask row (fetch_wide_rest_kernel takes the others).
enum : int { kBatches, kWholeWindows, kWindowParts };

// windows_pay by one wave for the block.
template <typename T, typename IdxT, int LAYOUT>
__device__ __forceinline__ bool block_windows_pay(const FetchParams &p, int rows)
{
    __shared__ int pay;
    if (wave_in_block_id() == 0) {
        const bool yes = windows_pay<T, IdxT, LAYOUT>(p, rows);
        if (lane_id() == 0) pay = yes;
    }
    __syncthreads();
    return readfirstlane((int64_t)pay) != 0;
}

// Batches (windows) of rows_per_batch rows.  team > 1: a block is one team;
// team = 1 (not with windows): each of a block's waves takes its own batches.
template <typename T, typename IdxT, int LAYOUT, bool NT, int TAKE>
__global__ __launch_bounds__(64 * kWideMaxTeam, 4) void fetch_wide_kernel(FetchParams p, int team, int rows_per_batch)
{
    __shared__ uint32_t lds[kWideSolo][kWideLdsWords];
    __shared__ __align__(8) uint32_t window[TAKE == kBatches ? 1 : kWindowLdsWords];
    const int wib = wave_in_block_id();
    if constexpr (TAKE == kWindowParts) {
        if (!block_windows_pay<T, IdxT, LAYOUT>(p, rows_per_batch)) return;
    }
    const int64_t first = team > 1 ? (int64_t)blockIdx.x : global_wave_id();
    const int64_t step = team > 1 ? (int64_t)gridDim.x : (int64_t)gridDim.x * (blockDim.x / kWave);
    for (int64_t b = first * rows_per_batch; b < p.n; b += step * rows_per_batch) {
        const int64_t e = b + rows_per_batch < p.n ? b + rows_per_batch : p.n;
        if constexpr (TAKE == kBatches)
            fetch_wide_batch<T, IdxT, LAYOUT, NT>(p, b, e, team, team > 1 ? wib : 0, lds[team > 1 ? 0 : wib]);
        else
            fetch_wide_window<T, IdxT, LAYOUT, NT, TAKE == kWholeWindows>(p, b, e, team, wib, lds[0], window);
    }
}

// A wave per row for the rows of windows of `rows` rows (a power of two) that
// the teams leave, which is all of them where windows do not pay.  (In the
// teams' kernel they had half the waves in flight, and their code cost it
// scratch memory: 8192 rows of 800 doubles of 16 evenly used mask rows 56 us, so
// 43, to which the launch that finds nothing to do adds 3; a wave per row 40.)
template <typename T, typename IdxT, int LAYOUT>
__global__ __launch_bounds__(256) void fetch_wide_rest_kernel(FetchParams p, int rows)
{
    const bool teams = block_windows_pay<T, IdxT, LAYOUT>(p, rows);
    const int64_t nwaves = (int64_t)gridDim.x * (blockDim.x / kWave);
    if (!teams) {
        fetch_large_range<T, IdxT, LAYOUT>(p, global_wave_id(), p.n, nwaves);
        return;
    }
    for (int64_t i = global_wave_id(); i < p.n; i += nwaves) {
        const int64_t b = i & ~(int64_t)(rows - 1);
        const int r = (int)(i - b);
        WideWindow<T> win;
        win.template load_window<IdxT, LAYOUT>(p, b, b + rows < p.n ? b + rows : p.n);
        if ((win.alike_rows(kWindowAlike) >> r) & 1) continue; // uniform
        fetch_large_row<T>(p, i, [&] { return win.row(r); });
    }
}

namespace {

template <typename T, typename IdxT, int LAYOUT>
void launch_stores(const FetchParams &p, const WideShape &w, int nblks, hipStream_t s)
{
    const dim3 g((unsigned)w.grid), b((unsigned)w.block);
    const int team = w.team, rows = w.rows;
    auto take = [&](auto how) {
        constexpr int TAKE = decltype(how)::value;
        if ((p.vec_size * (int64_t)sizeof(T)) % 128 == 0) // rows_fill_lines
            hipLaunchKernelGGL((fetch_wide_kernel<T, IdxT, LAYOUT, true, TAKE>), g, b, 0, s, p, team, rows);
        else
            hipLaunchKernelGGL((fetch_wide_kernel<T, IdxT, LAYOUT, false, TAKE>), g, b, 0, s, p, team, rows);
    };
    if constexpr ((LAYOUT & kLayoutClustered) != 0) {
        if (rows > kWideRows) {
            take(std::integral_constant<int, kWindowParts>());
            const int block = w.block < 256 ? w.block : 256;
            const int64_t waves = p.n < (int64_t)1 << 20 ? p.n : (int64_t)1 << 20;
            const int64_t blocks = nblks > 0 ? nblks : (waves * kWave + block - 1) / block;
            hipLaunchKernelGGL((fetch_wide_rest_kernel<T, IdxT, LAYOUT>), dim3((unsigned)blocks), dim3((unsigned)block), 0,
                               s, p, rows);
            return;
        }
        if (rows > 1) {
            take(std::integral_constant<int, kWholeWindows>());
            return;
        }
    }
    take(std::integral_constant<int, kBatches>());
}

template <typename T, typename IdxT>
void launch_layout(const FetchParams &p, int layout, const WideShape &w, int nblks, hipStream_t s)
{
    switch (layout) {
    case kLayoutSlots: launch_stores<T, IdxT, kLayoutSlots>(p, w, nblks, s); break;
    case kLayoutCondensed: launch_stores<T, IdxT, kLayoutCondensed>(p, w, nblks, s); break;
    case kLayoutClustered: launch_stores<T, IdxT, kLayoutClustered>(p, w, nblks, s); break;
    default: launch_stores<T, IdxT, kLayoutCondensed | kLayoutClustered>(p, w, nblks, s); break;
    }
}

} // namespace

// A batch's setup and barriers have to be earned.  One mask row: from 512
// columns on always (200 rows of 600 words: a wave per row 8.8 us, teams 5.9;
// of 400: 7.0 and 8.1 at 1000 rows), below from 8 MB of rows on (60,000 rows of
// 118 words 28 and 22 us, 8000 6.8 and 9.5; 12,000 rows of 256 words 12.8 and
// 9.6, 4000 6.6 and 8.5).  A mask row per cluster: rows of 6 KB and more.  All
// rows of one mask row (weights, node features, embeddings mostly): 2000, 4096
// and 30,000 rows of 800 doubles 16, 23 and 130 us by a wave per row and 13, 15
// and 87 by teams, of 2752 doubles (16,000) 51, 75 and 240 and 24, 33 and 135.
// Sixteen evenly used: 16, 24, 130 and 15, 25, 140; 52, 76, 239 and 38, 76, 241;
// two (12,000 rows) 58 and 54, 181 and 112.
// (With blocks of one wave, by nthreads, a window has no team.)
// Over PCIe rows of up to three chunks of 64-bit words stay with a wave per row,
// whose reads of a row come from one wave in address order (20,000 and 60,000
// embeddings of 66 doubles in a stream 145 and 385 us, by teams 159 and 404, of
// 100 188 and 508, 195 and 532; of 129 221 and 594, 229 and 630; of 160 it turns:
// 259 and 709, 245 and 672).  Of 32-bit words teams are as fast or faster.
bool fetch_wide_pays(const FetchParams &p, int layout, int elem_bytes, int nthreads)
{
    if (p.vec_size <= kWave || elem_bytes < 4) return false;
    const int64_t row_bytes = p.vec_size * elem_bytes;
    if (layout & kLayoutClustered) return row_bytes >= 6144 && (nthreads <= 0 || nthreads >= 2 * kWave);
    if (p.host_rows && elem_bytes == 8 && p.vec_size < 160) return false;
    return p.vec_size >= 512 || p.n >= ((int64_t)8 << 20) / row_bytes;
}

WideShape fetch_wide_shape(const FetchParams &p, int layout, int elem_bytes, int nblks, int nthreads)
{
    const DeviceInfo &dev = device_info();
    const int64_t nchunks = (p.vec_size * elem_bytes + 511) / 512;
    // The smallest batches (windows, with clusters) that run in one round of
    // 16 waves per CU with teams of eight, and the smallest team that gives
    // the chip twice that, since a smaller team shares fewer barriers (20,000
    // rows of eight chunks: teams of 2, 4, 8 take 32.9, 29.8, 34.4 us; 4096
    // rows of 43 chunks: teams of 4 and 8 take 53 and 45 us).
    // Of five to seven chunks teams of eight leave waves idle, which many rows
    // feel (16,000 rows of 600 words 36 us, by teams of four 26; 2000 rows 9.2
    // and 10.3).
    int most = nchunks <= 1 ? 1 : nchunks <= 2 ? 2 : nchunks <= 4 ? 4 : kWideMaxTeam;
    if (nchunks < most && p.n >= (int64_t)dev.num_cus * 24) most = 4;
    while (nthreads > 0 && most > 1 && most * kWave > nthreads) most /= 2;
    const bool clustered = (layout & kLayoutClustered) != 0;
    const int most_rows = clustered ? kWideWindow : kWideRows;
    WideShape w{0, 0, most < 2 ? most : 2, 1};
    // With clusters and four waves or more for a row, rows by themselves: which
    // mask rows they use does not matter then (1000 rows of 800 and 2752
    // doubles: 10 and 19 us; windows of two rows of other mask rows 14 and 31).
    if (clustered && p.n * 4 <= (int64_t)dev.num_cus * 16) {
        while (w.team < most && p.n * w.team * 2 <= (int64_t)dev.num_cus * 16) w.team *= 2;
    } else {
        while (w.rows < most_rows && (p.n + w.rows - 1) / w.rows * most > (int64_t)dev.num_cus * 16) w.rows *= 2;
        while (w.team < most && (p.n + w.rows - 1) / w.rows * w.team < (int64_t)dev.num_cus * 32) w.team *= 2;
    }
    int waves = w.team > 1 ? w.team : kWideSolo;
    if (nthreads > 0 && waves * kWave > nthreads) waves = nthreads / kWave;
    w.block = waves * kWave;
    w.grid = ((p.n + w.rows - 1) / w.rows * w.team + waves - 1) / waves;
    if (w.grid > (int64_t)1 << 20) w.grid = (int64_t)1 << 20;
    if (nblks > 0) w.grid = nblks;
    if (w.grid < 1) w.grid = 1;
    return w;
}

int fetch_wide_launch(const FetchParams &p, int layout, int elem_bytes, int index_bytes, int nblks, const WideShape &w,
                      hipStream_t stream)
{
    const bool i32 = p.index != nullptr && index_bytes == 4;
    if (elem_bytes == 8) {
        if (i32) launch_layout<uint64_t, int32_t>(p, layout, w, nblks, stream);
        else launch_layout<uint64_t, int64_t>(p, layout, w, nblks, stream);
    } else {
        if (i32) launch_layout<uint32_t, int32_t>(p, layout, w, nblks, stream);
        else launch_layout<uint32_t, int64_t>(p, layout, w, nblks, stream);
    }
    IBP_LAUNCH_CHECK();
    return IBP_OK;
}

} // namespace ibp
