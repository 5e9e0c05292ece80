// ibp_fetch_wide.hip -- the plain fetch of rows of more than 64 elements of 4 or 8 bytes
// (ibp_fetch_wide.h), in every layout.
#include "ibp_fetch_wide.h"
#include "ibp_internal.h"

namespace ibp {

// Batches of rows_per_batch rows.  team > 1: a block is one team; team = 1:
// each of a block's waves takes its own batches.
template <typename T, typename IdxT, int LAYOUT, bool NT>
__global__ __launch_bounds__(64 * kWideMaxTeam, 4) void fetch_wide_kernel(FetchParams p, int team, int rows_per_batch)
{
    __shared__ uint32_t lds[kWideSolo][kWideLdsWords];
    // With clusters: fewer rows of one mask row cost more in a batch than in a
    // wave each, unless their window is so small that the team's other waves
    // would have none (500 rows of 2752 words: 18 us against 51).
    const int least = rows_per_batch <= 2 ? 1 : rows_per_batch <= 4 ? 2 : 4;
    const int wib = wave_in_block_id();
    const int64_t first = team > 1 ? (int64_t)blockIdx.x : global_wave_id();
    const int64_t step = team > 1 ? (int64_t)gridDim.x : (int64_t)gridDim.x * (blockDim.x / kWave);
    for (int64_t b = first * rows_per_batch; b < p.n; b += step * rows_per_batch) {
        const int64_t e = b + rows_per_batch < p.n ? b + rows_per_batch : p.n;
        fetch_wide_batch<T, IdxT, LAYOUT, NT>(p, b, e, team, team > 1 ? wib : 0,
                                              lds[team > 1 ? 0 : wib], least);
    }
}

namespace {

template <typename T, typename IdxT, int LAYOUT>
void launch_stores(const FetchParams &p, dim3 g, dim3 b, int team, int rows, hipStream_t s)
{
    if ((p.vec_size * (int64_t)sizeof(T)) % 128 == 0) // rows_fill_lines
        hipLaunchKernelGGL((fetch_wide_kernel<T, IdxT, LAYOUT, true>), g, b, 0, s, p, team, rows);
    else
        hipLaunchKernelGGL((fetch_wide_kernel<T, IdxT, LAYOUT, false>), g, b, 0, s, p, team, rows);
}

template <typename T, typename IdxT>
void launch_layout(const FetchParams &p, int layout, dim3 g, dim3 b, int team, int rows, hipStream_t s)
{
    switch (layout) {
    case kLayoutSlots: launch_stores<T, IdxT, kLayoutSlots>(p, g, b, team, rows, s); break;
    case kLayoutCondensed: launch_stores<T, IdxT, kLayoutCondensed>(p, g, b, team, rows, s); break;
    case kLayoutClustered: launch_stores<T, IdxT, kLayoutClustered>(p, g, b, team, rows, s); break;
    default: launch_stores<T, IdxT, kLayoutCondensed | kLayoutClustered>(p, g, b, team, rows, s); break;
    }
}

} // namespace

// A batch's setup and barriers have to be earned.  One mask row: from 512
// columns on always (200 rows of 600 words: a wave per row 8.8 us, teams 5.9;
// of 400: 7.0 and 8.1 at 1000 rows), below from 8 MB of rows on (60,000 rows of
// 118 words 28 and 22 us, 8000 6.8 and 9.5; 12,000 rows of 256 words 12.8 and
// 9.6, 4000 6.6 and 8.5).  A mask row per cluster: rows of 6 KB and more
// (8192 rows of 2500 doubles with 16 of them: 135 and 85, 249 and 96, 120 and
// 82 us on weights, node features and embeddings, whose rows mostly share few
// mask rows; 107 and 140 where the sixteen are evenly used; of 500 doubles 34
// and 38).
bool fetch_wide_pays(const FetchParams &p, int layout, int elem_bytes)
{
    if (p.vec_size <= kWave || elem_bytes < 4) return false;
    const int64_t row_bytes = p.vec_size * elem_bytes;
    if (layout & kLayoutClustered) return row_bytes >= 6144;
    return p.vec_size >= 512 || p.n >= ((int64_t)8 << 20) / row_bytes;
}

int fetch_wide_launch(const FetchParams &p, int layout, int elem_bytes, int index_bytes, int nblks, hipStream_t stream)
{
    const DeviceInfo &dev = device_info();
    const int64_t nchunks = (p.vec_size * elem_bytes + 511) / 512;
    // The smallest batches (windows, with clusters) that run in one round of
    // 16 waves per CU with teams of eight, and the smallest team that gives
    // the chip twice that, since a smaller team shares fewer barriers (20,000
    // rows of eight chunks: teams of 2, 4, 8 take 32.9, 29.8, 34.4 us; 4096
    // rows of 43 chunks: teams of 4 and 8 take 53 and 45 us).
    const int most = nchunks <= 1 ? 1 : nchunks <= 2 ? 2 : nchunks <= 4 ? 4 : kWideMaxTeam;
    const int most_rows = (layout & kLayoutClustered) ? kWideWindow : kWideRows;
    int rows = 1;
    while (rows < most_rows && (p.n + rows - 1) / rows * most > (int64_t)dev.num_cus * 16) rows *= 2;
    int team = most < 2 ? most : 2;
    while (team < most && (p.n + rows - 1) / rows * team < (int64_t)dev.num_cus * 32) team *= 2;
    const int waves = team > 1 ? team : kWideSolo;
    int64_t grid = ((p.n + rows - 1) / rows * team + waves - 1) / waves;
    if (grid > (int64_t)1 << 20) grid = (int64_t)1 << 20;
    if (nblks > 0) grid = nblks;
    if (grid < 1) grid = 1;
    const dim3 g((unsigned)grid), b((unsigned)(waves * kWave));
    const bool i32 = p.index != nullptr && index_bytes == 4;
    if (elem_bytes == 8) {
        if (i32) launch_layout<uint64_t, int32_t>(p, layout, g, b, team, rows, stream);
        else launch_layout<uint64_t, int64_t>(p, layout, g, b, team, rows, stream);
    } else {
        if (i32) launch_layout<uint32_t, int32_t>(p, layout, g, b, team, rows, stream);
        else launch_layout<uint32_t, int64_t>(p, layout, g, b, team, rows, stream);
    }
    IBP_LAUNCH_CHECK();
    return IBP_OK;
}

} // namespace ibp
