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
    const int wib = wave_in_block_id();
    const int64_t first = team > 1 ? (int64_t)blockIdx.x : global_wave_id();
    const int64_t step = team > 1 ? (int64_t)gridDim.x : (int64_t)gridDim.x * (blockDim.x / kWave);
    for (int64_t b = first * rows_per_batch; b < p.n; b += step * rows_per_batch) {
        const int64_t e = b + rows_per_batch < p.n ? b + rows_per_batch : p.n;
        fetch_wide_batch<T, IdxT, LAYOUT, NT>(p, b, e, team, team > 1 ? wib : 0,
                                            lds[team > 1 ? 0 : wib]);
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

int fetch_wide_launch(const FetchParams &p, int layout, int elem_bytes, int index_bytes, int nblks, hipStream_t stream)
{
    const DeviceInfo &dev = device_info();
    const int64_t nchunks = (p.vec_size * elem_bytes + 511) / 512;
    // Full batches where they still give the chip its 16 waves per CU with
    // teams of eight, and the smallest team that gives it twice that, since a
    // smaller team shares fewer barriers (20,000 rows of eight chunks: teams
    // of 2, 4, 8 take 32.9, 29.8, 34.4 us; 4096 rows of 43 chunks: teams of 4
    // and 8 take 53 and 45 us).
    const int most = nchunks <= 1 ? 1 : nchunks <= 2 ? 2 : nchunks <= 4 ? 4 : kWideMaxTeam;
    int rows = kWideRows;
    while (rows > 1 && (p.n + rows - 1) / rows * most < (int64_t)dev.num_cus * 16) rows /= 2;
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
