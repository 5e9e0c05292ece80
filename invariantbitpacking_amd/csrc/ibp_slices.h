// ibp_slices.h -- rows of a row-major table read with lane <-> row, for rows of
// any length of 4-byte words from 16 bytes on: shared by the kernels that score
// or size whole rows.
//
// 64 rows (a tile) are read in slices of S chunks (16 bytes).  A slice's loads
// are 64 chunks of consecutive rows each; they go to registers while the slice
// before is worked on, then to the wave's own LDS, where lane r reads row r
// back chunk by chunk (an odd stride of chunks: no bank conflicts).  SPLIT
// waves share a tile's slices.  The last chunk of a row ends with it: where
// the row is not whole chunks, it overlaps the chunk before.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "ibp_wave.h"

namespace ibp {

__host__ __device__ constexpr int64_t row_chunks(int w, int64_t V) { return (V * w + 15) / 16; }

typedef uint32_t slice_chunk_t __attribute__((ext_vector_type(4), aligned(4)));

template <int S>
struct Slice {
    static constexpr int STRIDE = S | 1; // chunks of a row in LDS
    static_assert(S % 2 || kWave % S == 0, "");
    uint32_t offset[S]; // of load i: chunk g % S of tile row g / S, g = i * 64 + lane
    uint4 r[S];

    __device__ __forceinline__ void init(uint32_t row_bytes, int lane)
    {
#pragma unroll
        for (int i = 0; i < S; ++i) {
            const uint32_t g = (uint32_t)(i * kWave + lane);
            offset[i] = g / S * row_bytes + g % S * 16;
        }
    }
    // Starts the loads of slice s of `nslices` of a tile of `ntiles`.
    __device__ __forceinline__ void load(const void *data, int64_t rows, uint32_t row_bytes, int tile, int ntiles, int s,
                                         int nslices, int lane)
    {
        const char *base = reinterpret_cast<const char *>(data) + tile * (int64_t)kWave * (int64_t)row_bytes;
        const uint32_t at = (uint32_t)(s * S) * 16;
        if (s + 1 < nslices && tile + 1 < ntiles) { // whole (uniform)
            base += at;
#pragma unroll
            for (int i = 0; i < S; ++i) take(i, base + offset[i]);
        } else {
            // rows past the table: the last one again; the row's last chunk ends with it
            const int64_t left = rows - tile * (int64_t)kWave;
            const uint32_t last_row = left < kWave ? (uint32_t)left - 1 : kWave - 1;
            int l = lane;
            asm volatile("" : "+v"(l)); // computed here, not kept in registers
#pragma unroll
            for (int i = 0; i < S; ++i) {
                const uint32_t g = (uint32_t)(i * kWave + l);
                uint32_t row = g / S, c = at + g % S * 16;
                row = row < last_row ? row : last_row;
                c = c < row_bytes - 16 ? c : row_bytes - 16;
                take(i, base + (row * row_bytes + c));
            }
        }
    }
    __device__ __forceinline__ void store(uint4 *mine, int lane) const
    {
#pragma unroll
        for (int i = 0; i < S; ++i)
            mine[S % 2 ? i * kWave + lane : (i * (kWave / S) + lane / S) * STRIDE + lane % S] = r[i];
    }

private:
    __device__ __forceinline__ void take(int i, const char *p)
    {
        const slice_chunk_t v = *reinterpret_cast<const slice_chunk_t *>(p);
        r[i] = make_uint4(v.x, v.y, v.z, v.w);
    }
};

// f(S, SPLIT) for rows of C chunks, as integral constants: as few waves per
// tile as hold its rows in slices of at most 8 chunks, so a block loads whole
// rows at once (up to 32 chunks; 512 bytes of each row beyond); 16 waves where
// rows of more than 1 KB are so few that their tiles leave CUs idle
// (preprocess of 2292 x 741 doubles: 232 -> 104 us).
template <typename F>
void with_slices(int64_t C, int64_t ntiles, int num_cus, F f)
{
    using std::integral_constant;
    if (C <= 5) f(integral_constant<int, 5>(), integral_constant<int, 1>());
    else if (C <= 8) f(integral_constant<int, 8>(), integral_constant<int, 1>());
    else if (C <= 10) f(integral_constant<int, 5>(), integral_constant<int, 2>());
    else if (C <= 14) f(integral_constant<int, 7>(), integral_constant<int, 2>());
    else if (C <= 16) f(integral_constant<int, 8>(), integral_constant<int, 2>());
    else if (C <= 20) f(integral_constant<int, 5>(), integral_constant<int, 4>());
    else if (C <= 28) f(integral_constant<int, 7>(), integral_constant<int, 4>());
    else if (C <= 64 || ntiles > (int64_t)num_cus * 2) f(integral_constant<int, 8>(), integral_constant<int, 4>());
    else f(integral_constant<int, 8>(), integral_constant<int, 16>());
}

} // namespace ibp
