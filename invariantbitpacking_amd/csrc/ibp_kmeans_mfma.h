// ibp_kmeans_mfma.h -- bitwise k-means on the matrix units, for up to 16
// clusters: the assignment and the per-cluster bit counts are products of
// 0/1 matrices.
//
// A dword of 32 bits becomes four dwords of eight 4-bit floats (E2M1): part p
// holds bits p, p + 4, p + 8, ..., each where its nibble has it, so that most
// parts cost one AND: 0.5, 1.0, 2.0 for bits 0, 1, 2 of a nibble, and bit 3
// moved down to 2.0.  The other operand's parts hold the reciprocals, so each
// product of two set bits is exactly 1.0, and sums of them stay exact in the
// 32-bit float accumulators (below 2^24).  v_mfma_f32_16x16x128 then multiplies
// 16 x 32 x 4 bits with 16 x 32 x 4 bits: lane l holds the 32 bits of row (or
// column) l % 16 that belong to block l / 16 of the inner dimension; in which
// order they stand there does not matter, since both operands use the same.
// (Vector units: an XOR and a popcount-accumulate per 32 bits and centroid, 32
// operations against 5 here.)
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "ibp_wave.h"

namespace ibp {

constexpr int kMfmaK = 16; // clusters

typedef int km_frag_t __attribute__((ext_vector_type(8)));
typedef float km_acc_t __attribute__((ext_vector_type(4)));
typedef uint32_t km_load_t __attribute__((ext_vector_type(4), aligned(4)));

// 32 bits as the first operand's parts.
__device__ __forceinline__ km_frag_t frag_a(uint32_t w)
{
    km_frag_t f = {};
    f[0] = (int)(w & 0x11111111u);
    f[1] = (int)(w & 0x22222222u);
    f[2] = (int)(w & 0x44444444u);
    f[3] = (int)((w >> 1) & 0x44444444u);
    return f;
}
// ... as the second operand's: the reciprocals.
__device__ __forceinline__ km_frag_t frag_b(uint32_t w)
{
    km_frag_t f = {};
    f[0] = (int)((w << 2) & 0x44444444u);
    f[1] = (int)(w & 0x22222222u);
    f[2] = (int)((w >> 2) & 0x11111111u);
    f[3] = (int)((w >> 3) & 0x11111111u);
    return f;
}
// acc[i] of lane l: row 4 (l / 16) + i of the first operand, column l % 16 of the second.
__device__ __forceinline__ km_acc_t mfma_bits(km_frag_t a, km_frag_t b, km_acc_t c)
{
    return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b, c, 4, 4, 0, 0, 0, 0); // both 4-bit, no scales
}

// Lane l's 4 dwords of a step (16 dwords, 4 per lane group) of the row at
// `row`; `left` dwords of the row from the step's first one on.
__device__ __forceinline__ km_load_t load_step(const uint32_t *row, int64_t at, int64_t left)
{
    const int q = 4 * (lane_id() / 16);
    if (left >= 16) return *reinterpret_cast<const km_load_t *>(row + at + q); // uniform
    km_load_t v = {0u, 0u, 0u, 0u};
#pragma unroll
    for (int k = 0; k < 4; ++k)
        if (q + k < left) v[k] = row[at + q + k];
    return v;
}

// Nearest centroid of each row: the least popc(c) - 2 popc(x & c), the Hamming
// distance less the row's own popcount (pops: the centroids' popcounts); equal
// distances go to the highest index.  A tile of 16 rows per SPLIT waves, which
// share its columns (their sums meet in LDS); with SPLIT = 1 a block's four
// waves take a tile each.  Also writes the tile's members as bits: 16 rows in
// hot[c][tile].
//
// What bounds it: the rows once from L2 or memory, and the centroids once per
// tile from L2.  Against a lane per row on the vector units (with partial
// distances per column group and a kernel that sums them): 4096 rows of 8 KiB,
// 16 centroids, 15.0 + 4.7 -> 11 us.
template <int SPLIT>
__global__ __launch_bounds__(SPLIT == 1 ? 256 : 64 * SPLIT) void km_assign_mfma_kernel(
    const uint32_t *__restrict__ data, int64_t N, int64_t VD, const uint32_t *__restrict__ cent,
    const int32_t *__restrict__ pops, int K, int32_t *__restrict__ cluster, uint16_t *__restrict__ hot,
    int64_t hot_stride)
{
    constexpr int U = SPLIT == 16 ? 8 : 4; // steps whose loads are in flight together
    __shared__ int32_t sums[SPLIT > 1 ? SPLIT : 1][SPLIT > 1 ? 256 : 1];
    __shared__ uint32_t members[16];
    const int lane = lane_id(), wv = wave_in_block_id();
    const int n = lane % 16, q = lane / 16;
    const int64_t tile = SPLIT > 1 ? (int64_t)blockIdx.x : (int64_t)blockIdx.x * 4 + wv;
    if (tile * 16 >= N) { // uniform: a tile of the last 128 rows that holds none
        if (tile < hot_stride && (SPLIT == 1 || wv == 0) && lane < 16) hot[(int64_t)lane * hot_stride + tile] = 0;
        return;
    }
    if (SPLIT > 1 && threadIdx.x < 16) members[threadIdx.x] = 0;
    int64_t r = tile * 16 + n;
    if (r >= N) r = N - 1; // its result is dropped
    const uint32_t *row = data + r * VD, *ce = cent + (int64_t)(n < K ? n : 0) * VD;
    const int64_t nsteps = (VD + 15) / 16;
    km_acc_t acc = {0.f, 0.f, 0.f, 0.f};
    for (int64_t s0 = SPLIT > 1 ? wv : 0; s0 < nsteps; s0 += (int64_t)U * SPLIT) {
        km_load_t x[U], y[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int64_t at = (s0 + (int64_t)u * SPLIT) * 16;
            x[u] = load_step(row, at < VD ? at : 0, VD - at);
            y[u] = load_step(ce, at < VD ? at : 0, VD - at);
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int k = 0; k < 4; ++k) acc = mfma_bits(frag_a(x[u][k]), frag_b(y[u][k]), acc);
    }
    const int pop = n < K ? pops[n] : 0;
    // Rows 4 q + i of the tile with the products dot against centroid n: the
    // nearest one in all 16 lanes, its member bit in its lane.
    auto nearest = [&](int dot, int i) -> uint32_t {
        int key = n < K ? (pop - 2 * dot) * 16 + (15 - n) : 0x7fffffff;
#pragma unroll
        for (int m = 1; m < 16; m <<= 1) {
            const int o = (int)shfl((uint32_t)key, lane ^ m);
            key = o < key ? o : key;
        }
        const int best = 15 - (key & 15), j = 4 * q + i;
        const bool in = tile * 16 + j < N;
        if (n == 0 && in) cluster[tile * 16 + j] = best;
        return n == best && in ? 1u << j : 0u;
    };
    auto over_groups = [&](uint32_t bits) {
        bits |= shfl(bits, lane ^ 16);
        return bits | shfl(bits, lane ^ 32);
    };
    uint32_t bits = 0;
    if constexpr (SPLIT > 1) {
#pragma unroll
        for (int i = 0; i < 4; ++i) sums[wv][i * kWave + lane] = (int)acc[i];
        __syncthreads();
        if (wv < 4) { // wave i: rows 4 q + i
            int dot = 0;
#pragma unroll
            for (int w = 0; w < SPLIT; ++w) dot += sums[w][wv * kWave + lane];
            bits = over_groups(nearest(dot, wv));
            if (lane < 16 && bits) atomicOr(&members[lane], bits);
        }
        __syncthreads();
        if (threadIdx.x < 16) hot[(int64_t)threadIdx.x * hot_stride + tile] = (uint16_t)members[threadIdx.x];
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) bits |= nearest((int)acc[i], i);
        bits = over_groups(bits);
        if (lane < 16) hot[(int64_t)lane * hot_stride + tile] = (uint16_t)bits;
    }
}

// The first centroids: rows r[0..K) of the data, and their popcounts (a block
// per centroid).
struct KmStart {
    int64_t r[kMfmaK]; // -1: zero
};
__global__ __launch_bounds__(1024) void km_start_kernel(const uint32_t *__restrict__ data, int64_t VD, KmStart rows,
                                                        uint32_t *__restrict__ cent, int32_t *__restrict__ pops)
{
    __shared__ int32_t total;
    if (threadIdx.x == 0) total = 0;
    __syncthreads();
    const int64_t r = rows.r[blockIdx.x];
    int pop = 0;
    for (int64_t j = threadIdx.x; j < VD; j += blockDim.x) {
        const uint32_t w = r >= 0 ? data[r * VD + j] : 0u;
        cent[blockIdx.x * VD + j] = w;
        pop += __builtin_popcount(w);
    }
    pop = wave_sum(pop);
    if (lane_id() == 0) atomicAdd(&total, pop);
    __syncthreads();
    if (threadIdx.x == 0) pops[blockIdx.x] = total;
}

// r[k] holds 16 bits of row k (low half) and of row k + 16 (high half), k < 16;
// afterwards r[b] holds bit b of rows 0..31: the last four stages of a 32 x 32
// bit transpose in a lane.
__device__ __forceinline__ void transpose16x32(uint32_t (&r)[16])
{
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        const uint32_t x = r[k], y = r[k + 8];
        r[k] = __builtin_amdgcn_perm(y, x, 0x06020400u);     // even bytes of both
        r[k + 8] = __builtin_amdgcn_perm(y, x, 0x07030501u); // odd bytes
    }
    auto stage = [&](auto shift, uint32_t m) {
        constexpr int S = decltype(shift)::value;
#pragma unroll
        for (int g = 0; g < 16; g += 2 * S)
#pragma unroll
            for (int k = g; k < g + S; ++k) {
                const uint32_t x = r[k], y = r[k + S];
                r[k] = __builtin_amdgcn_bitop3_b32(x, y << S, m, 0xe4);     // m ? x : y << S
                r[k + S] = __builtin_amdgcn_bitop3_b32(x >> S, y, m, 0xe4); // m ? x >> S : y
            }
    };
    stage(std::integral_constant<int, 4>(), 0x0f0f0f0fu);
    stage(std::integral_constant<int, 2>(), 0x33333333u);
    stage(std::integral_constant<int, 1>(), 0x55555555u);
}

// The rows as bit planes: plane word of (16 dword columns ct, 128 rows b, bit k
// of the dword, lane l): bit k of column l % 16 in the 32 rows of group l / 16.
// Words are kept [ct][b][k / 4][l][k % 4], so a lane takes four bits in one
// 16-byte load and a wave 1 KB.  Rows past N repeat the last one (no cluster
// holds them), columns past the row its last one.
__global__ __launch_bounds__(256) void km_planes_kernel(const uint32_t *__restrict__ data, int64_t N, int64_t VD,
                                                        int64_t row_blocks, uint32_t *__restrict__ planes)
{
    const int lane = lane_id(), n = lane % 16, g = lane / 16;
    const int64_t b = (int64_t)blockIdx.y * 4 + wave_in_block_id();
    if (b >= row_blocks) return;
    const int64_t ct = blockIdx.x;
    const int64_t col = ct * 16 + n < VD ? ct * 16 + n : VD - 1;
    uint32_t r[32];
    if (b * 128 + 128 <= N) { // uniform: scalar row addresses
        const uint32_t *rows = data + b * 128 * VD;
        const uint32_t at = (uint32_t)(32 * g * VD + col); // below 2^32: rows are below 2^24 bytes
#pragma unroll
        for (int j = 0; j < 32; ++j) r[j] = (rows + j * VD)[at];
    } else {
        const int64_t r0 = b * 128 + 32 * g;
#pragma unroll
        for (int j = 0; j < 32; ++j) r[j] = data[(r0 + j < N ? r0 + j : N - 1) * VD + col];
    }
    uint32_t lo[16], hi[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) {
        lo[k] = __builtin_amdgcn_perm(r[k + 16], r[k], 0x05040100u); // bits 0..15 of rows k and k + 16
        hi[k] = __builtin_amdgcn_perm(r[k + 16], r[k], 0x07060302u); // bits 16..31
    }
    transpose16x32(lo);
    transpose16x32(hi);
    uint4 *out = reinterpret_cast<uint4 *>(planes + ((ct * row_blocks + b) * 32 * kWave)) + lane;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        out[k * kWave] = make_uint4(lo[4 * k], lo[4 * k + 1], lo[4 * k + 2], lo[4 * k + 3]);
        out[(k + 4) * kWave] = make_uint4(hi[4 * k], hi[4 * k + 1], hi[4 * k + 2], hi[4 * k + 3]);
    }
}

// Bit counts of every cluster in half (16 bits) of 16 dword columns:
// bits[c][dword][bit] = rows of cluster c that have it.  Block x takes half
// x % 2 of the columns 16 (x / 2) .. in the rows of part blockIdx.y; its waves
// take 128 rows at a time: lane l column l % 16 of the 32 rows of group l / 16,
// plane word b bit b of 32 rows.  One product per bit with the members' bits
// (hot) adds 128 rows to the counters of 16 clusters and 16 columns.  Rows are
// read in order, whatever their cluster, and nothing is sorted.
//
// One part (gridDim.y = 1): the block has whole counts and writes its halves of
// the majority words (bit set iff more than half of the members have it) or,
// with `masks` given (the last iteration), of the masks and bitvals at threshold
// t (km_mask_bit).  More parts (few columns, many rows): counts and members are
// added to zeroed arrays, and words are left to km_majority_kernel and
// km_masks_kernel.
//
// What bounds it: reading the planes once from L2 or memory.  Reading the rows
// instead, 64 bytes of each (a wave's load touches four rows), and transposing
// them here takes 24 us where this takes 9.3, so the planes, written once in
// 16, pay from the second of the ten iterations on.  Against the sort by
// cluster, carry-save counters over gathered rows and a pass that sums the
// chunks: 4096 rows of 8 KiB, 16 clusters, 8.9 + 17.3 + 5.4 -> 9.3 us.  (Row
// parts whose last block adds up: 70 us, its fences write back L2.)
// A bit that `set` of a cluster's members have (ibp_preproc_kmeans.cuh:273-293):
// 2: in mask and bitval (float(set) >= hi = t * float(members)); 1: in the mask
// (double(set) <= lo = (1.0 - t) * members); 0: in neither.
__device__ __forceinline__ int km_mask_bit(int32_t set, float hi, double lo)
{
    const float f = (float)set;
    return f >= hi ? 2 : (double)f <= lo ? 1 : 0;
}

constexpr int kCountWaves = 8;
constexpr int kCountStride = 256 + 20; // counters of a cluster, padded: pairs of clusters on different banks

__global__ __launch_bounds__(64 * kCountWaves) void km_count_mfma_kernel(
    const uint32_t *__restrict__ planes, int64_t N, int64_t VD, const uint32_t *__restrict__ hot, int64_t hot_words, int K,
    int64_t blocks_per_part, float t, uint16_t *__restrict__ masks, uint16_t *__restrict__ bitvals,
    int32_t *__restrict__ count, int32_t *__restrict__ bits, uint16_t *__restrict__ maj)
{
    __shared__ int32_t sum[kMfmaK * kCountStride]; // [cluster][bit][column]
    __shared__ int32_t members[kMfmaK];
    const int lane = lane_id(), wv = wave_in_block_id();
    const int n = lane % 16, g = lane / 16, half = (int)(blockIdx.x & 1);
    for (int i = threadIdx.x; i < kMfmaK * kCountStride; i += blockDim.x) sum[i] = 0;
    if (threadIdx.x < kMfmaK) members[threadIdx.x] = 0;
    const int64_t col0 = (int64_t)(blockIdx.x / 2) * 16;
    const int64_t nblocks = (N + 127) / 128;
    const int64_t b0 = (int64_t)blockIdx.y * blocks_per_part;
    const int64_t b1 = b0 + blocks_per_part < nblocks ? b0 + blocks_per_part : nblocks;
    km_acc_t acc[16];
#pragma unroll
    for (int b = 0; b < 16; ++b) acc[b] = km_acc_t{0.f, 0.f, 0.f, 0.f};
    int mem = 0;
    uint4 next[4];
    uint32_t nhot = 0;
    auto load = [&](int64_t b) {
        nhot = n < K ? hot[n * hot_words + b * 4 + g] : 0u;
        const uint4 *p =
            reinterpret_cast<const uint4 *>(planes + (((int64_t)(blockIdx.x / 2) * nblocks + b) * 32 + 16 * half) * kWave);
#pragma unroll
        for (int k = 0; k < 4; ++k) next[k] = p[k * kWave + lane];
    };
    if (b0 + wv < b1) load(b0 + wv);
    for (int64_t b = b0 + wv; b < b1; b += kCountWaves) {
        uint32_t x[16];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            x[4 * k] = next[k].x;
            x[4 * k + 1] = next[k].y;
            x[4 * k + 2] = next[k].z;
            x[4 * k + 3] = next[k].w;
        }
        const uint32_t h = nhot;
        if (b + kCountWaves < b1) load(b + kCountWaves);
        mem += __builtin_popcount(h);
        const km_frag_t fa = frag_a(h);
#pragma unroll
        for (int k = 0; k < 16; ++k) acc[k] = mfma_bits(fa, frag_b(x[k]), acc[k]);
    }
    __syncthreads();
    // Every wave's counters to LDS; two clusters' in a word where the block's
    // rows allow it, since the atomics are what this costs.
    const bool pairs = (b1 - b0) * 128 < 65536; // uniform
    if (pairs) {
#pragma unroll
        for (int k = 0; k < 16; ++k)
#pragma unroll
            for (int i = 0; i < 4; i += 2)
                atomicAdd(&sum[(4 * g + i) * kCountStride + k * 16 + n], (int)acc[k][i] | ((int)acc[k][i + 1] << 16));
    } else {
#pragma unroll
        for (int k = 0; k < 16; ++k)
#pragma unroll
            for (int i = 0; i < 4; ++i) atomicAdd(&sum[(4 * g + i) * kCountStride + k * 16 + n], (int)acc[k][i]);
    }
    if (mem) atomicAdd(&members[n], mem);
    __syncthreads();
    auto counter = [&](int c, int k, int d) -> int32_t { // cluster, bit, column
        if (!pairs) return sum[c * kCountStride + k * 16 + d];
        const uint32_t w = (uint32_t)sum[(c & ~1) * kCountStride + k * 16 + d];
        return (int32_t)((c & 1) ? w >> 16 : w & 0xffffu);
    };
    if (gridDim.y == 1) {
        for (int i = threadIdx.x; i < K * 16; i += blockDim.x) {
            const int c = i / 16, d = i % 16;
            if (col0 + d >= VD) continue;
            const int64_t to = 2 * (c * VD + col0 + d) + half;
            if (!masks) {
                const int most = members[c] / 2;
                uint32_t w = 0;
#pragma unroll
                for (int k = 0; k < 16; ++k) w |= counter(c, k, d) > most ? 1u << k : 0u;
                maj[to] = (uint16_t)w;
            } else {
                const float hi = __fmul_rn(t, (float)members[c]);
                const double lo = __dmul_rn(1.0 - (double)t, (double)members[c]);
                uint32_t m = 0, v = 0;
#pragma unroll
                for (int k = 0; k < 16; ++k) {
                    const int in = km_mask_bit(counter(c, k, d), hi, lo);
                    m |= in ? 1u << k : 0u;
                    v |= in > 1 ? 1u << k : 0u;
                }
                masks[to] = (uint16_t)m;
                bitvals[to] = (uint16_t)v;
            }
        }
    } else {
        if (blockIdx.x == 0 && (int)threadIdx.x < K && members[threadIdx.x])
            atomicAdd(&count[threadIdx.x], members[threadIdx.x]);
        for (int i = threadIdx.x; i < K * 256; i += blockDim.x) {
            const int c = i / 256, d = (i % 256) / 16, k = i % 16;
            const int32_t v = col0 + d < VD ? counter(c, k, d) : 0;
            if (v) atomicAdd(bits + ((int64_t)c * VD + col0 + d) * 32 + 16 * half + k, v);
        }
    }
}

} // namespace ibp
