// ibp_preproc.hip -- mask/bitval selection (preprocess).
//
// Replaces src/preprocess.cu:17-76 and ibp::preproc_data
// (include/preproc/ibp_preproc_host.cuh:24-115) with its kernels count_bit_kernel,
// create_mask and check_feats (include/preproc/ibp_preproc_kernels.cuh:8-77).
//
// Differences by design (values are identical):
//  * all thresholds of the sweep are scored in ONE pass over the data instead
//    of one pass plus a host synchronisation per threshold;
//  * the choice (first strict maximum, compared as double) is made on the
//    device, so the call is asynchronous and never copies to the host.
#include <stddef.h>

#include <vector>

#include "ibp_bits.h"
#include "ibp_internal.h"
#include "ibp_slices.h"
#include "ibp_tile.h"
#include "ibp_wave.h"

namespace ibp {

constexpr int kMaxThresholds = 8;
constexpr int kSweep = 7; // thresholds of the sweep: 0.70, 0.75, ... 1.00

// Sums that the kernels of one call add to, cleared by the first of them.
struct Sums {
    unsigned long long score[kMaxThresholds]; // bits saved
    unsigned int blocks; // scoring blocks that are done
    // Bits of all columns' masks: kCopies partial sums in lines of their own
    // (one line for the 512 blocks of a table of 1024 columns: 47 us of atomics)
    static constexpr int kCopies = 16;
    struct alignas(128) Flagged {
        unsigned long long t[kMaxThresholds];
    } flagged[kCopies];
};
__device__ __forceinline__ void clear_sums(Sums *sums)
{
    static_assert(sizeof(Sums) % 8 == 0, "");
    for (int i = threadIdx.x; i < (int)(sizeof(Sums) / 8); i += blockDim.x) reinterpret_cast<unsigned long long *>(sums)[i] = 0;
}

struct Thresholds {
    float t[kMaxThresholds];
    int count;
};

template <typename T>
using WideT = typename std::conditional<sizeof(T) == 8, uint64_t, uint32_t>::type;

// Column-bit counts of the row block blockIdx.x and the 64-column tile
// blockIdx.y: part[blockIdx.x][j*B + k] = rows of the block whose column j has
// bit k set.  Lane <-> column; the block's waves split the rows; every thread
// keeps its B counters in registers.  Rows of fewer than 32 elements take
// G = 64 / V rows per load (lane l: column l % V of row l / V, so a load reads
// G * V consecutive elements), and the G lanes of a column meet in the LDS sum.  Rows are taken 16 at a time (16 loads in
// flight) and added into bit-sliced counters (VCounter), folded into the B
// counters every 240 rows.  The waves' counters are summed in LDS and stored
// once per block (no global atomics: every block writes its own partial
// counts, masks_kernel adds them up).
template <typename T>
__global__ __launch_bounds__(256) void count_bits_kernel(const T *data, int64_t num_vecs, int64_t V,
                                                         int64_t rows_per_block, int32_t *part, Sums *sums)
{
    constexpr int STRIDE = kWave + 1; // of a bit's counts: read back column by column
    constexpr int B = 8 * (int)sizeof(T);
    constexpr int CHUNK = 16;
    using W = WideT<T>;
    __shared__ int32_t sum[B * STRIDE];
    if (blockIdx.x == 0 && blockIdx.y == 0) clear_sums(sums);
    const int lane = lane_id();
    const int wave_in_block = wave_in_block_id();
    const int waves = blockDim.x / kWave;
    const int G = V < kWave / 2 ? (int)(kWave / V) : 1; // rows per load
    const int lcol = G > 1 ? lane % (int)V : lane;
    const int lrow = G > 1 ? lane / (int)V : 0;
    const int64_t j = (int64_t)blockIdx.y * kWave + lcol;
    const bool col = j < V && lrow < G;
    const int64_t r0 = (int64_t)blockIdx.x * rows_per_block;
    int64_t r1 = r0 + rows_per_block;
    if (r1 > num_vecs) r1 = num_vecs;
    for (int i = threadIdx.x; i < B * STRIDE; i += blockDim.x) sum[i] = 0;
    int32_t c[B];
#pragma unroll
    for (int k = 0; k < B; ++k) c[k] = 0;
    VCounter<W, B> vc;
    const int64_t step = (int64_t)waves * G; // rows between a wave's loads
    for (int64_t r = r0 + (int64_t)wave_in_block * G; r < r1; r += CHUNK * step) {
        W x[CHUNK];
#pragma unroll
        for (int q = 0; q < CHUNK; ++q) {
            const int64_t rr = r + (int64_t)q * step + lrow;
            x[q] = (col && rr < r1) ? (W)data[rr * V + j] : W(0);
        }
        vc.add16(x, c);
    }
    vc.flush(c);
    __syncthreads();
#pragma unroll
    for (int k = 0; k < B; ++k)
        if (c[k]) atomicAdd(&sum[k * STRIDE + lcol], c[k]);
    __syncthreads();
    int32_t *out = part + (int64_t)blockIdx.x * V * B;
    for (int i = threadIdx.x; i < B * kWave; i += blockDim.x) {
        const int64_t jj = (int64_t)blockIdx.y * kWave + i / B;
        if (jj < V) out[jj * B + i % B] = sum[(i % B) * STRIDE + i / B];
    }
}

// The constants of one score unit (score_slices_kernel): one 8-byte or two
// 4-byte columns, half a 16-byte chunk, under NT thresholds.  In dwords:
// 8 bytes: masks (low, high), popcounts, bitval (low, high); 4 bytes: masks,
// popcounts and bitval of the first column, then of the second.  One bitval
// serves every threshold: a list of more than one ascends from 0.7, so a bit in
// threshold t's mask is in every earlier mask with the same value (a count
// above t*N is above every smaller t*N; one below (1-t)*N <= N/2 is below every
// larger (1-t)*N and cannot exceed t'*N >= N/2): bitval[t] = bitval[0] & mask[t].
template <typename T, int NT>
struct ScoreRec {
    static constexpr int EPC = 16 / (int)sizeof(T); // columns of a chunk
    static constexpr int EPU = EPC / 2;             // ... of a unit
    static constexpr int MASK = (int)sizeof(T) / 4; // dwords of a mask
    static constexpr int COL = (MASK + 1) * NT + MASK;
    static constexpr int STRIDE = (COL * EPU + 3) / 4 * 4;
    // Where column element e of chunk c stands (the row's last chunk ends
    // with it; columns that it shares with the one before are zero there).
    static __device__ __forceinline__ int64_t at(int64_t c, int e)
    {
        return (c * 2 + e / EPU) * STRIDE + (e % EPU) * COL;
    }
};
template <typename T, int NT>
__device__ __forceinline__ void store_rec(uint32_t *recs, int64_t V, int64_t j, const T (&m)[kMaxThresholds], T b)
{
    using R = ScoreRec<T, NT>;
    const int64_t C = row_chunks((int)sizeof(T), V);
    auto put = [&](int64_t c, int e, bool zero) {
        uint32_t *r = recs + R::at(c, e);
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const uint64_t x = zero ? 0 : (uint64_t)m[t];
#pragma unroll
            for (int q = 0; q < R::MASK; ++q) r[t * R::MASK + q] = (uint32_t)(x >> (32 * q));
            r[R::MASK * NT + t] = (uint32_t)__builtin_popcountll(x);
        }
#pragma unroll
        for (int q = 0; q < R::MASK; ++q) r[(R::MASK + 1) * NT + q] = (uint32_t)((uint64_t)b >> (32 * q));
    };
    const bool tail = j >= (C - 1) * R::EPC;
    put(tail ? C - 1 : j / R::EPC, (int)(tail ? j - (V - R::EPC) : j % R::EPC), false);
    if (j == V - 1)
        for (int e = 0; V - R::EPC + e < (C - 1) * R::EPC; ++e) put(C - 1, e, true);
}

// Adds up the row blocks' counts and makes the masks of every threshold t
// (ibp_preproc_kernels.cuh:34-51): bit in mask and bitval if
// float(cnt) > float(t) * float(N); in the mask only if
// double(cnt) < (1.0 - double(t)) * double(N).  Writes masks[t*V + j],
// bitvals[t*V + j], the masks' bits per threshold and, where the rows are
// scored from them (recs), the score units.
//
// A block of 16 waves owns 64 consecutive counts (lane = count), the bits of
// one 8-byte column or of 64 / B narrower ones: its waves each sum every 16th
// row block, 16 loads in flight, the partial sums meet in LDS, and a mask is
// the lanes' ballot.  (Counts, masks and units in kernels of their own: 10.6 +
// 10.5 + 4.6 us for 3200 counts of 1024 row blocks, where this takes 9.7 of 512.)
constexpr int kReduceWaves = 16;
template <typename T>
__global__ __launch_bounds__(1024) void masks_kernel(const int32_t *part, int64_t blocks, int64_t num_vecs, int64_t V,
                                                     Thresholds th, T *masks, T *bitvals, uint32_t *recs, Sums *total)
{
    constexpr int B = 8 * (int)sizeof(T);
    constexpr int COLS = kWave / B;
    constexpr int U = 16;
    __shared__ int32_t sums[kReduceWaves][kWave];
    const int64_t n = V * B;
    const int lane = lane_id();
    const int wv = wave_in_block_id();
    const int64_t i = (int64_t)blockIdx.x * kWave + lane;
    const bool ok = i < n;
    int32_t a[U] = {};
    int64_t b = wv;
    for (; b + (U - 1) * kReduceWaves < blocks; b += U * kReduceWaves)
        if (ok)
#pragma unroll
            for (int u = 0; u < U; ++u) a[u] += part[(b + u * kReduceWaves) * n + i];
    for (; b < blocks; b += kReduceWaves)
        if (ok) a[0] += part[b * n + i];
#pragma unroll
    for (int u = 1; u < U; ++u) a[0] += a[u];
    sums[wv][lane] = a[0];
    __syncthreads();
    if (wv != 0) return;
    int32_t cnt = 0;
#pragma unroll
    for (int q = 0; q < kReduceWaves; ++q) cnt += sums[q][lane];
    T m[kMaxThresholds];
    T b0 = T(0);
    const int64_t j = (int64_t)blockIdx.x * COLS + lane;
    const int sh = B * (lane & (COLS - 1)); // lane l < COLS writes column j
#pragma unroll
    for (int t = 0; t < kMaxThresholds; ++t) {
        m[t] = T(0);
        if (t >= th.count) continue; // uniform
        const float thr = th.t[t];
        const float hi = __fmul_rn(thr, (float)(uint64_t)num_vecs);
        const double lo = __dmul_rn(1.0 - (double)thr, (double)(uint64_t)num_vecs);
        const uint64_t ones = __ballot(ok && (float)cnt > hi);
        const uint64_t all = ones | __ballot(ok && (double)cnt < lo);
        m[t] = (T)(all >> sh);
        const T v = (T)(ones >> sh);
        if (t == 0) b0 = v;
        if (lane < COLS && j < V) {
            masks[t * V + j] = m[t];
            bitvals[t * V + j] = v;
        }
        if (recs && lane == 0) // only the slices' scores start from them
            atomicAdd(&total->flagged[blockIdx.x % Sums::kCopies].t[t], (unsigned long long)__builtin_popcountll(all));
    }
    if constexpr (sizeof(T) >= 4) {
        if (recs && lane < COLS && j < V) {
            if (th.count == 1) store_rec<T, 1>(recs, V, j, m, b0);
            else store_rec<T, kSweep>(recs, V, j, m, b0);
        }
    }
}

// scores[t] += sum over rows of max(0, S_t(row) - V), S_t = bits of the
// elements flagged under threshold t's mask (ibp_preproc_kernels.cuh:54-77).
template <typename T, int NT>
__global__ __launch_bounds__(256) void score_kernel(const T *data, int64_t num_vecs, int64_t V, const T *masks,
                                                    const T *bitvals, int nt, unsigned long long *scores)
{
    const int lane = lane_id();
    const int64_t wave = global_wave_id();
    const int64_t nwaves = ((int64_t)gridDim.x * blockDim.x) / kWave;
    unsigned long long saved[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) saved[t] = 0;
    if (V <= kWave) {
        // Rows of <= 64 elements: every lane keeps its column's masks in
        // registers; 4 rows in flight per wave; two thresholds share one
        // 32-bit reduction (a row's sum is at most 64 * 64 < 2^16).
        constexpr int R = 4;
        constexpr int NP = (NT + 1) / 2;
        T m_reg[NT], b_reg[NT];
        uint32_t pc_reg[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const bool ok = t < nt && lane < V;
            m_reg[t] = ok ? masks[t * V + lane] : T(0);
            b_reg[t] = ok ? bitvals[t * V + lane] : T(0);
            // a lane past the row (or a threshold past nt) never adds anything
            pc_reg[t] = ok ? (uint32_t)popc((WideT<T>)m_reg[t]) << (16 * (t & 1)) : 0u;
        }
        for (int64_t r = wave * R; r < num_vecs; r += nwaves * R) {
            T x[R];
#pragma unroll
            for (int i = 0; i < R; ++i) x[i] = (r + i < num_vecs && lane < V) ? data[(r + i) * V + lane] : T(0);
#pragma unroll
            for (int i = 0; i < R; ++i) {
                if (r + i >= num_vecs) break; // uniform
                uint32_t acc[NP];
#pragma unroll
                for (int q = 0; q < NP; ++q) acc[q] = 0;
#pragma unroll
                for (int t = 0; t < NT; ++t)
                    if ((T)(x[i] & m_reg[t]) == b_reg[t]) acc[t >> 1] += pc_reg[t];
#pragma unroll
                for (int q = 0; q < NP; ++q) {
                    const uint32_t sum = (uint32_t)wave_sum((int)acc[q]);
                    const int64_t s0 = sum & 0xffffu, s1 = sum >> 16;
                    if (s0 > V) saved[2 * q] += (unsigned long long)(s0 - V);
                    if (2 * q + 1 < NT && s1 > V) saved[2 * q + 1] += (unsigned long long)(s1 - V);
                }
            }
        }
    } else {
        for (int64_t r = wave; r < num_vecs; r += nwaves) {
            int acc[NT];
#pragma unroll
            for (int t = 0; t < NT; ++t) acc[t] = 0;
            for (int64_t j = lane; j < V; j += kWave) {
                const T x = data[r * V + j];
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    if (t >= nt) break;
                    const T m = masks[t * V + j];
                    if ((T)(x & m) == bitvals[t * V + j]) acc[t] += popc((WideT<T>)m);
                }
            }
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                if (t >= nt) break;
                const int64_t s = wave_sum(acc[t]);
                if (s > V) saved[t] += (unsigned long long)(s - V);
            }
        }
    }
    if (lane == 0)
#pragma unroll
        for (int t = 0; t < NT; ++t)
            if (t < nt && saved[t]) atomicAdd(&scores[t], saved[t]);
}

// First strict maximum of the scores compared as double
// (ibp_preproc_host.cuh:64,92-99); copies that threshold's mask/bitval out.
// Threads first, first + step, ...
template <typename T>
__device__ __forceinline__ void select_mask(const unsigned long long (&scores)[kMaxThresholds], int nt, const T *masks,
                                            const T *bitvals, int64_t V, T *mask_out, T *bitval_out, int32_t *chosen,
                                            int64_t first, int64_t step)
{
    int best = -1;
    double max_saved = 0;
#pragma unroll
    for (int t = 0; t < kMaxThresholds; ++t)
        if (t < nt && (double)scores[t] > max_saved) {
            max_saved = (double)scores[t];
            best = t;
        }
    if (chosen && first == 0) *chosen = best;
    if (best < 0) return;
    for (int64_t j = first; j < V; j += step) {
        mask_out[j] = masks[best * V + j];
        bitval_out[j] = bitvals[best * V + j];
    }
}
template <typename T>
__global__ void select_kernel(const Sums *sums, int nt, const T *masks, const T *bitvals, int64_t V, T *mask_out,
                              T *bitval_out, int32_t *chosen)
{
    unsigned long long scores[kMaxThresholds];
#pragma unroll
    for (int t = 0; t < kMaxThresholds; ++t) scores[t] = sums->score[t];
    select_mask<T>(scores, nt, masks, bitvals, V, mask_out, bitval_out, chosen,
                   (int64_t)blockIdx.x * blockDim.x + threadIdx.x, (int64_t)gridDim.x * blockDim.x);
}

__global__ void clear_kernel(Sums *sums) { clear_sums(sums); }

// The same scores with lane <-> row, for rows of 4- or 8-byte elements and at
// least 16 bytes.  Per row and threshold a lane adds up the popcounts of the
// columns that are NOT flagged, so S_t = (sum of popcounts) - lost_t needs no
// cross-lane reduction.
//
// Work: tiles of 64 rows in slices (ibp_slices.h).  The columns' constants are
// uniform, two units per chunk by scalar loads, each issued before the unit in
// front of it is scored.  The SPLIT waves of a tile
// meet in LDS.  NT = thresholds of the records; only the first ones, up to the
// last that flags any bit, are scored (of the sweep over float data, 1.0 and
// often 0.95 flag nothing).  The tiles are taken from the last one
// back: the counts have just read the table's end, so the last-level cache
// holds it.  The block that finishes last picks the threshold and writes the
// mask.
//
// What bounds it: reading the table once.  2,449,029 x 50 doubles, sweep: 180
// us, 5.4 TB/s (a plain read: 165 us); the vector work alone takes 126 and
// overlaps it.  Before, four waves staged a tile in LDS together and split the
// thresholds, each reading all of it: 237 us; rows that are not whole chunks
// went lane <-> column with a wave reduction per row: 32,299 x 50 floats, the
// whole call, 614 -> 38 us.  Slices of one wave per tile, whatever the row: 240
// us; a row's slices follow each other too late to find its lines in L2, so
// the waves that share a tile load its whole rows together.
template <typename T, int NT, int S, int SPLIT>
__global__ __launch_bounds__(SPLIT == 1 ? 256 : 64 * SPLIT) void score_slices_kernel(
    const T *__restrict__ data, int64_t num_vecs, int64_t V, int nslices, const uint32_t *__restrict__ recs,
    const Sums::Flagged *__restrict__ flagged, int nt, Sums *sums, const T *__restrict__ masks,
    const T *__restrict__ bitvals, T *mask_out, T *bitval_out, int32_t *chosen)
{
    using R = ScoreRec<T, NT>;
    constexpr int WAVES = SPLIT == 1 ? 4 : SPLIT;
    constexpr int STRIDE = Slice<S>::STRIDE;
    __shared__ uint4 lds[WAVES][kWave * STRIDE];
    __shared__ unsigned long long bsum[kMaxThresholds];
    __shared__ unsigned int ticket;
    if (threadIdx.x < kMaxThresholds) bsum[threadIdx.x] = 0;
    __syncthreads();
    const int lane = lane_id(), wv = wave_in_block_id();
    uint4 *const mine = lds[wv];
    const int C = (int)row_chunks((int)sizeof(T), V);
    const uint32_t row_bytes = (uint32_t)(V * (int64_t)sizeof(T));
    const int ntiles = (int)((num_vecs + kWave - 1) / kWave);
    const int step = SPLIT == 1 ? (int)gridDim.x * WAVES : (int)gridDim.x;
    const int first = SPLIT == 1 ? (int)blockIdx.x * WAVES + wv : (int)blockIdx.x;
    const int s0 = SPLIT == 1 ? 0 : wv; // this wave's slices: s0, s0 + SPLIT, ...

    Slice<S> slice;
    slice.init(row_bytes, lane);
    auto load = [&](int n, int s) { // slice s of the n-th tile from the end
        slice.load(data, num_vecs, row_bytes, ntiles - 1 - n, ntiles, s, nslices, lane);
    };

    uint32_t all[NT]; // bits of all columns' masks
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        all[t] = 0;
        for (int k = 0; k < Sums::kCopies; ++k) all[t] += (uint32_t)flagged[k].t[t];
    }

    auto run = [&](auto na_tag) {
        constexpr int NA = decltype(na_tag)::value;
        uint32_t total[NA];
        unsigned long long saved[NA];
#pragma unroll
        for (int t = 0; t < NA; ++t) {
            total[t] = all[t];
            asm volatile("" : "+v"(total[t])); // the scalar registers are for the units
            saved[t] = 0;
        }
        struct Unit {
            T m[R::EPU][NA];
            uint32_t p[R::EPU][NA];
            T b[R::EPU];
        };
        auto fetch = [&](int u, Unit &x) {
            const uint32_t *r = recs + (uint32_t)(u * R::STRIDE);
#pragma unroll
            for (int e = 0; e < R::EPU; ++e) {
#pragma unroll
                for (int t = 0; t < NA; ++t) {
                    if constexpr (sizeof(T) == 8)
                        x.m[e][t] = (T)r[e * R::COL + 2 * t] | ((T)((uint64_t)r[e * R::COL + 2 * t + 1] << 32));
                    else
                        x.m[e][t] = r[e * R::COL + t];
                    x.p[e][t] = r[e * R::COL + R::MASK * NT + t];
                }
                const uint32_t *rb = r + e * R::COL + (R::MASK + 1) * NT;
                if constexpr (sizeof(T) == 8) x.b[e] = (T)rb[0] | ((T)((uint64_t)rb[1] << 32));
                else x.b[e] = rb[0];
            }
        };
        // Empty asm that needs the unit in SGPRs: the wait for its scalar loads
        // (which complete in any order: lgkmcnt(0), LDS reads included) is here.
        auto need = [&](const Unit &x) {
#pragma unroll
            for (int e = 0; e < R::EPU; ++e) {
#pragma unroll
                for (int t = 0; t < NA; ++t) asm volatile("" ::"s"(x.m[e][t]), "s"(x.p[e][t]));
                asm volatile("" ::"s"(x.b[e]));
            }
        };
        uint32_t lost[NA];
        auto score = [&](uint32_t x0, uint32_t x1, const Unit &x) {
            if constexpr (sizeof(T) == 8) {
                const T d = xor_ordered((T)x0 | ((T)((uint64_t)x1 << 32)), x.b[0]);
#pragma unroll
                for (int t = 0; t < NA; ++t) lost[t] = lost_step(d, x.m[0][t], x.p[0][t], lost[t]);
            } else {
                const T d0 = xor_ordered((T)x0, x.b[0]), d1 = xor_ordered((T)x1, x.b[R::EPU - 1]);
#pragma unroll
                for (int t = 0; t < NA; ++t) {
                    lost[t] = lost_step(d0, x.m[0][t], x.p[0][t], lost[t]);
                    lost[t] = lost_step(d1, x.m[R::EPU - 1][t], x.p[R::EPU - 1][t], lost[t]);
                }
            }
        };
        int n = first;
        const bool any = s0 < nslices;
        Unit ua, ub;
        if (any && n < ntiles) {
            load(n, s0);
            fetch(s0 * S * 2, ua);
        }
        for (; n < ntiles; n += step) {
#pragma unroll
            for (int t = 0; t < NA; ++t) lost[t] = 0;
            for (int s = s0; s < nslices; s += SPLIT) {
                slice.store(mine, lane);
                __builtin_amdgcn_wave_barrier();
                const bool more = s + SPLIT < nslices;
                const int ns = more ? s + SPLIT : s0;
                if (more) load(n, ns);
                else if (n + step < ntiles) load(n + step, ns);
                const int c0 = s * S, nc = C - c0 < S ? C - c0 : S, next = ns * S;
                const uint4 *row = mine + lane * STRIDE;
                // chunk c of the slice, its first unit in ua
                auto chunk = [&](const uint4 &v, uint4 &vn, int c) {
                    need(ua);
                    asm volatile("" ::"v"(v.x), "v"(v.y), "v"(v.z), "v"(v.w));
                    fetch((c0 + c) * 2 + 1, ub);
                    vn = row[c + 1 < nc ? c + 1 : c];
                    score(v.x, v.y, ua);
                    need(ub);
                    fetch((c + 1 < nc ? c0 + c + 1 : next) * 2, ua);
                    score(v.z, v.w, ub);
                };
                uint4 va = row[0], vb;
                int c = 0;
                for (; c + 1 < nc; c += 2) {
                    chunk(va, vb, c);
                    chunk(vb, va, c + 1);
                }
                if (c < nc) chunk(va, vb, c);
                __builtin_amdgcn_wave_barrier();
            }
            const int64_t row = (int64_t)(ntiles - 1 - n) * kWave + lane;
            if constexpr (SPLIT == 1) {
                if (row < num_vecs) {
#pragma unroll
                    for (int t = 0; t < NA; ++t) {
                        const uint32_t st = total[t] - lost[t];
                        if (st > (uint32_t)V) saved[t] += st - (uint32_t)V;
                    }
                }
            } else {
                // every wave's part of the rows' losses, in its own LDS
                uint32_t *const part = reinterpret_cast<uint32_t *>(mine);
                static_assert(sizeof(lds[0]) >= kMaxThresholds * kWave * sizeof(uint32_t), "");
#pragma unroll
                for (int t = 0; t < NA; ++t) part[t * kWave + lane] = lost[t];
                __syncthreads();
                if (row < num_vecs) {
#pragma unroll
                    for (int t = 0; t < NA; ++t) {
                        if (t % SPLIT != wv) continue; // uniform
                        uint32_t st = total[t];
#pragma unroll
                        for (int q = 0; q < SPLIT; ++q) st -= reinterpret_cast<const uint32_t *>(lds[q])[t * kWave + lane];
                        if (st > (uint32_t)V) saved[t] += st - (uint32_t)V;
                    }
                }
                __syncthreads();
            }
        }
        // The lanes' savings as 24-bit low parts and the rest (each sum of 64
        // fits 32 bits as long as a lane's saving is below 2^49).
#pragma unroll
        for (int t = 0; t < NA; ++t) {
            const uint32_t lo = (uint32_t)wave_sum((int)(uint32_t)(saved[t] & 0xffffffull));
            const uint32_t hi = (uint32_t)wave_sum((int)(uint32_t)(saved[t] >> 24));
            if (lane == 0) atomicAdd(&bsum[t], (unsigned long long)lo + ((unsigned long long)hi << 24));
        }
    };
    int na = 0;
#pragma unroll
    for (int t = 0; t < NT; ++t)
        if (t < nt && all[t]) na = t + 1;
    if constexpr (NT == 1) {
        if (na) run(std::integral_constant<int, 1>());
    } else {
        if (na > 6) run(std::integral_constant<int, 7>());
        else if (na > 4) run(std::integral_constant<int, 6>());
        else if (na) run(std::integral_constant<int, 4>());
    }
    __syncthreads();
    // One atomic per threshold and block.  Their results are awaited before
    // the block's ticket, so the last ticket's block finds every sum (atomics
    // at agent scope and atomic loads: no fence, which would write back L2).
    unsigned long long was = 0;
    if ((int)threadIdx.x < na)
        was = __hip_atomic_fetch_add(&sums->score[threadIdx.x], bsum[threadIdx.x], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    asm volatile("s_waitcnt vmcnt(0)" ::"v"(was) : "memory");
    __syncthreads();
    if (threadIdx.x == 0)
        ticket = __hip_atomic_fetch_add(&sums->blocks, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    if (ticket != gridDim.x - 1) return;
    unsigned long long scores[kMaxThresholds];
#pragma unroll
    for (int t = 0; t < kMaxThresholds; ++t)
        scores[t] = __hip_atomic_load(&sums->score[t], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    select_mask<T>(scores, nt, masks, bitvals, V, mask_out, bitval_out, chosen, threadIdx.x, blockDim.x);
}

// Launch for nt thresholds (1, or the sweep), N > 0.  Four waves per SIMD fit
// (the sweep takes 84 to 128 registers, by the slice); a fifth gave nothing.
template <typename T>
void launch_score_slices(const T *data, int64_t N, int64_t V, const uint32_t *recs, int nt, Sums *sums, const T *masks,
                         const T *bitvals, T *mask, T *bitval, int32_t *chosen, int num_cus, hipStream_t stream)
{
    const int64_t C = row_chunks((int)sizeof(T), V), ntiles = (N + kWave - 1) / kWave;
    auto by_size = [&](auto nt_tag) {
        with_slices(C, ntiles, num_cus, [&](auto s_tag, auto split_tag) {
            constexpr int NT = decltype(nt_tag)::value, S = decltype(s_tag)::value, SPLIT = decltype(split_tag)::value;
            constexpr int WAVES = SPLIT == 1 ? 4 : SPLIT;
            const Sums::Flagged *flagged = sums->flagged;
            const int64_t blocks = SPLIT == 1 ? (ntiles + 3) / 4 : ntiles, most = (int64_t)num_cus * (16 / WAVES);
            hipLaunchKernelGGL((score_slices_kernel<T, NT, S, SPLIT>), dim3((unsigned)(blocks < most ? blocks : most)),
                               dim3(kWave * WAVES), 0, stream, data, N, V, (int)((C + S - 1) / S), recs, flagged, nt,
                               sums, masks, bitvals, mask, bitval, chosen);
        });
    };
    if (nt == 1) by_size(std::integral_constant<int, 1>());
    else by_size(std::integral_constant<int, kSweep>());
}

// The thresholds the reference tries (ibp_preproc_host.cuh:61-67): only
// `threshold` if it is >= 0, else 0.7f, then t = float(double(t) + 0.05) while
// t <= 1.0f.
Thresholds threshold_list(float threshold)
{
    Thresholds th;
    th.count = 0;
    const float lo = threshold < 0 ? 0.7f : threshold;
    const float hi = threshold < 0 ? 1.0f : threshold;
    for (volatile float t = lo; t <= hi && th.count < kMaxThresholds; t = (float)((double)t + 0.05))
        th.t[th.count++] = t;
    return th;
}

namespace {

struct PreWorkspace {
    size_t masks_off, bitvals_off, recs_off, sums_off, part_off, total;
};

// Row blocks of count_bits_kernel: as many blocks as the chip holds at once
// (two per CU of a 256-CU device with 8-byte elements, whose counters take 190
// registers, else three), at least one per 64-column tile, at least 64 rows
// each.  (2,449,029 x 50 doubles: 512 blocks 173 us, 1024 blocks 180.)
constexpr int64_t count_blocks(int w) { return w == 8 ? 512 : 768; }
int64_t max_count_row_blocks(int w, int64_t V)
{
    const int64_t tiles = (V + kWave - 1) / kWave;
    return count_blocks(w) / tiles > 1 ? count_blocks(w) / tiles : 1;
}
int64_t count_row_blocks(int w, int64_t N, int64_t V, int64_t *rows_per_block)
{
    const int64_t want = max_count_row_blocks(w, V);
    int64_t rpb = (N + want - 1) / want;
    if (rpb < 64) rpb = 64;
    *rows_per_block = rpb;
    return N > 0 ? (N + rpb - 1) / rpb : 0;
}

// Bytes of the score units for nt thresholds.
size_t score_recs_bytes(int w, int64_t V, int nt)
{
    if (w < 4) return 0;
    const int stride = w == 8 ? (nt == 1 ? ScoreRec<uint64_t, 1>::STRIDE : ScoreRec<uint64_t, kSweep>::STRIDE)
                              : (nt == 1 ? ScoreRec<uint32_t, 1>::STRIDE : ScoreRec<uint32_t, kSweep>::STRIDE);
    return sizeof(uint32_t) * (size_t)(row_chunks(w, V) * 2 * stride);
}

PreWorkspace layout(int w, int64_t V, int nt)
{
    auto al = [](size_t x) { return (x + 255) / 256 * 256; };
    PreWorkspace L;
    L.masks_off = 0;
    L.bitvals_off = al(L.masks_off + (size_t)w * V * nt);
    L.recs_off = al(L.bitvals_off + (size_t)w * V * nt);
    L.sums_off = al(L.recs_off + score_recs_bytes(w, V, nt));
    L.part_off = al(L.sums_off + sizeof(Sums));
    L.total = al(L.part_off + sizeof(int32_t) * (size_t)max_count_row_blocks(w, V) * V * 8 * w);
    return L;
}

template <typename T>
int preprocess_typed(const void *data, int64_t N, int64_t V, const Thresholds &th, void *mask, void *bitval,
                     int32_t *chosen, unsigned char *ws, hipStream_t stream)
{
    const DeviceInfo &dev = device_info();
    const PreWorkspace L = layout((int)sizeof(T), V, th.count);
    T *masks = (T *)(ws + L.masks_off);
    T *bitvals = (T *)(ws + L.bitvals_off);
    uint32_t *recs = (uint32_t *)(ws + L.recs_off);
    Sums *sums = (Sums *)(ws + L.sums_off);
    int32_t *part = (int32_t *)(ws + L.part_off);
    const int64_t ncnt = V * 8 * (int64_t)sizeof(T);
    int64_t rows_per_block = 0;
    const int64_t row_blocks = count_row_blocks((int)sizeof(T), N, V, &rows_per_block);
    if (row_blocks > 0) {
        const int64_t tiles = (V + kWave - 1) / kWave;
        hipLaunchKernelGGL((count_bits_kernel<T>), dim3((unsigned)row_blocks, (unsigned)tiles), dim3(256), 0, stream,
                           (const T *)data, N, V, rows_per_block, part, sums);
    } else {
        hipLaunchKernelGGL(clear_kernel, dim3(1), dim3(64), 0, stream, sums);
    }
    IBP_LAUNCH_CHECK();
    // Rows of 4- or 8-byte elements and at least 16 bytes: lane <-> row, from
    // the score units; narrower ones: lane <-> column.  So too, with one
    // threshold, tables of very wide rows that are few: a wave per row, where a
    // tile's waves walk its slices in turn (100 x 4096 doubles: 59 us per call
    // and 76, 400 x 8000 109 and 133, 1000 x 2752 76 and 62; 20 x 20,000 floats
    // 138 and 150, 400 162 and 160).
    const bool few_wide = th.count == 1 && V > 2048 && N * (sizeof(T) == 8 ? 6 : 256) < V;
    // And rows of 320 bytes and more in host memory, which a wave reads end to
    // end: PCIe carries slices of many rows 15% slower (200,000 x 50 doubles 3.20
    // ms per call, so 2.88; 5000 x 2752 4.44 and 3.85; 200,000 x 75 floats,
    // sweep, 2.40 and 2.49).
    const bool over_pcie = V * (int64_t)sizeof(T) >= 320 && N > 0 && pointer_is_host(data);
    const bool slices = sizeof(T) >= 4 && N > 0 && V * (int64_t)sizeof(T) >= 16 && V <= (int64_t)1 << 20 &&
                        (uintptr_t)data % 4 == 0 && (th.count == 1 || th.count == kSweep) && !few_wide && !over_pcie;
    const int64_t rgrid = (ncnt + kWave - 1) / kWave;
    hipLaunchKernelGGL((masks_kernel<T>), dim3((unsigned)rgrid), dim3(kWave * kReduceWaves), 0, stream,
                       (const int32_t *)part, row_blocks, N, V, th, masks, bitvals, slices ? recs : nullptr, sums);
    IBP_LAUNCH_CHECK();
    if constexpr (sizeof(T) >= 4) {
        if (slices) {
            launch_score_slices<T>((const T *)data, N, V, recs, th.count, sums, masks, bitvals, (T *)mask, (T *)bitval,
                                   chosen, dev.num_cus, stream);
            IBP_LAUNCH_CHECK();
            return IBP_OK;
        }
    }
    if (N > 0) {
        int64_t grid = (N * kWave + 255) / 256;
        if (grid > (int64_t)dev.num_cus * 8) grid = (int64_t)dev.num_cus * 8;
        if (th.count <= 1)
            hipLaunchKernelGGL((score_kernel<T, 1>), dim3((unsigned)grid), dim3(256), 0, stream, (const T *)data, N, V,
                               masks, bitvals, th.count, sums->score);
        else
            hipLaunchKernelGGL((score_kernel<T, kMaxThresholds>), dim3((unsigned)grid), dim3(256), 0, stream,
                               (const T *)data, N, V, masks, bitvals, th.count, sums->score);
        IBP_LAUNCH_CHECK();
    }
    unsigned sel_grid = (unsigned)((V + 255) / 256);
    if (sel_grid > 256) sel_grid = 256;
    hipLaunchKernelGGL((select_kernel<T>), dim3(sel_grid), dim3(256), 0, stream, sums, th.count, masks, bitvals, V,
                       (T *)mask, (T *)bitval, chosen);
    IBP_LAUNCH_CHECK();
    return IBP_OK;
}

} // namespace

} // namespace ibp

using namespace ibp;

extern "C" size_t ibp_preprocess_workspace_size(int elem_bytes, int64_t vec_size, float threshold)
{
    return layout(elem_bytes, vec_size, threshold_list(threshold).count).total;
}

extern "C" int ibp_preprocess(int elem_bytes, const void *data, int64_t num_vecs, int64_t vec_size, float threshold,
                              void *mask, void *bitval, int32_t *chosen_step, void *workspace,
                              size_t workspace_bytes, void *stream)
{
    IBP_TRACE("ibp_preprocess");
    IBP_CHECK(elem_bytes == 1 || elem_bytes == 2 || elem_bytes == 4 || elem_bytes == 8,
              "Input tensor must be 1, 2, 4, or 8-byte datatype (got %d)", elem_bytes);
    IBP_CHECK(vec_size > 0 && num_vecs >= 0, "invalid shape");
    IBP_CHECK(mask && bitval && (data || num_vecs == 0), "null pointer argument");
    IBP_CHECK(num_vecs < (int64_t)1 << 31, "num_vecs must fit the int32 bit counters");
    const Thresholds th = threshold_list(threshold);
    const size_t need = layout(elem_bytes, vec_size, th.count).total;
    hipStream_t s = as_stream(stream);
    unsigned char *ws = (unsigned char *)workspace;
    bool own = false;
    if (ws == nullptr) {
        IBP_HIP(hipMallocAsync((void **)&ws, need, s));
        own = true;
    } else {
        IBP_CHECK(workspace_bytes >= need, "workspace too small (%zu < %zu)", workspace_bytes, need);
    }
    int st;
    switch (elem_bytes) {
    case 1: st = preprocess_typed<uint8_t>(data, num_vecs, vec_size, th, mask, bitval, chosen_step, ws, s); break;
    case 2: st = preprocess_typed<uint16_t>(data, num_vecs, vec_size, th, mask, bitval, chosen_step, ws, s); break;
    case 4: st = preprocess_typed<uint32_t>(data, num_vecs, vec_size, th, mask, bitval, chosen_step, ws, s); break;
    default: st = preprocess_typed<uint64_t>(data, num_vecs, vec_size, th, mask, bitval, chosen_step, ws, s); break;
    }
    if (st == IBP_OK && debug_enabled()) {
        // Debug mode reports what the reference's sweep prints
        // (ibp_preproc_host.cuh:66,89-98): the bits each threshold saves, and
        // each new best with its expected compressed length in elements.
        // This synchronises the stream; without debug the call stays
        // asynchronous.
        unsigned long long sc[kMaxThresholds] = {0};
        const PreWorkspace L = layout(elem_bytes, vec_size, th.count);
        if (hipMemcpyAsync(sc, ws + L.sums_off + offsetof(Sums, score), sizeof(sc), hipMemcpyDeviceToHost, s) == hipSuccess &&
            hipStreamSynchronize(s) == hipSuccess) {
            const double total = (double)num_vecs * (double)vec_size * 8.0 * elem_bytes;
            dprintf("Num elems: %lld\n", (long long)num_vecs);
            double best = 0;
            for (int t = 0; t < th.count; ++t) {
                dprintf("Threshold %.2f: Saved bits per element: %llu (Total %.0f, %.3f%%)\n", th.t[t], sc[t], total,
                        total > 0 ? (double)sc[t] * 100.0 / total : 0.0);
                if ((double)sc[t] > best) {
                    best = (double)sc[t];
                    const int len = total > 0 ? (int)((double)vec_size * (total - (double)sc[t]) / total) + 1 : 0;
                    dprintf("Selected threshold %.2f; compress_len %d\n", th.t[t], len);
                }
            }
        } else {
            (void)hipGetLastError();
        }
    }
    if (own) {
        hipError_t e = hipFreeAsync(ws, s);
        if (st == IBP_OK && e != hipSuccess) return set_error(IBP_ERR_HIP, "hipFreeAsync: %s", hipGetErrorString(e));
    }
    if (st == IBP_OK) dprintf("[ibp] preprocess: %d threshold(s), V=%lld, N=%lld\n", th.count, (long long)vec_size,
                              (long long)num_vecs);
    return st;
}
