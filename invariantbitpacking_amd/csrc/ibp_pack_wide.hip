// ibp_pack_wide.hip -- the pack of rows of more than 64 elements of 4 or 8
// bytes and at most 32 KiB (compress_inplace and compress_condensed; the slot
// format is described in ibp_fetch_dev.h), with one mask or a mask row per row.
//
// As in ibp_fetch_wide.h a row is cut into chunks of 512 bytes in which lane l
// owns 8 bytes, handled as two 32-bit halves in stream order, and a team of
// waves packs a row together:
//   A. every wave loads its chunks (kept in registers: a row is read once,
//      which matters for tables in host memory) and counts their free bits,
//   B. the chunks' counts give their positions and the row's size,
//   C. the free bits go to their places in the slot, put together in LDS,
//      which then leaves in one coalesced pass.
//
// What bounds it, and why this shape.  A wave per row walks its chunks one by
// one, and a bitmask word per block leaves 4096 rows on 128 blocks: 200 us for
// a 4096 x 2752 block of 8-byte words, 180 MB at 0.9 TB/s.  Here a row's chunks
// are loaded together by up to eight waves, blocks take single rows, and the
// bitmask, zeroed beforehand, is put together with one atomic per packed row:
// 86 us; 284,138 rows of 196 4-byte words 324 -> 204 us, 40,000 rows of 512
// 8-byte words 178 -> 108 us.  Now the vector work per chunk and the rows in
// flight per CU (100 registers at eight chunks a wave: 16 waves) bound it.
#include "ibp_fetch_dev.h"
#include "ibp_internal.h"
#include "ibp_pack.h"
#include "ibp_wave.h"

namespace ibp {

namespace {

constexpr int kMaxChunks = 8; // chunks a wave keeps in registers, at most
constexpr int kMaxTeam = 8;
constexpr int kSoloWaves = 4; // waves of a block of one-wave teams
static_assert(kPackWideMaxBytes == kMaxChunks * kMaxTeam * 512);

typedef uint32_t pack8_t __attribute__((ext_vector_type(2), aligned(4)));

// A lane's 8 bytes of a chunk, as the half that comes first in the stream and
// the other; `words` of the chunk's 32-bit words are in the row (0 for others).
template <typename T>
__device__ __forceinline__ void load_halves(const T *cols, int lane, int words, uint32_t &first, uint32_t &second)
{
    pack8_t v = {0u, 0u};
    if (words == 2 * kWave) { // uniform
        v = reinterpret_cast<const pack8_t *>(cols)[lane];
    } else {
        const uint32_t *w = reinterpret_cast<const uint32_t *>(cols) + 2 * lane;
        if (2 * lane < words) v.x = w[0];
        if (2 * lane + 1 < words) v.y = w[1];
    }
    first = sizeof(T) == 8 ? v.y : v.x;
    second = sizeof(T) == 8 ? v.x : v.y;
}

// Closes the highest run of masked bits of m in v: the bits of v below the run
// move up over it.  m loses the run (its lower runs move up too).  With m = 0
// nothing moves; the ORs keep the counts below 32, and a mask of 32 bits is
// used up in two steps.
__device__ __forceinline__ void close_run(uint32_t &v, uint32_t &m)
{
    const int s = __builtin_clz(m | 1u);
    const uint32_t low = 0xffffffffu >> s;
    const int g = __builtin_clz(~(m << s) | 1u);
    v = __builtin_amdgcn_bitop3_b32(v << g, v, low, 0xe4); // low ? v << g : v
    m = (m << g) & low;
}

// CPW: chunks per wave, at most; fewer leave registers for more waves.
constexpr int pack_waves(int cpw) { return cpw <= 2 ? 8 : cpw <= 4 ? 6 : 4; }

template <typename T, typename IdxT, bool CONDENSED, int CPW>
__global__ __launch_bounds__(64 * kMaxTeam, pack_waves(CPW)) void pack_wide_kernel(PackParams p, int team)
{
    constexpr int W = (int)sizeof(T);
    constexpr int kCols = 512 / W;
    extern __shared__ __align__(16) uint32_t lds[];
    const int lane = lane_id();
    const int slot = team > 1 ? wave_in_block_id() : 0;
    const int V = (int)p.V;
    const int row_words = V * (W / 4);              // 32-bit words of a row
    const int buf_words = (row_words + 3) / 4 * 4;  // the slot, zero between rows
    uint32_t *buf = lds + (team > 1 ? 0 : wave_in_block_id() * (buf_words + kWave));
    uint32_t *tot = buf + buf_words;                // free bits per chunk
    const int nchunks = (V + kCols - 1) / kCols;
    const int hdr_words = (int)header_bytes(V, W) / 4;
    const bool in_place = !CONDENSED && p.in == (const void *)p.out && p.index == nullptr;
    const int threads = team * kWave, tid = slot * kWave + lane;
    unsigned long long bad = 0;
    auto sync = [&]() {
        if (team > 1) {
            __syncthreads();
        } else {
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        }
    };
    for (int k = tid; k < buf_words; k += threads) buf[k] = 0u;

    const int64_t first = team > 1 ? (int64_t)blockIdx.x : global_wave_id();
    const int64_t step = team > 1 ? (int64_t)gridDim.x : (int64_t)gridDim.x * (blockDim.x / kWave);
    for (int64_t i = first; i < p.n; i += step) {
        const int64_t r = p.index ? readfirstlane((int64_t)((const IdxT *)p.index)[i]) : i;
        int64_t c = r >= 0 && r < p.num_vecs ? 0 : -1;
        if (c == 0 && p.clusters) {
            c = readfirstlane(p.clusters[r]);
            if (c >= p.num_clusters) c = -1;
        }
        if (c < 0) { // uniform for the team
            ++bad;
            continue;
        }
        const T *src = (const T *)p.in + r * V;
        const T *mask = (const T *)p.mask + c * V, *bitval = (const T *)p.bitval + c * V;

        // A. x: the elements; m: their column's mask where the element has the
        // masked bits (flagged), else 0; f: the halves' flags.
        uint32_t x0[CPW], x1[CPW], m0[CPW], m1[CPW];
        uint32_t b0[CPW], b1[CPW];
        int before[CPW]; // free bits of the chunk's columns before this lane's
        uint32_t f = 0;
#pragma unroll
        for (int u = 0; u < CPW; ++u) {
            const int k = slot + u * team;
            x0[u] = x1[u] = m0[u] = m1[u] = b0[u] = b1[u] = 0;
            before[u] = 0;
            if (k < nchunks) { // uniform
                const int words = (V - k * kCols < kCols ? V - k * kCols : kCols) * (W / 4);
                load_halves<T>(src + k * kCols, lane, words, x0[u], x1[u]);
                load_halves<T>(mask + k * kCols, lane, words, m0[u], m1[u]);
                load_halves<T>(bitval + k * kCols, lane, words, b0[u], b1[u]);
            }
        }
#pragma unroll
        for (int u = 0; u < CPW; ++u) {
            const int k = slot + u * team;
            if (k < nchunks) { // uniform
                const int words = (V - k * kCols < kCols ? V - k * kCols : kCols) * (W / 4);
                bool g0 = (x0[u] & m0[u]) == b0[u], g1 = (x1[u] & m1[u]) == b1[u];
                if constexpr (W == 8) g0 = g1 = g0 && g1;
                const bool in0 = 2 * lane < words, in1 = 2 * lane + 1 < words;
                g0 = g0 && in0;
                g1 = g1 && in1;
                f |= (g0 ? 1u << (2 * u) : 0u) | (g1 ? 2u << (2 * u) : 0u);
                m0[u] = g0 ? m0[u] : 0u;
                m1[u] = g1 ? m1[u] : 0u;
                const int L = (in0 ? 32 : 0) + (in1 ? 32 : 0) - __builtin_popcount(m0[u]) - __builtin_popcount(m1[u]);
                const int incl = wave_incl_scan(L);
                before[u] = incl - L;
                if (lane == kWave - 1) tot[k] = (uint32_t)incl;
            }
        }
        sync(); // the counts are there (and the slot before this one is out)

        // B. Positions (lane k: chunk k's) and the size.
        const int mine = lane < nchunks ? (int)tot[lane] : 0;
        const int incl = wave_incl_scan(mine);
        const int bits = readlane(incl, kWave - 1);
        const int64_t size = slot_size(V, W, (int64_t)V * 8 * W - bits);
        bool row_ok = true;
        unsigned char *dst;
        if constexpr (CONDENSED) {
            const int64_t lo = i > 0 ? readfirstlane(p.offsets[i - 1]) : 0;
            const int64_t hi = readfirstlane(p.offsets[i]);
            // The stored length must be this row's size: offsets from another
            // dataset or mask never make a write leave the row.
            row_ok = lo >= 0 && hi - lo == size && hi <= p.stream_bytes && (lo % W) == 0;
            dst = (unsigned char *)p.out + lo;
            if (!row_ok) ++bad;
        } else {
            dst = (unsigned char *)p.out + i * (int64_t)V * W;
        }
        const bool packed = row_ok && size < (int64_t)V * W;
        if (packed) {
            // C. The free bits, highest first, from bit `pos` of the payload
            // on: 64 bits at most, over three words of the stream.
#pragma unroll
            for (int u = 0; u < CPW; ++u) {
                const int k = slot + u * team;
                if (k >= nchunks) break; // uniform
                const int words = (V - k * kCols < kCols ? V - k * kCols : kCols) * (W / 4);
                const uint32_t g0 = (f >> (2 * u)) & 1u, g1 = (f >> (2 * u + 1)) & 1u;
                if constexpr (W == 8) {
                    const uint64_t hb = ballot(g0 != 0);
                    if (lane < 2 && 2 * k + lane < hdr_words) buf[2 * k + lane] = (uint32_t)(hb >> (32 * lane));
                } else {
                    // 16 lanes hold 32 flags
                    uint32_t h = (g0 | g1 << 1) << (2 * (lane & 15));
                    h |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)h, 0x111, 0xf, 0xf, true);
                    h |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)h, 0x112, 0xf, 0xf, true);
                    h |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)h, 0x114, 0xf, 0xf, true);
                    h |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)h, 0x118, 0xf, 0xf, true);
                    if ((lane & 15) == 15 && 4 * k + (lane >> 4) < hdr_words) buf[4 * k + (lane >> 4)] = h;
                }
                const int n0 = (2 * lane < words ? 32 : 0) - __builtin_popcount(m0[u]);
                const int pos = readlane(incl, k) - readlane(mine, k) + before[u];
                uint32_t v0 = x0[u] & ~m0[u], v1 = x1[u] & ~m1[u], e0 = m0[u], e1 = m1[u];
                while (ballot((e0 | e1) != 0)) {
                    close_run(v0, e0);
                    close_run(v1, e1);
                }
                // below the free bits only zeros: closing moves zeros in
                const uint64_t v = ((uint64_t)v0 << 32) | (((uint64_t)v1 << 32) >> n0);
                const uint32_t hi = (uint32_t)(v >> 32), lo = (uint32_t)v, o = (uint32_t)pos & 31u;
                const uint32_t t = (uint32_t)pos >> 5;
                uint32_t *pay = buf + hdr_words;
                // stream word s is word s of 4-byte slots, word s ^ 1 of 8-byte ones
                auto put = [&](uint32_t s, uint32_t w) {
                    if (w) __hip_atomic_fetch_or(&pay[W == 8 ? s ^ 1u : s], w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                };
                put(t, hi >> o);
                put(t + 1, __builtin_amdgcn_alignbit(hi, lo, o));
                put(t + 2, __builtin_amdgcn_alignbit(lo, 0u, o));
            }
        }
        sync(); // the slot is complete
        if (packed) {
            const int out_words = CONDENSED ? (int)(size / 4) : row_words; // the rest of a slot is zero
            for (int k = 2 * tid; k < row_words; k += 2 * threads) {
                const pack8_t v = {buf[k], buf[k + 1]};
                buf[k] = buf[k + 1] = 0u;
                if (k + 2 <= out_words) {
                    *reinterpret_cast<pack8_t *>(dst + 4 * k) = v;
                } else if (k < out_words) {
                    *reinterpret_cast<uint32_t *>(dst + 4 * k) = v.x;
                }
            }
            if (p.bitmask && tid == 0) atomicOr(&p.bitmask[i >> 5], 1u << (i & 31));
        } else if (row_ok && !in_place) { // a raw row, from the registers
#pragma unroll
            for (int u = 0; u < CPW; ++u) {
                const int k = slot + u * team;
                if (k >= nchunks) break; // uniform
                const int words = (V - k * kCols < kCols ? V - k * kCols : kCols) * (W / 4);
                const pack8_t v = W == 8 ? (pack8_t){x1[u], x0[u]} : (pack8_t){x0[u], x1[u]};
                uint32_t *d = reinterpret_cast<uint32_t *>(dst + k * 512) + 2 * lane;
                if (2 * lane + 1 < words) *reinterpret_cast<pack8_t *>(d) = v;
                else if (2 * lane < words) d[0] = v.x;
            }
        }
    }
    if (p.err && bad && slot == 0 && lane == 0) atomicAdd(p.err, bad);
}

__global__ void zero_words_kernel(uint32_t *p, int64_t n)
{
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        p[i] = 0u;
}

template <typename T, typename IdxT, bool CONDENSED>
void launch_chunks(const PackParams &p, int cpw, dim3 g, dim3 b, size_t lds, int team, hipStream_t s)
{
    if (cpw <= 2) hipLaunchKernelGGL((pack_wide_kernel<T, IdxT, CONDENSED, 2>), g, b, lds, s, p, team);
    else if (cpw <= 4) hipLaunchKernelGGL((pack_wide_kernel<T, IdxT, CONDENSED, 4>), g, b, lds, s, p, team);
    else hipLaunchKernelGGL((pack_wide_kernel<T, IdxT, CONDENSED, kMaxChunks>), g, b, lds, s, p, team);
}

template <typename T>
void launch(const PackParams &p, bool i32, bool condensed, int cpw, dim3 g, dim3 b, size_t lds, int team, hipStream_t s)
{
    if (condensed) {
        if (i32) launch_chunks<T, int32_t, true>(p, cpw, g, b, lds, team, s);
        else launch_chunks<T, int64_t, true>(p, cpw, g, b, lds, team, s);
    } else {
        if (i32) launch_chunks<T, int32_t, false>(p, cpw, g, b, lds, team, s);
        else launch_chunks<T, int64_t, false>(p, cpw, g, b, lds, team, s);
    }
}

} // namespace

int pack_wide_launch(const PackParams &p, int elem_bytes, int index_bytes, hipStream_t stream)
{
    const DeviceInfo &dev = device_info();
    const int64_t row_bytes = p.V * elem_bytes;
    const int nchunks = (int)((row_bytes + 511) / 512);
    // Two chunks per wave (39 registers, all 32 waves of a CU: 60,000 rows of
    // eight chunks 161 us against 176 with four), more only past eight waves;
    // larger teams when the rows are too few for 16 waves per CU.
    int team = 1;
    while (team < kMaxTeam && team < nchunks && (nchunks > 2 * team || p.n * team < (int64_t)dev.num_cus * 16)) team *= 2;
    const int cpw = (nchunks + team - 1) / team;
    const int waves = team > 1 ? team : kSoloWaves;
    const size_t lds = (size_t)((row_bytes + 15) / 16 * 16 + kWave * 4) * (team > 1 ? 1 : waves);
    int64_t grid = (p.n * team + waves - 1) / waves;
    // A small team's block takes more rows while they are few, since its start
    // costs more than a row (8000 and 16,000 rows of 600 words: 32 waves' blocks
    // per CU 51.7 and 70.0 us, 128 waves' 55.0 and 72.9; 48,000 rows 145.6 and
    // 141.2; 8000 rows of 1200 doubles 113 and 103).
    const bool few = team <= 4 && p.n * team <= (int64_t)dev.num_cus * 256;
    const int64_t cap = (int64_t)dev.num_cus * (few ? 32 : 128) / waves;
    if (grid > cap) grid = cap;
    if (p.bitmask) {
        const int64_t words = (p.n + 31) / 32;
        hipLaunchKernelGGL(zero_words_kernel, dim3((unsigned)(words < 65536 ? (words + 255) / 256 : 256)), dim3(256), 0,
                           stream, p.bitmask, words);
        IBP_LAUNCH_CHECK();
    }
    dprintf("[ibp] compress: team of %d waves per row, V=%lld, w=%d, n=%lld, grid %lld x %d\n", team, (long long)p.V,
            elem_bytes, (long long)p.n, (long long)grid, waves * kWave);
    const dim3 g((unsigned)grid), b((unsigned)(waves * kWave));
    const bool i32 = p.index && index_bytes == 4, condensed = p.offsets != nullptr;
    if (elem_bytes == 8) launch<uint64_t>(p, i32, condensed, cpw, g, b, lds, team, stream);
    else launch<uint32_t>(p, i32, condensed, cpw, g, b, lds, team, stream);
    IBP_LAUNCH_CHECK();
    return IBP_OK;
}

} // namespace ibp
