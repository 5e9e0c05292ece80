// ibp_fetch_wide.h -- fetch and unpack of rows of more than 64 elements of 4 or
// 8 bytes (the slot format is described in ibp_fetch_dev.h).
//
// A row is cut into chunks of 512 output bytes.  In a chunk lane l owns 8
// bytes: one 8-byte column, or two adjacent 4-byte columns.  Either way they
// are two 32-bit halves, decoded with 32-bit operations: the high half of an
// 8-byte element comes first in the MSB-first stream, so a half of an element
// takes the free bits of its half of the mask.
//
// A team of waves takes a batch of up to kWideRows rows of one mask row; wave
// w of the team takes chunks w, w + team, ... of every row:
//   A. the free bits of each chunk of each row (header flags and mask only),
//   B. their prefix sums: where each chunk's bits begin,
//   C. each chunk of each row unpacked.
//
// What bounds it, and why this shape.  Where a chunk's bits begin depends on
// all chunks before it.  A wave that walks a row chunk by chunk waits out a
// memory latency per chunk, and works out where a column's masked bits lie
// anew for every row: 119 to 130 vector operations per chunk and row.  Here no
// load depends on another chunk's payload, the loads of up to eight rows are
// in flight per wave, and a column's layout is worked out once per batch: 70
// operations.  Measured against the wave per row: 20,000 random 4 KiB rows of
// 4-byte words (40% packed) 70.0 -> 31.1 us (115 MB: 3.7 TB/s; a device copy
// runs at 5.0), a 4096 x 2752 block of 8-byte words whose rows share one of 16
// mask rows 92 -> 47 us, 27,000 rows of 99 words with scattered masks 32.6 -> 21.5 us.
//
// With a mask row per cluster the team looks through a window of rows and
// batches those of one mask row (raw rows need none) where such rows are most of
// the call's; the others go to a wave per row, or to two.
#pragma once

#include "ibp_fetch_dev.h"

namespace ibp {

constexpr int kWideRows = 8;    // rows of a batch, at most
constexpr int kWideWindow = 64; // rows among which those of one mask row are looked for, at most
constexpr int kWideSpan = 64;   // chunks whose positions are worked out together
constexpr int kWideMaxTeam = 8; // waves of a team, at most
constexpr int kWideSolo = 4;    // waves of a block of one-wave teams
// A team's LDS: per row of the batch the positions of a span's chunks and its bits.
constexpr int kWideStride = kWideSpan + 1;
constexpr int kWideLdsWords = kWideRows * kWideStride;

// Rows start at multiples of the element size only.
typedef uint32_t wide8_t __attribute__((ext_vector_type(2), aligned(4)));
typedef uint32_t wide12_t __attribute__((ext_vector_type(3), aligned(4)));
typedef uint32_t wide16_t __attribute__((ext_vector_type(4), aligned(8)));
typedef uint32_t raw16_t __attribute__((ext_vector_type(4), aligned(4)));

// A lane's 8 bytes of mask or bitval in a chunk, as the half that comes first
// in the stream and the other; `left` of the chunk's columns are in the row
// (the others are not read, and give 0).
template <typename T>
__device__ __forceinline__ void load_wide_cols(const T *cols, int left, uint32_t &first, uint32_t &second)
{
    const int lane = lane_id();
    wide8_t v = {0u, 0u};
    if (left == 512 / (int)sizeof(T)) { // uniform
        v = reinterpret_cast<const wide8_t *>(cols)[lane];
    } else {
        const uint32_t *w = reinterpret_cast<const uint32_t *>(cols) + 2 * lane;
        const int words = left * (int)(sizeof(T) / 4);
        if (2 * lane < words) v.x = w[0];
        if (2 * lane + 1 < words) v.y = w[1];
    }
    first = sizeof(T) == 8 ? v.y : v.x;
    second = sizeof(T) == 8 ? v.x : v.y;
}

// a where mask has a bit, else b.
__device__ __forceinline__ uint32_t bit_select(uint32_t mask, uint32_t a, uint32_t b)
{
    return __builtin_amdgcn_bitop3_b32(a, b, mask, 0xe4);
}

// How the top-aligned free bits of a half spread to the zero bits of its mask,
// built once per batch of rows and applied to each of them.
//  * Two runs (no half of the wave has more than two runs of masked bits, the
//    usual case): opening a run moves the bits below its start, a[0] (a[2]),
//    down by its length, a[1] (a[3]): two operations a run.  A half with fewer
//    runs has entries that move nothing.
//  * Otherwise the expand operation of Warren's Hacker's Delight (7-5),
//    mirrored to fill from the top: step i moves the bits of a[i] down by 2^i,
//    ten operations whatever the mask.
struct WideCode {
    uint32_t a[5];
};

// The highest run of m; m loses it.  With m = 0: low = 1, g = 0 (nothing
// moves).  A mask of 32 bits is used up in two steps; the ORs keep the counts
// below 32.
__device__ __forceinline__ void next_run(uint32_t &m, uint32_t &low, uint32_t &g)
{
    const int s = __builtin_clz(m | 1u);
    low = 0xffffffffu >> s;
    g = (uint32_t)__builtin_clz(~(m << s) | 1u);
    m &= low >> g;
}

__device__ __forceinline__ void expand_steps(uint32_t mask, WideCode &c)
{
    uint32_t m = ~mask, mk = mask >> 1;
#pragma unroll
    for (int i = 0; i < 5; ++i) {
        uint32_t mp = mk ^ (mk >> 1);
        mp ^= mp >> 2;
        mp ^= mp >> 4;
        mp ^= mp >> 8;
        mp ^= mp >> 16;
        c.a[i] = mp & m;
        m = (m ^ c.a[i]) | (c.a[i] << (1 << i));
        mk &= ~mp;
    }
}

// true: the codes are the two-run form (uniform).
__device__ __forceinline__ bool wide_codes(uint32_t m0, uint32_t m1, WideCode &c0, WideCode &c1)
{
    uint32_t e0 = m0, e1 = m1;
    next_run(e0, c0.a[0], c0.a[1]);
    next_run(e1, c1.a[0], c1.a[1]);
    next_run(e0, c0.a[2], c0.a[3]);
    next_run(e1, c1.a[2], c1.a[3]);
    c0.a[4] = c1.a[4] = 0;
    if (ballot((e0 | e1) != 0) == 0) return true;
    expand_steps(m0, c0);
    expand_steps(m1, c1);
    return false;
}

template <bool TWO>
__device__ __forceinline__ uint32_t wide_spread(uint32_t v, const WideCode &c)
{
    if constexpr (TWO) {
        v = bit_select(c.a[0], v >> c.a[1], v);
        v = bit_select(c.a[2], v >> c.a[3], v);
    } else {
#pragma unroll
        for (int i = 4; i >= 0; --i) v = bit_select(c.a[i], v >> (1 << i), v);
    }
    return v;
}

// Sums of eight values over the wave's lanes.  Two exchanges between halves
// and quarters of the wave leave two registers: lane 16 k + 15 of z0 holds sum
// 2 k, of z1 sum 2 k + 1 (20 operations; eight scans would take 48).
__device__ __forceinline__ int row16_sum(int x) // at lane 15 of each 16 lanes
{
    x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, true);
    x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, true);
    x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, true);
    x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, true);
    return x;
}
__device__ __forceinline__ void wave_sum8(const int (&x)[8], int &z0, int &z1)
{
    uint32_t y[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) { // lanes below 32: sum k, the others: sum k + 4
        const auto s = __builtin_amdgcn_permlane32_swap((uint32_t)x[k], (uint32_t)x[k + 4], false, false);
        y[k] = s[0] + s[1];
    }
    const auto a = __builtin_amdgcn_permlane16_swap(y[0], y[2], false, false); // quarters: sums 0, 2, 4, 6
    const auto b = __builtin_amdgcn_permlane16_swap(y[1], y[3], false, false); // 1, 3, 5, 7
    z0 = row16_sum((int)(a[0] + a[1]));
    z1 = row16_sum((int)(b[0] + b[1]));
}

// The batch's rows: lane r (and r + 8, r + 16, ...) holds row r's.
// (Offsets from the compressed data, not pointers: an address put together
// from exchanged lanes would be loaded with flat instructions.)
struct WideRow {
    int64_t row;    // where the stored row starts
    int64_t stored; // its bytes
    int64_t cursor; // the span's first bit in it
    int out;        // its output row, from the batch's first one (mask row per cluster)
};

// The same rows' stretches of a span: a stretch starts a word before the
// span's first bit, so that bit (position - 1) of every position is in it.
struct WideStretch {
    int64_t base;
    uint32_t room; // stored bytes from there, clamped to 2^31 - 1
    uint32_t q;    // chunk: the bit before its first one
};

// NT: the store policy (rows_fill_lines).  SUB: rows unpacked together, at most:
// 8, 4, or 1 (batches are single rows).  LOCKSTEP: teams of one block run rows
// of their own together, so every wave passes every barrier, whatever its row.
template <typename T, int LAYOUT, bool NT, int SUB, bool LOCKSTEP = false>
struct WideBatch {
    static constexpr bool ONE = SUB == 1;
    static constexpr int W = (int)sizeof(T);
    static constexpr int kCols = 512 / W; // columns of a chunk
    enum : int { kAny, kFast, kWhole };
    template <int N>
    using Int = std::integral_constant<int, N>;

    const FetchParams &p;
    const unsigned char *const comp;
    const int team, slot;  // waves of the team, this wave's place in it
    uint32_t *const lds;   // kWideLdsWords words shared by the team
    const int lane;

    __device__ __forceinline__ WideBatch(const FetchParams &p_, int team_, int slot_, uint32_t *lds_)
        : p(p_), comp((const unsigned char *)p_.comp), team(team_), slot(slot_), lds(lds_),
          lane(lane_id())
    {
    }

    // The lane number as a value of its own: what is computed from it stays
    // where it is used (hoisted to the batch loop it fills the registers).
    static __device__ __forceinline__ int fresh_lane()
    {
        int l = lane_id();
        asm volatile("" : "+v"(l));
        return l;
    }

    // Orders the team's LDS accesses: a block barrier, unless the team is one wave.
    __device__ __forceinline__ void sync() const
    {
        if (team > 1) {
            __syncthreads();
        } else {
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        }
    }

    // Header flags of chunk c for the rows in `rows`: lane 8 k + r holds 32-bit
    // word k of row r's flags (2 words per chunk of 8-byte elements, 4 of
    // 4-byte ones).
    __device__ __forceinline__ uint32_t load_flags(const WideRow &me, int64_t c, uint32_t rows) const
    {
        constexpr int kWords = kCols / 32;
        const int64_t hdr = header_bytes(p.vec_size, W);
        const int64_t at = c * (kCols / 8) + (lane >> 3) * 4;
        const bool ok = lane < 8 * kWords && ((rows >> (lane & 7)) & 1) && at + 4 <= (hdr < me.stored ? hdr : me.stored);
        return ok ? *reinterpret_cast<const uint32_t *>(comp + me.row + at) : 0u;
    }

    // Row r's flags of this lane's columns: 8-byte elements: all ones or zero;
    // 4-byte elements: the 32 flags that hold them (bits 2 (l % 16) and the
    // next one of word l / 16).
    __device__ __forceinline__ uint32_t lane_flags(int lane, uint32_t flags, int r) const
    {
        if constexpr (W == 8) {
            const uint64_t hw = ((uint64_t)readlane(flags, 8 + r) << 32) | readlane(flags, r);
            return __builtin_amdgcn_inverse_ballot_w64(hw) ? 0xffffffffu : 0u;
        } else {
            return shfl(flags, (lane >> 4) * 8 + r);
        }
    }
    // ... as a mask of the first half (k = 0) or of the second.
    __device__ __forceinline__ uint32_t half_flag(int lane, uint32_t f, int k) const
    {
        return W == 8 ? f : (uint32_t)__builtin_amdgcn_sbfe((int)f, 2 * (lane & 15) + k, 1);
    }
    // Bits that masked columns save in this lane (s0, s1: of the halves).
    __device__ __forceinline__ int lane_saved(int lane, uint32_t f, int s0, int s1) const
    {
        if constexpr (W == 8) return (s0 + s1) & (int)f;
        else return (s0 & (int)half_flag(lane, f, 0)) + (s1 & (int)half_flag(lane, f, 1));
    }

    // 64 bits of the stream from bit q + 1 of the stretch at `base` (first bit
    // at the top), for every lane.  INSIDE: the chunk's windows end within the
    // stretch's `room` bytes; otherwise words past them read as zero.
    struct Window {
        uint32_t d0, d1, d2, d3;
    };
    template <bool INSIDE>
    static __device__ __forceinline__ Window load_window(const unsigned char *base, uint32_t q, uint32_t room)
    {
        Window w{0u, 0u, 0u, 0u};
        if constexpr (W == 4) {
            const uint32_t off = (q >> 5) * 4;
            if constexpr (INSIDE) {
                const wide12_t v = *reinterpret_cast<const wide12_t *>(base + off);
                w = {v.x, v.y, v.z, 0u};
            } else {
                const uint32_t *d = reinterpret_cast<const uint32_t *>(base + off);
                if (off + 4 <= room) w.d0 = d[0];
                if (off + 8 <= room) w.d1 = d[1];
                if (off + 12 <= room) w.d2 = d[2];
            }
        } else {
            const uint32_t off = (q >> 6) * 8;
            if constexpr (INSIDE) {
                const wide16_t v = *reinterpret_cast<const wide16_t *>(base + off);
                w = {v.x, v.y, v.z, v.w};
            } else {
                const uint32_t *d = reinterpret_cast<const uint32_t *>(base + off);
                if (off + 8 <= room) {
                    w.d0 = d[0];
                    w.d1 = d[1];
                }
                if (off + 16 <= room) {
                    w.d2 = d[2];
                    w.d3 = d[3];
                }
            }
        }
        return w;
    }
    static __device__ __forceinline__ uint64_t window_bits(const Window &w, uint32_t q)
    {
        uint32_t s0, s1, s2; // stream words from the one that holds bit q
        if constexpr (W == 4) {
            s0 = w.d0;
            s1 = w.d1;
            s2 = w.d2;
        } else { // 8-byte words: the high half comes first
            const bool odd = (q >> 5) & 1u;
            s0 = odd ? w.d0 : w.d1;
            s1 = odd ? w.d3 : w.d0;
            s2 = odd ? w.d2 : w.d3;
        }
        // shifted right by the bits that follow the window's first 32: -(q + 1) mod 32
        const uint32_t hi = __builtin_amdgcn_alignbit(s0, s1, ~q), lo = __builtin_amdgcn_alignbit(s1, s2, ~q);
        return ((uint64_t)hi << 32) | lo;
    }

    // Phase C for rows [r0, r0 + N) of the batch, chunk c: m, b the
    // column's mask and bitval halves, w their codes (TWO: the two-run
    // form); pk, raw, live: the rows'
    // kinds; out: the chunk of output row 0.  kAny: rows of any kind.
    // kFast: every row is packed and its windows lie inside the stored row;
    // kWhole: and the chunk is whole.
    template <int MODE, bool TWO, int N, int r0>
    __device__ __forceinline__ void unpack_rows(const WideRow &me, const WideStretch &st, uint32_t pk,
                                                uint32_t raw, uint32_t live, uint32_t inside, unsigned char *out,
                                                int64_t c, int left, uint32_t flags, const WideCode &w0,
                                                const WideCode &w1, uint32_t m0, uint32_t m1, uint32_t b0,
                                                uint32_t b1) const
    {
        constexpr bool FAST = MODE != kAny;
        const int lane = fresh_lane();
        const int saved0 = __builtin_popcount(m0), saved1 = __builtin_popcount(m1);
        const int words = left * (W / 4);
        // bits of this lane's columns
        const int full = MODE == kWhole || 2 * lane + 2 <= words ? 64 : 2 * lane < words ? 32 : 0;
        Window win[N];
        uint32_t q[N], f[N];
#pragma unroll
        for (int u = 0; u < N; ++u) {
            const int r = r0 + u;
            win[u] = {0u, 0u, 0u, 0u};
            q[u] = f[u] = 0;
            if (FAST || ((pk >> r) & 1)) { // uniform
                f[u] = lane_flags(lane, flags, r);
                const int L = full - lane_saved(lane, f[u], saved0, saved1);
                q[u] = readlane(st.q, r) + (uint32_t)(wave_incl_scan(L) - L);
                const unsigned char *base = comp + readlane(st.base, r);
                if (FAST || ((inside >> r) & 1))
                    win[u] = load_window<true>(base, q[u], 0);
                else
                    win[u] = load_window<false>(base, q[u], readlane(st.room, r));
            } else if ((raw >> r) & 1) {
                const unsigned char *row = comp + readlane(me.row, r) + c * 512;
                if (left == kCols) {
                    const wide8_t v = reinterpret_cast<const wide8_t *>(row)[lane];
                    win[u].d0 = v.x;
                    win[u].d1 = v.y;
                } else {
                    const uint32_t *d = reinterpret_cast<const uint32_t *>(row) + 2 * lane;
                    if (2 * lane < words) win[u].d0 = d[0];
                    if (2 * lane + 1 < words) win[u].d1 = d[1];
                }
            }
        }
#pragma unroll
        for (int u = 0; u < N; ++u) {
            const int r = r0 + u;
            if (MODE != kWhole && !((live >> r) & 1)) continue; // uniform
            wide8_t o = {win[u].d0, win[u].d1};
            if (FAST || ((pk >> r) & 1)) {
                const uint32_t f0 = half_flag(lane, f[u], 0), f1 = half_flag(lane, f[u], 1);
                const uint64_t v = window_bits(win[u], q[u]);
                const uint32_t v0 = (uint32_t)(v >> 32);
                const uint32_t v1 = (uint32_t)((v << (32 - (saved0 & f0))) >> 32);
                uint32_t x0 = wide_spread<TWO>(v0, w0), x1 = wide_spread<TWO>(v1, w1);
                x0 = bit_select(f0, (x0 & ~m0) | b0, v0);
                x1 = bit_select(f1, (x1 & ~m1) | b1, v1);
                o = W == 8 ? (wide8_t){x1, x0} : (wide8_t){x0, x1};
            }
            unsigned char *d = out + ((LAYOUT & kLayoutClustered) ? readlane(me.out, r) : r) * (p.vec_size * W);
            if (MODE == kWhole || left == kCols) {
                wide8_t *e = reinterpret_cast<wide8_t *>(d) + lane;
                if constexpr (NT) __builtin_nontemporal_store(o, e);
                else *e = o;
            } else {
                uint32_t *e = reinterpret_cast<uint32_t *>(d) + 2 * lane;
                if (2 * lane < words) store_row_word<uint32_t, NT>(e, o.x);
                if (2 * lane + 1 < words) store_row_word<uint32_t, NT>(e + 1, o.y);
            }
        }
    }

    // A batch without a packed row: its rows as they are stored (raw) or zero,
    // in pieces of 4 KiB spread over the team, four 16-byte loads in flight per
    // lane (4096 raw rows of 1024 and 2752 doubles by chunks 1431 GB/s, so 2165).
    __device__ __forceinline__ void copy_rows(const WideRow &me, int nrows, uint32_t raw, unsigned char *out) const
    {
        const int64_t bytes = p.vec_size * W;
        int turn = 0;
        for (int r = 0; r < nrows; ++r) {
            const unsigned char *src = comp + readlane(me.row, r);
            unsigned char *dst = out + ((LAYOUT & kLayoutClustered) ? readlane(me.out, r) : r) * bytes;
            const bool stored = (raw >> r) & 1;
            for (int64_t at = 0; at < bytes; at += 4096, turn = turn + 1 == team ? 0 : turn + 1) {
                if (turn != slot) continue; // uniform
                const int64_t o = at + fresh_lane() * 16;
                wide16_t v[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    v[u] = (wide16_t){0u, 0u, 0u, 0u};
                    if (stored && o + u * 1024 + 16 <= bytes)
                        v[u] = *reinterpret_cast<const raw16_t *>(src + o + u * 1024);
                }
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const int64_t k = o + u * 1024;
                    if (k + 16 <= bytes) {
                        raw16_t *e = reinterpret_cast<raw16_t *>(dst + k);
                        if constexpr (NT) __builtin_nontemporal_store((raw16_t)v[u], e);
                        else *e = v[u];
                    } else { // the row's last words
                        for (int64_t i = k; i < bytes; i += 4)
                            *reinterpret_cast<uint32_t *>(dst + i) =
                                stored ? *reinterpret_cast<const uint32_t *>(src + i) : 0u;
                    }
                }
            }
        }
    }

    // Rows [0, nrows) of the batch (output rows out0, out0 + 1, ...; with
    // clusters me.out) of mask row cl: pk, raw: the packed and the raw rows (the others become zero).
    __device__ __forceinline__ void run(WideRow me, int nrows, uint32_t pk, uint32_t raw, int64_t cl, int64_t out0) const
    {
        const int64_t V = p.vec_size;
        const T *mask = (const T *)p.mask + cl * V, *bitval = (const T *)p.bitval + cl * V;
        const int64_t nchunks = (V + kCols - 1) / kCols;
        const uint32_t live = (1u << nrows) - 1;
        unsigned char *out = (unsigned char *)p.out + out0 * (V * W);
        const bool copied = !pk && !p.host_rows; // uniform for the team (over PCIe by chunks: 57 against 55 GB/s)
        if (copied) {
            copy_rows(me, nrows, raw, out);
            if constexpr (!LOCKSTEP) return;
        }
        auto cols_left = [&](int64_t c) { return V - c * kCols < kCols ? (int)(V - c * kCols) : kCols; };
        for (int64_t c0 = 0; c0 < nchunks; c0 += kWideSpan) {
            const int nc = nchunks - c0 < kWideSpan ? (int)(nchunks - c0) : kWideSpan;
            if (LOCKSTEP || pk) { // uniform for the team
                sync(); // the positions before these have been read
                for (int k = pk ? slot : nc; k < nc; k += team) {
                    const int lane = fresh_lane();
                    const int left = cols_left(c0 + k);
                    uint32_t m0, m1;
                    load_wide_cols<T>(mask + (c0 + k) * kCols, left, m0, m1);
                    const uint32_t flags = load_flags(me, c0 + k, pk);
                    const int s0 = __builtin_popcount(m0), s1 = __builtin_popcount(m1);
                    if constexpr (ONE) {
                        const int z = wave_sum(lane_saved(lane, lane_flags(lane, flags, 0), s0, s1));
                        if (lane == 0) lds[k] = (uint32_t)(left * W * 8 - z);
                    } else {
                        int x[kWideRows], z0, z1;
#pragma unroll
                        for (int r = 0; r < kWideRows; ++r) {
                            x[r] = lane_saved(lane, lane_flags(lane, flags, r), s0, s1);
                        }
                        wave_sum8(x, z0, z1);
                        if ((lane & 15) == 15) {
                            uint32_t *t = lds + 2 * (lane >> 4) * kWideStride + k;
                            t[0] = (uint32_t)(left * W * 8 - z0);
                            t[kWideStride] = (uint32_t)(left * W * 8 - z1);
                        }
                    }
                }
                sync();
                for (int r = pk ? slot : kWideRows; r < (ONE ? 1 : kWideRows); r += team) {
                    uint32_t *t = lds + r * kWideStride;
                    const int x = lane < nc ? (int)t[lane] : 0;
                    const int incl = wave_incl_scan(x);
                    t[lane] = (uint32_t)(incl - x);
                    if (lane == kWave - 1) t[kWideSpan] = (uint32_t)incl;
                }
                sync();
            }
            if (LOCKSTEP && (copied || nrows == 0)) continue;
            const uint32_t *mine = lds + (ONE ? 0 : (lane & 7) * kWideStride); // this lane's row's positions
            WideStretch st;
            const int64_t at = (me.cursor >> (W == 8 ? 6 : 5)) * W - W;
            const int64_t room = me.stored - at;
            const uint32_t rel = (uint32_t)(me.cursor - at * 8);
            st.base = me.row + at;
            st.room = room <= 0 ? 0u : room < 0x7fffffff ? (uint32_t)room : 0x7fffffffu;
            st.q = 0;
            for (int k = slot; k < nc; k += team) {
                const int64_t c = c0 + k;
                const int left = cols_left(c);
                uint32_t m0, m1, b0, b1, flags = 0, inside = 0;
                m0 = m1 = b0 = b1 = 0;
                WideCode w0{}, w1{};
                bool two = true;
                if (pk) {
                    load_wide_cols<T>(mask + c * kCols, left, m0, m1);
                    load_wide_cols<T>(bitval + c * kCols, left, b0, b1);
                    flags = load_flags(me, c, pk);
                    st.q = rel + mine[k] - 1u;
                    // no window of the chunk ends past its last bit's byte + 16
                    const uint32_t end = rel + (k + 1 < nc ? mine[k + 1] : mine[kWideSpan]);
                    inside = (uint32_t)ballot(end / 8 + 16 <= st.room);
                    two = wide_codes(m0, m1, w0, w1);
                }
                // Rows r0, r0 + 1, ... of the batch (places past nrows stand
                // for row 0 again: only `live` tells them apart).
                auto go = [&](auto mode, auto form, auto sub, auto r0) {
                    unpack_rows<decltype(mode)::value, decltype(form)::value, decltype(sub)::value, decltype(r0)::value>(
                        me, st, pk, raw, live, inside, out + c * 512, c, left, flags, w0, w1, m0, m1, b0, b1);
                };
                auto rows = [&](auto mode, auto form) {
                    constexpr int kSub = SUB < 8 || (decltype(mode)::value == kWhole && decltype(form)::value) ? SUB : 4;
                    go(mode, form, Int<kSub>(), Int<0>());
                    if constexpr (kSub == 4)
                        if (nrows > 4) go(mode, form, Int<kSub>(), Int<4>());
                };
                auto go_mode = [&](auto mode) {
                    if (two) rows(mode, std::true_type());
                    else rows(mode, std::false_type());
                };
                const bool fast = (pk & inside & 0xffu) == 0xffu;
                if (fast && (ONE || nrows == kWideRows) && left == kCols) go_mode(Int<kWhole>());
                else if (fast) go_mode(Int<kFast>());
                else go_mode(Int<kAny>());
            }
            if (pk && c0 + kWideSpan < nchunks) me.cursor += mine[kWideSpan];
        }
    }
};

template <typename T>
__device__ __forceinline__ WideRow wide_row(const FetchParams &p, const RowMeta &m)
{
    WideRow r;
    r.row = m.word * (int64_t)sizeof(T);
    r.stored = m.len * (int64_t)sizeof(T);
    r.cursor = header_bytes(p.vec_size, (int)sizeof(T)) * 8;
    r.out = 0;
    return r;
}

// Reads the headers of packed pinned rows in one go before their words are read by
// chunk (the team waits in run()): their lines then cross PCIe once.
__device__ __forceinline__ void touch_headers(const FetchParams &p, int w, const WideRow &me, uint64_t packed, int nrows, int team,
                                              int slot)
{
    const int64_t words = header_bytes(p.vec_size, w) / 4;
    for (int t = slot; t < nrows; t += team) {
        if (!((packed >> t) & 1)) continue; // uniform
        const uint32_t *h = (const uint32_t *)((const unsigned char *)p.comp + readlane(me.row, t));
        const int64_t n = readlane(me.stored, t) / 4 < words ? readlane(me.stored, t) / 4 : words;
        for (int64_t i = lane_id(); i < n; i += kWave) {
            const uint32_t x = h[i];
            asm volatile("" ::"v"(x)); // the read is the point
        }
    }
}

// Output rows [b, e) by a team of waves (called by every wave of the team with
// the same arguments but slot; team > 1: the waves of a block): kWideRows at
// most make a batch.
template <typename T, typename IdxT, int LAYOUT, bool NT>
__device__ __forceinline__ void fetch_wide_batch(const FetchParams &p, int64_t b, int64_t e, int team, int slot,
                                                 uint32_t *lds)
{
    const int nrows = e - b < kWideRows ? (int)(e - b) : kWideRows;
    // places past the last row stand for row 0 again
    const int r = (lane_id() & (kWideRows - 1)) < nrows ? lane_id() & (kWideRows - 1) : 0;
    const int64_t s = load_index<IdxT>(p.index, b + r);
    const RowMeta m = decode_meta<T, LAYOUT>(p, s, true, load_meta<LAYOUT>(p, s, true));
    const WideRow me = wide_row<T>(p, m);
    if (p.host_rows && p.vec_size * (int64_t)sizeof(T) > 2048)
        touch_headers(p, (int)sizeof(T), me, ballot(m.ok && m.packed), nrows, team, slot);
    const WideBatch<T, LAYOUT, NT, (LAYOUT & kLayoutClustered) ? 1 : 8> batch(p, team, slot, lds);
    constexpr uint32_t kLow = (1u << kWideRows) - 1;
    const uint32_t ok = (uint32_t)ballot(m.ok) & kLow, pk = (uint32_t)ballot(m.ok && m.packed) & kLow;
    if (p.err && slot == 0 && lane_id() == 0) {
        const int bad = nrows - (int)__builtin_popcount(ok & ((1u << nrows) - 1));
        if (bad) atomicAdd(p.err, (unsigned long long)bad);
    }
    // (with clusters: one row)
    batch.run(me, nrows, pk, ok & ~pk, (LAYOUT & kLayoutClustered) ? readlane(m.cl, 0) : 0, b);
}

// With a mask row per cluster: the rows [b, e) of a window, lane r: row r.
template <typename T>
struct WideWindow {
    RowMeta m;
    int key;     // what rows of one batch share: the mask row, -1 for raw rows, which need none; -2: refused
    uint64_t ok; // the rows that are not refused
    int nrows;

    // i: this lane's output row (places past the last one: any row).
    template <typename IdxT, int LAYOUT>
    __device__ __forceinline__ void load(const FetchParams &p, int64_t i, int rows)
    {
        nrows = rows;
        const int64_t s = load_index<IdxT>(p.index, i);
        m = decode_meta<T, LAYOUT>(p, s, true, load_meta<LAYOUT>(p, s, true));
        key = !m.ok ? -2 : m.packed ? m.cl : -1;
        count();
    }
    template <typename IdxT, int LAYOUT>
    __device__ __forceinline__ void load_window(const FetchParams &p, int64_t b, int64_t e)
    {
        load<IdxT, LAYOUT>(p, b + (lane_id() < (int)(e - b) ? lane_id() : 0), (int)(e - b));
    }
    __device__ __forceinline__ void count()
    {
        ok = ballot(key != -2) & (nrows == kWave ? ~0ull : (1ull << nrows) - 1);
    }
    // Row r, which is the same for the whole wave.
    __device__ __forceinline__ RowMeta row(int r) const
    {
        RowMeta me;
        me.word = readlane(m.word, r);
        me.len = readlane(m.len, r);
        me.cl = readlane(m.cl, r);
        me.ok = (ok >> r) & 1;
        me.packed = me.ok && readlane(key, r) >= 0;
        return me;
    }
    // The rows that one batch may hold beside row r, which is not refused.
    __device__ __forceinline__ uint64_t alike(int r) const { return ballot(key == readlane(key, r)) & ok; }
    // The raw rows and those of mask rows with `each` rows or more, or with all
    // but a quarter of the window's together with the raw ones.
    __device__ __forceinline__ uint64_t alike_rows(int each) const
    {
        const uint64_t raw = ballot(key == -1) & ok;
        uint64_t take = raw, left = ok & ~raw;
        const int nraw = __builtin_popcountll(raw);
        while (__builtin_popcountll(left) >= each || __builtin_popcountll(left | raw) * 4 >= nrows * 3) { // uniform
            if (!left) break;
            const uint64_t same = alike(__builtin_ctzll(left));
            const int n = __builtin_popcountll(same);
            left &= ~same;
            if (n >= each || (n + nraw) * 4 >= nrows * 3) take |= same;
        }
        return take;
    }
    // Whether all rows go together: one mask row, and raw ones.  (Without a
    // branch, which takes a register more.)
    __device__ __forceinline__ bool uniform() const
    {
        const uint64_t packed = ballot(key >= 0) & ok;
        return __builtin_popcountll(ok) >= nrows &&
               (packed == 0 || alike(__builtin_ctzll(packed | 1ull << 63)) == packed);
    }
};

// Whether windows of `rows` rows (more than kWideRows) go to teams at all, from
// 64 rows of the call (four stretches of 16): mask rows that a window is to hold
// twelve rows of have to make three quarters of them; of windows of 16, one
// mask row nearly all of them.  Every wave that asks finds the same answer.
// (By each window for itself, chance gives the teams a few windows of tables
// whose rows should all go to a wave each, which then wait for them: 8192 rows of
// 800 doubles of two mask rows 62 us, a wave per row 40, now 45.)
template <typename T, typename IdxT, int LAYOUT>
__device__ __forceinline__ bool windows_pay(const FetchParams &p, int rows)
{
    WideWindow<T> sample;
    const int64_t i = lane_id() / 16 * (p.n / 4) + lane_id() % 16;
    sample.template load<IdxT, LAYOUT>(p, i < p.n ? i : p.n - 1, kWave);
    const uint64_t raw = ballot(sample.key == -1);
    const int each = rows <= 16 ? 60 : kWave * 12 / rows, least = rows <= 16 ? 60 : 48;
    uint64_t left = sample.ok & ~raw;
    const int nraw = __builtin_popcountll(raw);
    int take = nraw;
    while (left && take + __builtin_popcountll(left) >= least) { // uniform
        const uint64_t same = sample.alike(__builtin_ctzll(left));
        const int n = __builtin_popcountll(same);
        left &= ~same;
        if (n >= each || n + nraw >= least) take += n;
    }
    return take >= least;
}

// A window's rows in the team's LDS: where the stored rows start, their bytes,
// their keys.
constexpr int kWindowLdsWords = 5 * kWideWindow;
constexpr int kWindowAlike = 6; // rows of one mask row that a team takes from a window, at least

// The part of a window that a team of two waves or more takes, in batches of
// rows alike.  WHOLE (windows of kWideRows at most): all of it, in batches if all
// its rows go together, else two waves per row.  One wave reads the rows'
// metadata for the team.
//
// Batches of few rows cost as much as full ones, and a window's rows that go by
// themselves wait for its batches: taken from two or four alike rows on, windows
// of 16 evenly used mask rows lost up to 2.1 times a wave per row (2000 rows of
// 1600 words 22 us against 46, now 16).  A batch's rows are unpacked four at a
// time: with what the window keeps, eight put 22 to 28 registers in scratch
// memory.  (Two at a time: 4096 x 2752 doubles from HBM 56 us, four 48.)
template <typename T, typename IdxT, int LAYOUT, bool NT, bool WHOLE>
__device__ __forceinline__ void fetch_wide_window(const FetchParams &p, int64_t b, int64_t e, int team, int slot,
                                                  uint32_t *lds, uint32_t *rows)
{
    const WideBatch<T, LAYOUT, NT, 4> batch(p, team, slot, lds);
    int64_t *const start = reinterpret_cast<int64_t *>(rows), *const stored = start + kWideWindow;
    int *const keys = reinterpret_cast<int *>(stored + kWideWindow);
    WideWindow<T> win;
    batch.sync(); // the window before this one is done
    if (slot == 0) {
        win.template load_window<IdxT, LAYOUT>(p, b, e);
        start[lane_id()] = win.m.word * (int64_t)sizeof(T);
        stored[lane_id()] = win.m.len * (int64_t)sizeof(T);
        keys[lane_id()] = win.key;
    }
    batch.sync();
    win.nrows = (int)(e - b);
    win.key = keys[lane_id()];
    win.count();
    if constexpr (WHOLE) {
        if (!win.uniform()) {
            // Two waves a row.
            const WideBatch<T, LAYOUT, NT, 1, true> one(p, 2, slot & 1, lds + (slot >> 1) * kWideStride);
            for (int r0 = 0; r0 < win.nrows; r0 += team / 2) {
                const int r = r0 + (slot >> 1);
                const bool row = r < win.nrows; // the last pairs may have none
                const int kind = row ? readlane(win.key, r) : -2;
                WideRow part;
                part.row = start[row ? r : 0];
                part.stored = stored[row ? r : 0];
                part.cursor = header_bytes(p.vec_size, (int)sizeof(T)) * 8;
                part.out = 0;
                if (p.host_rows && kind >= 0 && p.vec_size * (int64_t)sizeof(T) > 2048)
                    touch_headers(p, (int)sizeof(T), part, 1, 1, 2, slot & 1);
                if (row && kind == -2 && p.err && (slot & 1) == 0 && lane_id() == 0) atomicAdd(p.err, 1ull);
                one.run(part, row ? 1 : 0, kind >= 0 ? 0xffu : 0u, kind == -1 ? 0xffu : 0u, kind < 0 ? 0 : kind, b + r);
            }
            return;
        }
    }
    for (uint64_t left = WHOLE ? win.ok : win.alike_rows(kWindowAlike); left;) {
        const int head = __builtin_ctzll(left);
        uint64_t alike = win.alike(head) & left;
        left &= ~alike;
        const int kind = readlane(win.key, head), cl = kind < 0 ? 0 : kind;
        while (alike) {
            // place k of the batch: the k-th of them; places past the last stand for the first
            const int place = lane_id() & (kWideRows - 1);
            int from = __builtin_ctzll(alike), n = 0;
#pragma unroll
            for (int k = 0; k < kWideRows; ++k) {
                if (!alike) break; // uniform
                const int at = __builtin_ctzll(alike);
                alike &= alike - 1;
                from = place == k ? at : from;
                ++n;
            }
            WideRow part;
            part.row = start[from];
            part.stored = stored[from];
            part.cursor = header_bytes(p.vec_size, (int)sizeof(T)) * 8;
            part.out = from;
            constexpr uint32_t kLow = (1u << kWideRows) - 1;
            if (p.host_rows && kind >= 0 && p.vec_size * (int64_t)sizeof(T) > 2048)
                touch_headers(p, (int)sizeof(T), part, kLow, n, team, slot);
            batch.run(part, n, kind < 0 ? 0u : kLow, kind < 0 ? kLow : 0u, cl, b);
        }
    }
}

// Whether teams of waves are the faster way (else a wave per row).
bool fetch_wide_pays(const FetchParams &p, int layout, int elem_bytes, int nthreads);
// The plain fetch's launch for rows of more than 64 elements of 4 or 8 bytes
// (ibp_fetch_wide.hip).  nblks <= 0: a grid for the rows; nthreads > 0: threads
// of a block, at most.
struct WideShape {
    int64_t grid;
    int block; // threads
    int team;  // waves
    int rows;  // of a batch, or of a window
};
WideShape fetch_wide_shape(const FetchParams &p, int layout, int elem_bytes, int nblks, int nthreads);
int fetch_wide_launch(const FetchParams &p, int layout, int elem_bytes, int index_bytes, int nblks,
                      const WideShape &shape, hipStream_t stream);

} // namespace ibp
