// ibp_pack.h -- parameters of the pack kernels, shared by ibp_pack.hip and
// ibp_pack_wide.hip.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace ibp {

struct PackParams {
    const void *in;
    void *out;
    int64_t num_vecs;
    int64_t V;
    const void *mask;
    const void *bitval;
    const int32_t *clusters; // mask row per source row, or nullptr
    int64_t num_clusters;
    const int64_t *offsets;  // condensed output: inclusive end byte offset per output row
    int64_t stream_bytes;
    const void *index;
    int64_t n;
    uint32_t *bitmask; // may be nullptr with a condensed output
    void *gbuf;        // per-wave slot buffers when they do not fit LDS
    unsigned long long *err;
    int split = 1;     // waves of a block sharing one 32-row group (1: a wave per group)
};

// Rows of more than 64 elements of 4 or 8 bytes and at most kPackWideMaxBytes
// (ibp_pack_wide.hip); p.gbuf and p.split are not used.
constexpr int64_t kPackWideMaxBytes = 32768;
int pack_wide_launch(const PackParams &p, int elem_bytes, int index_bytes, hipStream_t stream);

} // namespace ibp
