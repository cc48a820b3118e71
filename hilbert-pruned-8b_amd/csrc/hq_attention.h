// hq_attention.h - causal attention over the backend's fp32 KV cache (hq_attention.hip).
#ifndef HQ_ATTENTION_H
#define HQ_ATTENTION_H

#include <hip/hip_runtime.h>
#include <stddef.h>

struct HqAttnArgs {
    const float *qr;       // [T, nh, hd] rotated queries
    const float *qb;       // [T, qw] raw query rows (the output gate of head j at 2 hd j + hd), read when gated
    const float *kc, *vc;  // [positions, nkv * hd] caches; positions 0 .. pos0 + T - 1 hold keys and values
    _Float16 *out;         // [T, nh * hd]
    float *part;           // hq_attn_work_bytes(): partial rows of split blocks
    int *counters;         // HQ_ATTN_MAX_BLOCKS counters, zero when idle (each launch leaves them zero)
    int T, nh, nkv, hd, qw, gated, pos0;
    float scale;
};

// Row blocks that may split their positions over workgroups, and the partials' size in bytes.
constexpr int HQ_ATTN_MAX_BLOCKS = 1024;
size_t hq_attn_work_bytes(int hd, int n_cu);
hipError_t hq_launch_attention(const HqAttnArgs &a, int n_cu, hipStream_t st);

#endif
