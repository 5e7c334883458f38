// Shared between the int8 attention's two paths: attention.hip (step by step, a head's scores in
// memory) and attention_fused.hip (one launch, no scores in memory).
#pragma once

#include "common.h"

namespace fg {

// Q7b32 levels of four values at scale d (quant.rs:143-150: rne(x / d) clamped to ±63 through the
// saturating cast), packed as one dword of device levels.
__device__ __forceinline__ int q7_levels4(const float (&x)[4], float d)
{
    int l[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const float v = __builtin_rintf(x[j] / d);
        const int level = v != v ? 0 : v >= 127.0f ? 127 : v <= -128.0f ? -128 : int(v);
        l[j] = level < -63 ? -63 : (level > 63 ? 63 : level);
    }
    return pack4(l[0], l[1], l[2], l[3]);
}

// The fused path's scratch for a call, and its launches over it: head_dim at most 128.
size_t attend_fused_bytes(const fg_attention *c);
int launch_attend_fused(const fg_attention *c, float *out, void *workspace, hipStream_t s);

}  // namespace fg
