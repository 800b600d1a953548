// The matrix-core kernels of self_attention (self_attention_mfma.hip), as
// self_attention.hip dispatches to them.
#pragma once

#include "launch.hpp"

namespace llaisys::kernels {

constexpr int kSelfAttentionMaxSplits = 16; // key splits the merge kernel takes

struct SelfAttentionPlan {
    int shape;  // which workgroup shape
    int splits; // key splits over workgroups (> 1: partials, then the merge kernel)
};

// Whether the matrix-core kernels take this call (else the general kernel).
bool selfAttentionMfmaTakes(ElemType type, int L, int S, int nkvh, int d, int dv, float scale);
SelfAttentionPlan planSelfAttentionMfma(ElemType type, int L, int S, int nh, int nkvh, int cus);
void selfAttentionMfma(void *out, const void *q, const void *k, const void *v, ElemType type, int L, int S, int nh,
                       int nkvh, int d, float scale, const SelfAttentionPlan &plan, float *part, void *stream);

} // namespace llaisys::kernels
