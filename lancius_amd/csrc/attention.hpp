// What the attention translation units share.
#pragma once

#include "common.hpp"
#include "kernels.hpp"

namespace lancius {

struct AttnParams {
    float* O[LANCIUS_HIP_MAX_GROUP];
    const float* Q[LANCIUS_HIP_MAX_GROUP];
    const float* K[LANCIUS_HIP_MAX_GROUP];
    const float* V[LANCIUS_HIP_MAX_GROUP];
    int batch;  // batches per group entry
    int S, H, D;   // queries per sequence, query heads, head dim
    int Skv, Hkv;  // keys per sequence, K/V heads (query head h reads K/V head h / (H / Hkv))
    int causal;    // query i sees keys j <= i + (Skv - S)
    float qscale;  // scale * log2(e)
    int q_tiles;
    int pair_tiles;  // causal grid small enough to be resident at once (see attention_mfma)
    int Z;         // count * batch independent problems
};

// 2^x as the one v_exp_f32.  exp2f adds a range fix-up (compare, select,
// add, select, ldexp: five more instructions) that only changes results
// below 2^-126; the softmax exponents here are <= 0 and a probability under
// 2^-126 does not move a sum that is >= 1.
__device__ __forceinline__ float exp2_raw(float x) { return __builtin_amdgcn_exp2f(x); }

// The split-product kernel (attention_split.hip): D = 32, 64, 96 or 128,
// 16-byte aligned operands whose K/V rows of a sequence stay under 2 GiB, p
// filled but for the grid order.
int launch_attention_split(lancius_hip_ctx* ctx, AttnParams& p);

}  // namespace lancius
