// Per-head q / k RMSNorm + neox RoPE shared by the attention kernels (paged_attn.hip) and the code-predictor chain
// (cp_chain.hip): one arithmetic, the same bits in both.
#pragma once
#include "common.cuh"

#define LOG2E 1.4426950408889634f

// one wave, one 128-wide head; lane owns elements l and l + 64 (the RoPE pair): x0 / x1 = the raw bf16 values, w0 / w1 the norm weights, c / s the row
// of the cos / sin table
__device__ __forceinline__ void head_norm_rope_with(float x0, float x1, float w0, float w1, float c, float s, float eps, float& y0, float& y1) {
    const float ss = wave_sum(x0 * x0 + x1 * x1);
    const float rstd = 1.0f / sqrtf(ss * (1.0f / 128.0f) + eps);
    const float n0 = bfround(w0 * bfround(x0 * rstd));
    const float n1 = bfround(w1 * bfround(x1 * rstd));
    y0 = bfround(bfround(n0 * c) + bfround(-n1 * s));
    y1 = bfround(bfround(n1 * c) + bfround(n0 * s));
}
__device__ __forceinline__ void head_norm_rope_vals(float x0, float x1, const uint16_t* nw, const uint16_t* cs, float eps,
                                                    int lane, float& y0, float& y1) {
    head_norm_rope_with(x0, x1, bf2f(nw[lane]), bf2f(nw[lane + 64]), bf2f(cs[lane]), bf2f(cs[64 + lane]), eps, y0, y1);
}
__device__ __forceinline__ void head_norm_rope(const uint16_t* src, const uint16_t* nw, const uint16_t* cs, float eps,
                                               int lane, float& y0, float& y1) {
    head_norm_rope_vals(bf2f(src[lane]), bf2f(src[lane + 64]), nw, cs, eps, lane, y0, y1);
}
