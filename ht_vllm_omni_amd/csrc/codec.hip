// Code2Wav (12 Hz speech-tokenizer decoder) kernels that are not GEMM-shaped.  Every convolution / linear layer of the decoder
// runs on omni_gemm_tile (gemm_prefill.hip) over TIME-major activations [T, C]; this file holds the rest:
//   codec_rvq_embed    residual-VQ code lookup: sum over the quantizers of one row of a folded table (codebook / usage, times the
//                      1x1 output projection, folded at load) -> bf16 [T, C]
//   codec_rmsnorm      RMSNorm of the fp32 residual stream -> bf16 GEMM operand
//   codec_rope         rotate-half RoPE on the q / k heads of a fused qkv row, in place
//   codec_window_attn  causal sliding-window attention, one wave per (frame, head): <= window keys
//   codec_dwconv_ln    ConvNeXt front: depthwise causal conv (7 taps) + LayerNorm over channels, fp32 stream -> bf16
//   codec_out_conv     last layer: causal conv to ONE channel + clamp to [-1, 1], bf16 -> fp32 waveform
// All HBM-bound element / row work: coalesced 16-byte accesses along the channel dimension, reductions by DPP / permlane
// (common.cuh), no LDS except where rows are shared.
// Reference: tokenizer_12hz/modeling_qwen3_tts_tokenizer_v2.py (Qwen3TTSTokenizerV2Decoder.forward :1009-1027 and the modules
// it calls); oracle: oracle/code2wav_oracle.py.
#include "common.cuh"
#include "kernels.h"

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

// ---------------------------------------------------------------- residual VQ lookup
// out[t, :] = bf16( sum_q table[q][clamp(codes[q, t])][:] ), table fp32 [Q][bins][C]
// A frame is a chain of two trips to memory, the ids and then their rows: lane q of a wave fetches quantizer q's id (64 of them at a time) and eight rows
// are in flight at once (50 frames, 16 quantizers, 512 channels: 8.1 -> 3.3 us).
__global__ __launch_bounds__(256) void codec_rvq_embed_kernel(const int64_t* __restrict__ codes, int ld_codes, const float* __restrict__ table,
                                                              uint16_t* __restrict__ out, int T, int Q, int bins, int C) {
    const int t = blockIdx.x, lane = threadIdx.x & 63;
    for (int c0 = 0; c0 < C; c0 += blockDim.x * 4) {
        const int c = c0 + threadIdx.x * 4, cc = min(c, C - 4);
        f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
        for (int q0 = 0; q0 < Q; q0 += 64) {
            const int nq = min(64, Q - q0);
            long long id = codes[(size_t)(q0 + min(lane, nq - 1)) * ld_codes + t];
            const int bin = (int)(id < 0 ? 0 : (id >= bins ? bins - 1 : id));      // memory safety only: the caller validates the range
            for (int q = 0; q < nq; q += 8) {
                f32x4 r[8];
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    r[e] = *reinterpret_cast<const f32x4*>(table + ((size_t)(q0 + min(q + e, nq - 1)) * bins + __builtin_amdgcn_readlane(bin, min(q + e, nq - 1))) * C + cc);
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    if (q + e < nq) acc += r[e];
            }
        }
        if (c >= C) continue;
        uint2 pk;
        pk.x = pack_bf2(acc[0], acc[1]);
        pk.y = pack_bf2(acc[2], acc[3]);
        *reinterpret_cast<uint2*>(out + (size_t)t * C + c) = pk;
    }
}

extern "C" int omni_codec_rvq_embed(const int64_t* codes, int ld_codes, const float* table, void* out, int T, int Q, int bins, int C,
                                    void* stream) {
    OMNI_CHECK_ARG(codes && table && out && T > 0 && Q > 0 && bins > 0 && C > 0 && C % 4 == 0, "omni_codec_rvq_embed: T=%d Q=%d bins=%d C=%d", T, Q, bins, C);
    hipLaunchKernelGGL(codec_rvq_embed_kernel, dim3(T), dim3(C >= 1024 ? 256 : C > 256 ? 128 : 64), 0, (hipStream_t)stream, codes, ld_codes, table,
                       (uint16_t*)out, T, Q, bins, C);
    OMNI_CHECK_LAUNCH("omni_codec_rvq_embed");
    return OMNI_OK;
}

// ---------------------------------------------------------------- RMSNorm of the fp32 stream: one wave per row
// The row and the weights are asked for at once and stay in registers (PIECES of 256 columns; the row was walked twice, a wait per piece).  Measured in the
// decode of 50 frames, 17 of these launches over 50 rows of 1024: 1158 -> 1143 us.  Wider rows take the kernel that walks them.
// ADD: what the sublayer in front left joins the row first: partial sums of a product whose few tiles would each walk all of K alone (omni_gemm_tile k_splits).
// A row to a workgroup: four of them on one CU wait for its intake (with four partial sums a row is 28 KB).  Us, four rows / one of 1024, behind the kernel that wrote them, without partial
// sums, with one, with four: 50 rows 2.0 / 1.8, 3.6 / 2.0, 3.4 / 2.6; 325 2.5 / 2.0, 3.9 / 2.6, 5.8 / 4.1; 1024 3.9 / 2.6, 7.9 / 3.9, 11.5 / 3.5; 8192 12.2 / 8.5, 18.6 / 16.9.
struct CodecAdd { float* x; const float* y; const float* scale; int slabs; long long stride; };
template <int PIECES, bool ADD>
__global__ __launch_bounds__(64) void codec_rmsnorm_kernel(const float* x, int ldx, const float* __restrict__ w, float eps,
                                                           uint16_t* __restrict__ out, int H, const CodecAdd add) {
    const int lane = threadIdx.x, t = blockIdx.x;
    const float* xr = x + (size_t)t * ldx;
    f32x4 v[PIECES], g[PIECES];
#pragma unroll
    for (int i = 0; i < PIECES; ++i) v[i] = *reinterpret_cast<const f32x4*>(xr + min(lane * 4 + 256 * i, H - 4));
#pragma unroll
    for (int i = 0; i < PIECES; ++i) g[i] = *reinterpret_cast<const f32x4*>(w + min(lane * 4 + 256 * i, H - 4));
    if constexpr (ADD) {
        constexpr int S = 4;                               // all partial sums leave at once (past the last: that one again, not added)
        f32x4 y[PIECES][S], sc[PIECES];
#pragma unroll
        for (int i = 0; i < PIECES; ++i)
#pragma unroll
            for (int s = 0; s < S; ++s) y[i][s] = *reinterpret_cast<const f32x4*>(add.y + min(s, add.slabs - 1) * add.stride + (size_t)t * H + min(lane * 4 + 256 * i, H - 4));
#pragma unroll
        for (int i = 0; i < PIECES; ++i) sc[i] = *reinterpret_cast<const f32x4*>(add.scale + min(lane * 4 + 256 * i, H - 4));
#pragma unroll
        for (int i = 0; i < PIECES; ++i) {
#pragma unroll
            for (int s = 1; s < S; ++s)
#pragma unroll
                for (int e = 0; e < 4; ++e) y[i][0][e] += s < add.slabs ? y[i][s][e] : 0.f;
#pragma unroll
            for (int e = 0; e < 4; ++e) v[i][e] = fmaf(y[i][0][e], sc[i][e], v[i][e]);
            if (lane * 4 + 256 * i < H) *reinterpret_cast<f32x4*>(add.x + (size_t)t * ldx + lane * 4 + 256 * i) = v[i];
        }
    }
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < PIECES; ++i)
        if (lane * 4 + 256 * i < H) ss += v[i][0] * v[i][0] + v[i][1] * v[i][1] + v[i][2] * v[i][2] + v[i][3] * v[i][3];
    const float rstd = rsqrtf(wave_sum(ss) / (float)H + eps);
#pragma unroll
    for (int i = 0; i < PIECES; ++i) {
        const int c = lane * 4 + 256 * i;
        if (c >= H) continue;
        uint2 pk;
        pk.x = pack_bf2(g[i][0] * (v[i][0] * rstd), g[i][1] * (v[i][1] * rstd));
        pk.y = pack_bf2(g[i][2] * (v[i][2] * rstd), g[i][3] * (v[i][3] * rstd));
        *reinterpret_cast<uint2*>(out + (size_t)t * H + c) = pk;
    }
}

__global__ __launch_bounds__(256) void codec_rmsnorm_wide_kernel(const float* __restrict__ x, int ldx, const float* __restrict__ w, float eps,
                                                            uint16_t* __restrict__ out, int T, int H) {
    const int lane = threadIdx.x & 63;
    const int t = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (t >= T) return;
    const float* xr = x + (size_t)t * ldx;
    float ss = 0.f;
    for (int c = lane * 4; c < H; c += 256) {
        const f32x4 v = *reinterpret_cast<const f32x4*>(xr + c);
        ss += v[0] * v[0] + v[1] * v[1] + v[2] * v[2] + v[3] * v[3];
    }
    const float rstd = rsqrtf(wave_sum(ss) / (float)H + eps);
    for (int c = lane * 4; c < H; c += 256) {
        const f32x4 v = *reinterpret_cast<const f32x4*>(xr + c);
        const f32x4 g = *reinterpret_cast<const f32x4*>(w + c);
        uint2 pk;
        pk.x = pack_bf2(g[0] * (v[0] * rstd), g[1] * (v[1] * rstd));
        pk.y = pack_bf2(g[2] * (v[2] * rstd), g[3] * (v[3] * rstd));
        *reinterpret_cast<uint2*>(out + (size_t)t * H + c) = pk;
    }
}

extern "C" int omni_codec_rmsnorm(const float* x, int ldx, const float* w, float eps, void* out, int T, int H, void* stream) {
    OMNI_CHECK_ARG(x && w && out && T > 0 && H > 0 && H % 4 == 0 && ldx >= H && ldx % 4 == 0, "omni_codec_rmsnorm: T=%d H=%d ldx=%d", T, H, ldx);
    const dim3 grid(T), block(64);
    if (H <= 512) hipLaunchKernelGGL((codec_rmsnorm_kernel<2, false>), grid, block, 0, (hipStream_t)stream, x, ldx, w, eps, (uint16_t*)out, H, CodecAdd{});
    else if (H <= 1024) hipLaunchKernelGGL((codec_rmsnorm_kernel<4, false>), grid, block, 0, (hipStream_t)stream, x, ldx, w, eps, (uint16_t*)out, H, CodecAdd{});
    else hipLaunchKernelGGL(codec_rmsnorm_wide_kernel, dim3((T + 3) / 4), dim3(256), 0, (hipStream_t)stream, x, ldx, w, eps, (uint16_t*)out, T, H);
    OMNI_CHECK_LAUNCH("omni_codec_rmsnorm");
    return OMNI_OK;
}

extern "C" int omni_codec_add_rmsnorm(float* x, int ldx, const float* y, int slabs, int64_t slab_stride, const float* scale, const float* w, float eps, void* out, int T, int H, void* stream) {
    OMNI_CHECK_ARG(x && y && scale && w && out && T > 0 && H > 0 && H % 4 == 0 && H <= 1024 && ldx >= H && ldx % 4 == 0 && slabs >= 1 && slabs <= 4 &&
                   (slabs == 1 || slab_stride >= (int64_t)T * H) && slab_stride % 4 == 0, "omni_codec_add_rmsnorm: T=%d H=%d (<= 1024) ldx=%d slabs=%d (<= 4)", T, H, ldx, slabs);
    const dim3 grid(T), block(64);
    const CodecAdd add{x, y, scale, slabs, slab_stride};
    if (H <= 512) hipLaunchKernelGGL((codec_rmsnorm_kernel<2, true>), grid, block, 0, (hipStream_t)stream, x, ldx, w, eps, (uint16_t*)out, H, add);
    else hipLaunchKernelGGL((codec_rmsnorm_kernel<4, true>), grid, block, 0, (hipStream_t)stream, x, ldx, w, eps, (uint16_t*)out, H, add);
    OMNI_CHECK_LAUNCH("omni_codec_add_rmsnorm");
    return OMNI_OK;
}

// ---------------------------------------------------------------- RoPE (rotate-half) on the q and k heads of qkv rows, in place
// position = row index; angle(d) = t * theta^(-2 d / hd), d < hd / 2; (x1, x2) = (x[d], x[d + hd/2]) -> (x1 cos - x2 sin, x2 cos + x1 sin)
__global__ __launch_bounds__(256) void codec_rope_kernel(uint16_t* __restrict__ qkv, int ld, int T, int heads /* q + k heads */, int hd,
                                                         float log2_theta) {
    const int half = hd >> 1;
    const int per_row = heads * half;
    const long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (long long)T * per_row) return;
    const int t = (int)(idx / per_row), r = (int)(idx - (long long)t * per_row);
    const int h = r / half, d = r - h * half;
    const float inv = exp2f(-log2_theta * (float)(2 * d) / (float)hd);
    float sn, cs;
    sincosf((float)t * inv, &sn, &cs);
    uint16_t* p = qkv + (size_t)t * ld + h * hd + d;
    const float x1 = bf2f(p[0]), x2 = bf2f(p[half]);
    p[0] = f2bf(x1 * cs - x2 * sn);
    p[half] = f2bf(x2 * cs + x1 * sn);
}

extern "C" int omni_codec_rope(void* qkv, int ld, int T, int q_heads, int kv_heads, int head_dim, float theta, void* stream) {
    OMNI_CHECK_ARG(qkv && T > 0 && q_heads > 0 && kv_heads > 0 && head_dim % 2 == 0 && theta > 0.f, "omni_codec_rope: bad shape");
    const long long n = (long long)T * (q_heads + kv_heads) * (head_dim / 2);
    hipLaunchKernelGGL(codec_rope_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream, (uint16_t*)qkv, ld, T,
                       q_heads + kv_heads, head_dim, log2f(theta));
    OMNI_CHECK_LAUNCH("omni_codec_rope");
    return OMNI_OK;
}

// ---------------------------------------------------------------- causal sliding-window attention, one wave per (frame, head)
// qkv row = [q heads | k heads | v heads] x hd, already rotated.  Keys j in [max(0, t - window + 1), t], 64 per chunk: lane = key
// for the scores (q broadcast by v_readlane), online softmax across chunks; P.V: lane = (key & 7, 8 columns), folded over the keys at the end.
// Few keys and many waves: what bounds a wave is its trips to memory.  A chunk's keys and values are all asked for before the first is used, in 16-byte
// pieces (50 frames, 16 heads of 64: one value row after the other 15.2 us, so 4.4; 325 frames 18.0 -> 14.7).  VPL = hd / 64.
template <int VPL>
__global__ __launch_bounds__(64) void codec_window_attn_kernel(const uint16_t* __restrict__ qkv, int ld, uint16_t* __restrict__ out, int ldo,
                                                               int nh, int nkv, int window, float scale) {
    constexpr int HD = 64 * VPL;
    const int t = blockIdx.x, h = blockIdx.y, lane = threadIdx.x;
    const int key = lane >> 3, col = (lane & 7) * 8;
    const int kvh = h / (nh / nkv);
    const uint16_t* qp = qkv + (size_t)t * ld + h * HD;
    const size_t koff = (size_t)(nh + kvh) * HD, voff = (size_t)(nh + nkv + kvh) * HD;
    int qv[VPL];                                          // q[lane + 64 v] * scale as raw bits (v_readlane works on b32)
#pragma unroll
    for (int v = 0; v < VPL; ++v) qv[v] = __float_as_int(bf2f(qp[lane + 64 * v]) * scale);
    const int j0 = max(0, t - window + 1);
    float m = -INFINITY, l = 0.f, acc[VPL][8];
#pragma unroll
    for (int v = 0; v < VPL; ++v)
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[v][e] = 0.f;
    for (int jb = j0; jb <= t; jb += 64) {
        const int cnt = min(64, t - jb + 1);
        u32x4 K[VPL][8], V[VPL][8];
#pragma unroll
        for (int v = 0; v < VPL; ++v)
#pragma unroll
            for (int i = 0; i < 8; ++i) K[v][i] = *reinterpret_cast<const u32x4*>(qkv + (size_t)min(jb + lane, t) * ld + koff + 64 * v + i * 8);     // lanes past the window: key t, masked below
#pragma unroll
        for (int v = 0; v < VPL; ++v)
#pragma unroll
            for (int i = 0; i < 8; ++i) V[v][i] = *reinterpret_cast<const u32x4*>(qkv + (size_t)min(jb + 8 * i + key, t) * ld + voff + 64 * v + col);
        float dot = 0.f;
#pragma unroll
        for (int v = 0; v < VPL; ++v)
#pragma unroll
            for (int d8 = 0; d8 < 8; ++d8)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float q0 = __int_as_float(__builtin_amdgcn_readlane(qv[v], d8 * 8 + 2 * e));
                    const float q1 = __int_as_float(__builtin_amdgcn_readlane(qv[v], d8 * 8 + 2 * e + 1));
                    dot += q0 * bf_lo(K[v][d8][e]) + q1 * bf_hi(K[v][d8][e]);
                }
        const float s = lane < cnt ? dot : -INFINITY;
        const float m_new = fmaxf(m, wave_max(s));
        const float corr = __expf(m - m_new);             // first chunk: exp(-inf) = 0
        const float p = lane < cnt ? __expf(s - m_new) : 0.f;
        l = l * corr + wave_sum(p);
        m = m_new;
#pragma unroll
        for (int v = 0; v < VPL; ++v)
#pragma unroll
            for (int e = 0; e < 8; ++e) acc[v][e] *= corr;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float pj = __shfl(p, 8 * i + key);      // zero past the window
#pragma unroll
            for (int v = 0; v < VPL; ++v)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    acc[v][2 * e] += pj * bf_lo(V[v][i][e]);
                    acc[v][2 * e + 1] += pj * bf_hi(V[v][i][e]);
                }
        }
    }
    const float inv = 1.0f / l;
#pragma unroll
    for (int v = 0; v < VPL; ++v) {
#pragma unroll
        for (int e = 0; e < 8; ++e)
#pragma unroll
            for (int o = 8; o < 64; o *= 2) acc[v][e] += __shfl_xor(acc[v][e], o);
        if (key == 0) {
            uint16_t* d = out + (size_t)t * ldo + h * HD + 64 * v + col;
            u32x4 o;
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = pack_bf2(acc[v][2 * e] * inv, acc[v][2 * e + 1] * inv);
            if (((size_t)d & 15) == 0) {
                *reinterpret_cast<u32x4*>(d) = o;
            } else {                                       // rows of any pitch and address
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    d[2 * e] = (uint16_t)o[e];
                    d[2 * e + 1] = (uint16_t)(o[e] >> 16);
                }
            }
        }
    }
}

extern "C" int omni_codec_window_attn(const void* qkv, int ld, void* out, int ldo, int T, int q_heads, int kv_heads, int head_dim,
                                      int window, float scale, void* stream) {
    OMNI_CHECK_ARG(qkv && out && T > 0 && q_heads > 0 && kv_heads > 0 && q_heads % kv_heads == 0 && window > 0, "omni_codec_window_attn: bad shape");
    OMNI_CHECK_ARG(head_dim == 64 || head_dim == 128, "omni_codec_window_attn: head_dim=%d (64 | 128)", head_dim);
    OMNI_CHECK_ARG(ld % 8 == 0 && ld >= (q_heads + 2 * kv_heads) * head_dim, "omni_codec_window_attn: ld=%d", ld);
    const dim3 grid(T, q_heads);
    if (head_dim == 64)
        hipLaunchKernelGGL(codec_window_attn_kernel<1>, grid, dim3(64), 0, (hipStream_t)stream, (const uint16_t*)qkv, ld, (uint16_t*)out, ldo,
                           q_heads, kv_heads, window, scale);
    else
        hipLaunchKernelGGL(codec_window_attn_kernel<2>, grid, dim3(64), 0, (hipStream_t)stream, (const uint16_t*)qkv, ld, (uint16_t*)out, ldo,
                           q_heads, kv_heads, window, scale);
    OMNI_CHECK_LAUNCH("omni_codec_window_attn");
    return OMNI_OK;
}

// ---------------------------------------------------------------- ConvNeXt front: depthwise causal conv + LayerNorm over channels
// y[t, c] = b[c] + sum_j w[c][j] x[t - (taps - 1) + j][c] (rows < 0 are zero);  out = bf16(LN(y) * g + beta).  One workgroup per frame.
// Seven taps: the channels of seven rows, their weights, gains and offsets are asked for at once (a channel and a tap after the other, a wait each: 11.8 us
// for 100 frames of 1024, so 3.9); the same sums.  TAPS 0: any number.
template <int TAPS>
__global__ __launch_bounds__(256) void codec_dwconv_ln_kernel(const float* __restrict__ x, int ldx, const float* __restrict__ w,
                                                              const float* __restrict__ b, const float* __restrict__ ln_w,
                                                              const float* __restrict__ ln_b, float eps, uint16_t* __restrict__ out,
                                                              int T, int C, int taps) {
    __shared__ float red[2][4];
    const int t = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    float y[4], g[4], o[4];                               // C <= 1024: channel tid + 256 i
    float sum = 0.f;
    if constexpr (TAPS > 0) {
        float xv[4][TAPS], wq[4][TAPS];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int c = min(tid + 256 * i, C - 1);
#pragma unroll
            for (int j = 0; j < TAPS; ++j) {
                xv[i][j] = x[(size_t)max(t - (TAPS - 1) + j, 0) * ldx + c];
                wq[i][j] = w[c * TAPS + j];
            }
            y[i] = b[c]; g[i] = ln_w[c]; o[i] = ln_b[c];
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
#pragma unroll
            for (int j = 0; j < TAPS; ++j)
                if (t - (TAPS - 1) + j >= 0) y[i] += wq[i][j] * xv[i][j];
            if (tid + 256 * i >= C) y[i] = 0.f;
            else sum += y[i];
        }
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int c = tid + 256 * i;
            y[i] = g[i] = o[i] = 0.f;
            if (c < C) {
                float a = b[c];
                for (int j = 0; j < taps; ++j) {
                    const int r = t - (taps - 1) + j;
                    if (r >= 0) a += w[c * taps + j] * x[(size_t)r * ldx + c];
                }
                y[i] = a; g[i] = ln_w[c]; o[i] = ln_b[c];
                sum += a;
            }
        }
    }
    sum = wave_sum(sum);
    if (lane == 0) red[0][wv] = sum;
    __syncthreads();
    const float mean = (red[0][0] + red[0][1] + red[0][2] + red[0][3]) / (float)C;
    float var = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i)
        if (tid + 256 * i < C) var += (y[i] - mean) * (y[i] - mean);
    var = wave_sum(var);
    if (lane == 0) red[1][wv] = var;
    __syncthreads();
    const float rstd = rsqrtf((red[1][0] + red[1][1] + red[1][2] + red[1][3]) / (float)C + eps);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int c = tid + 256 * i;
        if (c < C) out[(size_t)t * C + c] = f2bf((y[i] - mean) * rstd * g[i] + o[i]);
    }
}

extern "C" int omni_codec_dwconv_ln(const float* x, int ldx, const float* w, const float* b, const float* ln_w, const float* ln_b, float eps,
                                    void* out, int T, int C, int taps, void* stream) {
    OMNI_CHECK_ARG(x && w && b && ln_w && ln_b && out && T > 0 && C > 0 && C <= 1024 && taps > 0 && ldx >= C, "omni_codec_dwconv_ln: T=%d C=%d (<= 1024)", T, C);
    if (taps == 7) hipLaunchKernelGGL(codec_dwconv_ln_kernel<7>, dim3(T), dim3(256), 0, (hipStream_t)stream, x, ldx, w, b, ln_w, ln_b, eps, (uint16_t*)out, T, C, taps);
    else hipLaunchKernelGGL(codec_dwconv_ln_kernel<0>, dim3(T), dim3(256), 0, (hipStream_t)stream, x, ldx, w, b, ln_w, ln_b, eps, (uint16_t*)out, T, C, taps);
    OMNI_CHECK_LAUNCH("omni_codec_dwconv_ln");
    return OMNI_OK;
}

// ---------------------------------------------------------------- last layer: causal conv to one channel + clamp
// wav[t] = clamp(b + sum_{j, c} w[j][c] x[t - (taps - 1) + j][c], -1, 1); x bf16 [T, C] (already through the last snake), w fp32 [taps][C].
// A lane's sample needs `taps` whole rows, and neighbouring lanes' rows are neighbours: lanes that fetch a row each take 16 bytes out of as many lines as there
// are lanes, `taps` times over.  So a block's rows go to LDS once, in whole lines (pitch of an odd number of 16-byte pieces: 16 rows lie in 16 different
// bank groups), all pieces of a thread asked for at once, and the weights, the same for every lane, behind them.  A sample is one chain of sums, taps outer, channels
// inner, whatever the width.  Us, out of cold caches with the events around it, weights by scalar loads 32 at a time and rows a piece after the other / this: 23040 samples of 96
// channels, 7 taps, 23.3 / 11.7, 96000 23.7 / 14.0, 624000 71 / 55.  Every row times every tap on the matrix cores takes 7.5, 9.5 and 25, but adds up in another order: not kept.
#define OC_ROWS 256
// xr: 16-byte pieces; wr: in LDS, 16-byte aligned
__device__ __forceinline__ float oc_piece(u32x4 v, const float* wr, float acc) {
    const f32x4 a = *reinterpret_cast<const f32x4*>(wr), b = *reinterpret_cast<const f32x4*>(wr + 4);
    acc += bf_lo(v[0]) * a[0] + bf_hi(v[0]) * a[1];
    acc += bf_lo(v[1]) * a[2] + bf_hi(v[1]) * a[3];
    acc += bf_lo(v[2]) * b[0] + bf_hi(v[2]) * b[1];
    acc += bf_lo(v[3]) * b[2] + bf_hi(v[3]) * b[3];
    return acc;
}
__device__ __forceinline__ float oc_row(const uint16_t* xr, const float* wr, int C, float acc) {
    int c = 0;
    for (; c + 32 <= C; c += 32) {                        // (four pieces of the row and of the weights per wait)
        u32x4 v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = *reinterpret_cast<const u32x4*>(xr + c + 8 * i);
#pragma unroll
        for (int i = 0; i < 4; ++i) acc = oc_piece(v[i], wr + c + 8 * i, acc);
    }
    for (; c < C; c += 8) acc = oc_piece(*reinterpret_cast<const u32x4*>(xr + c), wr + c, acc);
    return acc;
}
static inline __host__ __device__ int oc_pitch(int C) { return 16 * ((C / 8) | 1); }

__global__ __launch_bounds__(OC_ROWS) void codec_out_conv_kernel(const uint16_t* __restrict__ x, const float* __restrict__ w, float bias,
                                                                 float* __restrict__ wav, int T, int C, int taps) {
    extern __shared__ __attribute__((aligned(16))) uint8_t rows[];
    const int t0 = blockIdx.x * OC_ROWS, r0 = t0 - (taps - 1), ch = C / 8, pitch = oc_pitch(C), total = (min(OC_ROWS, T - t0) + taps - 1) * ch;
    float* wl = reinterpret_cast<float*>(rows + (OC_ROWS + taps - 1) * pitch);
    constexpr int P = 16;                                 // pieces of a thread in flight: 7 taps of 96 channels are 13
    for (int first = 0; first < total; first += P * OC_ROWS) {
        const int base = first + threadIdx.x;
        u32x4 v[P];
#pragma unroll
        for (int i = 0; i < P; ++i) {                     // (rows in front of the first: its first piece, not used; past the last: that one again)
            const int64_t at = (int64_t)r0 * ch + min(base + i * OC_ROWS, total - 1);
            v[i] = *reinterpret_cast<const u32x4*>(x + (at < 0 ? 0 : at) * 8);
        }
        if (first == 0)
            for (int i = threadIdx.x; i < taps * C; i += OC_ROWS) wl[i] = w[i];
#pragma unroll
        for (int i = 0; i < P; ++i) {
            const int id = base + i * OC_ROWS, lr = id / ch;
            if (id < total) *reinterpret_cast<u32x4*>(rows + lr * pitch + (id - lr * ch) * 16) = v[i];
        }
    }
    __syncthreads();
    const int t = t0 + threadIdx.x;
    if (t >= T) return;
    float acc = bias;
    for (int j = 0; j < taps; ++j)
        if (t - (taps - 1) + j >= 0) acc = oc_row(reinterpret_cast<const uint16_t*>(rows + (threadIdx.x + j) * pitch), wl + j * C, C, acc);
    wav[t] = fminf(fmaxf(acc, -1.0f), 1.0f);
}

// rows too wide for LDS: straight from memory, the weights in LDS
__global__ __launch_bounds__(256) void codec_out_conv_wide_kernel(const uint16_t* __restrict__ x, const float* __restrict__ w, float bias,
                                                                  float* __restrict__ wav, int T, int C, int taps) {
    extern __shared__ __attribute__((aligned(16))) float wl[];                         // [taps * C]
    for (int i = threadIdx.x; i < taps * C; i += blockDim.x) wl[i] = w[i];
    __syncthreads();
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= T) return;
    float acc = bias;
    for (int j = 0; j < taps; ++j)
        if (t - (taps - 1) + j >= 0) acc = oc_row(x + (size_t)(t - (taps - 1) + j) * C, wl + j * C, C, acc);
    wav[t] = fminf(fmaxf(acc, -1.0f), 1.0f);
}

extern "C" int omni_codec_out_conv(const void* x, const float* w, float bias, float* wav, int T, int C, int taps, void* stream) {
    OMNI_CHECK_ARG(x && w && wav && T > 0 && C > 0 && C % 8 == 0 && taps > 0 && taps * C * 4 <= 64 * 1024, "omni_codec_out_conv: T=%d C=%d taps=%d", T, C, taps);
    const int rows = (OC_ROWS + taps - 1) * oc_pitch(C), weights = taps * C * (int)sizeof(float);
    if (rows <= 64 * 1024) {
        if (rows + weights > 64 * 1024) {
            static const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(codec_out_conv_kernel), hipFuncAttributeMaxDynamicSharedMemorySize, 128 * 1024);
            if (e != hipSuccess) { omni_set_error("omni_codec_out_conv: LDS attribute: %s", hipGetErrorString(e)); return OMNI_EHIP; }
        }
        hipLaunchKernelGGL(codec_out_conv_kernel, dim3((T + OC_ROWS - 1) / OC_ROWS), dim3(OC_ROWS), (size_t)(rows + weights), (hipStream_t)stream,
                           (const uint16_t*)x, w, bias, wav, T, C, taps);
    } else
        hipLaunchKernelGGL(codec_out_conv_wide_kernel, dim3((T + 255) / 256), dim3(256), taps * C * sizeof(float), (hipStream_t)stream,
                           (const uint16_t*)x, w, bias, wav, T, C, taps);
    OMNI_CHECK_LAUNCH("omni_codec_out_conv");
    return OMNI_OK;
}
