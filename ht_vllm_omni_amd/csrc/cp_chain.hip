// The code predictor's layer stack as ONE persistent launch (reference: the 5-layer decoder that
// qwen3_tts_code_predictor_vllm.py:480-561 re-runs for each of the 15 residual code groups of a talker step).
//
// Launch-per-op, a predictor pass is 25 dependent launches (5 layers x { qkv, attention, o_proj, gate_up, down_proj }) of
// ~5.5 us each although a workgroup's share of a GEMM is 16-48 KB of weights and a few MFMAs: a dependent launch pays the
// kernel boundary (1.65 us), a cold weight fetch, a cold activation fetch and a store drain, one after the other.
// Here the stages run inside one grid of 256 co-resident workgroups (one per CU):
//   * a stage's WEIGHT slice does not depend on its predecessor: every wave loads its whole slice before it looks for its operands;
//   * cp_chain_kernel (passes 2 .. 15, their heads and samplers) hands activations over by content: an operand is there when none of its words
//     is EMPTY (chain_flow.cuh).  No drain, no flag, no barrier between a stage's last store and its successor's first MFMA.  What bounds it is
//     that chain of dependent trips: 27 stages a pass of about 2.6 us at 5 rows (69 us a pass) and 3.3 at 64 (89), of which 0.6 to 1.6 us are a stage's own
//     arithmetic, LDS combine and epilogue and the rest the operands' way (profiles/talker_step_timeline.txt).  Behind flags (coherent.cuh) a pass took
//     104 / 110 us;
//   * cp_pair_kernel (positions 0 and 1, group 1) likewise, over both positions' rows; a decode step of 64 / of 5 rows, us, behind flags 2886 / 1859, by
//     content 2860 / 1784 (the stages of up to 16 rows over all 256 workgroups: 64 of them owned every column of qkv);
//   * what a stage may read without waiting (besides weights): bytes that were final two or more stages earlier -- the K / V history of the
//     private cache, the old residual values of a residual epilogue.
// K-step ownership of the 8 waves, accumulation order, LDS combine order and every rounding point are those of
// gemm_skinny_kernel / attn_tiny_dense_kernel: the chain is bit-identical to the launch-per-op path (tests/test_gpu_chain.py).
// Bounded spins: a grid that is not co-resident times out into an error word (never a hang).
#include "attn_common.cuh"
#include "coherent.cuh"
#include "common.cuh"
#include "gemm_frag.cuh"
#include "chain_gemm.cuh"
#include "chain_flow.cuh"
#include "kernels.h"
#include "sampler_body.cuh"

#define CH_MAX_LAYERS 8
#define CH_LDS_FLOATS ((CH_WAVES * 6 * 4 * 64) + CH_WAVES * 64)      // combine slots of the widest stage (NT * MT = 6) + rstd area

struct ChainLayer {
    const uint16_t *ln1, *wqkv, *qnorm, *knorm, *wo, *ln2, *wgu, *wdown;
    uint16_t *kc, *vc;                    // this layer's private K / V cache [B][bs][kv_heads][128] bf16
};
struct ChainArgs {
    ChainLayer layer[CH_MAX_LAYERS];
    int layers, B, bs, np_in;
    int g0, g1;                           // passes = buffer positions g0 .. g1 - 1 (1 <= g0, g1 <= 16); with_head: each pass ends in
    int with_head;                        // the group's head GEMM + sampler (+ gather of the next pass's input row)
    int q_heads, kv_heads;
    float eps, sm_scale;
    uint16_t* resid;                      // fragment-major residual stream [64][Hc]
    float* part;                          // sum(r^2) slabs [np][64]
    const uint16_t* cos_sin;
    // head + sampler of pass g (group g): logits row b at logits + b * logits_ld + (g - 1) * logits_pass
    const uint16_t *cp_norm, *lm_head;    // lm_head: [Q - 1][codebook][Hc] fragment-major per group
    float* logits; int logits_ld, logits_pass;
    int greedy, top_k, Q, codebook; float temperature, top_p; uint32_t seed;
    const int32_t* steps; const uint32_t* row_seed;
    int32_t* codes;                       // [B][Q]
    const uint16_t* ptab;                 // folded projection tables [Q - 1][codebook][Hc]: pass g < Q - 1 gathers row `code` of table g - 1
    uint32_t* flags;
    int32_t* err;
    // tail of the all-pass launch: input assembly of the backbone by the last sampler stage's row owners, then layer 0's qkv
    struct Tail {
        const int32_t* input_ids; const uint16_t* embed; int vocab; const uint16_t* cp_embed; const uint16_t* text_step;
        uint16_t* x_out; uint16_t* resid; float* part; int64_t* audio_codes; int H;
        const uint16_t* wqkv; const uint16_t* ln1; uint16_t* qkv; int NQ;
        int enabled;
    } tail;
    char* flow;                           // hand-off buffers: FLOW_COPIES copies of CP_COPY (all-pass launch) or PP_COPY bytes (pair launch)
    int Bp;                               // pair kernel: rows of position 1 start at Bp (B rounded up to 16) in the 128-row stream
    unsigned long long* stamps;           // debug library only: [stage][CH_NSTAMP][256] s_memrealtime ticks (100 MHz) of wave 0, or NULL
};

// ---- the backbone's input row of batch row b (mtp_finalize_kernel, capi.hip: x[t+1] = bf16(bf16(sum_fp32(e0, emb_1 .. emb_{Q-1})) + text_step), an
// invalid layer-0 id -> a frame of zeros; qwen3_tts_talker.py:1630-1641) by the workgroup that just drew the row's last code: the same 256 threads,
// the same order of additions, the same slab value.  Row-major copy (inputs_embeds: the step's output) by plain stores, the residual stream and its
// slab by write-through stores (the qkv stage behind the flags reads them)
// (a real call, not inlined: compiled into the sampler stage its code changed the register allocation of the whole pass loop -- the all-pass
//  launch ran 4.5 us per pass slower with the tail inlined, profiles/r06 NOTEBOOK)
struct ChainFinArgs { ChainArgs::Tail T; const int32_t* codes; int Q, codebook; };
__device__ __attribute__((noinline)) void chain_finalize_row(const ChainFinArgs fa, int b, int last_code, float* lds) {
    const ChainArgs::Tail& T = fa.T;
    struct { const int32_t* codes; int Q, codebook; } a{fa.codes, fa.Q, fa.codebook};
    const int Q = a.Q, H = T.H, tid = threadIdx.x;
    int* cg = reinterpret_cast<int*>(lds + CH_LDS_FLOATS - 128);          // [64] codes of the row | [4] wave sums (past the sampler's carve)
    float* red = lds + CH_LDS_FLOATS - 64;
    const int c0 = T.input_ids[b];
    const bool invalid0 = c0 < 0 || c0 >= a.codebook;
    if (tid < Q) {
        int c = tid == 0 ? c0 : (tid == Q - 1 ? last_code : (int)coh_ld4(coh_rsrc(a.codes), ((uint32_t)b * Q + tid) * 4));
        if (invalid0) c = 0;
        cg[tid] = c;
        T.audio_codes[(size_t)b * Q + tid] = (int64_t)c;
    }
    __syncthreads();
    float ss = 0.f;
    if (tid < 256) {
        const coh_rsrc_t rrs = coh_rsrc(T.resid);
        for (int v = tid; v < H / 8; v += 256) {
            float s[8];
            {
                const bool ok = c0 >= 0 && c0 < T.vocab;
                const u32x4 e = ok ? ld16(T.embed + (size_t)c0 * H + v * 8) : (u32x4){0u, 0u, 0u, 0u};
#pragma unroll
                for (int j = 0; j < 4; ++j) { s[2 * j] = bf_lo(e[j]); s[2 * j + 1] = bf_hi(e[j]); }
            }
#pragma unroll 4
            for (int g = 1; g < Q; ++g) {
                const u32x4 e = ld16(T.cp_embed + ((size_t)(g - 1) * a.codebook + cg[g]) * H + v * 8);
#pragma unroll
                for (int j = 0; j < 4; ++j) { s[2 * j] += bf_lo(e[j]); s[2 * j + 1] += bf_hi(e[j]); }
            }
            const u32x4 tx = ld16(T.text_step + (size_t)b * H + v * 8);
            u32x4 o;
#pragma unroll
            for (int j = 0; j < 4; ++j) o[j] = pack_bf2(bfround(s[2 * j]) + bf_lo(tx[j]), bfround(s[2 * j + 1]) + bf_hi(tx[j]));
            *reinterpret_cast<u32x4*>(T.x_out + (size_t)b * H + v * 8) = o;
#pragma unroll
            for (int j = 0; j < 4; ++j) ss += bf_lo(o[j]) * bf_lo(o[j]) + bf_hi(o[j]) * bf_hi(o[j]);
            coh_st16(rrs, (uint32_t)frag_off(b, v * 8, H) * 2, o);
        }
        ss = wave_sum(ss);
        if ((tid & 63) == 0) red[tid >> 6] = ss;
    }
    __syncthreads();
    if (tid == 0) coh_st4(coh_rsrc(T.part), (uint32_t)b * 4, __float_as_uint(red[0] + red[1] + red[2] + red[3]));
}

// ---- the all-pass launch: passes 2 .. 15 of every row, hand-offs by content (chain_flow.cuh)
// hand-off buffers of one copy, bytes from its base (64 rows)
enum : uint32_t {
    CP_QKV = 0,                           // 4096 columns, 16 x 16 tiles
    CP_ATT = CP_QKV + 64 * 4096 * 2,      // fragment-major, 2048 columns
    CP_RA = CP_ATT + 64 * 2048 * 2,       // residual stream behind o_proj, fragment-major, + its slabs
    CP_PA = CP_RA + 64 * 1024 * 2,
    CP_ACT = CP_PA + 64 * 64 * 4,         // fragment-major, 3072 columns
    CP_RB = CP_ACT + 64 * 3072 * 2,       // residual stream behind down_proj + its slabs
    CP_PB = CP_RB + 64 * 1024 * 2,
    CP_R0 = CP_PB + 64 * 64 * 4,          // a pass's input rows (the sampler's gather) + their one slab
    CP_P0 = CP_R0 + 64 * 1024 * 2,
    CP_LOG = CP_P0 + 1024,                // 2048 logits a row, 16 x 16 tiles
    CP_COPY = CP_LOG + 64 * 2048 * 4
};
#define CP_FLOW_BYTES ((size_t)FLOW_COPIES * CP_COPY)
// ... and of one copy of the pair launch: the same for 128 rows; its logits, written once, lie behind the copies
enum : uint32_t {
    PP_QKV = 0,
    PP_ATT = PP_QKV + 128 * 4096 * 2,
    PP_RA = PP_ATT + 128 * 2048 * 2,
    PP_PA = PP_RA + 128 * 1024 * 2,
    PP_ACT = PP_PA + 64 * 128 * 4,
    PP_RB = PP_ACT + 128 * 3072 * 2,
    PP_PB = PP_RB + 128 * 1024 * 2,
    PP_COPY = PP_PB + 64 * 128 * 4
};
#define PP_FLOW_BYTES ((size_t)FLOW_COPIES * PP_COPY + 64 * 2048 * 4)
size_t k_cp_flow_bytes() { return CP_FLOW_BYTES > PP_FLOW_BYTES ? CP_FLOW_BYTES : PP_FLOW_BYTES; }       // (the two launches run one behind the other)

// LDS of the launch: two combine halves, a KB per wave for the attention, the sampler's working set, one word
#define CPF_ATTN_FLOATS (2 * FLOW_HALF_FLOATS)
#define CPF_SMP_FLOATS (CPF_ATTN_FLOATS + CH_WAVES * 256)
#define CPF_LAST ((SMP_LDS_BYTES(8) + 15) / 16 * 4)                  // the drawn code's word, floats behind the sampler's working set
#define CPF_LDS_BYTES ((CPF_SMP_FLOATS + CPF_LAST + 4) * 4)

// attention at buffer position pos <= 15 (dense private cache: row b owns block b): one wave per (row, q head), the work layout of
// attn_tiny_dense_kernel (paged_attn.hip).  A kv head's q heads are waves of ONE workgroup, in every pass the same one: the K / V rows that the
// first of them writes are read, passes later, behind that workgroup's own barriers.
// a wave's history rows: lane = (token lane / 4, quarter lane % 4) of K, a dword of every token of V; and what the norm and the rotation multiply by (asked for
// behind the wait, the trip stood between q and the scores: a decode step of 64 rows 2817 -> 2787 us, of 5 rows 1739 -> 1720).
// Rows from pos on hold what an earlier step left there, possibly NaN or infinity, which a weight of 0 does not mask: V's descriptor ends at row pos,
// past which a load returns 0 (K's scores are replaced)
struct FlowHist { u32x4 k[4]; uint32_t v[16]; uint16_t qn[2], kn[2], cs[2]; };
__device__ __forceinline__ void flow_history(const ChainArgs& a, const ChainLayer& L, int pos, int pair, FlowHist& hist) {
    int lane = threadIdx.x & 63;
    asm volatile("" : "+v"(lane));
    const int row = __builtin_amdgcn_readfirstlane(pair / a.q_heads), kvh = (pair - row * a.q_heads) / (a.q_heads / a.kv_heads);
    const coh_rsrc_t krs = coh_rsrc(L.kc), vrs = coh_rsrc(L.vc + (size_t)row * a.bs * a.kv_heads * 128, pos * a.kv_heads * 256);
    const uint32_t hrow = ((uint32_t)(row * a.bs + (lane >> 2)) * a.kv_heads + kvh) * 128;
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        hist.qn[e] = L.qnorm[lane + 64 * e];
        hist.kn[e] = L.knorm[lane + 64 * e];
        hist.cs[e] = a.cos_sin[(size_t)pos * 128 + lane + 64 * e];
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) hist.k[j] = coh_ld16(krs, (hrow + (lane & 3) * 32 + j * 8) * 2);
#pragma unroll
    for (int u = 0; u < 16; ++u) hist.v[u] = coh_ld4(vrs, ((uint32_t)(u * a.kv_heads + kvh) * 128 + 2 * lane) * 2);
}
__device__ __forceinline__ void flow_attn(const ChainArgs& a, const ChainLayer& L, int pos, int pair, float* sq, const char* in, char* out, char* clr,
                                          const FlowHist& hist, FlowWait& fw, int code, unsigned long long* stamps) {
    const int sidx = ((code & 255) >> 4) * 5 + (code & 15) - 1;
    CH_STAMP_BY(stamps, sidx, 0, 256);
    int lane = threadIdx.x & 63;
    asm volatile("" : "+v"(lane));      // opaque per call (flow_gemm)
    const int q_heads = a.q_heads, kv_heads = a.kv_heads, bs = a.bs;
    const int row = pair / q_heads, h = pair - row * q_heads;
    const int ratio = q_heads / kv_heads, kvh = h / ratio;
    const int tiles = (q_heads + 2 * kv_heads) * 8;
    const int t = lane >> 2, qd = lane & 3;
    const coh_rsrc_t krs = coh_rsrc(L.kc), vrs = coh_rsrc(L.vc), qrs = coh_rsrc(in + CP_QKV), ars = coh_rsrc(out + CP_ATT);
    if (lane < 16) flow_clear16(coh_rsrc(clr + CP_ATT), (uint32_t)frag_off(row, h * 128 + 8 * lane, q_heads * 128) * 2);
    const u32x4 (&kq)[4] = hist.k;
    const uint32_t (&vq)[16] = hist.v;
    CH_STAMP_BY(stamps, sidx, 1, 256);
    // ---- this row's q / k / v heads out of the qkv stage's tiles, one dword per lane each; the (l, l + 64) pairing of the norm + RoPE is
    // restored through LDS
    const uint32_t base = (uint32_t)(row >> 4) * tiles * 512 + (row & 15) * 32 + (lane >> 3) * 512 + (lane & 7) * 4;
    uint32_t qw, kw, vnew;
    {
        unsigned spins = 0;
        unsigned long long t0 = 0;
        bool go = true;
        do {
            qw = coh_ld4(qrs, base + h * 4096);
            kw = coh_ld4(qrs, base + (q_heads + kvh) * 4096);
            vnew = coh_ld4(qrs, base + (q_heads + kv_heads + kvh) * 4096);
        } while (__builtin_amdgcn_ballot_w64(max(max(qw, kw), vnew) == FLOW_EMPTY) != 0 && go && (go = flow_again(fw, code, spins, t0)));
    }
    if (fw.dead) { qw = flow_or0(qw); kw = flow_or0(kw); vnew = flow_or0(vnew); }
    CH_STAMP_BY(stamps, sidx, 2, 256);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");      // the clearing is complete before this use's rows go out (chain_flow.cuh)
    uint32_t* raw = reinterpret_cast<uint32_t*>(sq + 128);        // sq: [0, 128) q in the score layout; [128, 256) raw q | k dwords
    raw[lane] = qw;
    raw[64 + lane] = kw;
    __builtin_amdgcn_wave_barrier();
    const uint16_t* rq = reinterpret_cast<const uint16_t*>(raw);
    const uint16_t* rk = rq + 128;
    float q0, q1, k0, k1;
    const float co = bf2f(hist.cs[0]), si = bf2f(hist.cs[1]);
    head_norm_rope_with(bf2f(rq[lane]), bf2f(rq[lane + 64]), bf2f(hist.qn[0]), bf2f(hist.qn[1]), co, si, a.eps, q0, q1);
    head_norm_rope_with(bf2f(rk[lane]), bf2f(rk[lane + 64]), bf2f(hist.kn[0]), bf2f(hist.kn[1]), co, si, a.eps, k0, k1);
    if (h % ratio == 0) {
        // the new token's K / V into the private cache: one dword per lane (even lanes elements l, l + 1 of the first half, odd lanes l + 63,
        // l + 64 of the second), written through for the later passes
        const uint32_t crow = ((uint32_t)(row * bs + pos) * kv_heads + kvh) * 128;
        const uint32_t kb0 = f2bf(k0), kb1 = f2bf(k1);
        const uint32_t n0 = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)kb0, OMNI_DPP_XOR1, 0xF, 0xF, true);
        const uint32_t n1 = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)kb1, OMNI_DPP_XOR1, 0xF, 0xF, true);
        const bool odd = (lane & 1) != 0;
        const uint32_t word = odd ? (n1 | (kb1 << 16)) : (kb0 | (n0 << 16));
        const uint32_t elem = odd ? 64 + lane - 1 : lane;
        coh_st4(krs, (crow + elem) * 2, word);
        coh_st4(vrs, (crow + 2 * lane) * 2, vnew);
    }
    const float qs = a.sm_scale * LOG2E;
    const float s_new = wave_sum(fmaf(q0 * qs, k0, (q1 * qs) * k1));
    sq[lane] = q0 * qs;
    sq[lane + 64] = q1 * qs;
    __builtin_amdgcn_wave_barrier();
    float d = 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const f32x4 qa = *reinterpret_cast<const f32x4*>(&sq[qd * 32 + j * 8]);
        const f32x4 qb = *reinterpret_cast<const f32x4*>(&sq[qd * 32 + j * 8 + 4]);
        d = fmaf(qa[0], bf_lo(kq[j][0]), d); d = fmaf(qa[1], bf_hi(kq[j][0]), d);
        d = fmaf(qa[2], bf_lo(kq[j][1]), d); d = fmaf(qa[3], bf_hi(kq[j][1]), d);
        d = fmaf(qb[0], bf_lo(kq[j][2]), d); d = fmaf(qb[1], bf_hi(kq[j][2]), d);
        d = fmaf(qb[2], bf_lo(kq[j][3]), d); d = fmaf(qb[3], bf_hi(kq[j][3]), d);
    }
    d += dpp_f<OMNI_DPP_XOR1>(d);
    d += dpp_f<OMNI_DPP_XOR2>(d);
    const float s = t < pos ? d : -INFINITY;
    float m = fmaxf(s, dpp_f<OMNI_DPP_HALF_MIRROR>(s));
    m = fmaxf(m, dpp_f<OMNI_DPP_MIRROR>(m));
    m = xor32_max(xor16_max(m));
    m = fmaxf(m, s_new);
    const float p = exp2f(s - m);
    const float p_new = exp2f(s_new - m);
    float lsum = p + dpp_f<OMNI_DPP_HALF_MIRROR>(p);
    lsum += dpp_f<OMNI_DPP_MIRROR>(lsum);
    lsum = xor32_sum(xor16_sum(lsum));
    const float inv = 1.0f / (lsum + p_new);
    float o0 = p_new * bf_lo(vnew), o1 = p_new * bf_hi(vnew);
#pragma unroll
    for (int u = 0; u < 16; ++u) {
        const float pu = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(p), 4 * u));
        o0 = fmaf(pu, bf_lo(vq[u]), o0);
        o1 = fmaf(pu, bf_hi(vq[u]), o1);
    }
    coh_st4(ars, (uint32_t)frag_off(row, h * 128 + 2 * lane, q_heads * 128) * 2, flow_word(pack_bf2(o0 * inv, o1 * inv)));
    CH_STAMP_BY(stamps, sidx, 6, 256);
    CH_STAMP_BY(stamps, sidx, 7, 256);
}

// the sampler stage of pass g by the workgroup that owns batch row b: draws code g of row b from the head stage's logits and, unless this was the
// last group, gathers the folded embedding -> projection row of the drawn code as the next pass's input (slab 0 = its sum of squares).  The pick
// is wave 0's alone (sampler_body.cuh smp_pick_wave); rows that ask for top-p take the four-wave pick
// logits: 16 x 16 fp32 tiles; r0, p0: where the next pass's input rows and their slab go; c0, cl: the same places in the copy to clear, NULL: none
template <bool TAIL>
__device__ __forceinline__ void flow_sample(const ChainArgs& a, int g, int b, float* lds, float* smp, const void* logits, void* r0, void* p0, void* c0, void* cl,
                                            FlowWait& fw, int code, unsigned long long* stamps) {
    const int sidx = 26;
    int* const last_code = reinterpret_cast<int*>(smp + CPF_LAST);
    CH_STAMP(stamps, sidx, 0);
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));       // opaque per call (flow_gemm)
    const int lane = tid & 63;
    const bool more = g < a.Q - 1 && a.ptab != nullptr;
    const int V = a.codebook, Hc = 1024;
    const coh_rsrc_t lrs = coh_rsrc(logits), rrs = coh_rsrc(r0), prs = coh_rsrc(p0);
    const uint32_t base = (uint32_t)(b >> 4) * 128 * 1024 + (b & 15) * 64;        // logit i of the row: base + (i / 16) * 1024 + (i % 16) * 4
    if (tid < 64 && c0 != nullptr) {
        const coh_rsrc_t crs = coh_rsrc(c0);
        flow_clear16(crs, (uint32_t)frag_off(b, lane * 8, Hc) * 2);
        flow_clear16(crs, (uint32_t)frag_off(b, (lane + 64) * 8, Hc) * 2);
        if (lane == 0) coh_st4(coh_rsrc(cl), (uint32_t)b * 4, FLOW_EMPTY);
    }
    const uint32_t seed = a.row_seed ? a.row_seed[b] : a.seed;
    const uint32_t step = (uint32_t)(a.steps ? a.steps[b] * a.Q + g : g);
    CH_STAMP(stamps, sidx, 1);
    // workgroup-uniform: kernel arguments only
    const bool wave_path = a.greedy || !(a.top_p > 0.f && a.top_p < 1.f);
    const SmpLds S = smp_carve<8>(smp);
    int pick = 0;
    if (wave_path) {
        if (tid < 64) {
            // a moderate temperature keeps the head GEMM's bf16-exact logits strictly ordered under the division: select first, divide the kept
            const bool late = !a.greedy && a.temperature >= 1.0f / 64 && a.temperature <= 64.0f;
            float xr[32];
            unsigned spins = 0;
            unsigned long long t0 = 0;
            for (;;) {
                uint32_t w = 0;
#pragma unroll
                for (int j8 = 0; j8 < 8; ++j8) {
                    const u32x4 v4 = coh_ld16(lrs, base + (j8 * 16 + (lane >> 2)) * 1024 + (lane & 3) * 16);
                    w = max(w, flow_max(v4));
#pragma unroll
                    for (int c = 0; c < 4; ++c) xr[j8 * 4 + c] = __uint_as_float(v4[c]);
                }
                if (__builtin_amdgcn_ballot_w64(w == FLOW_EMPTY) == 0 || !flow_again(fw, code, spins, t0)) break;
            }
            if (fw.dead) {
#pragma unroll
                for (int e = 0; e < 32; ++e) xr[e] = flow_or0(xr[e]);
            }
            CH_STAMP(stamps, sidx, 2);
            // (both fix-ups behind wave-uniform branches the optimiser cannot turn into 32 selects: as straight-line code they were 32 IEEE
            //  divisions on every pick)
            if (V < 2048) {
                asm volatile("" ::: "memory");
#pragma unroll
                for (int e = 0; e < 32; ++e)
                    if ((e >> 2) * 256 + 4 * lane + (e & 3) >= V) xr[e] = -INFINITY;
            }
            if (!a.greedy && !late) {
                asm volatile("" ::: "memory");
#pragma unroll
                for (int e = 0; e < 32; ++e) xr[e] = xr[e] / a.temperature;
            }
            pick = smp_pick_wave<32>(xr, V, a.greedy, a.top_k, late, a.temperature, seed, step, S.ckey);
        }
    } else {
        constexpr int NPT = 8;
        const bool live = tid < SMP_THREADS;
        float xr[NPT];
        unsigned spins = 0;
        unsigned long long t0 = 0;
        for (;;) {
            uint32_t w = 0;
#pragma unroll
            for (int e = 0; e < NPT; ++e) {
                const int i = tid + e * SMP_THREADS;
                uint32_t v = __float_as_uint(-INFINITY);
                if (live && i < V) v = coh_ld4(lrs, base + (i >> 4) * 1024 + (i & 15) * 4);
                w = max(w, v);
                xr[e] = __uint_as_float(v);
            }
            if (__builtin_amdgcn_ballot_w64(w == FLOW_EMPTY) == 0 || !flow_again(fw, code, spins, t0)) break;
        }
        if (fw.dead) {
#pragma unroll
            for (int e = 0; e < NPT; ++e) xr[e] = flow_or0(xr[e]);
        }
        if (!a.greedy) {
#pragma unroll
            for (int e = 0; e < NPT; ++e) {
                const int i = tid + e * SMP_THREADS;
                if (live && i < V) xr[e] = xr[e] / a.temperature;
            }
        }
        pick = smp_pick<NPT>(xr, V, a.greedy, a.top_k, a.top_p, seed, step, S, live, stamps);
    }
    CH_STAMP(stamps, sidx, 4);
    if (tid < 64) {
        if (more) {
            // the folded embedding -> projection row of the drawn code: lane l moves 16-byte pieces l and l + 64 of the 2 KB row; the slab value in
            // sample_kernel's order of additions (piece sums, one wave_sum per 64 pieces, then the two halves)
            const uint16_t* tab = a.ptab + ((size_t)(g - 1) * a.codebook + pick) * Hc;
            float ss2[2];
            u32x4 w4[2];
#pragma unroll
            for (int h2 = 0; h2 < 2; ++h2) w4[h2] = ld16(tab + (lane + 64 * h2) * 8);
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");      // the clearing is complete (chain_flow.cuh)
#pragma unroll
            for (int h2 = 0; h2 < 2; ++h2) {
                u32x4 o;
#pragma unroll
                for (int j = 0; j < 4; ++j) o[j] = flow_word(w4[h2][j]);
                coh_st16(rrs, (uint32_t)frag_off(b, (lane + 64 * h2) * 8, Hc) * 2, o);
                float ss = 0.f;
#pragma unroll
                for (int j = 0; j < 4; ++j) ss += bf_lo(w4[h2][j]) * bf_lo(w4[h2][j]) + bf_hi(w4[h2][j]) * bf_hi(w4[h2][j]);
                ss2[h2] = wave_sum(ss);
            }
            if (lane == 0) coh_st4(prs, (uint32_t)b * 4, flow_word(__float_as_uint(((ss2[0] + ss2[1]) + 0.f) + 0.f)));
        }
        if (lane == 0) {
            coh_st4(coh_rsrc(a.codes), ((uint32_t)b * a.Q + g) * 4, (uint32_t)pick);
            last_code[0] = pick;
        }
    }
    if (TAIL && g == a.Q - 1 && a.tail.enabled) {
        // the row's frame is complete: its owner assembles the backbone's input row right here (no hand-off: the last code is its own)
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        chain_finalize_row(ChainFinArgs{a.tail, a.codes, a.Q, a.codebook}, b, last_code[0], lds);
    }
    CH_STAMP(stamps, sidx, 6);
    CH_STAMP(stamps, sidx, 7);
}

// ---- positions 0 and 1 of the predictor: the two-block stream of cp_forward_pair01 (capi.hip) -- rows [0, B) = position 0 (the talker's last hidden
// state), rows [Bp, Bp + B) = position 1 (the layer-0 code embedding), slabs 128 rows wide -- through the layers { qkv, pair attention, o_proj, gate_up,
// down_proj }, then the group-1 head GEMM on the position-1 rows and the sampler, which gathers the input of pass 2 into rows [0, B).
// The pair attention: a wave per (row, q head) as attn_pair01_kernel (paged_attn.hip) -- position 0 attends to itself (output = its V row), position 1
// to both; K / V of both positions go to the private cache.  The rows between B and Bp pass through the stages of position 0 like the others (their
// consumers wait for whole tiles); nothing of them is kept.
__device__ __forceinline__ void flow_attn_pair(const ChainArgs& a, const ChainLayer& L, int pair, float* sq, char* buf, char* clr, FlowWait& fw, int code,
                                               unsigned long long* stamps) {
    const int sidx = ((code & 255) >> 4) * 5 + (code & 15) - 1;
    CH_STAMP_BY(stamps, sidx, 0, 256);
    int lane = threadIdx.x & 63;
    asm volatile("" : "+v"(lane));      // opaque per call (flow_gemm)
    const int q_heads = a.q_heads, kv_heads = a.kv_heads, bs = a.bs, width = q_heads * 128;
    const int row = pair / q_heads, h = pair - row * q_heads;
    const int ratio = q_heads / kv_heads, kvh = h / ratio;
    const int tiles = (q_heads + 2 * kv_heads) * 8;
    const bool both = row < a.B;
    const coh_rsrc_t krs = coh_rsrc(L.kc), vrs = coh_rsrc(L.vc), qrs = coh_rsrc(buf + PP_QKV), ars = coh_rsrc(buf + PP_ATT), crs = coh_rsrc(clr + PP_ATT);
    if (lane < 16) flow_clear16(crs, (uint32_t)frag_off(row, h * 128 + 8 * lane, width) * 2);
    else if (lane < 32 && both) flow_clear16(crs, (uint32_t)frag_off(a.Bp + row, h * 128 + 8 * (lane - 16), width) * 2);
    // what the norm and the rotation multiply by, ahead of the wait (FlowHist)
    uint16_t qn[2], kn[2], cs[4];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        qn[e] = L.qnorm[lane + 64 * e];
        kn[e] = L.knorm[lane + 64 * e];
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) cs[e] = a.cos_sin[lane + 64 * e];
    CH_STAMP_BY(stamps, sidx, 1, 256);
    // elements 2 l, 2 l + 1 of the heads out of the qkv stage's tiles
    auto at = [&](int m, int head) -> uint32_t { return (uint32_t)((m >> 4) * tiles * 512 + (m & 15) * 32 + (lane >> 3) * 512 + (lane & 7) * 4 + head * 4096); };
    uint32_t k0w = 0, k1w = 0, q1w = 0, v0w, v1w = 0;
    {
        unsigned spins = 0;
        unsigned long long t0 = 0;
        for (;;) {
            v0w = coh_ld4(qrs, at(row, q_heads + kv_heads + kvh));
            if (both) {
                k0w = coh_ld4(qrs, at(row, q_heads + kvh));
                k1w = coh_ld4(qrs, at(a.Bp + row, q_heads + kvh));
                q1w = coh_ld4(qrs, at(a.Bp + row, h));
                v1w = coh_ld4(qrs, at(a.Bp + row, q_heads + kv_heads + kvh));
            }
            if (__builtin_amdgcn_ballot_w64(max(max(max(k0w, k1w), max(q1w, v0w)), v1w) == FLOW_EMPTY) == 0 || !flow_again(fw, code, spins, t0)) break;
        }
    }
    if (fw.dead) { k0w = flow_or0(k0w); k1w = flow_or0(k1w); q1w = flow_or0(q1w); v0w = flow_or0(v0w); v1w = flow_or0(v1w); }
    CH_STAMP_BY(stamps, sidx, 2, 256);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");      // the clearing is complete before this use's rows go out (chain_flow.cuh)
    const int col = h * 128 + 2 * lane;
    coh_st4(ars, (uint32_t)frag_off(row, col, width) * 2, v0w);
    if (both) {
        uint32_t* raw = reinterpret_cast<uint32_t*>(sq);        // three heads of raw dwords: k(pos 0) | k(pos 1) | q(pos 1); the (l, l + 64) pairing through LDS
        raw[lane] = k0w; raw[64 + lane] = k1w; raw[128 + lane] = q1w;
        __builtin_amdgcn_wave_barrier();
        const uint16_t* rh = reinterpret_cast<const uint16_t*>(raw);
        float k00, k01, k10, k11, q0, q1;
        const float w0 = bf2f(kn[0]), w1 = bf2f(kn[1]), c1 = bf2f(cs[2]), s1_ = bf2f(cs[3]);
        head_norm_rope_with(bf2f(rh[lane]), bf2f(rh[lane + 64]), w0, w1, bf2f(cs[0]), bf2f(cs[1]), a.eps, k00, k01);
        head_norm_rope_with(bf2f(rh[128 + lane]), bf2f(rh[128 + lane + 64]), w0, w1, c1, s1_, a.eps, k10, k11);
        head_norm_rope_with(bf2f(rh[256 + lane]), bf2f(rh[256 + lane + 64]), bf2f(qn[0]), bf2f(qn[1]), c1, s1_, a.eps, q0, q1);
        __builtin_amdgcn_wave_barrier();
        const float qs = a.sm_scale * LOG2E;
        const float s0 = wave_sum(fmaf(q0 * qs, k00, (q1 * qs) * k01));
        const float s1 = wave_sum(fmaf(q0 * qs, k10, (q1 * qs) * k11));
        const float m = fmaxf(s0, s1);
        const float p0 = exp2f(s0 - m), p1 = exp2f(s1 - m);
        const float inv = 1.0f / (p0 + p1);
        coh_st4(ars, (uint32_t)frag_off(a.Bp + row, col, width) * 2,
                flow_word(pack_bf2(fmaf(p1, bf_lo(v1w), p0 * bf_lo(v0w)) * inv, fmaf(p1, bf_hi(v1w), p0 * bf_hi(v0w)) * inv)));
        if (h % ratio == 0) {
            // K / V of both positions into the private cache, one dword per lane (flow_attn's pairing of the two halves)
            const bool odd = (lane & 1) != 0;
            const uint32_t elem = odd ? 64 + lane - 1 : lane;
#pragma unroll
            for (int pz = 0; pz < 2; ++pz) {
                const uint32_t crow = ((uint32_t)(row * bs + pz) * kv_heads + kvh) * 128;
                const uint32_t kb0 = f2bf(pz ? k10 : k00), kb1 = f2bf(pz ? k11 : k01);
                const uint32_t n0 = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)kb0, OMNI_DPP_XOR1, 0xF, 0xF, true);
                const uint32_t n1 = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)kb1, OMNI_DPP_XOR1, 0xF, 0xF, true);
                coh_st4(krs, (crow + elem) * 2, odd ? (n1 | (kb1 << 16)) : (kb0 | (n0 << 16)));
                coh_st4(vrs, (crow + 2 * lane) * 2, pz ? v1w : v0w);
            }
        }
    }
    CH_STAMP_BY(stamps, sidx, 6, 256);
    CH_STAMP_BY(stamps, sidx, 7, 256);
}

// combine areas of the pair launch, in floats: o_proj | down_proj | qkv, gate_up and head.  A workgroup's o_proj and down_proj barriers stand between two uses
// of the last; one without o_proj rows meets once more in front of each
#define PP_AREA(tiles) (CH_WAVES * (tiles) * 256 + CH_WAVES * 64)
#define PP_BIG_FLOATS (2 * PP_AREA(2))
#define PP_ATTN_FLOATS (PP_BIG_FLOATS + PP_AREA(12))
#define PP_LDS_BYTES ((PP_ATTN_FLOATS + CH_WAVES * 256) * 4)
static_assert((CPF_LAST + 4) <= PP_ATTN_FLOATS, "the sampler's working set lies over the combine areas");

// R: the most stream rows (both positions) of the launch's split of a stage over the 256 workgroups
//   32   qkv 16 columns x 32 rows each; o_proj / down_proj 16 x 16 on 128 workgroups, gate_up 24 activation columns x 32 rows on the others
//   64   qkv 32 x 32, o_proj / down_proj 16 x 16, gate_up 24 x 32
//   128  qkv 64 x 32, o_proj / down_proj 16 x 32, gate_up 24 x 64
template <int R>
__global__ __launch_bounds__(CH_THREADS) void cp_pair_kernel(const ChainArgs a) {
    extern __shared__ __attribute__((aligned(16))) float lds[];
    ChainGate g;
    chain_gate_init(g, a.flags, a.err);
    constexpr int Hc = 1024, NQ = 4096, NI = 3072;
    constexpr bool SPLIT = R == 32;
    constexpr int QM = 2, QN = R == 32 ? 1 : R / 32, OM = R == 128 ? 2 : 1, GM = R == 128 ? 4 : 2, QC = NQ / 16 / QN;
    const int B = a.B, Bp = a.Bp, M2 = Bp + B;
    const int wg0 = blockIdx.x, wave = threadIdx.x >> 6;
    FlowWait fw{a.err, g.dead ? 1 : 0};
    // ---- this workgroup's part of each stage
    const bool does_q = (wg0 / QC) * QM * 16 < M2;
    const bool does_o = (!SPLIT || wg0 < 128) && (wg0 >> 6) * OM * 16 < M2;
    const bool does_gu = SPLIT ? wg0 >= 128 : (wg0 >> 7) * GM * 16 < M2;
    constexpr int HM = R == 64 ? 2 : 1, HN = R == 128 ? 2 : 1;
    const int hbx = R == 128 ? wg0 & 63 : wg0 - 128, hby = R == 128 ? wg0 >> 6 : 0;
    const bool does_head = hbx >= 0 && hby * HM * 16 < B;
    const int smp_row = R == 128 ? ((wg0 & 63) < 16 ? (wg0 >> 6) * 16 + (wg0 & 63) : 64) : wg0;
    constexpr int PPW = R == 128 ? 4 : 2;                        // (row, q head) pairs per workgroup: waves 4 .. 4 + PPW - 1
    const int pair = (SPLIT ? wg0 - 128 : wg0) * PPW + wave - 4;
    const bool does_attn = wave >= 4 && wave < 4 + PPW && pair >= 0 && pair < Bp * a.q_heads;
    char* const logits = a.flow + (size_t)FLOW_COPIES * PP_COPY;
    float *const lo = lds, *const ld = lds + PP_AREA(2), *const big = lds + PP_BIG_FLOATS;
    // ---- empty this workgroup's tiles of every copy; the launch's first gate tells the others (chain_flow.cuh)
    auto fill = [&](char* p, int pieces) {
        const coh_rsrc_t rs = coh_rsrc(p);
        for (int i = threadIdx.x; i < pieces; i += CH_THREADS) flow_clear16(rs, i * 16);
    };
    for (int c = 0; c < FLOW_COPIES; ++c) {
        char* const cb = a.flow + (size_t)c * PP_COPY;
        if (does_q)
            for (int i = 0; i < QM; ++i) fill(cb + PP_QKV + ((wg0 / QC) * QM + i) * (NQ / 16 * 512) + (wg0 % QC) * QN * 512, QN * 32);
        if (does_attn && (threadIdx.x & 63) < 32) {
            const int row = pair / a.q_heads, m = (threadIdx.x & 16) ? Bp + row : row;
            if (m == row || row < B)
                flow_clear16(coh_rsrc(cb + PP_ATT), (uint32_t)frag_off(m, (pair % a.q_heads) * 128 + 8 * (threadIdx.x & 15), a.q_heads * 128) * 2);
        }
        if (does_o) {
            const int bx = wg0 & 63, by = wg0 >> 6;
            for (int i = 0; i < OM; ++i) { fill(cb + PP_RA + (by * OM + i) * 32768 + bx * 512, 32); fill(cb + PP_RB + (by * OM + i) * 32768 + bx * 512, 32); }
            fill(cb + PP_PA + (bx * 128 + by * OM * 16) * 4, OM * 4);
            fill(cb + PP_PB + (bx * 128 + by * OM * 16) * 4, OM * 4);
        }
        if (does_gu)
            for (int i = 0; i < GM; ++i) fill(cb + PP_ACT + ((SPLIT ? 0 : wg0 >> 7) * GM + i) * 98304 + (wg0 & 127) * 768, 48);
    }
    if (does_head)
        for (int i = 0; i < HM; ++i) fill(logits + (hby * HM + i) * 131072 + hbx * HN * 1024, HN * 64);
    chain_gate_arrive(g);

    u32x2 res = (u32x2){0u, 0u}, none = res;
    char *last = nullptr, *lb = a.flow;
    for (int l = 0; l < a.layers; ++l) {
        const ChainLayer& L = a.layer[l];
        int wg = blockIdx.x;                 // opaque per layer (cp_chain_kernel)
        asm volatile("" : "+s"(wg));
        char* const nb = l % FLOW_COPIES == FLOW_COPIES - 1 ? a.flow : lb + PP_COPY;
        if (does_q) {
            if (!does_o) __syncthreads();
            if (l == 0)
                flow_gemm<QM, QN, 4, 3, OMNI_EPI_BF16, 0, false, 128>(L.wqkv, L.ln1, a.resid, a.part, a.np_in, lb + PP_QKV, nullptr, nb + PP_QKV, nullptr, M2, NQ, a.eps,
                                                                      wg % QC, wg / QC, big, none, fw, 0x0100 | (16 * l + 1), a.stamps, true);
            else
                flow_gemm<QM, QN, 4, 4, OMNI_EPI_BF16, 0, false, 128>(L.wqkv, nullptr, last + PP_RB, (const float*)(last + PP_PB), Hc / 16, lb + PP_QKV, nullptr,
                                                                      nb + PP_QKV, nullptr, M2, NQ, a.eps, wg % QC, wg / QC, big, none, fw, 0x0100 | (16 * l + 1),
                                                                      a.stamps);
        }
        if (l == 0) {                        // everybody's tiles are empty: the first content that is waited for lies behind this
            chain_gate_wait(g, 0x0102);
            fw.dead = flow_failed(a.err);
        }
        if (does_attn) flow_attn_pair(a, L, pair, lds + PP_ATTN_FLOATS + wave * 256, lb, nb, fw, 0x0100 | (16 * l + 2), a.stamps);
        const int bx = wg & 63, by = wg >> 6;
        if (does_o) {
            if (l == 0) {
                const int m = by * OM * 16 + (threadIdx.x >> 6) * 16 + (threadIdx.x & 15);
                if (threadIdx.x < OM * 64 && m < M2) res = coh_ld8(coh_rsrc(a.resid), (uint32_t)frag_off(m, bx * 16 + 4 * ((threadIdx.x & 63) >> 4), Hc) * 2);
            }
            flow_gemm<OM, 1, 8, 0, OMNI_EPI_RESID, 0, false, 128>(L.wo, L.ln2, lb + PP_ATT, nullptr, 0, lb + PP_RA, (float*)(lb + PP_PA), nb + PP_RA, (float*)(nb + PP_PA),
                                                                  M2, Hc, a.eps, bx, by, lo, res, fw, 0x0100 | (16 * l + 3), a.stamps);
        }
        if (does_gu) {
            if (!does_o) __syncthreads();
            flow_gemm<GM, 3, 4, 4, OMNI_EPI_SILU_MUL_GU8, 0, false, 128>(L.wgu, nullptr, lb + PP_RA, (const float*)(lb + PP_PA), Hc / 16, lb + PP_ACT, nullptr, nb + PP_ACT,
                                                                         nullptr, M2, NI, a.eps, wg & 127, SPLIT ? 0 : wg >> 7, big, none, fw,
                                                                         0x0100 | (16 * l + 4), a.stamps);
        }
        if (does_o)
            flow_gemm<OM, 1, 12, 0, OMNI_EPI_RESID, 0, false, 128>(L.wdown, l < a.layers - 1 ? a.layer[l + 1].ln1 : nullptr, lb + PP_ACT, nullptr, 0, lb + PP_RB,
                                                                   (float*)(lb + PP_PB), nb + PP_RB, (float*)(nb + PP_PB), M2, Hc, a.eps, bx, by, ld, res, fw,
                                                                   0x0100 | (16 * l + 5), a.stamps);
        last = lb;
        lb = nb;
    }
    // group 1 on the position-1 rows (tiles Bp / 16 onwards; their slabs start at row Bp)
    if (does_head) {
        if (!does_o) __syncthreads();
        flow_gemm<HM, HN, 4, 2, OMNI_EPI_F32_BF16RND, 0, false, 128>(a.lm_head, a.cp_norm, last + PP_RB + (size_t)Bp * Hc * 2, (const float*)(last + PP_PB) + Bp, Hc / 16,
                                                                     logits, nullptr, nullptr, nullptr, B, a.codebook, a.eps, hbx, hby, big, none, fw, 0x0156, a.stamps,
                                                                     false, a.logits_pass ? a.logits : nullptr, a.logits_ld);
    }
    if (smp_row < B) {
        __syncthreads();                     // the combine areas are read
        flow_sample<false>(a, 1, smp_row, lds, lds, logits, a.resid, a.part, nullptr, nullptr, fw, 0x01F2, a.stamps);
    }
}

// the tail's qkv stage as a real call on a copy of the gate (the launch ends behind it: nothing reads the gate afterwards)
template <int KHT>
__device__ __attribute__((noinline)) void chain_tail_qkv(const ChainArgs::Tail T, int B, float eps, float* lds, ChainGate g, int code) {
    g.dom = 8;
    const int nc_q = T.NQ >> 5;
    chain_gemm<2, 2, KHT, 3, OMNI_EPI_BF16, 4>(T.wqkv, T.ln1, T.resid, T.part, 1, T.qkv, T.NQ, nullptr, B, T.NQ, eps, blockIdx.x % nc_q, blockIdx.x / nc_q, lds, g,
                                               true, code, nullptr);
}

// ROWS: the most rows the launch's split of a stage over the 256 workgroups is for
//   16   every stage but o_proj / down_proj over (nearly) all workgroups: qkv 16 columns each, gate_up 16 activation columns on 192, head 16 on
//        128; o_proj / down_proj (64 tiles of 16 columns) on the other 64, whose weights then wait in registers before gate_up has begun.  (64
//        workgroups for everything, the other 192 idle, pull four times as much each: a pass 104 us behind flags)
//   32   qkv 16 columns x 32 rows each; o_proj / down_proj on 128 workgroups, gate_up (24 activation columns x 32 rows) and head on the others
//   48, 64  a row group of 16 owns 64 workgroups (gate_up at 64: 24 activation columns x 32 rows): three row groups divide no better, four fill the
//        chip
// KHT: 0, or hidden / 256 of the backbone whose first qkv stage closes the launch (the tail)
template <int ROWS, int KHT = 0>
__global__ __launch_bounds__(CH_THREADS) void cp_chain_kernel(const ChainArgs a) {
    extern __shared__ __attribute__((aligned(16))) float lds[];
    static_assert(KHT == 0 || ROWS == 64, "the tail needs every row group live");
    ChainGate g;
    chain_gate_init(g, a.flags, a.err);
    const int Hc = 1024, NQ = 4096, NI = 3072, B = a.B;
    const int wg0 = blockIdx.x, wave = threadIdx.x >> 6;
    constexpr bool SPLIT = ROWS <= 32;
    constexpr int NO = ROWS == 16 ? 64 : 128;                    // SPLIT: workgroups of o_proj / down_proj; the others do gate_up
    if (!SPLIT && (wg0 >> 6) * 16 >= B) {                        // a row group without rows: nobody waits for it beyond the launch's first gate
        if (threadIdx.x < 64) chain_flag_publish(g.frs, wg0, g.epoch + 1u);
        return;
    }
    FlowWait fw{a.err, g.dead ? 1 : 0, !SPLIT};
    float* const attn_lds = lds + CPF_ATTN_FLOATS + wave * 256;
    // ---- this workgroup's part of each stage
    const bool does_o = !SPLIT || wg0 < NO, does_gu = !SPLIT || wg0 >= NO;
    const bool does_head = a.with_head && (!SPLIT || wg0 >= 128);
    const int smp_row = ROWS == 16 ? wg0 - 64 : (ROWS == 32 ? wg0 : ((wg0 & 63) < 16 ? (wg0 >> 6) * 16 + (wg0 & 63) : 64));
    const bool does_smp = a.with_head && smp_row >= 0 && smp_row < B;
    constexpr int PPW = SPLIT ? 2 : 4;                           // (row, q head) pairs per workgroup: waves 4 .. 4 + PPW - 1
    const int pair = (ROWS == 16 ? wg0 - 64 : wg0) * PPW + wave - 4;
    const bool does_attn = wave >= 4 && wave < 4 + PPW && pair >= 0 && pair < B * a.q_heads;
    // ---- empty this workgroup's tiles of every copy; the launch's first gate tells the others (chain_flow.cuh)
    for (int c = 0; c < FLOW_COPIES; ++c) {
        char* const cb = a.flow + (size_t)c * CP_COPY;
        const int tid = threadIdx.x;
        auto fill = [&](uint32_t off, int pieces) {
            const coh_rsrc_t rs = coh_rsrc(cb + off);
            for (int i = tid; i < pieces; i += CH_THREADS) flow_clear16(rs, i * 16);
        };
        if (ROWS == 16) fill(CP_QKV + wg0 * 512, 32);
        else if (ROWS == 32) { fill(CP_QKV + wg0 * 512, 32); fill(CP_QKV + 256 * 512 + wg0 * 512, 32); }
        else fill(CP_QKV + (wg0 >> 6) * 256 * 512 + (wg0 & 63) * 2048, 128);
        if (does_attn && (tid & 63) < 16) flow_clear16(coh_rsrc(cb + CP_ATT), (uint32_t)frag_off(pair / a.q_heads, (pair % a.q_heads) * 128 + 8 * (tid & 15), a.q_heads * 128) * 2);
        if (does_o) {
            const int bx = wg0 & 63, by = wg0 >> 6;
            fill(CP_RA + by * 32768 + bx * 512, 32); fill(CP_RB + by * 32768 + bx * 512, 32);
            fill(CP_PA + (bx * 64 + by * 16) * 4, 4); fill(CP_PB + (bx * 64 + by * 16) * 4, 4);
        }
        if (does_gu) {
            if (ROWS == 16) fill(CP_ACT + (wg0 - NO) * 512, 32);
            else if (ROWS == 48) fill(CP_ACT + (wg0 >> 6) * 98304 + (wg0 & 63) * 1536, 96);
            else {
                const int bx = ROWS == 32 ? wg0 - NO : wg0 & 127, by = ROWS == 32 ? 0 : wg0 >> 7;
                fill(CP_ACT + by * 196608 + bx * 768, 48); fill(CP_ACT + by * 196608 + 98304 + bx * 768, 48);
            }
        }
        if (does_head) {
            if (ROWS == 16) fill(CP_LOG + (wg0 - 128) * 1024, 64);
            else if (ROWS == 32) { fill(CP_LOG + (wg0 - 128) * 1024, 64); fill(CP_LOG + 131072 + (wg0 - 128) * 1024, 64); }
            else fill(CP_LOG + (wg0 >> 6) * 131072 + (wg0 & 63) * 2048, 128);
        }
        if (does_smp && tid < 128) {
            flow_clear16(coh_rsrc(cb + CP_R0), (uint32_t)frag_off(smp_row, tid * 8, Hc) * 2);
            if (tid == 0) coh_st4(coh_rsrc(cb + CP_P0), smp_row * 4, FLOW_EMPTY);
        }
    }
    chain_gate_arrive(g);

    int cl = 0, cp = 0, half = 0;                                // copies of this layer's and this pass's hand-offs; LDS half of the next combine
    bool open = false;                                           // the launch's first gate is behind us
    u32x2 res = (u32x2){0u, 0u}, none = res;
    constexpr int QMT = ROWS == 32 ? 2 : 1, QNT = SPLIT ? 1 : 4;
    // Up to 16 rows the workgroups of o_proj / down_proj ask for their qkv slice ahead of down_proj, not behind it: the heads they own were the last that
    // the attention waited for.  A decode step, 5 rows of the 0.6B talker 1720 -> 1702 us, 7 of the 1.7B one 2067 -> 2049; at up to 32 rows, where all
    // of down_proj's operands queue behind it, 2362 -> 2373.
    constexpr bool ASK = ROWS == 16;
    u32x4 Wn[4][QNT];
    for (int pass = a.g0; pass < a.g1; ++pass) {
        const int pc = pass << 8;            // error-word stage codes: (pass << 8) | (16 * layer + stage + 1); head 0x56, sampler 0xF2
        // debug library: every pass stamps its own block of CH_STAMP_PASS words
        unsigned long long* const st = a.stamps ? a.stamps + (size_t)pass * CH_STAMP_PASS : nullptr;
        const int cpn = cp == FLOW_COPIES - 1 ? 0 : cp + 1, cpl = cp == 0 ? FLOW_COPIES - 1 : cp - 1;
        char *const pb = a.flow + (size_t)cp * CP_COPY, *const pbn = a.flow + (size_t)cpn * CP_COPY, *const pbl = a.flow + (size_t)cpl * CP_COPY;
        const bool first = pass == a.g0;
        char* last = nullptr;                                    // copy of the previous layer
        for (int l = 0; l < a.layers; ++l) {
            const ChainLayer& L = a.layer[l];
            // the workgroup index, opaque per layer: hipcc otherwise hoists every tile / k-step offset of every stage (they depend on
            // blockIdx only) out of both loops and parks them in VGPR lanes for the whole launch (v_writelane / v_readlane; some 240 other
            // SGPRs, mostly arguments and descriptors, still lie there, in 4 VGPRs)
            int wg = blockIdx.x;
            asm volatile("" : "+s"(wg));
            const int cn = cl == FLOW_COPIES - 1 ? 0 : cl + 1;
            char *const lb = a.flow + (size_t)cl * CP_COPY, *const nb = a.flow + (size_t)cn * CP_COPY;
            auto area = [&]() -> float* { half ^= 1; return lds + half * FLOW_HALF_FLOATS; };
            // the pass's own input: raw rows; behind o_proj and down_proj the stream travels as bf16(w r) of the norm in front of its consumer
            const void* xin = first ? (const void*)a.resid : (const void*)(pbl + CP_R0);
            const float* pin = first ? a.part : (const float*)(pbl + CP_P0);
            const int np = first ? a.np_in : 1;
            const bool given = first;
            // the attention's history (written by earlier passes, rows >= pass hold stale bytes and are masked): there before its q / k / v
            if (ASK && (!does_o || (first && l == 0))) flow_ask<QNT, 4>(L.wqkv, wg, Wn);
            FlowHist hist;
            if (does_attn) flow_history(a, L, pass, pair, hist);
            if (l == 0)
                flow_gemm<QMT, QNT, 4, 3, OMNI_EPI_BF16, 0, false, 64, 0, 0, ASK>(L.wqkv, L.ln1, xin, pin, np, lb + CP_QKV, nullptr, nb + CP_QKV, nullptr, B, NQ, a.eps,
                                                         SPLIT ? wg : wg & 63, SPLIT ? 0 : wg >> 6, area(), none, fw, pc | (16 * l + 1), st, given, nullptr, 0, FlowPlain{}, Wn);
            else
                flow_gemm<QMT, QNT, 4, 4, OMNI_EPI_BF16, 0, false, 64, 0, 0, ASK>(L.wqkv, nullptr, last + CP_RB, (const float*)(last + CP_PB), Hc / 16, lb + CP_QKV, nullptr, nb + CP_QKV,
                                                         nullptr, B, NQ, a.eps, SPLIT ? wg : wg & 63, SPLIT ? 0 : wg >> 6, area(), none, fw, pc | (16 * l + 1), st, false, nullptr, 0, FlowPlain{},
                                                         Wn);
            if (!open) {                                         // everybody's tiles are empty: the first content that is waited for lies behind this
                chain_gate_wait(g, pc | (16 * l + 2));
                fw.dead = flow_failed(a.err);
                open = true;
            }
            if (does_attn) flow_attn(a, L, pass, pair, attn_lds, lb, lb, nb, hist, fw, pc | (16 * l + 2), st);
            const bool to_plain = !a.with_head && l == a.layers - 1;       // the stream leaves the launch
            if (does_o) {
                const int bx = wg & 63, by = wg >> 6;
                // this thread's residual values: kept in registers from stage to stage, the pass's own from its input rows
                if (l == 0 && threadIdx.x < 64 && by * 16 + (threadIdx.x & 15) < B) {
                    res = coh_ld8(coh_rsrc(xin), (uint32_t)frag_off(by * 16 + (threadIdx.x & 15), bx * 16 + 4 * (threadIdx.x >> 4), Hc) * 2);
                    if (fw.dead) res = (u32x2){flow_or0(res[0]), flow_or0(res[1])};
                }
                flow_gemm<1, 1, 8, 0, OMNI_EPI_RESID>(L.wo, L.ln2, lb + CP_ATT, nullptr, 0, lb + CP_RA, (float*)(lb + CP_PA), nb + CP_RA, (float*)(nb + CP_PA), B,
                                                      Hc, a.eps, bx, by, area(), res, fw, pc | (16 * l + 3), st);
            }
            if (does_gu) {
                if (ROWS == 16)
                    flow_gemm<1, 2, 4, 4, OMNI_EPI_SILU_MUL_GU8>(L.wgu, nullptr, lb + CP_RA, (const float*)(lb + CP_PA), Hc / 16, lb + CP_ACT, nullptr, nb + CP_ACT,
                                                                 nullptr, B, NI, a.eps, wg - NO, 0, area(), none, fw, pc | (16 * l + 4), st);
                else if (ROWS == 48)
                    flow_gemm<1, 6, 4, 4, OMNI_EPI_SILU_MUL_GU8>(L.wgu, nullptr, lb + CP_RA, (const float*)(lb + CP_PA), Hc / 16, lb + CP_ACT, nullptr, nb + CP_ACT,
                                                                 nullptr, B, NI, a.eps, wg & 63, wg >> 6, area(), none, fw, pc | (16 * l + 4), st);
                else
                    flow_gemm<2, 3, 4, 4, OMNI_EPI_SILU_MUL_GU8>(L.wgu, nullptr, lb + CP_RA, (const float*)(lb + CP_PA), Hc / 16, lb + CP_ACT, nullptr, nb + CP_ACT,
                                                                 nullptr, B, NI, a.eps, ROWS == 32 ? wg - NO : wg & 127, ROWS == 32 ? 0 : wg >> 7, area(), none, fw,
                                                                 pc | (16 * l + 4), st);
            }
            if (ASK && does_o) flow_ask<QNT, 4>(a.layer[l < a.layers - 1 ? l + 1 : 0].wqkv, wg, Wn);
            if (does_o)
                flow_gemm<1, 1, 12, 0, OMNI_EPI_RESID>(L.wdown, l < a.layers - 1 ? a.layer[l + 1].ln1 : nullptr, lb + CP_ACT, nullptr, 0, to_plain ? (void*)a.resid : lb + CP_RB,
                                                       to_plain ? a.part : (float*)(lb + CP_PB), nb + CP_RB, (float*)(nb + CP_PB), B, Hc, a.eps, wg & 63, wg >> 6,
                                                       area(), res, fw, pc | (16 * l + 5), st);
            last = lb;
            cl = cn;
        }
        if (!a.with_head) continue;
        int wg = blockIdx.x;
        asm volatile("" : "+s"(wg));
        // group `pass`: final norm folded into the head GEMM (2048 logits per row), then one workgroup per row samples
        if (does_head) {
            half ^= 1;
            constexpr int HMT = ROWS == 32 ? 2 : 1, HNT = SPLIT ? 1 : 2;
            flow_gemm<HMT, HNT, 4, 2, OMNI_EPI_F32_BF16RND>(a.lm_head + (size_t)(pass - 1) * a.codebook * Hc, a.cp_norm, last + CP_RB, (const float*)(last + CP_PB),
                                                            Hc / 16, pb + CP_LOG, nullptr, pbn + CP_LOG, nullptr, B, a.codebook, a.eps, SPLIT ? wg - 128 : wg & 63,
                                                            SPLIT ? 0 : wg >> 6, lds + half * FLOW_HALF_FLOATS, none, fw, pc | 0x56, st, false,
                                                            a.logits_pass ? a.logits + (size_t)(pass - 1) * a.logits_pass : nullptr, a.logits_ld);
        }
        if (does_smp) flow_sample<(KHT > 0)>(a, pass, smp_row, lds, lds + CPF_SMP_FLOATS, pb + CP_LOG, pb + CP_R0, pb + CP_P0, pbn + CP_R0, pbn + CP_P0, fw, pc | 0xF2, st);
        cp = cpn;
    }
    if constexpr (KHT > 0) {
        if (a.tail.enabled) {
            // layer 0's qkv rows of the backbone, behind EVERY row's input assembly (flag domain: all 256 workgroups); gemm_skinny_kernel's
            // norm-fused arithmetic on 32 x 32 tiles (the bits do not depend on the tile shape: gemm_frag.cuh SlabOrder)
            chain_gate_arrive(g);
            chain_tail_qkv<KHT>(a.tail, B, a.eps, lds, g, ((a.g1 - 1) << 8) | 0x62);
        }
    }
}

// ---- host
OMNI_KNOB g_cp_chain = 1, g_chain_split48 = 0, g_chain_span = 2, g_chain_pair = 1;
#ifdef OMNI_DEBUG_HOOKS
// wide 0: above 48 rows too the 48-row split of the stages (16-row gate_up tiles); the other two were the flag domain and the poll pause
extern "C" void omni_debug_chain_mode(int, int wide, int) { g_chain_split48 = wide == 0; }
extern "C" void omni_debug_chain_pair(int on) { g_chain_pair = on; }            // positions 0 / 1 + group 1 as a persistent launch (0: the launch path's pair pass)
static unsigned long long* g_chain_stamps = nullptr;
// 0: launch per op; 1: one persistent launch per pass (layer stack only); 2: one persistent launch for all passes incl. heads + samplers
extern "C" void omni_debug_cp_chain(int on) { g_cp_chain = on != 0; g_chain_span = on; }
// device buffer of 16 blocks (one per predictor pass; block 0: the pair kernel) of 40 * CH_NSTAMP * 256 uint64 that every following chain
// launch overwrites (NULL: off)
extern "C" void omni_debug_chain_stamps(void* buf) { g_chain_stamps = (unsigned long long*)buf; }
#endif

bool k_cp_chain_supported(const omni_talker_desc& d, int pos) {
    static int cus = -1;
    if (cus < 0) {
        int dev = 0;
        hipDeviceProp_t p;
        cus = (hipGetDevice(&dev) == hipSuccess && hipGetDeviceProperties(&p, dev) == hipSuccess) ? p.multiProcessorCount : 0;
    }
    return g_cp_chain && cus >= OMNI_CHAIN_WGS && d.cp_fused_norm && d.frag_layout && d.cp_hidden == 1024 && d.cp_head_dim == 128 &&
           d.cp_q_heads * 128 == 2048 && (d.cp_q_heads + 2 * d.cp_kv_heads) * 128 == 4096 && d.cp_inter == 3072 &&
           d.cp_layers >= 1 && d.cp_layers <= CH_MAX_LAYERS && pos >= 1 && pos <= 15 && d.num_code_groups + 1 >= 16 &&
           d.max_batch <= 64;
}
// all passes g0 .. Q - 1 with their heads and samplers in ONE launch: additionally the 2048-entry codebook the in-chain sampler is
// built for, the folded projection tables (the next pass's input is a gather) and top-k within the sampler's fast path
bool k_cp_chain_all_supported(const omni_talker_desc& d, int g0, int greedy, int top_k, float top_p) {
    return g_chain_span >= 2 && k_cp_chain_supported(d, g0) && d.codebook == 2048 && d.cp_proj_table != nullptr && d.cp_lm_head != nullptr &&
           d.num_code_groups <= 16 && (greedy || !(top_p > 0.f && top_p < 1.f) || (top_k > 0 && top_k <= SMP_PCAP));
}

// positions 0 / 1 of every row + group 1's head and sampler as ONE persistent launch (cp_pair_kernel); supported where the all-pass
// chain is, with the projected inputs already in the two-block stream (capi.hip run_code_predictor)
bool k_cp_pair_supported(const omni_talker_desc& d, int B, int greedy, int top_k, float top_p) {
    return g_chain_pair && k_cp_chain_all_supported(d, 1, greedy, top_k, top_p) && d.cp_layers <= CH_MAX_LAYERS && B >= 1 && ((B + 15) & ~15) + B <= 128;
}
template <int R>
static int cp_pair_launch(const ChainArgs& a, hipStream_t stream) {
    static const hipError_t attr = hipFuncSetAttribute((const void*)cp_pair_kernel<R>, hipFuncAttributeMaxDynamicSharedMemorySize, PP_LDS_BYTES);
    (void)attr;
    hipLaunchKernelGGL(cp_pair_kernel<R>, dim3(OMNI_CHAIN_WGS), dim3(CH_THREADS), PP_LDS_BYTES, stream, a);
    OMNI_CHECK_LAUNCH("cp_pair");
    return OMNI_OK;
}
int k_cp_pair(const omni_talker_desc& d, const omni_layer_weights* layers, uint16_t* const* k_cache, uint16_t* const* v_cache, int B, int np_in,
              uint16_t* resid, float* part, uint32_t* flags, int32_t* err, void* flow, const omni_chain_head* head, void* stream) {
    ChainArgs a{};
    for (int l = 0; l < d.cp_layers; ++l) {
        const omni_layer_weights& w = layers[l];
        a.layer[l] = ChainLayer{(const uint16_t*)w.ln1, (const uint16_t*)w.wqkv, (const uint16_t*)w.qnorm, (const uint16_t*)w.knorm,
                                (const uint16_t*)w.wo, (const uint16_t*)w.ln2, (const uint16_t*)w.wgu, (const uint16_t*)w.wdown,
                                k_cache[l], v_cache[l]};
    }
    a.layers = d.cp_layers; a.B = B; a.Bp = (B + 15) & ~15; a.g0 = 0; a.g1 = 2; a.bs = d.num_code_groups + 1; a.np_in = np_in;
    a.q_heads = d.cp_q_heads; a.kv_heads = d.cp_kv_heads;
    a.eps = d.eps; a.sm_scale = 1.0f / sqrtf((float)d.cp_head_dim);
    a.resid = resid; a.part = part; a.flow = (char*)flow;
    a.cos_sin = (const uint16_t*)d.cp_cos_sin;
    a.flags = flags; a.err = err;
    a.with_head = 1;
    a.cp_norm = (const uint16_t*)d.cp_norm; a.lm_head = (const uint16_t*)d.cp_lm_head;
    a.logits = head->logits; a.logits_ld = head->logits_ld; a.logits_pass = head->logits_pass;
    a.greedy = head->greedy; a.top_k = head->top_k; a.Q = d.num_code_groups; a.codebook = d.codebook;
    a.temperature = head->temperature; a.top_p = head->top_p; a.seed = head->seed;
    a.steps = head->steps; a.row_seed = head->row_seed; a.codes = head->codes;
    a.ptab = (const uint16_t*)d.cp_proj_table;
#ifdef OMNI_DEBUG_HOOKS
    a.stamps = g_chain_stamps;            // block 0 of the stamp buffer (the chain's passes 2 .. 15 stamp blocks 2 .. 15)
#endif
    const int rows = a.Bp + B;
    if (rows <= 32) return cp_pair_launch<32>(a, (hipStream_t)stream);
    if (rows <= 64) return cp_pair_launch<64>(a, (hipStream_t)stream);
    return cp_pair_launch<128>(a, (hipStream_t)stream);
}

// backbone widths (hidden / 256) the tail's qkv stage is instantiated for: those of bb_chain.hip's BB_SHAPES
#define CP_TAIL_WIDTHS(X) X(8) X(6)
OMNI_KNOB g_chain_tail = 1;
#ifdef OMNI_DEBUG_HOOKS
extern "C" void omni_debug_chain_tail(int on) { g_chain_tail = on; }      // 0: mtp_finalize and the first qkv as launches of their own
#endif
bool k_cp_chain_tail_supported(const omni_talker_desc& d, int B) {
    bool listed = false;
#define X(KH_) listed = listed || d.hidden == KH_ * 256;
    CP_TAIL_WIDTHS(X)
#undef X
    const int NQ = (d.q_heads + 2 * d.kv_heads) * 128;
    // every row group live (B > 48: no workgroup leaves at launch start, all of them own a qkv tile with rows), the norm-free stream, the
    // qkv stage's 32 x 32 tile grid inside the 256 workgroups
    return g_chain_tail && !g_chain_split48 && g_cp_chain && g_chain_span >= 2 && listed && B > 48 && B <= 64 && d.fused_norm && d.frag_layout && d.moe_experts == 0 && d.head_dim == 128 &&
           NQ % 32 == 0 && (NQ / 32) * 2 <= OMNI_CHAIN_WGS && d.hidden % 8 == 0;
}

int k_cp_chain(const omni_talker_desc& d, const omni_layer_weights* layers, uint16_t* const* k_cache, uint16_t* const* v_cache, int B,
               int g0, int g1, int np_in, uint16_t* resid, float* part, uint32_t* flags,
               int32_t* err, void* flow, const omni_chain_head* head, void* stream) {
    ChainArgs a{};
    for (int l = 0; l < d.cp_layers; ++l) {
        const omni_layer_weights& w = layers[l];
        a.layer[l] = ChainLayer{(const uint16_t*)w.ln1, (const uint16_t*)w.wqkv, (const uint16_t*)w.qnorm, (const uint16_t*)w.knorm,
                                (const uint16_t*)w.wo, (const uint16_t*)w.ln2, (const uint16_t*)w.wgu, (const uint16_t*)w.wdown,
                                k_cache[l], v_cache[l]};
    }
    a.layers = d.cp_layers; a.B = B; a.g0 = g0; a.g1 = g1; a.bs = d.num_code_groups + 1; a.np_in = np_in;
    a.q_heads = d.cp_q_heads; a.kv_heads = d.cp_kv_heads;
    a.eps = d.eps; a.sm_scale = 1.0f / sqrtf((float)d.cp_head_dim);
    a.resid = resid; a.part = part; a.flow = (char*)flow;
    a.cos_sin = (const uint16_t*)d.cp_cos_sin;
    a.flags = flags; a.err = err;
    if (head) {
        a.with_head = 1;
        a.cp_norm = (const uint16_t*)d.cp_norm; a.lm_head = (const uint16_t*)d.cp_lm_head;
        a.logits = head->logits; a.logits_ld = head->logits_ld; a.logits_pass = head->logits_pass;
        a.greedy = head->greedy; a.top_k = head->top_k; a.Q = d.num_code_groups; a.codebook = d.codebook;
        a.temperature = head->temperature; a.top_p = head->top_p; a.seed = head->seed;
        a.steps = head->steps; a.row_seed = head->row_seed; a.codes = head->codes;
        a.ptab = (const uint16_t*)d.cp_proj_table;
    }
#ifdef OMNI_DEBUG_HOOKS
    a.stamps = g_chain_stamps;
#endif
    static bool attr = false;
    if (!attr) {
        (void)hipFuncSetAttribute((const void*)cp_chain_kernel<16>, hipFuncAttributeMaxDynamicSharedMemorySize, CPF_LDS_BYTES);
        (void)hipFuncSetAttribute((const void*)cp_chain_kernel<32>, hipFuncAttributeMaxDynamicSharedMemorySize, CPF_LDS_BYTES);
        (void)hipFuncSetAttribute((const void*)cp_chain_kernel<48>, hipFuncAttributeMaxDynamicSharedMemorySize, CPF_LDS_BYTES);
        (void)hipFuncSetAttribute((const void*)cp_chain_kernel<64>, hipFuncAttributeMaxDynamicSharedMemorySize, CPF_LDS_BYTES);
#define X(KH_) (void)hipFuncSetAttribute((const void*)cp_chain_kernel<64, KH_>, hipFuncAttributeMaxDynamicSharedMemorySize, CPF_LDS_BYTES);
        CP_TAIL_WIDTHS(X)
#undef X
        attr = true;
    }
#define CP_LAUNCH(...)                                                                                                                              \
    do {                                                                                                                                             \
        hipLaunchKernelGGL((cp_chain_kernel<__VA_ARGS__>), dim3(OMNI_CHAIN_WGS), dim3(CH_THREADS), CPF_LDS_BYTES, (hipStream_t)stream, a);           \
        OMNI_CHECK_LAUNCH("cp_chain");                                                                                                               \
        return OMNI_OK;                                                                                                                              \
    } while (0)
    if (head && head->tail && g1 == d.num_code_groups && k_cp_chain_tail_supported(d, B)) {
        // the launch ends in the step's input assembly + layer 0's qkv (instantiated per backbone width: CP_TAIL_WIDTHS)
        const omni_chain_tail& T = *head->tail;
        a.tail = ChainArgs::Tail{T.input_ids, (const uint16_t*)T.embed, T.vocab, (const uint16_t*)T.cp_embed, (const uint16_t*)T.text_step,
                                 (uint16_t*)T.x_out, (uint16_t*)T.resid, T.part, T.audio_codes, T.H,
                                 (const uint16_t*)T.wqkv, (const uint16_t*)T.ln1, (uint16_t*)T.qkv, T.NQ, 1};
#define X(KH_) if (d.hidden == KH_ * 256) CP_LAUNCH(64, KH_);
        CP_TAIL_WIDTHS(X)
#undef X
    }
    if (B <= 16) CP_LAUNCH(16);
    if (B <= 32) CP_LAUNCH(32);
    if (B <= 48 || g_chain_split48) CP_LAUNCH(48);
    CP_LAUNCH(64);
#undef CP_LAUNCH
}
