// The talker backbone between two attention launches as ONE persistent launch per decoder layer:
//     o_proj(l) -> gate_up(l) -> down_proj(l) -> qkv_proj(l + 1)
// (reference: the vLLM Qwen3 decoder layer reached through qwen3_tts_talker.py:341,414-422; four of the five launches of
// a layer on the launch-per-op path).  A stage's weight slice -- 64-196 KB per workgroup, 32-96 VGPRs per lane -- goes out before the
// stage looks for its operands, so the HBM stream keeps running through the hand-off instead of stopping for a kernel boundary (1.65 us)
// plus a cold first fetch.
//   bb_flow_kernel, bb_flow_small_kernel   one rank, the whole chip: activations cross by content (chain_flow.cuh)
//   bb_chain_kernel                        a tensor-parallel rank (AR), the half grid (HALF): behind flags (chain_gemm.cuh)
// K-step ownership, combine order and rounding points are the launch path's: results are bit-identical.
// A decode step, behind flags and by content, one card: 64 rows of the 1.7B shape 3050 -> 2886 us, 5 rows of the 0.6B one 2091 -> 1859.
// Of a 64-row launch (32 us, 100 MB) gate_up takes 13 us, in which its 50 MB come out of HBM; a wave's loads return in order, so half of a wave's
// slice goes out in front of the first look at the operands and half behind the first of them (down_proj: half of its 24 k-steps, x twelve deep): 64 rows
// 2807 -> 2771 us a step, 24 rows 2354 -> 2342.  Slices with a single reader are loaded past the caches, which leaves the last-level cache to the predictor's
// weights (157 MB): 64 rows 2786 -> 2771, 24 rows 2352 -> 2342, 7 rows 2079 -> 2031, 0.6B, 5 rows 1750 -> 1717; those that the two row halves share are not
// (64 rows 2817 -> 2839).  The splits for few rows alone: 24 rows 2488 -> 2342, 7 rows 2310 -> 2031, 0.6B, 5 rows 2030 -> 1717 (with the predictor's;
// profiles/talker_step_sweeps.txt, talker_step_timeline.txt).
// Tried: gate_up's slice asked for by o_proj's waves (their combine waits for the queue: the same), half of qkv's behind the look (64 rows + 10 us).
// Shapes are parameters, not literals (the checkpoint decides them, configuration_qwen3_tts.py:192-216): the stage set is a template
// on the k-steps per wave of its three reduction widths -- KO = q_heads * 128 / 256 (o_proj), KH = hidden / 256 (gate_up, qkv), KI =
// intermediate / 256 (down_proj); BB_SHAPES lists the instantiated triples: the released 1.7B shape (8, 8, 24) and (6, 6, 18) = hidden 1536 /
// intermediate 4608 / 12 q heads, a shape no released checkpoint has (tests/test_gpu_chain.py).  A shape runs here when its triple is listed
// and every stage's tile grid fits the 256 workgroups (k_bb_chain_supported); the 0.6B shape has the code predictor's layer dimensions and its
// split of the stages; every other configuration stays on the launch path.
#include "bb_areas.h"
#include "chain_flow.cuh"
#include "common.cuh"
#include "kernels.h"

#define BB_LDS_BYTES ((CH_WAVES * 12 * 64 * 16) + CH_WAVES * 64 * 4)      // bb_chain_kernel: combine slots (gate_up: 12 tiles) + rstd area

struct BbArgs {
    const uint16_t *wo, *ln2, *wgu, *wdown, *ln1_next, *wqkv_next;      // *_next == NULL: last layer, no qkv stage
    const uint16_t* attn;               // fragment-major [64][2048]: the attention launch's output
    uint16_t* resid; float* part;       // fragment-major residual stream [64][2048] + sum(r^2) slabs [128][64]
    uint16_t* act;                      // fragment-major [64][6144]
    uint16_t* qkv;                      // row-major [B][NQ]
    int H, I, NQ;                       // output widths: hidden, intermediate, (q_heads + 2 kv_heads) * 128
    // the LAST layer's launch (no next qkv) may end in the talker's own head instead: final norm folded into the lm_head GEMM, its
    // normalised rows = h[t + 1] (row-major, rows below *num_live), logits fp32 [B][V] holding bf16-rounded values, the codec mask applied
    const uint16_t *lm_head, *final_norm; float* logits; uint16_t* last_hidden; const uint8_t* mask; const int32_t* num_live; float mask_fill; int V;
    int B; float eps;
    uint32_t* flags; int32_t* err;
    unsigned long long* stamps;
    // tensor-parallel rank: o_proj and down_proj are row-parallel partials; their all-reduce rides in the two residual epilogues
    // (chain_gemm AR).  ar_epoch = allreduce.hip's epoch / ticket words: this launch makes calls epoch + 1 (o_proj) and epoch + 2 (down_proj)
    ChainAr ar_o, ar_dn;
    uint32_t* ar_epoch;
    // hand-offs by content: this launch's buffers, the ones it empties for the next layer's launch (NULL: none behind it), 1: the step's first launch
    char *flow, *flow_next;
    int first;
};
static_assert(BB_WAVES == CH_WAVES, "bb_areas.h");

// Rings: gate_up's activations and weights two k-steps deep, down_proj's and qkv's activations four.  gate_up's 12 tiles combine in one pass, the RMSNorm's
// rstd is applied in the epilogues (chain_gemm PRO 3).
// HEAD: the instantiation the LAST layer launches when the step's head rides along (its own code object entry: the other 27 launches keep the
// leaner kernel -- with the head stage compiled into every launch the segment cost 0.9 us more per layer, register allocation of the shared stages)
// AR: the instantiation of a tensor-parallel rank (the all-reduces inside the o_proj / down_proj stages); HALF: 128 workgroups play the 256 of the
// stage grid, two VIRTUAL workgroups each, stage by stage (a virtual workgroup's stage needs only stages that every physical workgroup has
// already run or will run before it waits again: no cycle) -- two such launches of two processes fit the chip side by side, which is how the
// cross-process exchange is tested on one GPU (tests/test_gpu_tp.py) and how a co-located second engine keeps its backbone chain
template <int KO, int KH, int KI, bool HEAD, bool AR, bool HALF>
__global__ __launch_bounds__(CH_THREADS) void bb_chain_kernel(const BbArgs a) {
    extern __shared__ __attribute__((aligned(16))) float lds[];
    static_assert((AR || HALF) && !(HEAD && HALF), "bb_chain: one rank on the whole chip runs bb_flow_kernel; the half grid has no head stage");
    uint32_t e0 = 0;
    if constexpr (AR) e0 = __builtin_amdgcn_readfirstlane(__hip_atomic_load(a.ar_epoch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
    ChainGate g;
    chain_gate_init(g, a.flags, a.err);
    g.dom = 8;                          // gate_up's 64-row tiles tie every row group together
    const int wg = blockIdx.x;
    const int H = a.H, I = a.I, NQ = a.NQ;
    // workgroup -> tile: o_proj / down_proj 16 columns x 32 rows, gate_up 24 activation columns x 64 rows, qkv 32 columns x 32 rows; a
    // workgroup past a stage's grid (column tiles x row tiles < 256 at widths below the 1.7B shape's) publishes the stage and runs ahead
    const int nc_h = H >> 4, nc_gu = I / 24, nc_q = NQ >> 5;
    // stage codes (error word): 0x1001 .. 0x1005
    // the four stages of (virtual) workgroup WG_ behind gate G_
#define BB_O(WG_, G_)                                                                                                                                   \
    chain_gemm<2, 1, KO, 0, OMNI_EPI_RESID, 0, 0, ChainNoPrefetch, false, AR>(a.wo, nullptr, a.attn, nullptr, 0, a.resid, 0, a.part, a.B, H, a.eps,         \
                                                                              (WG_) % nc_h, (WG_) / nc_h, lds, G_, false, 0x1001, a.stamps,                \
                                                                              ChainNoPrefetch(), nullptr, nullptr, 0.f, nullptr, &a.ar_o, e0 + 1u)
#define BB_GU(WG_, G_)                                                                                                                                  \
    do {                                                                                                                                                \
        if ((WG_) < nc_gu)                                                                                                                              \
            chain_gemm<4, 3, KH, 3, OMNI_EPI_SILU_MUL_GU8, 2, 1, ChainNoPrefetch, true>(a.wgu, a.ln2, a.resid, a.part, H / 16, a.act, 0, nullptr, a.B, I,   \
                                                                                        a.eps, WG_, 0, lds, G_, true, 0x1002, a.stamps);                   \
        else                                                                                                                                            \
            chain_gate_skip(G_);                                                                                                                        \
    } while (0)
#define BB_DN(WG_, G_)                                                                                                                                  \
    chain_gemm<2, 1, KI, 0, OMNI_EPI_RESID, 4, 0, ChainNoPrefetch, false, AR>(a.wdown, nullptr, a.act, nullptr, 0, a.resid, 0, a.part, a.B, H, a.eps,        \
                                                                              (WG_) % nc_h, (WG_) / nc_h, lds, G_, true, 0x1003, a.stamps,                 \
                                                                              ChainNoPrefetch(), nullptr, nullptr, 0.f, nullptr, &a.ar_dn, e0 + 2u)
#define BB_QK(WG_, G_)                                                                                                                                  \
    chain_gemm<2, 2, KH, 3, OMNI_EPI_BF16, 4>(a.wqkv_next, a.ln1_next, a.resid, a.part, H / 16, a.qkv, NQ, nullptr, a.B, NQ, a.eps, (WG_) % nc_q,            \
                                              (WG_) / nc_q, lds, G_, true, 0x1004, a.stamps)
    if constexpr (HALF) {
        ChainGate g2;
        chain_gate_init(g2, a.flags, a.err, wg + OMNI_CHAIN_WGS / 2);
        g2.dom = 8;
        const int wg2 = wg + OMNI_CHAIN_WGS / 2;
        BB_O(wg, g); BB_O(wg2, g2);
        BB_GU(wg, g); BB_GU(wg2, g2);
        BB_DN(wg, g); BB_DN(wg2, g2);
        if (a.wqkv_next) { BB_QK(wg, g); BB_QK(wg2, g2); }
    } else {
    BB_O(wg, g);
    BB_GU(wg, g);
    BB_DN(wg, g);
    if (a.wqkv_next)
        BB_QK(wg, g);
    else if (HEAD && a.lm_head) {
        // the step's head as the last stage of its last backbone launch (one launch and one cold start less: 9.8 us + a boundary -> a stage):
        // gemm_skinny_kernel<2, 2, PRO 2, F32_BF16RND>'s tile and arithmetic (exact norm: its normalised rows are h[t + 1])
        const int nc_v = a.V >> 5;
        chain_gemm<2, 2, KH, 2, OMNI_EPI_F32_BF16RND, 4>(a.lm_head, a.final_norm, a.resid, a.part, H / 16, a.logits, a.V, nullptr, a.B, a.V, a.eps, wg % nc_v,
                                                         wg / nc_v, lds, g, true, 0x1005, a.stamps, ChainNoPrefetch(), a.last_hidden, a.mask, a.mask_fill,
                                                         a.num_live);
    }
    }
#undef BB_O
#undef BB_GU
#undef BB_DN
#undef BB_QK
    if constexpr (AR) {
        // the last workgroup out closes the launch's two all-reduce calls (allreduce.hip's epoch word: every workgroup read it at its start)
        __syncthreads();
        if (threadIdx.x == 0) {
            const uint32_t t = atomicAdd(a.ar_epoch + 1, 1u);
            if (t == gridDim.x - 1) {
                __hip_atomic_store(a.ar_epoch + 1, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                __hip_atomic_store(a.ar_epoch, e0 + 2u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
    }
}

// ---- the single-rank launches: hand-offs by content (chain_flow.cuh).  What bounds a stage here is the trip from its predecessor's last store to its
// own operands and what a CU can take in (wide shape, 64 rows: 0.2 to 0.6 MB of weights and activations a stage); behind flags every stage paid a
// drain, a barrier, a flag, a poll and another barrier on top.
// Two copies of the hand-off buffers: a launch uses one, empty when it starts, and empties its own tiles of the other for the launch behind it (the
// last layer's has none).  The first layer's launch empties its own copy itself and is the only one that meets at a gate: whatever an earlier, broken
// off step left there does not matter.
struct BbFlowMap {                          // byte offsets within a copy (64 rows)
    uint32_t ra, pa, act, rb, pb, copy;
    __host__ __device__ constexpr BbFlowMap(int H, int I)
        : ra(0), pa(64 * H * 2), act(pa + H / 16 * 64 * 4), rb(act + 64 * I * 2), pb(rb + 64 * H * 2), copy(pb + H / 16 * 64 * 4) {}
};
// the attention's rows are the launch's input: taken as they are
#define BB_GIVEN true

// ROWS: 64 (33 to 64 rows: o_proj / down_proj 16 columns x 32 rows a workgroup, gate_up 24 activation columns x 64, qkv 32 x 32), 32 (o_proj / down_proj
// 16 x 16, qkv 16 x 32) or 16 (one row tile: o_proj / down_proj on half of the workgroups); gate_up takes 24 activation columns of all rows
template <int KO, int KH, int KI, int ROWS, bool HEAD>
__global__ __launch_bounds__(CH_THREADS) void bb_flow_kernel(const BbArgs a) {
    extern __shared__ __attribute__((aligned(16))) float lds[];
    constexpr int H = KH * 256, I = KI * 256, MO = ROWS == 64 ? 2 : 1, MG = ROWS / 16, NQT = ROWS == 64 ? 2 : 1, MQ = ROWS == 16 ? 1 : 2;
    constexpr BbFlowMap F(H, I);
    constexpr BbAreas A = bb_areas_wide(ROWS);
    constexpr int nc_h = H / 16, nc_gu = I / 24;
    static_assert(ROWS == 16 || nc_gu <= 2 * nc_h, "bb_areas_wide: whoever runs gate_up runs down_proj");
    static_assert(A.gate_up == bb_area(MO) && A.down == A.gate_up + bb_area(3 * MG) && A.last + bb_area(MQ * NQT) <= A.total, "bb_areas_wide: tiles");
    // weight slices that one workgroup alone reads go past the caches (a step's weights do not fit them, the predictor's do)
    constexpr int NO = ROWS == 16 ? OMNI_AUX_NT : 0, NQA = ROWS <= 32 ? OMNI_AUX_NT : 0;
    static_assert(nc_h * (ROWS == 16 ? 1 : 2) <= OMNI_CHAIN_WGS && nc_gu <= OMNI_CHAIN_WGS && I % 24 == 0, "bb_flow: tiles");
    const int B = a.B, wg = blockIdx.x;
    const int bxo = wg % nc_h, byo = wg / nc_h;
    const bool does_o = byo < (ROWS == 16 ? 1 : 2) && byo * MO * 16 < B, does_gu = wg < nc_gu;
    char *const fl = a.flow, *const nx = a.flow_next;
    ChainGate g;
    FlowWait fw{a.err, 0};
    u32x2 res = (u32x2){0u, 0u}, none = res;
    if (a.first) {
        chain_gate_init(g, a.flags, a.err);
        fw.dead = g.dead;
        auto fill = [&](uint32_t off, int pieces) {
            const coh_rsrc_t rs = coh_rsrc(fl + off);
            for (int i = threadIdx.x; i < pieces; i += CH_THREADS) flow_clear16(rs, i * 16);
        };
        if (does_o) {
            for (int i = 0; i < MO; ++i) {
                fill(F.ra + (byo * MO + i) * 32 * H + bxo * 512, 32);
                fill(F.rb + (byo * MO + i) * 32 * H + bxo * 512, 32);
            }
            fill(F.pa + (bxo * 64 + byo * MO * 16) * 4, MO * 4);
            fill(F.pb + (bxo * 64 + byo * MO * 16) * 4, MO * 4);
        }
        if (does_gu)
            for (int i = 0; i < MG; ++i) fill(F.act + i * 32 * I + wg * 768, 48);
        chain_gate_arrive(g);
    }
    auto next = [&](uint32_t off) -> char* { return nx != nullptr ? nx + off : nullptr; };
    float *const lo = lds + A.o, *const lg = lds + A.gate_up, *const ld = lds + A.down, *const ll = lds + A.last;
    if (does_o) {
        if (threadIdx.x < MO * 64 && byo * MO * 16 + (int)threadIdx.x / 64 * 16 + (threadIdx.x & 15) < B)
            res = coh_ld8(coh_rsrc(a.resid), (uint32_t)frag_off(byo * MO * 16 + threadIdx.x / 64 * 16 + (threadIdx.x & 15), bxo * 16 + 4 * ((threadIdx.x & 63) >> 4), H) * 2);
        flow_gemm<MO, 1, KO, 0, OMNI_EPI_RESID, 0, false, 64, 0, NO>(a.wo, a.ln2, a.attn, nullptr, 0, fl + F.ra, (float*)(fl + F.pa), next(F.ra), (float*)next(F.pa), B, H, a.eps, bxo,
                                                byo, lo, res, fw, 0x1001, a.stamps, BB_GIVEN);
    }
    if (a.first) {
        chain_gate_wait(g, 0x1002);
        fw.dead = flow_failed(a.err);
    }
    if (does_gu)
        flow_gemm<MG, 3, KH, 4, OMNI_EPI_SILU_MUL_GU8, ROWS == 64 ? 4 : 0, false, 64, 4, OMNI_AUX_NT>(a.wgu, nullptr, fl + F.ra, (const float*)(fl + F.pa), H / 16, fl + F.act, nullptr, next(F.act),
                                                                          nullptr, B, I, a.eps, wg, 0, lg, none, fw, 0x1002, a.stamps);
    const bool qkv = a.wqkv_next != nullptr, head = HEAD && !qkv && a.lm_head != nullptr;
    if (does_o)
        // raw values for the next launch; bf16(w r) for the qkv stage, the values themselves for the head (its norm is exact)
        flow_gemm<MO, 1, KI, 0, OMNI_EPI_RESID, ROWS == 64 ? 12 : 8, false, 64, ROWS == 64 ? 12 : 0, NO>(a.wdown, qkv ? a.ln1_next : nullptr, fl + F.act, nullptr, 0, qkv || head ? fl + F.rb : nullptr,
                                                                    (float*)(fl + F.pb), next(F.rb), (float*)next(F.pb), B, H, a.eps, bxo, byo, ld, res, fw, 0x1003,
                                                                    a.stamps, false, nullptr, 0, FlowPlain{nullptr, a.resid, a.part});
    if (qkv) {
        const int nc_q = a.NQ / (16 * NQT), bx = wg % nc_q, by = wg / nc_q;
        if (by * MQ * 16 < B && by < 4 / MQ)
            flow_gemm<MQ, NQT, KH, 4, OMNI_EPI_BF16, 0, true, 64, 0, NQA>(a.wqkv_next, nullptr, fl + F.rb, (const float*)(fl + F.pb), H / 16, nullptr, nullptr, nullptr, nullptr, B,
                                                              a.NQ, a.eps, bx, by, ll, none, fw, 0x1004, a.stamps, false, nullptr, a.NQ, FlowPlain{a.qkv});
    } else if (head) {
        const int nc_v = a.V / (16 * NQT), bx = wg % nc_v, by = wg / nc_v;
        if (by * MQ * 16 < B && by < 4 / MQ)
            flow_gemm<MQ, NQT, KH, 2, OMNI_EPI_F32_BF16RND, 0, true>(a.lm_head, a.final_norm, fl + F.rb, (const float*)(fl + F.pb), H / 16, nullptr, nullptr, nullptr,
                                                                     nullptr, B, a.V, a.eps, bx, by, ll, none, fw, 0x1005, a.stamps, false, a.logits, a.V,
                                                                     FlowPlain{nullptr, nullptr, nullptr, a.last_hidden, a.num_live, a.mask, a.mask_fill});
    }
}

// ---- the 0.6B backbone shape (hidden 1024, 16 x 128 attention width over 8 kv heads, intermediate 3072): the dimensions of the code predictor's
// layers, and its split of the stages over the 256 workgroups by rows (cp_chain.hip cp_chain_kernel).
template <int ROWS>
__global__ __launch_bounds__(CH_THREADS) void bb_flow_small_kernel(const BbArgs a) {
    extern __shared__ __attribute__((aligned(16))) float lds[];
    constexpr int H = 1024, I = 3072, NQ = 4096;
    constexpr BbFlowMap F(H, I);
    constexpr BbAreas A = bb_areas_small(ROWS);
    constexpr bool SPLIT = ROWS <= 32;
    constexpr int NO = ROWS == 16 ? 64 : 128;                    // SPLIT: workgroups of o_proj / down_proj; the others do gate_up
    const int B = a.B, wg = blockIdx.x;
    if (!SPLIT && (wg >> 6) * 16 >= B) {                         // a row group without rows: nobody waits for it beyond the first launch's gate
        if (a.first && threadIdx.x < 64) {
            ChainGate g;
            chain_gate_init(g, a.flags, a.err);
            chain_flag_publish(g.frs, wg, g.epoch + 1u);
        }
        return;
    }
    const bool does_o = (!SPLIT || wg < NO) && (wg >> 6) * 16 < B, does_gu = !SPLIT || wg >= NO;
    const int bxo = wg & 63, byo = wg >> 6;
    char *const fl = a.flow, *const nx = a.flow_next;
    ChainGate g;
    FlowWait fw{a.err, 0};
    u32x2 res = (u32x2){0u, 0u}, none = res;
    constexpr int GM = ROWS == 16 || ROWS == 48 ? 1 : 2, GN = ROWS == 16 ? 2 : (ROWS == 48 ? 6 : 3);       // gate_up's tiles
    constexpr int QM = ROWS == 32 ? 2 : 1, QN = SPLIT ? 1 : 4;
    static_assert(A.gate_up == bb_area(1) && A.down == A.gate_up + bb_area(ROWS == 16 ? 2 : 6) && GM * GN <= 6 && A.last + bb_area(QM * QN) <= A.total, "bb_areas_small: tiles");
    const int bxg = SPLIT ? wg - NO : (ROWS == 48 ? wg & 63 : wg & 127), byg = SPLIT ? 0 : (ROWS == 48 ? wg >> 6 : wg >> 7);
    if (a.first) {
        chain_gate_init(g, a.flags, a.err);
        fw.dead = g.dead;
        auto fill = [&](uint32_t off, int pieces) {
            const coh_rsrc_t rs = coh_rsrc(fl + off);
            for (int i = threadIdx.x; i < pieces; i += CH_THREADS) flow_clear16(rs, i * 16);
        };
        if (does_o) {
            fill(F.ra + byo * 32 * H + bxo * 512, 32); fill(F.rb + byo * 32 * H + bxo * 512, 32);
            fill(F.pa + (bxo * 64 + byo * 16) * 4, 4); fill(F.pb + (bxo * 64 + byo * 16) * 4, 4);
        }
        if (does_gu)
            for (int i = 0; i < GM; ++i) fill(F.act + (byg * GM + i) * 32 * I + bxg * GN * 256, GN * 16);
        chain_gate_arrive(g);
    }
    auto next = [&](uint32_t off) -> char* { return nx != nullptr ? nx + off : nullptr; };
    float *const lo = lds + A.o, *const lg = lds + A.gate_up, *const ld = lds + A.down, *const ll = lds + A.last;
    if (does_o) {
        if (threadIdx.x < 64 && byo * 16 + (int)(threadIdx.x & 15) < B)
            res = coh_ld8(coh_rsrc(a.resid), (uint32_t)frag_off(byo * 16 + (threadIdx.x & 15), bxo * 16 + 4 * (threadIdx.x >> 4), H) * 2);
        flow_gemm<1, 1, 8, 0, OMNI_EPI_RESID, 0, false, 64, 0, ROWS == 16 ? OMNI_AUX_NT : 0>(a.wo, a.ln2, a.attn, nullptr, 0, fl + F.ra, (float*)(fl + F.pa), next(F.ra), (float*)next(F.pa), B, H, a.eps, bxo, byo,
                                              lo, res, fw, 0x1001, a.stamps, BB_GIVEN);
    }
    if (a.first) {
        chain_gate_wait(g, 0x1002);
        fw.dead = flow_failed(a.err);
    }
    if (does_gu)
        flow_gemm<GM, GN, 4, 4, OMNI_EPI_SILU_MUL_GU8, 0, false, 64, 0, SPLIT ? OMNI_AUX_NT : 0>(a.wgu, nullptr, fl + F.ra, (const float*)(fl + F.pa), H / 16, fl + F.act, nullptr, next(F.act), nullptr, B, I,
                                                       a.eps, bxg, byg, lg, none, fw, 0x1002, a.stamps);
    const bool qkv = a.wqkv_next != nullptr;
    if (does_o)
        flow_gemm<1, 1, 12, 0, OMNI_EPI_RESID, 0, false, 64, 0, ROWS == 16 ? OMNI_AUX_NT : 0>(a.wdown, qkv ? a.ln1_next : nullptr, fl + F.act, nullptr, 0, qkv ? fl + F.rb : nullptr, (float*)(fl + F.pb), next(F.rb),
                                               (float*)next(F.pb), B, H, a.eps, bxo, byo, ld, res, fw, 0x1003, a.stamps, false, nullptr, 0,
                                               FlowPlain{nullptr, a.resid, a.part});
    if (qkv) {
        flow_gemm<QM, QN, 4, 4, OMNI_EPI_BF16, 0, true, 64, 0, SPLIT ? OMNI_AUX_NT : 0>(a.wqkv_next, nullptr, fl + F.rb, (const float*)(fl + F.pb), H / 16, nullptr, nullptr, nullptr, nullptr, B, NQ,
                                                        a.eps, SPLIT ? wg : wg & 63, SPLIT ? 0 : wg >> 6, ll, none, fw, 0x1004, a.stamps, false, nullptr, NQ,
                                                        FlowPlain{a.qkv});
    }
}

size_t k_bb_flow_bytes(const omni_talker_desc& d) { return 2 * (size_t)BbFlowMap(d.hidden, d.inter).copy; }

OMNI_KNOB g_bb_chain = 1, g_bb_min_rows = 33, g_bb_b32 = 1, g_bb_ar = 1;
#ifdef OMNI_DEBUG_HOOKS
static unsigned long long* g_bb_stamps = nullptr;
extern "C" void omni_debug_bb_chain(int on) { g_bb_chain = on; }
extern "C" void omni_debug_bb_stamps(void* buf) { g_bb_stamps = (unsigned long long*)buf; }
extern "C" void omni_debug_bb_deep(int) {}                                  // the arms that it chose timed a launch that is gone
extern "C" void omni_debug_bb_ar(int on) { g_bb_ar = on; }                  // 0: tensor-parallel ranks keep the launch-per-op backbone
extern "C" void omni_debug_bb_min_rows(int rows) { g_bb_min_rows = rows; g_bb_b32 = rows <= 49; }      // smallest batch of the 64-row split
#endif

// the instantiated shape triples (KO, KH, KI) = (q_heads * 128, hidden, intermediate) / 256: the released 1.7B shape and one no released
// checkpoint has (hidden 1536, intermediate 4608, 12 q heads: tests/test_gpu_chain.py, tests/test_gpu_engine.py); a new width = one more line
#define BB_SHAPES(X) X(8, 8, 24) X(6, 6, 18)
// ... and the triples of a tensor-parallel RANK (the all-reduce instantiations, full and half grid): the 1.7B shape whole (a one-rank group:
// bench.py --tp-force), over 2 ranks (8 q / 4 kv heads, intermediate 3072), over 4 and over the 8 GPUs of a node (2 q / 1 kv head, 768)
#define BB_AR_SHAPES(X) X(8, 8, 24) X(4, 8, 12) X(2, 8, 6) X(1, 8, 3)

// ar: the rank's peer table (NULL = not tensor parallel); half: the 128-workgroup grid (omni_talker_set_chains(t, 2))
bool k_bb_chain_supported(const omni_talker_desc& d, int B, const omni_ar_peers* ar, bool half) {
    static int cus = -1;
    if (cus < 0) {
        int dev = 0;
        hipDeviceProp_t p;
        cus = (hipGetDevice(&dev) == hipSuccess && hipGetDeviceProperties(&p, dev) == hipSuccess) ? p.multiProcessorCount : 0;
    }
    const bool has_ar = ar != nullptr;
    // a tensor-parallel rank: every peer's tile flags mapped (omni_ar_peers::tile_flags; a one-rank group exchanges nothing)
    bool ar_ok = has_ar && g_bb_ar;
    if (has_ar)
        for (int p = 0; p < ar->world; ++p) ar_ok = ar_ok && (ar->world == 1 || ar->tile_flags[p] != nullptr);
    const bool common = g_bb_chain && d.cp_chain && cus >= OMNI_CHAIN_WGS && d.fused_norm && d.frag_layout && (!has_ar || ar_ok) && d.moe_experts == 0 &&
                        d.head_dim == 128 && B <= 64;
    if (common && !has_ar && !half && k_bb_chain_small(d)) return B >= 1;      // 0.6B shape: 16-row tiles, every batch size
    const int H = d.hidden, I = d.inter, KOW = d.q_heads * 128, NQ = (d.q_heads + 2 * d.kv_heads) * 128;
    bool listed = false;
#define X(KO_, KH_, KI_) listed = listed || (KOW == KO_ * 256 && H == KH_ * 256 && I == KI_ * 256);
    if (has_ar) { BB_AR_SHAPES(X) }
    else if (half) { X(8, 8, 24) }
    else { BB_SHAPES(X) }
#undef X
    if (has_ar || half) return common && listed && I % 24 == 0 && NQ % 32 == 0 && B >= 33;      // the 64-row stage set only
    // every stage's tile grid inside the 256 workgroups: o_proj / down_proj 16 columns x 2 row tiles, gate_up 24 activation columns, qkv 32 x 2
    const bool grids = I % 24 == 0 && NQ % 32 == 0 && (H / 16) * 2 <= OMNI_CHAIN_WGS && I / 24 <= OMNI_CHAIN_WGS && (NQ / 32) * 2 <= OMNI_CHAIN_WGS;
    return common && listed && grids && (B >= g_bb_min_rows || (g_bb_b32 && B <= 32));
}
bool k_bb_chain_small(const omni_talker_desc& d) {
    return d.hidden == 1024 && d.inter == 3072 && d.q_heads * 128 == 2048 && (d.q_heads + 2 * d.kv_heads) * 128 == 4096;
}

// one shape's launches, by rows; the step's head rides along where the last layer's launch brings one
template <int KO, int KH, int KI, int ROWS, bool HEAD>
static int bb_launch_rows(const BbArgs& a, hipStream_t stream) {
    constexpr int bytes = bb_areas_wide(ROWS).total * 4;
    static const hipError_t attr = hipFuncSetAttribute((const void*)bb_flow_kernel<KO, KH, KI, ROWS, HEAD>, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    (void)attr;
    hipLaunchKernelGGL((bb_flow_kernel<KO, KH, KI, ROWS, HEAD>), dim3(OMNI_CHAIN_WGS), dim3(CH_THREADS), bytes, stream, a);
    OMNI_CHECK_LAUNCH("bb_flow");
    return OMNI_OK;
}
template <int KO, int KH, int KI>
static int bb_launch_shape(const BbArgs& a, int B, hipStream_t stream) {
    const bool head = a.lm_head != nullptr;
    if (B <= 16) return head ? bb_launch_rows<KO, KH, KI, 16, true>(a, stream) : bb_launch_rows<KO, KH, KI, 16, false>(a, stream);
    if (B <= 32) return head ? bb_launch_rows<KO, KH, KI, 32, true>(a, stream) : bb_launch_rows<KO, KH, KI, 32, false>(a, stream);
    return head ? bb_launch_rows<KO, KH, KI, 64, true>(a, stream) : bb_launch_rows<KO, KH, KI, 64, false>(a, stream);
}
template <int ROWS>
static int bb_launch_small(const BbArgs& a, hipStream_t stream) {
    constexpr int bytes = bb_areas_small(ROWS).total * 4;
    static const hipError_t attr = hipFuncSetAttribute((const void*)bb_flow_small_kernel<ROWS>, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    (void)attr;
    hipLaunchKernelGGL(bb_flow_small_kernel<ROWS>, dim3(OMNI_CHAIN_WGS), dim3(CH_THREADS), bytes, stream, a);
    OMNI_CHECK_LAUNCH("bb_flow_small");
    return OMNI_OK;
}

// the all-reduce / half-grid instantiations of one triple (64-row stage set)
template <int KO, int KH, int KI, bool HEAD, bool AR, bool HALF>
static int bb_launch_flags(const BbArgs& a, hipStream_t stream) {
    static const hipError_t attr = hipFuncSetAttribute((const void*)bb_chain_kernel<KO, KH, KI, HEAD, AR, HALF>, hipFuncAttributeMaxDynamicSharedMemorySize, BB_LDS_BYTES);
    (void)attr;
    hipLaunchKernelGGL((bb_chain_kernel<KO, KH, KI, HEAD, AR, HALF>), dim3(HALF ? OMNI_CHAIN_WGS / 2 : OMNI_CHAIN_WGS), dim3(CH_THREADS), BB_LDS_BYTES, stream, a);
    OMNI_CHECK_LAUNCH("bb_chain(all-reduce / half grid)");
    return OMNI_OK;
}
template <int KO, int KH, int KI>
static int bb_launch_ar(const BbArgs& a, bool half, hipStream_t stream) {
    if (half) return bb_launch_flags<KO, KH, KI, false, true, true>(a, stream);
    // a rank's last layer: the (replicated) lm_head as the launch's last stage
    return a.lm_head != nullptr ? bb_launch_flags<KO, KH, KI, true, true, false>(a, stream) : bb_launch_flags<KO, KH, KI, false, true, false>(a, stream);
}

static void bb_fill_ar(ChainAr& c, const omni_ar_peers& p) {
    c.world = p.world; c.rank = p.rank;
    const ptrdiff_t eoff = p.error - reinterpret_cast<int32_t*>(p.flags[p.rank]);      // the error word sits at the same offset in every rank's control block
    for (int r = 0; r < CH_AR_MAX_WORLD; ++r) {
        c.data[r] = r < p.world ? (const uint16_t*)p.data[r] : nullptr;
        c.tflags[r] = r < p.world ? p.tile_flags[r] : nullptr;
        c.error[r] = r < p.world ? (p.flags[r] ? reinterpret_cast<int32_t*>(p.flags[r]) + eoff : p.error) : nullptr;
    }
}

bool k_bb_chain_head_supported(const omni_talker_desc& d) {      // the lm_head stage's tile grid: 32 columns x 2 row tiles inside 256 workgroups
    return !k_bb_chain_small(d) && d.vocab % 32 == 0 && (d.vocab / 32) * 2 <= OMNI_CHAIN_WGS && d.lm_head != nullptr;
}

int k_bb_chain(const omni_talker_desc& d, const omni_layer_weights& w, const omni_layer_weights* next, const void* attn, void* resid, float* part,
               void* act, void* qkv, int B, float eps, uint32_t* flags, int32_t* err, void* stream, bool small, const omni_bb_head* head,
               const omni_bb_ar* ar, bool half, char* flow, int layer) {
    BbArgs a{};
    a.wo = (const uint16_t*)w.wo; a.ln2 = (const uint16_t*)w.ln2; a.wgu = (const uint16_t*)w.wgu; a.wdown = (const uint16_t*)w.wdown;
    a.ln1_next = next ? (const uint16_t*)next->ln1 : nullptr;
    a.wqkv_next = next ? (const uint16_t*)next->wqkv : nullptr;
    a.attn = (const uint16_t*)attn; a.resid = (uint16_t*)resid; a.part = part; a.act = (uint16_t*)act; a.qkv = (uint16_t*)qkv;
    a.H = d.hidden; a.I = d.inter; a.NQ = (d.q_heads + 2 * d.kv_heads) * 128;
    a.B = B; a.eps = eps; a.flags = flags; a.err = err;
    if (head != nullptr && next == nullptr && !small) {
        a.lm_head = (const uint16_t*)d.lm_head; a.final_norm = (const uint16_t*)d.final_norm; a.logits = head->logits; a.V = d.vocab;
        a.last_hidden = (uint16_t*)head->last_hidden; a.mask = (const uint8_t*)d.allowed_mask; a.mask_fill = head->mask_fill; a.num_live = head->num_live;
    }
#ifdef OMNI_DEBUG_HOOKS
    a.stamps = g_bb_stamps;
#endif
    if (flow != nullptr) {
        const size_t copy = BbFlowMap(a.H, a.I).copy;
        a.flow = flow + (layer & 1) * copy;
        a.flow_next = next ? flow + ((layer + 1) & 1) * copy : nullptr;
        a.first = layer == 0;
    }
    if (small) {
        if (B <= 16) return bb_launch_small<16>(a, (hipStream_t)stream);
        if (B <= 32) return bb_launch_small<32>(a, (hipStream_t)stream);
        if (B <= 48) return bb_launch_small<48>(a, (hipStream_t)stream);
        return bb_launch_small<64>(a, (hipStream_t)stream);
    }
    const int ko = d.q_heads * 128 / 256, kh = d.hidden / 256, ki = d.inter / 256;
    if (ar != nullptr || half) {
        OMNI_CHECK_ARG(!small && B > 32 && (a.lm_head == nullptr || (ar != nullptr && !half)), "bb_chain: the all-reduce / half-grid launches are the 64-row stage set; the half grid has no head stage");
        if (ar != nullptr) {
            OMNI_CHECK_ARG(ar->attn && ar->mlp && ar->attn->epoch == ar->mlp->epoch, "bb_chain: the two all-reduces share one epoch word");
            bb_fill_ar(a.ar_o, *ar->attn);
            bb_fill_ar(a.ar_dn, *ar->mlp);
            a.ar_epoch = ar->attn->epoch;
#define X(KO_, KH_, KI_) if (ko == KO_ && kh == KH_ && ki == KI_) return bb_launch_ar<KO_, KH_, KI_>(a, half, (hipStream_t)stream);
            BB_AR_SHAPES(X)
#undef X
        } else if (ko == 8 && kh == 8 && ki == 24) {
            return bb_launch_flags<8, 8, 24, false, false, true>(a, (hipStream_t)stream);
        }
        omni_set_error("bb_chain: no all-reduce / half-grid stage set for (q width, hidden, intermediate) = (%d, %d, %d)", d.q_heads * 128, d.hidden, d.inter);
        return OMNI_EINVAL;
    }
#define X(KO_, KH_, KI_) if (ko == KO_ && kh == KH_ && ki == KI_) return bb_launch_shape<KO_, KH_, KI_>(a, B, (hipStream_t)stream);
    BB_SHAPES(X)
#undef X
    omni_set_error("bb_chain: no stage set for (q width, hidden, intermediate) = (%d, %d, %d)", d.q_heads * 128, d.hidden, d.inter);
    return OMNI_EINVAL;
}
