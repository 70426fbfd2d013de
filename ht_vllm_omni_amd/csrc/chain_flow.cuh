// Hand-offs between the stages of a persistent launch in which the DATA is the flag (cp_chain.hip: the code predictor; bb_chain.hip: the
// backbone's layer segment).
//
// The flag protocol of coherent.cuh puts five dependent trips between a stage's last store and its successor's first MFMA: the stores'
// drain, a workgroup barrier, the flag's write-through, a poll that sees it, another barrier, and only then the activations' own fetch
// (3.1 us a stage of which the arithmetic is 0.3).  Here an output buffer is EMPTY (every 32-bit word FLOW_EMPTY) before its producers write
// it, and a consumer wave loads the very bytes it needs until none of their words is EMPTY: no drain, no flag, no barrier in front of the
// arithmetic, and a wave waits for its own operands only.
//
// Contract:
//   words     a producer never stores the word FLOW_EMPTY (flow_word turns it into another NaN payload: two bf16 NaNs, or an fp32 NaN); a
//             store is whole aligned words, so a word is either EMPTY or final
//   copies    every buffer exists FLOW_COPIES = 3 times; use number c of it (a layer, or a pass) goes to copy c % 3
//   clearing  when a workgroup enters a stage for use c it stores EMPTY over its own tile of copy (c + 1) % 3, and its outputs of use c go out
//             behind a barrier in front of which every wave has waited for all of its memory operations.  So
//               - who clears copy (c + 1) % 3, last used at c - 2, has finished use c - 1 of the same stage, i.e. has seen inputs that depend
//                 on every reader of use c - 2: nobody still reads what is cleared;
//               - who polls use c + 1 has seen use c of the same tiles before, whose stores came behind the clearing: it never meets the
//                 bytes of use c - 2.
//             The first polls of a launch wait once for all workgroups' flags: each has cleared its tiles of all three copies by then.
//             (A launch that uses each buffer once needs two copies: it clears the one that the launch behind it will use: bb_chain.hip.)
//   order     loads and stores of handed-off bytes carry sc1 (coherent.cuh): a completed store is what every later load returns
//   end       a wait is bounded by wall clock (coherent.cuh) and by the launch's error word: a wave that gives up records its stage code and
//             never waits again; the launch runs to its end on whatever it has loaded
#pragma once
#include "chain_gemm.cuh"

#define FLOW_EMPTY 0xffffffffu
#define FLOW_COPIES 3

__device__ __forceinline__ uint32_t flow_word(uint32_t w) { return w == FLOW_EMPTY ? FLOW_EMPTY - 1u : w; }
__device__ __forceinline__ uint32_t flow_max(u32x4 v) { return max(max(v[0], v[1]), max(v[2], v[3])); }
__device__ __forceinline__ void flow_clear16(coh_rsrc_t rs, uint32_t off) { coh_st16(rs, off, (u32x4){FLOW_EMPTY, FLOW_EMPTY, FLOW_EMPTY, FLOW_EMPTY}); }

// A wave that does not wait (any more) takes 0 for a word that is EMPTY, so a step that is thrown away computes on zeros and not on NaNs.  Nothing depends
// on it: what such a step leaves in a cache is written again before it is read
__device__ __forceinline__ uint32_t flow_or0(uint32_t w) { return w == FLOW_EMPTY ? 0u : w; }
__device__ __forceinline__ float flow_or0(float w) { return __uint_as_float(flow_or0(__float_as_uint(w))); }
struct FlowWait {
    int32_t* err;
    int dead;              // this wave gave up once (or the launch began with the error word set); wave-uniform
    int calm;              // looks further apart (constant: a launch's split of its stages)
};
__device__ __forceinline__ int flow_failed(const int32_t* err) {
    return __builtin_amdgcn_readfirstlane(__hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) != 0;
}
// another look at the operands is due: false = carry on with what is there.  (Looks at lines nobody has written since are served by the XCD's
// own L2.  The predictor's launch, pauses of 0 / 64 / 128 / 256 / 384 clocks: 64 rows 2807 / 2810 / 2781 / 2770 / 2785 us a step, 5 rows 1719 / 1717 / 1719 / 1722 and,
// on another card, 1697 / 1700 / 1705 (128 / 256 / 384): twice as long above 32 rows, where every workgroup waits in every stage.  That is little, and in every one of
// twelve pairs of runs: 64 rows 2779 -> 2776, 44 rows 2596 -> 2591, 40 rows of the 0.6B talker 2201 -> 2198, 64 rows 2298 -> 2289, runs of one side within 3 us
// (profiles/talker_step_sweeps.txt).  The backbone's layers: no difference.)
__device__ __forceinline__ bool flow_again(FlowWait& f, int code, unsigned& spins, unsigned long long& t0) {
    if (f.dead) return false;
    if (f.calm) __builtin_amdgcn_s_sleep(4);
    else __builtin_amdgcn_s_sleep(2);
    if (chain_wait_expired(++spins, t0)) {
        if ((threadIdx.x & 63) == 0) atomicCAS(f.err, 0, code);
        f.dead = 1;
    } else if ((spins & 1023u) == 0) {
        f.dead = flow_failed(f.err);
    }
    if (f.dead) return false;
    asm volatile("" ::: "memory");        // the operand loads are plain reads to the compiler: they stay inside the loop
    return true;
}
// every wave waits for all of its memory operations (contract: clearing), then the workgroup meets
__device__ __forceinline__ void flow_barrier() { asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// ---- LDS of a combine: one 1 KB block per (wave, tile) + the waves' row statistics; two of them alternate from stage to stage, so that a
// wave may write stage s + 1's partial sums while others still read stage s's (one barrier a stage).
// A block holds the 16 x 16 sums by rows, the four 16-byte pieces of a row turned by row / 4: writes (a lane = 4 columns of a row) and reads
// (a lane = 2 or 4 columns) meet no bank twice.
#define FLOW_TILES 6
#define FLOW_HALF_FLOATS (CH_WAVES * FLOW_TILES * 256 + CH_WAVES * 64)
__device__ __forceinline__ int flow_slot(int row, int piece) { return (row * 4 + (piece ^ ((row >> 2) & 3))) * 4; }        // in floats

// a later stage's weight slice, asked for ahead of it
template <int NT, int NTW>
__device__ __forceinline__ void flow_ask(const uint16_t* W, int bx, u32x4 (&Wq)[NTW][NT]) {
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));      // opaque per call (flow_gemm)
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const coh_rsrc_t rs = coh_rsrc(W);
#pragma unroll
    for (int d = 0; d < NTW; ++d)
#pragma unroll
        for (int j = 0; j < NT; ++j)
            Wq[d][j] = __builtin_amdgcn_raw_buffer_load_b128(rs, (tid & 63) * 16, (uint32_t)(((bx * NT + j) * NTW * CH_WAVES + wave + d * CH_WAVES) * 1024), 0);
}

// One skinny-GEMM stage: chain_gemm's k-steps per wave, accumulation, combine order and rounding points (the launch path's bits), its x and
// slabs awaited by content.  x: fragment-major, 32-column k-steps; `x` / `part_in` / `out` / `part_out` lie in this use's copy (or, the launch's
// first input, in the plain buffers its predecessor filled: never EMPTY).  clr / clr_part: the same places in the copy to clear, NULL: none.
// Output layouts (a workgroup's tiles lie together, so that no line of them has two writers; the slabs' 64-byte groups of 16 rows share lines):
//   RESID, GU8    fragment-major
//   BF16          16 x 16 bf16 tiles, 512 B: tile t of row group r at (r * (N / 16) + t) * 512, rows of 32 B
//   F32_BF16RND   16 x 16 fp32 tiles, 1 KB:  tile t of row group r at (r * (N / 16) + t) * 1024, rows of 64 B
// res: the residual values of this thread's item (RESID: threads < 64 MT), kept in registers from one residual stage to the next
// G: k-steps of x in flight (0: the wave's whole share).  A ring looks for EMPTY words step by step, in front of the step's MFMAs
// WA: k-steps of weights that go out in front of the first look at the operands (0: all); the others go out behind the first k-steps of x
// WP: the weight slice is in Wp already (flow_ask)
// WAUX: cache policy of the weights
// PS: rows per slab of sums of squares
// pl: what leaves the launch, by plain stores (FlowPlain); ROWS: the output goes there only (BF16 / F32 rows)
struct FlowPlain {
    uint16_t* rows;                       // BF16: row-major output, row m at rows + m * ldo
    uint16_t* resid; float* part;         // RESID: the residual values themselves (fragment-major) and their slabs
    uint16_t* normed; const int32_t* num_live;        // PRO 2: the normalised rows below *num_live, row-major
    const uint8_t* mask; float mask_fill;             // F32: logit n is mask_fill where mask[n] == 0
};
template <int MT, int NT, int NTW, int PRO, int EPI, int G = 0, bool ROWS = false, int PS = 64, int WA = 0, int WAUX = 0, bool WP = false>
__device__ __forceinline__ void flow_gemm(const uint16_t* __restrict__ W, const uint16_t* __restrict__ norm_w, const void* x, const float* part_in,
                                          int np_in, void* out, float* part_out, void* clr, float* clr_part, int M, int N, float eps, int bx, int by,
                                          float* lds, u32x2& res, FlowWait& fw, int code, unsigned long long* stamps,
                                          bool given = false /* x and the slabs were there before the launch: taken as they are, whatever their words */,
                                          float* logits_rows = nullptr /* F32: also row-major, row m at logits_rows + m * ldo */, int ldo = 0,
                                          const FlowPlain pl = FlowPlain{}, const u32x4 (*Wp)[NT] = nullptr) {
    const int sidx = ((code & 255) >> 4) * 5 + (code & 15) - 1;
    constexpr bool NORM = PRO == 2 || PRO == 3 || PRO == 4, DEFER = PRO == 3 || PRO == 4, NW = PRO == 2 || PRO == 3;
    constexpr bool GU8 = EPI == OMNI_EPI_SILU_MUL_GU8, RESID = EPI == OMNI_EPI_RESID, F32 = EPI == OMNI_EPI_F32_BF16RND;
    constexpr int K = NTW * CH_WAVES * 32, nsteps = K / 32;
    static_assert(EPI == OMNI_EPI_BF16 || RESID || F32 || GU8, "flow_gemm: epilogue");
    constexpr int XG = (G == 0 || G > NTW) ? NTW : G;
    constexpr bool RING = XG < NTW;
    static_assert(NT * MT <= 12 && (!RESID || (NT == 1 && PRO == 0)), "flow_gemm: tiles");
    static_assert(!RING || PRO == 0 || PRO == 4, "flow_gemm: a ring's x is multiplied as it is");
    // opaque per stage: hipcc otherwise hoists every stage's lane-dependent offsets out of the caller's loops and keeps them in scratch
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int q = lane >> 4;
    const int m_base = by * (MT * 16);
    const int Mloc = min(M - m_base, MT * 16);
    const coh_rsrc_t xrs = coh_rsrc(x), ors = coh_rsrc(out), wrs = coh_rsrc(W), nrs = coh_rsrc(NW || RESID ? norm_w : W);
    const uint32_t lane16 = lane * 16;
    CH_STAMP(stamps, sidx, 0);                                           // 0: stage entered

    // ---- clear this workgroup's tiles of the next use
    constexpr int TB = GU8 ? 256 : (F32 ? 1024 : 512);                   // bytes of an output tile
    constexpr int TP16 = TB / 16;                                        // 16-byte pieces
    auto tile_off = [&](int i, int j) -> uint32_t {
        const int mt = (m_base >> 4) + i;
        if (GU8) return (uint32_t)(mt * (N >> 5) * 1024 + (bx * NT + j) * 256);            // fragment-major: 8 columns = 256 B of a 1 KB k-step
        if (RESID) return (uint32_t)(mt * (N >> 5) * 1024 + bx * 512);
        return (uint32_t)((mt * (N >> 4) + bx * NT + j) * TB);
    };
    if (clr != nullptr) {
        const coh_rsrc_t crs = coh_rsrc(clr);
        for (int it = tid; it < NT * MT * TP16; it += CH_THREADS) {
            const int t = it / TP16;
            flow_clear16(crs, tile_off(t % MT, t / MT) + (it % TP16) * 16);
        }
        if (RESID && tid >= 256 && tid < 256 + MT * 4) flow_clear16(coh_rsrc(clr_part), (uint32_t)(bx * PS + m_base + (tid - 256) * 4) * 4);
    }

    // ---- what does not depend on the predecessor: the weight slice, the norm weights
    u32x4 Wq[NTW][NT], NWq[NW ? NTW : 1];
    auto load_w = [&](int d0, int d1) {
#pragma unroll
        for (int d = d0; d < d1; ++d) {
            const int ks = wave + d * CH_WAVES;
#pragma unroll
            for (int j = 0; j < NT; ++j) Wq[d][j] = WP ? Wp[d][j] : __builtin_amdgcn_raw_buffer_load_b128(wrs, lane16, (uint32_t)(((bx * NT + j) * nsteps + ks) * 1024), WAUX);
            if (NW) NWq[d] = __builtin_amdgcn_raw_buffer_load_b128(nrs, q * 16, ks * 64, 0);
        }
    };
    load_w(0, WA > 0 ? WA : NTW);
    u32x2 nwn = (u32x2){0x3f803f80u, 0x3f803f80u};                       // RESID: the next norm's weights of this thread's columns (1: none)
    if (RESID && norm_w != nullptr) nwn = __builtin_amdgcn_raw_buffer_load_b64(nrs, (bx * 16 + 4 * q) * 2, 0, 0);
    CH_STAMP(stamps, sidx, 1);                                           // 1: weight loads issued

    // ---- the activations and slabs, until none of their words is EMPTY (rows past the batch: zeros, no load)
    constexpr int XROWS = MT * 16;
    typedef SlabOrder<XROWS> SO;
    float pv[SO::PE];
    u32x4 Xq[XG][MT];
    const coh_rsrc_t prs = coh_rsrc(NORM ? (const void*)part_in : x);
    const int prow = lane % XROWS, psub = lane / XROWS;
    const uint32_t poff = (uint32_t)(m_base + prow) * 4;
#pragma unroll
    for (int e = 0; e < SO::PE; ++e) pv[e] = 0.f;
#pragma unroll
    for (int d = 0; d < XG; ++d)
#pragma unroll
        for (int i = 0; i < MT; ++i) Xq[d][i] = (u32x4){0u, 0u, 0u, 0u};
    auto load_p = [&]() {
        if (prow < Mloc) {
#pragma unroll
            for (int e = 0; e < SO::PE; ++e) pv[e] = coh_ldf(prs, (uint32_t)(min(SO::index(wave, psub, e), np_in - 1) * (PS * 4)) + poff);
        }
    };
    auto load_x = [&](int d0, int d1) {
#pragma unroll
        for (int i = 0; i < MT; ++i)
            if (i * 16 + (lane & 15) < Mloc) {
#pragma unroll
                for (int d = d0; d < d1; ++d)
                    Xq[d % XG][i] = __builtin_amdgcn_raw_buffer_load_b128(xrs, lane16, (uint32_t)((((m_base >> 4) + i) * nsteps + wave + d * CH_WAVES) * 1024), OMNI_AUX_SC1);
            }
    };
    // Waiting looks at ONE line, the first of the wave's first k-step; when that has come, at everything.  Waiting eats the bandwidth of those who
    // still work, and every copy of a line in a waiting XCD's L2 has to go before the store that fills it is done.  A decode step of 64 / of 5
    // rows, us: all operands again and again 3540 / 2300, one k-step (8 lines) 3276 / 2122, two lines 3043 / 2110, one line 3007 / 2074
    auto peek = [&]() -> bool {
        uint32_t w = 0;
        if (lane < min(Mloc, 8)) w = coh_ld4(xrs, lane16 + (uint32_t)(((m_base >> 4) * nsteps + wave) * 1024));
        return __builtin_amdgcn_ballot_w64(w == FLOW_EMPTY) != 0;
    };
    unsigned spins = 0;
    unsigned long long t0 = 0;
    bool go = !given;
    while (go && peek()) go = flow_again(fw, code, spins, t0);
    CH_STAMP(stamps, sidx, 2);                                           // 2: something is there
    if (NORM) load_p();
    load_x(0, XG);
    if (WA > 0) load_w(WA, NTW);
    while (!RING && go) {
        uint32_t w = 0;
        if (NORM) {
#pragma unroll
            for (int e = 0; e < SO::PE; ++e) w = max(w, __float_as_uint(pv[e]));
        }
#pragma unroll
        for (int d = 0; d < XG; ++d)
#pragma unroll
            for (int i = 0; i < MT; ++i) w = max(w, flow_max(Xq[d][i]));
        if (__builtin_amdgcn_ballot_w64(w == FLOW_EMPTY) == 0 || !(go = flow_again(fw, code, spins, t0))) break;
        if (NORM) load_p();
        load_x(0, XG);
    }
    if (!RING && fw.dead) {                                                     // (see flow_or0)
#pragma unroll
        for (int e = 0; e < SO::PE; ++e) pv[e] = flow_or0(pv[e]);
#pragma unroll
        for (int d = 0; d < XG; ++d)
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int c = 0; c < 4; ++c) Xq[d][i][c] = flow_or0(Xq[d][i][c]);
    }
    CH_STAMP(stamps, sidx, 3);                                           // 3: operands complete (a ring: asked for)
    auto short_p = [&]() {               // slabs past the last one
#pragma unroll
        for (int e = 0; e < SO::PE; ++e)
            if (SO::index(wave, psub, e) >= np_in) pv[e] = 0.f;
    };
    if (NORM && !RING) short_p();
    float* red = lds + CH_WAVES * NT * MT * 256;
    float rstd[MT];
    if (PRO == 2) {
        red[wave * 64 + lane] = SO::reduce(pv);
        flow_barrier();
        float t = 0.f;
#pragma unroll
        for (int w = 0; w < CH_WAVES; ++w) t += red[w * 64 + lane];
        const float rl = 1.0f / sqrtf(t / (float)K + eps);
#pragma unroll
        for (int i = 0; i < MT; ++i) rstd[i] = __shfl(rl, i * 16 + (lane & 15), 64);
    }
    f32x4 acc[NT][MT];
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int i = 0; i < MT; ++i) acc[j][i] = (f32x4){0.f, 0.f, 0.f, 0.f};
    if constexpr (RING) {
#pragma unroll
        for (int d = 0; d < NTW; ++d) {
            u32x4 (&X)[MT] = Xq[d % XG];
            auto empty = [&]() -> bool {
                uint32_t w = 0;
#pragma unroll
                for (int i = 0; i < MT; ++i) w = max(w, flow_max(X[i]));
                return __builtin_amdgcn_ballot_w64(w == FLOW_EMPTY) != 0;
            };
            if (!given && empty()) {
                while (flow_again(fw, code, spins, t0)) {
                    load_x(d, d + 1);
                    if (!empty()) break;
                }
                if (fw.dead) {
#pragma unroll
                    for (int i = 0; i < MT; ++i)
#pragma unroll
                        for (int c = 0; c < 4; ++c) X[i][c] = flow_or0(X[i][c]);
                }
            }
#pragma unroll
            for (int j = 0; j < NT; ++j)
#pragma unroll
                for (int i = 0; i < MT; ++i) acc[j][i] = mfma16(Wq[d][j], X[i], acc[j][i]);
            if (d + XG < NTW) load_x(d + XG, d + XG + 1);
        }
        if (NORM) {
            for (;;) {
                uint32_t w = 0;
#pragma unroll
                for (int e = 0; e < SO::PE; ++e) w = max(w, __float_as_uint(pv[e]));
                if (given || __builtin_amdgcn_ballot_w64(w == FLOW_EMPTY) == 0 || !flow_again(fw, code, spins, t0)) break;
                load_p();
            }
            if (fw.dead) {
#pragma unroll
                for (int e = 0; e < SO::PE; ++e) pv[e] = flow_or0(pv[e]);
            }
            short_p();
        }
    } else {
#pragma unroll
    for (int d = 0; d < NTW; ++d) {
        u32x4 Xn[MT];
#pragma unroll
        for (int i = 0; i < MT; ++i) Xn[i] = PRO == 2 ? xnorm_frag(Xq[d][i], NWq[NW ? d : 0], rstd[i]) : (PRO == 3 ? xw_frag(Xq[d][i], NWq[NW ? d : 0]) : Xq[d][i]);
        if (PRO == 2 && pl.normed != nullptr && bx < CH_WAVES && wave == bx) {
            // k-steps bx, bx + 8, ... leave through workgroup column bx (gemm_skinny_kernel)
            const int live = pl.num_live ? min(*pl.num_live, M) - m_base : Mloc;
#pragma unroll
            for (int i = 0; i < MT; ++i)
                if (i * 16 + (lane & 15) < min(Mloc, live))
                    *reinterpret_cast<u32x4*>(pl.normed + (size_t)(m_base + i * 16 + (lane & 15)) * K + (wave + d * CH_WAVES) * 32 + 8 * q) = Xn[i];
        }
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int i = 0; i < MT; ++i) acc[j][i] = mfma16(Wq[d][j], Xn[i], acc[j][i]);
    }
    }
    if (DEFER) red[wave * 64 + lane] = SO::reduce(pv);
    const int wslot = flow_slot(lane & 15, q);
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int i = 0; i < MT; ++i) *reinterpret_cast<f32x4*>(lds + (wave * (NT * MT) + j * MT + i) * 256 + wslot) = acc[j][i];
    CH_STAMP(stamps, sidx, 4);                                           // 4: partials in LDS
    flow_barrier();
    CH_STAMP(stamps, sidx, 5);                                           // 5: combine barrier passed

    if constexpr (RESID) {
        // a thread = four columns of a row (the slab's order of additions); whole waves: rows past Mloc add into lanes nobody stores
        if (tid < MT * 64) {
            const int i = tid >> 6, r = lane & 15, ml = i * 16 + r;
            f32x4 v[CH_WAVES], sum = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int w = 0; w < CH_WAVES; ++w) v[w] = *reinterpret_cast<const f32x4*>(lds + (w * MT + i) * 256 + wslot);
            __builtin_amdgcn_sched_barrier(0);                           // all eight reads in flight (left alone, hipcc waits for each)
#pragma unroll
            for (int w = 0; w < CH_WAVES; ++w) sum += v[w];
            float rv[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) rv[e] = bfround(sum[e]);
            rv[0] = bfround(bf_lo(res[0]) + rv[0]); rv[1] = bfround(bf_hi(res[0]) + rv[1]);
            rv[2] = bfround(bf_lo(res[1]) + rv[2]); rv[3] = bfround(bf_hi(res[1]) + rv[3]);
            res = (u32x2){pack_bf2(rv[0], rv[1]), pack_bf2(rv[2], rv[3])};
            float ss = sq4_sum(rv[0], rv[1], rv[2], rv[3]);
            ss = xor32_sum(xor16_sum(ss));
            if (ml < Mloc && pl.resid != nullptr) {
                *reinterpret_cast<u32x2*>(reinterpret_cast<char*>(pl.resid) + tile_off(i, 0) + (q >> 1) * 256 + r * 16 + (q & 1) * 8) = res;
                if (lane < 16) pl.part[bx * PS + m_base + ml] = ss;
            }
            if (ml < Mloc && out != nullptr) {
                // what the next norm's product takes: bf16(w r) (gemm_frag.cuh xw_frag); the residual values themselves stay here
                const u32x2 o = (u32x2){flow_word(pack_bf2(bf_lo(res[0]) * bf_lo(nwn[0]), bf_hi(res[0]) * bf_hi(nwn[0]))),
                                        flow_word(pack_bf2(bf_lo(res[1]) * bf_lo(nwn[1]), bf_hi(res[1]) * bf_hi(nwn[1])))};
                coh_st8(ors, tile_off(i, 0) + (q >> 1) * 256 + r * 16 + (q & 1) * 8, o);
                if (lane < 16) coh_st4(coh_rsrc(part_out), (uint32_t)(bx * PS + m_base + ml) * 4, flow_word(__float_as_uint(ss)));
            }
        }
    } else {
        // a thread = two columns of a row, neighbouring threads neighbouring bytes of the tile
        constexpr int PER = GU8 ? 64 : 128;                              // threads per tile
        for (int it = tid; it < NT * MT * PER; it += CH_THREADS) {
            const int t = it / PER, k = it % PER;
            const int i = t % MT, j = t / MT;
            const int r = GU8 ? k >> 2 : k >> 3, c2 = GU8 ? k & 3 : k & 7;      // columns 2 c2, 2 c2 + 1 of row r
            const int ml = i * 16 + r;
            if (ml >= Mloc) continue;
            const int at = (j * MT + i) * 256 + flow_slot(r, c2 >> 1) + (c2 & 1) * 2;
            f32x2 v[CH_WAVES], v2[GU8 ? CH_WAVES : 1], sum = (f32x2){0.f, 0.f}, sum2 = (f32x2){0.f, 0.f};
            float rs[DEFER ? CH_WAVES : 1];
            const int at2 = GU8 ? (j * MT + i) * 256 + flow_slot(r, 2 + (c2 >> 1)) + (c2 & 1) * 2 : 0;
#pragma unroll
            for (int w = 0; w < CH_WAVES; ++w) {
                if (DEFER) rs[w] = red[w * 64 + ml];
                v[w] = *reinterpret_cast<const f32x2*>(lds + w * (NT * MT * 256) + at);
                if (GU8) v2[w] = *reinterpret_cast<const f32x2*>(lds + w * (NT * MT * 256) + at2);
            }
            __builtin_amdgcn_sched_barrier(0);                           // all reads in flight
#pragma unroll
            for (int w = 0; w < CH_WAVES; ++w) {
                sum += v[w];
                if (GU8) sum2 += v2[w];
            }
            if (DEFER) {
                float t_ = 0.f;
#pragma unroll
                for (int w = 0; w < CH_WAVES; ++w) t_ += rs[w];
                const float rl = 1.0f / sqrtf(t_ / (float)K + eps);
                sum *= rl;
                if (GU8) sum2 *= rl;
            }
            if (GU8) {
                coh_st4(ors, tile_off(i, j) + k * 4, flow_word(pack_bf2(silu_mul_bf16(sum[0], sum2[0]), silu_mul_bf16(sum[1], sum2[1]))));
            } else if (F32) {
                // logits: fp32 cells holding bf16-rounded values (the reference's bf16 head output)
                float y0 = bfround(sum[0]), y1 = bfround(sum[1]);
                if (ROWS && pl.mask != nullptr) {
                    const int n = (bx * NT + j) * 16 + 2 * c2;
                    if (!pl.mask[n]) y0 = pl.mask_fill;
                    if (!pl.mask[n + 1]) y1 = pl.mask_fill;
                }
                if (!ROWS) coh_st8(ors, tile_off(i, j) + k * 8, (u32x2){flow_word(__float_as_uint(y0)), flow_word(__float_as_uint(y1))});
                if (logits_rows != nullptr) *reinterpret_cast<f32x2*>(logits_rows + (size_t)(m_base + ml) * ldo + (bx * NT + j) * 16 + 2 * c2) = (f32x2){y0, y1};
            } else if (ROWS) {
                *reinterpret_cast<uint32_t*>(pl.rows + (size_t)(m_base + ml) * ldo + (bx * NT + j) * 16 + 2 * c2) = pack_bf2(sum[0], sum[1]);
            } else {
                coh_st4(ors, tile_off(i, j) + k * 4, flow_word(pack_bf2(sum[0], sum[1])));
            }
        }
    }
    CH_STAMP(stamps, sidx, 6);                                           // 6: stores issued
    CH_STAMP(stamps, sidx, 7);
}
