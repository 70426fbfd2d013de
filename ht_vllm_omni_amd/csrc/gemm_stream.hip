// Weight-streaming GEMM of the language models' decode step: out[M <= 64, N] = x[M, K] . W[N, K]^T, both operands fragment-major
// (common.cuh frag_off), every W byte read once.
//
// A workgroup owns NT 16-column tiles for all rows and 1 / S of K (grid.y = S); its 8 waves take the k-steps round-robin, P steps of W and x in
// flight each, and combine through LDS in a fixed order.  What bounds the op at 64 rows is not only W: every workgroup reads all of
// x for its K range, 64 rows against its 16 NT columns of W, so wide tiles with K split over workgroups move the fewest bytes through L2.  The
// S partial sums leave as fp32 slabs [S][M][N]; the row kernels that consume them (decoder_rows.hip) add them up in slab order.
// A row or a few (the language models' smallest steps) are made by the product itself (gemm_behind_kernel): what comes before it is a launch of its own
// otherwise, and a launch is most of what such a step waits for.
//   out kinds: fp32 slabs (S >= 1) | bf16 row- or fragment-major | the same through an activation (common.cuh), possibly times a row table
#include "common.cuh"
#include "gemm_frag.cuh"
#include "stream_row.cuh"

#define GS_WAVES 8
#define GS_THREADS (GS_WAVES * 64)
enum { GS_F32 = 0, GS_BF16 = 1, GS_ACT = 2 };

struct StreamArgs {
    const uint16_t* x; const uint16_t* W; void* out;
    int M, N, nsteps, split_steps, oshuf;
    float ap, an;
    int act;
    omni_row_table rt;
};

// the waves' sums added up in a fixed order, and out
template <int MT, int NT, int KIND>
__device__ __forceinline__ void gs_store(const StreamArgs& a, const f32x4* part, int m0) {
    for (int it = threadIdx.x; it < NT * MT * 64; it += GS_THREADS) {
        const int l = it & 63, f = it >> 6, j = f / MT, i = f - j * MT;
        const int m = (m0 + i) * 16 + (l & 15), n = (blockIdx.x * NT + j) * 16 + 4 * (l >> 4);
        if (m >= a.M) continue;
        f32x4 v = part[f * 64 + l];
#pragma unroll
        for (int w = 1; w < GS_WAVES; ++w) v += part[(w * (NT * MT) + f) * 64 + l];
        if (KIND == GS_F32) {
            *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(a.out) + ((size_t)blockIdx.y * a.M + m) * a.N + n) = v;
        } else {
            if (KIND == GS_ACT) {
                if (a.act == OMNI_ACT_XIELU) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[e] = xielu(v[e], a.ap, a.an);
                } else if (a.act == OMNI_ACT_RELU2) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[e] = relu2(v[e]);
                } else {
                    const int id = a.rt.ids[m];
                    uint2 z = make_uint2(0, 0);
                    if (id >= 0 && id < a.rt.rows) z = *reinterpret_cast<const uint2*>(reinterpret_cast<const uint16_t*>(a.rt.table) + (size_t)id * a.rt.ld + n);
                    v[0] = gelu_tanh(v[0]) * bf_lo(z.x); v[1] = gelu_tanh(v[1]) * bf_hi(z.x);
                    v[2] = gelu_tanh(v[2]) * bf_lo(z.y); v[3] = gelu_tanh(v[3]) * bf_hi(z.y);
                }
            }
            uint16_t* d = reinterpret_cast<uint16_t*>(a.out) + (a.oshuf ? frag_off(m, n, a.N) : (size_t)m * a.N + n);
            *reinterpret_cast<uint2*>(d) = make_uint2(pack_bf2(v[0], v[1]), pack_bf2(v[2], v[3]));
        }
    }}

// P: k-steps in flight per wave: 2 on a grid that fills the chip (4 measured the same or slower at 1 .. 64 rows).
// grid.z: groups of MT row tiles (more than one where the columns alone leave CUs idle)
template <int MT, int NT, int KIND, int P>
__global__ __launch_bounds__(GS_THREADS) void gemm_stream_kernel(const StreamArgs a) {
    extern __shared__ __attribute__((aligned(16))) f32x4 part[];      // [wave][NT * MT][lane]
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int k0 = blockIdx.y * a.split_steps, nk = min(a.split_steps, a.nsteps - k0);
    const int m0 = blockIdx.z * MT;
    const uint16_t* wp[NT];
    const uint16_t* xp[MT];
#pragma unroll
    for (int j = 0; j < NT; ++j) wp[j] = a.W + ((size_t)(blockIdx.x * NT + j) * a.nsteps + k0 + wave) * 512 + lane * 8;
#pragma unroll
    for (int i = 0; i < MT; ++i) xp[i] = a.x + ((size_t)min(m0 + i, ((a.M + 15) >> 4) - 1) * a.nsteps + k0 + wave) * 512 + lane * 8;      // row tiles past M: re-read, discarded
    f32x4 acc[NT][MT];
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int i = 0; i < MT; ++i) acc[j][i] = (f32x4){0.f, 0.f, 0.f, 0.f};
    const int mine = nk > wave ? (nk - wave + GS_WAVES - 1) / GS_WAVES : 0;
    u32x4 W[P][NT], X[P][MT];
    auto load = [&](int d, int s) {
#pragma unroll
        for (int j = 0; j < NT; ++j) W[d][j] = ld16_nt(wp[j] + (size_t)s * (GS_WAVES * 512));
#pragma unroll
        for (int i = 0; i < MT; ++i) X[d][i] = ld16(xp[i] + (size_t)s * (GS_WAVES * 512));
    };
    auto mul = [&](int d) {
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int i = 0; i < MT; ++i) acc[j][i] = mfma16(W[d][j], X[d][i], acc[j][i]);
    };
    int s = 0;
    if (mine >= P) {                       // whole groups of P steps: no predicated load, each product waits for its own operands only
#pragma unroll
        for (int d = 0; d < P; ++d) load(d, d);
        for (; s + 2 * P <= mine; s += P) {
#pragma unroll
            for (int d = 0; d < P; ++d) {
                mul(d);
                load(d, s + P + d);
            }
        }
#pragma unroll
        for (int d = 0; d < P; ++d) mul(d);
        s += P;
    }
    if (s < mine) {                        // fewer than P steps left
#pragma unroll
        for (int d = 0; d < P - 1; ++d)
            if (s + d < mine) load(d, s + d);
#pragma unroll
        for (int d = 0; d < P - 1; ++d)
            if (s + d < mine) mul(d);
    }
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int i = 0; i < MT; ++i) part[(wave * (NT * MT) + j * MT + i) * 64 + lane] = acc[j][i];
    __syncthreads();
    gs_store<MT, NT, KIND>(a, part, m0);
}

// ---- products whose operand rows every workgroup makes for itself, into LDS, two at a time by 256 threads each.  What bounds them is trips to memory, not
// bytes: the first weights are asked for behind the rows' own pieces and arrive while those are summed, and the launch in front (2.5 - 3.5 us of some 40
// a layer) is gone.  One workgroup (`writer`) leaves what others read later.  Us, a decode step of 8 layers, launches of their own / rows made by the
// product: Zefedra, 1024 wide, 1 row 330 / 280 (its latents and the merge of attention's splits among them: rows of the stream alone 301), 2 rows 334 / 286,
// 2048 wide 457 / 400 and 464 / 413; Koronex 323 / 277, 330 / 284, 440 / 407, 444 / 416.
// How many rows it takes: a third and a fourth are summed behind the first two, which costs what it saves where a row is wide (3 rows of 2048: Zefedra 463 / 479), and for
// latents always (4 rows 347 / 363).  Which products are given theirs: omni_gemm_stream_joins.
constexpr int gs_joined_rows(int maxc) { return maxc == 1 ? OMNI_STREAM_JOINED_ROWS : 2; }
template <int MAXC, bool SHIFT>
struct RowsPro {                                          // a row of the residual stream (decoder_rows.hip stream_rows_kernel)
    using Args = omni_stream_rows;
    template <typename F>
    static __device__ __forceinline__ void run(const Args& a, uint16_t* xs, float* red, bool writer, F meanwhile) {
        const int half = threadIdx.x / DR_THREADS;
        StreamRow<uint16_t, MAXC, true> sr{a, (int)threadIdx.x % DR_THREADS, BlockSum{red + half * 2 * DR_WAVES, 0}};
        constexpr int PASSES = gs_joined_rows(MAXC) / 2;
        using Pieces = typename StreamRow<uint16_t, MAXC, true>::Pieces;
        auto token = [&](int i0) { const int i = min(i0 + half, a.rows - 1); return a.sel ? a.sel[i] : i; };
        Pieces now[PASSES];                               // every row's, ahead of all sums
        if (!a.ids) {
            sr.fetch(token(0), now[0]);
#pragma unroll
            for (int p = 1; p < PASSES; ++p)
                if (2 * p < a.rows) sr.fetch(token(2 * p), now[p]);
        }
        sr.weights(SHIFT);
        meanwhile();
        bool behind = false;                              // (uniform: barriers follow) some row's predecessor is a row of this batch
        if (SHIFT)
            for (int u = 1; u < a.rows; ++u) behind |= a.row_of_tok[u] == a.row_of_tok[u - 1];
#pragma unroll
        for (int p = 0; p < PASSES; ++p) {
            if (2 * p >= a.rows) break;
            const int i = 2 * p + half, t = token(2 * p);
            float cur[MAXC][4], prev[MAXC][4];
#pragma unroll
            for (int c = 0; c < MAXC; ++c) prev[c][0] = prev[c][1] = prev[c][2] = prev[c][3] = 0.f;
            if (SHIFT) {
                const int row = a.row_of_tok[t];
                const bool first = t == 0 || a.row_of_tok[t - 1] != row;
                if (behind) {
                    if (a.ids) {
                        sr.embed(max(t - 1, 0), prev);
                    } else {
                        Pieces before;
                        sr.fetch(max(t - 1, 0), before);
                        sr.join(before, prev);
                    }
                }
                if (first) {
#pragma unroll
                    for (int c = 0; c < MAXC; ++c) prev[c][0] = prev[c][1] = prev[c][2] = prev[c][3] = 0.f;
                    if (a.positions[t] != 0) sr.shifted_in(row, prev);
                }
            }
            if (a.ids) sr.embed(t, cur);
            else sr.join(now[p], cur);
            const float rf = !SHIFT && a.use_final ? sr.final_factor(cur) : 0.f;
            if (i >= a.rows) continue;                    // (no barrier below)
#pragma unroll
            for (int c = 0; c < MAXC; ++c) {
                const int k = (c * DR_THREADS + sr.tid) * 4;
                if (k >= a.wp) continue;
                if (a.x_out && writer) st4<float>(a.x_out + (size_t)t * a.wp + k, cur[c]);
                float h[4];
                sr.operand(SHIFT, c, cur[c], prev[c], rf, h);
                st4<uint16_t>(xs + (size_t)i * a.wp + k, h);
            }
        }
    }
};
template <int MAXC>
struct LatentPro {                                        // a token's query latent; cache row, gates and state by the writer (decoder_rows.hip latent_write_kernel)
    using Args = omni_latent_write;
    template <typename F>
    static __device__ __forceinline__ void run(const Args& a, uint16_t* xs, float* red, bool writer, F meanwhile) {
        const int half = threadIdx.x / DR_THREADS, tid = threadIdx.x % DR_THREADS, wave = tid >> 6;
        const uint16_t* qw = reinterpret_cast<const uint16_t*>(a.qw);
        const uint16_t* kw = reinterpret_cast<const uint16_t*>(a.kw);
        const int cols = writer ? a.ld : a.qp, norms = writer ? a.qp + a.rp : a.qp;
        const int t = min(half, a.T - 1);
        const bool mine = half < a.T;
        slab_pieces<MAXC, true> z;
        z.load(a.proj + (size_t)t * a.ld, a.slabs, a.slab_stride, [&](int c) { return min((c * DR_THREADS + tid) * 4, cols - 4); });
        raw4<uint16_t> w[MAXC];
#pragma unroll
        for (int c = 0; c < MAXC; ++c) {
            const int k = min((c * DR_THREADS + tid) * 4, norms - 4);
            w[c].load(k < a.qp ? qw + k : kw + (k - a.qp));
        }
        meanwhile();
        const int row = a.row_of_tok[t], pos = a.positions[t];
        const bool live = writer && mine && (!a.num_live || row < *a.num_live);
        if (live && a.state && (t == a.T - 1 || a.row_of_tok[t + 1] != row)) {
            const size_t to = (size_t)a.state_slot[row] * a.wp;
            for (int k = tid * 4; k < a.wp; k += DR_THREADS * 4)
                *reinterpret_cast<float4*>(a.state + to + k) = *reinterpret_cast<const float4*>(a.x + (size_t)t * a.wp + k);
        }
        float v[MAXC][4], sq = 0.f, sk = 0.f;
#pragma unroll
        for (int c = 0; c < MAXC; ++c) {
            const int k = (c * DR_THREADS + tid) * 4;
            z.sum(c, a.slabs, v[c]);
            const float ss = sq4_sum(v[c][0], v[c][1], v[c][2], v[c][3]);
            if (k < a.qp) sq += ss;
            else if (k < norms) sk += ss;
        }
        sq = wave_sum(sq);
        sk = wave_sum(sk);
        float* b = red + half * 2 * DR_WAVES;
        if ((tid & 63) == 0) { b[wave] = sq; b[DR_WAVES + wave] = sk; }
        __syncthreads();
        sq = sk = 0.f;
#pragma unroll
        for (int u = 0; u < DR_WAVES; ++u) { sq += b[u]; sk += b[DR_WAVES + u]; }
        if (!mine) return;                                // (no barrier below)
        const float rq = 1.0f / sqrtf(sq / (float)a.q_rank + a.eps), rk = 1.0f / sqrtf(sk / (float)a.kv_rank + a.eps);
        uint16_t* dst = nullptr;
        if (live) dst = reinterpret_cast<uint16_t*>(a.cache) + ((size_t)a.block_table[(size_t)row * a.bt_stride + pos / a.block_size] * a.block_size + pos % a.block_size) * a.rp;
#pragma unroll
        for (int c = 0; c < MAXC; ++c) {
            const int k = (c * DR_THREADS + tid) * 4;
            if (k >= cols) continue;
            float g[4], o[4];
            w[c].get(g);
            const float n = k < a.qp ? rq : rk;
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = v[c][e] * n * g[e];
            if (k < a.qp) st4<uint16_t>(xs + (size_t)t * a.qp + k, o);
            else if (k < a.qp + a.rp) {
                if (dst) st4<uint16_t>(dst + (k - a.qp), o);
            } else if (a.gate) {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (k - a.qp - a.rp + e < a.heads) a.gate[(size_t)t * a.heads + (k - a.qp - a.rp + e)] = 1.0f / (1.0f + expf(-v[c][e]));
            }
        }
    }
};

template <int NT, int KIND, class PRO>
__global__ __launch_bounds__(GS_THREADS) void gemm_behind_kernel(const StreamArgs a, const typename PRO::Args pa) {
    extern __shared__ __attribute__((aligned(16))) f32x4 part[];      // [wave][NT][lane] | the operand rows
    __shared__ float red[2 * 2 * DR_WAVES];
    constexpr int P = 4;                                  // k-steps in flight: 1024 deep, all of a wave's
    uint16_t* xs = reinterpret_cast<uint16_t*>(part + GS_WAVES * NT * 64);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int k0 = blockIdx.y * a.split_steps, nk = min(a.split_steps, a.nsteps - k0), mine = nk > wave ? (nk - wave + GS_WAVES - 1) / GS_WAVES : 0;
    u32x4 W[P][NT];
    auto load = [&](int d, int s) {                       // (past the last step: that one again, not used)
        const int step = k0 + min(wave + s * GS_WAVES, nk - 1);
#pragma unroll
        for (int j = 0; j < NT; ++j) W[d][j] = ld16_nt(a.W + ((size_t)(blockIdx.x * NT + j) * a.nsteps + step) * 512 + lane * 8);
    };
    PRO::run(pa, xs, red, blockIdx.x == 0 && blockIdx.y == 0, [&]() {
#pragma unroll
        for (int d = 0; d < P; ++d) load(d, d);
    });
    __syncthreads();
    f32x4 acc[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[j] = (f32x4){0.f, 0.f, 0.f, 0.f};
    const uint16_t* xp = xs + (size_t)min(lane & 15, a.M - 1) * (a.nsteps * 32) + (k0 + wave) * 32 + 8 * (lane >> 4);      // (rows past M: the last one again, discarded)
    for (int s = 0; s < mine; s += P) {
#pragma unroll
        for (int d = 0; d < P; ++d) {
            if (s + d >= mine) break;
            const u32x4 X = *reinterpret_cast<const u32x4*>(xp + (size_t)(s + d) * (GS_WAVES * 32));
#pragma unroll
            for (int j = 0; j < NT; ++j) acc[j] = mfma16(W[d][j], X, acc[j]);
            if (s + d + P < mine) load(d, s + d + P);
        }
    }
#pragma unroll
    for (int j = 0; j < NT; ++j) part[(wave * NT + j) * 64 + lane] = acc[j];
    __syncthreads();
    gs_store<1, NT, KIND>(a, part, 0);
}

// Columns per workgroup and K splits.  At more than 32 rows a workgroup's registers and LDS leave room for one per CU, so a grid runs in rounds of 256; below,
// several share a CU and a further round costs three quarters of the first.  A workgroup's time goes with the operand tiles it reads per k-step (NT of W; of x,
// which is in L2, three quarters of MT) plus its epilogue, NT * MT sums of eight waves through LDS; a split also costs its reader.
// The numbers are a fit with all rows in a workgroup, over 1 ... 64 rows x the weight shapes of the language models; gs_run then deals rows out.  As launched, over 297 products
// out of HBM and every choice of columns, splits and rows, the reader of partial sums at 30 ns and 8 TB/s a slab, it is 1.3 % behind the best on average (the rule before,
// rounds, MT and splits in full and a fifth of the epilogue: 4.2 %); table: profiles/gemm_stream_sweep.txt.  Us, before / now, 8 rows, columns x K: 8192 x 2048 8.6 / 7.4 (4 column
// tiles in 2 splits / 2 in one), 5120 x 2048 6.1 / 5.6, 1024 x 2048 3.2 / 2.8.  Slower: 2064 columns, 129 tiles, at 17 - 32 rows, 4.2 / 4.5.
// As before: 9216 x 2048 by 3 (192 workgroups; by 2, 288 of them, 2 us more), 2048 x 9216 by 2 in 4 splits.
static void gs_policy(int M, int N, int nsteps, bool slabs, int* nt, int* splits) {
    const int tiles = N / 16, mt = M > 32 ? 4 : (M > 16 ? 2 : 1);
    long best = -1;
    for (int n = 1; n <= 4; ++n) {
        if (tiles % n) continue;
        for (int s = 1; s <= (slabs ? OMNI_STREAM_MAX_SPLITS : 1); ++s) {
            if (s > 1 && nsteps / s < GS_WAVES) break;
            const long rounds = ((long)tiles / n * s + 255) / 256, quarters = mt == 4 ? 4 * rounds : 1 + 3 * rounds;
            const long cost = quarters * ((4 * n + 3 * mt) * ((nsteps + s - 1) / s) + (mt == 4 ? 44 : 80) * n * mt) + (mt == 4 ? 0 : 128) * s;
            if (best < 0 || cost < best) { best = cost; *nt = n; *splits = s; }
        }
    }
}

template <int MT, int NT, int KIND, int P>
static int gs_launch(const StreamArgs& a, int splits, hipStream_t st) {
    constexpr int LDS = GS_WAVES * NT * MT * 1024;
    if (LDS > 64 * 1024) {
        static const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_stream_kernel<MT, NT, KIND, P>), hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
        if (e != hipSuccess) { omni_set_error("omni_gemm_stream: LDS attribute: %s", hipGetErrorString(e)); return OMNI_EHIP; }
    }
    hipLaunchKernelGGL((gemm_stream_kernel<MT, NT, KIND, P>), dim3(a.N / (16 * NT), splits, ((a.M + 15) / 16 + MT - 1) / MT), dim3(GS_THREADS), LDS, st, a);
    OMNI_CHECK_LAUNCH("omni_gemm_stream");
    return OMNI_OK;
}

extern "C" int omni_gemm_stream_splits(int M, int N, int K) {
    int nt, s;
    gs_policy(M, N, K / 32, true, &nt, &s);
    return s;
}

static int gs_run(StreamArgs a, int kind, bool one, hipStream_t st) {
    int nt, splits;
    gs_policy(a.M, a.N, a.nsteps, kind == GS_F32 && !one, &nt, &splits);
    a.split_steps = (a.nsteps + splits - 1) / splits;
    int mt = a.M > 32 ? 4 : (a.M > 16 ? 2 : 1);
    // Where the columns leave half of the CUs idle the rows are dealt out as well: a workgroup's time goes with the x it pulls through its CU, and W is read by the
    // second group out of a cache.  The same sums.  Us, rows x columns x K, all rows / dealt out: 64 x 2048 x 1536 6.1 / 4.6, 64 x 2048 x 768 4.1 / 3.6, 32 x 2048 x 1536
    // 4.7 / 4.0, 64 x 1024 x 256 2.7 / 2.4; beyond one round of 256 workgroups the other way round: 64 x 4608 x 1024 6.3 / 7.0, 32 x 9216 x 2048 11.0 / 15.0.
    while (mt > 1 && a.N / 16 / nt * splits * (((a.M + 15) / 16 + mt / 2 - 1) / (mt / 2)) <= 256) mt /= 2;
    // a narrow product (a side input's gate), more steps in flight
    if (a.N / 16 * splits <= 32) {
        if (kind == GS_F32) return gs_launch<1, 1, GS_F32, 4>(a, splits, st);
        return kind == GS_BF16 ? gs_launch<1, 1, GS_BF16, 4>(a, splits, st) : gs_launch<1, 1, GS_ACT, 4>(a, splits, st);
    }
#define GS(MT_, NT_, K_) if (mt == MT_ && nt == NT_ && kind == K_) return gs_launch<MT_, NT_, K_, 2>(a, splits, st);
#define GS_NT(NT_, K_) GS(1, NT_, K_) GS(2, NT_, K_) GS(4, NT_, K_)
#define GS_ALL(K_) GS_NT(1, K_) GS_NT(2, K_) GS_NT(3, K_) GS_NT(4, K_)
    GS_ALL(GS_F32) GS_ALL(GS_BF16) GS_ALL(GS_ACT)
    omni_set_error("omni_gemm_stream: no tile for M=%d N=%d", a.M, a.N);
    return OMNI_EINVAL;
}

#define GS_CHECK(name)                                                                                                                              \
    OMNI_CHECK_ARG(x && w && out, name ": null pointer");                                                                                           \
    OMNI_CHECK_ARG(M >= 1 && M <= 64 && N > 0 && N % 16 == 0 && K > 0 && K % 32 == 0, name ": M=%d (<= 64) N=%d (%% 16) K=%d (%% 32)", M, N, K);    \
    OMNI_CHECK_ARG(!out_frag || N % 32 == 0, name ": out_frag needs N %% 32 == 0 (N=%d)", N)

extern "C" int omni_gemm_stream(const void* x, const void* w, void* out, int M, int N, int K, int kind, int one, float act_p, float act_n, int out_frag, void* stream) {
    GS_CHECK("omni_gemm_stream");
    OMNI_CHECK_ARG(kind >= 0 && kind <= 3 && (!out_frag || kind != GS_F32), "omni_gemm_stream: kind=%d out_frag=%d", kind, out_frag);
    StreamArgs a{(const uint16_t*)x, (const uint16_t*)w, out, M, N, K / 32, 0, out_frag, act_p, act_n, kind == 3 ? OMNI_ACT_RELU2 : OMNI_ACT_XIELU, {}};
    return gs_run(a, kind == 3 ? (int)GS_ACT : kind, one != 0, (hipStream_t)stream);
}

extern "C" int omni_gemm_stream_rows(const void* x, const void* w, void* out, int M, int N, int K, const omni_row_table* rt, int out_frag, void* stream) {
    GS_CHECK("omni_gemm_stream_rows");
    OMNI_CHECK_ARG(rt && rt->table && rt->ids && rt->rows > 0 && rt->ld >= N && rt->ld % 4 == 0, "omni_gemm_stream_rows: table of %d rows, ld %d", rt ? rt->rows : 0, rt ? rt->ld : 0);
    StreamArgs a{(const uint16_t*)x, (const uint16_t*)w, out, M, N, K / 32, 0, out_frag, 0.f, 0.f, OMNI_ACT_GELU_MUL, *rt};
    return gs_run(a, GS_ACT, true, (hipStream_t)stream);
}

// ---- up to OMNI_STREAM_JOINED_ROWS rows: the product makes them
template <int KIND, class PRO>
static int gs_behind(StreamArgs a, bool one, const typename PRO::Args& pa, hipStream_t st) {
    int nt, splits;
    gs_policy(a.M, a.N, a.nsteps, KIND == GS_F32 && !one, &nt, &splits);
    a.split_steps = (a.nsteps + splits - 1) / splits;
    if (a.N / 16 * splits <= 32) nt = 1;
#define GS(NT_)                                                                                                                                     \
    if (nt == NT_) {                                                                                                                                \
        hipLaunchKernelGGL((gemm_behind_kernel<NT_, KIND, PRO>), dim3(a.N / (16 * NT_), splits), dim3(GS_THREADS), GS_WAVES * NT_ * 1024 + a.M * a.nsteps * 64, st, a, pa); \
        OMNI_CHECK_LAUNCH("omni_gemm_stream(behind)");                                                                                              \
        return OMNI_OK;                                                                                                                             \
    }
    GS(1) GS(2) GS(3) GS(4)
#undef GS
    return OMNI_EINVAL;
}

// Every workgroup makes the rows: what the launch in front costs is saved once, what the rows cost is paid by every round of workgroups -- and hidden behind the weights
// of the round before where a row is as wide as those are long.  Us, rows made by the product against launches of their own, behind four partial sums, a row or two: up to
// 256 workgroups -1.2 ... -2.5 at every width; 512 -0.3 ... -0.7 (widths to 640), -1 ... -2.5 (wider); 768 of one column tile -0.0 ... -0.6, of two and more +1.4 ... +2.6
// (256 to 512 wide); 2374 +12 ... +22 (to 384), +5.4 (512), +3.9 (640), +0.4 (768), -0.5 (896), -1.2 ... -3.1 (1024 to 2048).  With the token shift, whose state is one more
// trip: 192 -0.6 ... -1.2, 512 and 576 -0.9 ... +3.2.  Three and four rows: 256 workgroups 0 ... -1.2, 288 and more +0.3 ... +1.9; with the shift +0.2 ... +6.6.
extern "C" int omni_gemm_stream_joins(int rows, int wp, int N, int shift, int sums) {
    if (rows < 1 || wp < 32 || wp % 32 || wp > 2 * DR_THREADS * 4 || rows > gs_joined_rows(wp > DR_THREADS * 4 ? 2 : 1) || N < 16 || N % 16 || (shift && rows > 2)) return 0;
    int nt, splits;
    gs_policy(rows, N, wp / 32, sums != 0, &nt, &splits);
    if (N / 16 * splits <= 32) nt = 1;
    const int wgs = N / 16 / nt * splits;
    if (shift || rows > 2) return wgs <= 256;
    return wp > 768 || wgs <= (nt == 1 ? 768 : 512);
}

extern "C" int omni_gemm_stream_joined(const omni_stream_rows* r, const void* w, void* out, int N, int kind, int one, float act_p, float act_n, const omni_row_table* rt, int out_frag, void* stream) {
    OMNI_CHECK_ARG(r && w && out, "omni_gemm_stream_joined: null pointer");
    const int rc = omni_stream_rows_check(r);
    if (rc != OMNI_OK) return rc;
    OMNI_CHECK_ARG(r->elem == 0 && r->rows >= 1 && r->wp <= 2 * DR_THREADS * 4 && r->rows <= gs_joined_rows(r->wp > DR_THREADS * 4 ? 2 : 1), "omni_gemm_stream_joined: %d rows of %d (bf16, <= %d of <= %d)", r->rows, r->wp,
                   gs_joined_rows(r->wp > DR_THREADS * 4 ? 2 : 1), 2 * DR_THREADS * 4);
    OMNI_CHECK_ARG(N > 0 && N % 16 == 0 && (!out_frag || N % 32 == 0) && kind >= 0 && kind <= 3 && kind != GS_BF16 && (!out_frag || kind != GS_F32), "omni_gemm_stream_joined: N=%d kind=%d out_frag=%d", N, kind, out_frag);
    OMNI_CHECK_ARG(!rt || (kind != GS_F32 && rt->table && rt->ids && rt->rows > 0 && rt->ld >= N && rt->ld % 4 == 0), "omni_gemm_stream_joined: table");
    OMNI_CHECK_ARG(!r->mu || kind == GS_F32, "omni_gemm_stream_joined: shifted rows are multiplied into fp32");
    StreamArgs a{nullptr, (const uint16_t*)w, out, r->rows, N, r->wp / 32, 0, out_frag, act_p, act_n, rt ? OMNI_ACT_GELU_MUL : kind == 3 ? OMNI_ACT_RELU2 : OMNI_ACT_XIELU, rt ? *rt : omni_row_table{}};
    hipStream_t st = (hipStream_t)stream;
    const bool wide = r->wp > DR_THREADS * 4;
    if (kind != GS_F32) return wide ? gs_behind<GS_ACT, RowsPro<2, false>>(a, true, *r, st) : gs_behind<GS_ACT, RowsPro<1, false>>(a, true, *r, st);
    if (r->mu) return wide ? gs_behind<GS_F32, RowsPro<2, true>>(a, one, *r, st) : gs_behind<GS_F32, RowsPro<1, true>>(a, one, *r, st);
    return wide ? gs_behind<GS_F32, RowsPro<2, false>>(a, one, *r, st) : gs_behind<GS_F32, RowsPro<1, false>>(a, one, *r, st);
}

extern "C" int omni_gemm_stream_latents(const omni_latent_write* r, const void* w, void* out, int N, void* stream) {
    OMNI_CHECK_ARG(r && w && out, "omni_gemm_stream_latents: null pointer");
    const int rc = omni_latent_write_check(r);
    if (rc != OMNI_OK) return rc;
    OMNI_CHECK_ARG(r->elem == 0 && r->T >= 1 && r->T <= OMNI_STREAM_LATENT_ROWS && r->ld <= 3 * DR_THREADS * 4 && N > 0 && N % 16 == 0, "omni_gemm_stream_latents: %d rows of %d, N=%d (bf16, <= %d of <= %d)", r->T, r->ld, N,
                   OMNI_STREAM_LATENT_ROWS, 3 * DR_THREADS * 4);
    StreamArgs a{nullptr, (const uint16_t*)w, out, r->T, N, r->qp / 32, 0, 0, 0.f, 0.f, 0, {}};
    return r->ld > 2 * DR_THREADS * 4 ? gs_behind<GS_BF16, LatentPro<3>>(a, true, *r, (hipStream_t)stream) : gs_behind<GS_BF16, LatentPro<2>>(a, true, *r, (hipStream_t)stream);
}
