// Row-wise kernels of the decoder-only language models (include/omni_decoder.h): everything between two matrix products of a layer.
// The residual stream is fp32; norms, gates and the token-shift state are fp32; only matrix operands are rounded (once) to bf16.
#include "stream_row.cuh"

// A workgroup walks `strip` consecutive tokens so that the token shift finds the previous token's NEW stream row in registers; only the
// strip's first token rebuilds its predecessor (or reads it from the sequence's state, or takes zeros).
// At decode sizes a row is a chain of trips to memory, not of bytes: the row's pieces, its partial sums and the weights of the norm and the shift are all
// asked for before anything is waited for; lanes past the row's end read its last piece.  Measured over all kernels of this file: a Koronex decode step
// of 64 rows (8 layers, 33 of these launches) 719 -> 697 us, of 8 rows 389 -> 378; prompts of 6870 tokens 6960 -> 6880.
// SPLIT: y arrives as more than one partial sum.
template <typename E, int MAXC, bool SHIFT, bool SPLIT>
__global__ __launch_bounds__(DR_THREADS) void stream_rows_kernel(const omni_stream_rows a, int strip) {
    __shared__ float red[2 * DR_WAVES];
    StreamRow<E, MAXC, SPLIT> sr{a, (int)threadIdx.x, BlockSum{red, 0}};
    using Pieces = typename StreamRow<E, MAXC, SPLIT>::Pieces;
    E* h_out = reinterpret_cast<E*>(a.h_out);
    const int wp = a.wp;
    const int i0 = blockIdx.x * strip, i1 = min(i0 + strip, a.rows);
    float cur[MAXC][4], prev[MAXC][4];
    for (int i = i0; i < i1; ++i) {
        const int t = a.sel ? a.sel[i] : i;
        Pieces now;
        if (!a.ids) sr.fetch(t, now);
        if (i == i0) sr.weights(SHIFT);
        if (SHIFT) {
            const int row = a.row_of_tok[t];
            const bool first = t == 0 || a.row_of_tok[t - 1] != row;
            if (first) {
                if (a.positions[t] == 0) {                 // zeros; the slot of a sequence that begins may not be set yet
#pragma unroll
                    for (int c = 0; c < MAXC; ++c) prev[c][0] = prev[c][1] = prev[c][2] = prev[c][3] = 0.f;
                } else {
                    sr.shifted_in(row, prev);
                }
            } else if (i == i0) {
                if (a.ids) {
                    sr.embed(t - 1, prev);
                } else {
                    Pieces before;
                    sr.fetch(t - 1, before);
                    sr.join(before, prev);
                }
            } else {
#pragma unroll
                for (int c = 0; c < MAXC; ++c)
#pragma unroll
                    for (int e = 0; e < 4; ++e) prev[c][e] = cur[c][e];
            }
        }
        if (a.ids) sr.embed(t, cur);
        else sr.join(now, cur);
        const float rf = !SHIFT && a.use_final ? sr.final_factor(cur) : 0.f;
#pragma unroll
        for (int c = 0; c < MAXC; ++c) {
            const int k = (c * DR_THREADS + threadIdx.x) * 4;
            if (k >= wp) continue;
            if (a.x_out) st4<float>(a.x_out + (size_t)t * wp + k, cur[c]);
            if (!h_out) continue;
            float h[4];
            sr.operand(SHIFT, c, cur[c], prev[c], rf, h);
            st4<E>(h_out + (a.frag ? frag_off(i, k, wp) : (size_t)i * wp + k), h);
        }
    }
}

template <typename E, int MAXC>
static void stream_rows_launch(const omni_stream_rows& a, int strip, hipStream_t st) {
    const dim3 grid((a.rows + strip - 1) / strip), block(DR_THREADS);
    const bool split = a.y && a.y_slabs > 1;
    if (a.mu && split) hipLaunchKernelGGL((stream_rows_kernel<E, MAXC, true, true>), grid, block, 0, st, a, strip);
    else if (a.mu) hipLaunchKernelGGL((stream_rows_kernel<E, MAXC, true, false>), grid, block, 0, st, a, strip);
    else if (split) hipLaunchKernelGGL((stream_rows_kernel<E, MAXC, false, true>), grid, block, 0, st, a, strip);
    else hipLaunchKernelGGL((stream_rows_kernel<E, MAXC, false, false>), grid, block, 0, st, a, strip);
}

template <typename E>
static int stream_rows_pick(const omni_stream_rows& a, int strip, hipStream_t st) {
    const int chunks = (a.wp / 4 + DR_THREADS - 1) / DR_THREADS;
    if (chunks <= 1) stream_rows_launch<E, 1>(a, strip, st);
    else if (chunks <= 2) stream_rows_launch<E, 2>(a, strip, st);
    else if (chunks <= 4) stream_rows_launch<E, 4>(a, strip, st);
    else stream_rows_launch<E, 8>(a, strip, st);
    OMNI_CHECK_LAUNCH("omni_stream_rows");
    return OMNI_OK;
}

int omni_stream_rows_check(const omni_stream_rows* p) {
    OMNI_CHECK_ARG(p && (p->ids ? p->table != nullptr : p->x_in != nullptr), "omni_stream_rows: null pointer");
    const omni_stream_rows& a = *p;
    OMNI_CHECK_ARG(a.width > 0 && a.wp >= a.width && a.wp % 32 == 0 && a.wp <= DR_THREADS * 4 * 8, "omni_stream_rows: width=%d wp=%d (multiple of 32, <= 8192)", a.width, a.wp);
    OMNI_CHECK_ARG(a.y_slabs <= OMNI_STREAM_MAX_SPLITS, "omni_stream_rows: y_slabs=%d", a.y_slabs);
    OMNI_CHECK_ARG(a.elem == 0 || a.elem == 1, "omni_stream_rows: elem=%d", a.elem);
    OMNI_CHECK_ARG(!a.frag || a.elem == 0, "omni_stream_rows: fragment-major output is bf16");
    OMNI_CHECK_ARG(!a.mu || (a.state && a.state_slot && a.row_of_tok && a.positions && !a.sel && !a.use_final), "omni_stream_rows: token shift needs state, rows and positions, and no selection");
    OMNI_CHECK_ARG(!a.sel || !a.x_out, "omni_stream_rows: a selection writes h only");
    OMNI_CHECK_ARG(!a.post || (a.y && !a.ids), "omni_stream_rows: the norm behind the sum needs y");
    // (a strip's first token and the shift read rows of x_in that another workgroup may already have rewritten: never in place)
    OMNI_CHECK_ARG(a.x_out == nullptr || a.x_out != a.x_in, "omni_stream_rows: x_out must not be x_in");
    return OMNI_OK;
}

extern "C" int omni_stream_rows_run(const omni_stream_rows* p, void* stream) {
    const int rc = omni_stream_rows_check(p);
    if (rc != OMNI_OK) return rc;
    const omni_stream_rows& a = *p;
    OMNI_CHECK_ARG(a.x_out || a.h_out, "omni_stream_rows: null pointer");
    if (a.rows <= 0) return OMNI_OK;
    const int strip = a.mu && a.rows > 1024 ? 4 : 1;
    return a.elem ? stream_rows_pick<float>(a, strip, (hipStream_t)stream) : stream_rows_pick<uint16_t>(a, strip, (hipStream_t)stream);
}

// ---- latents: norms, cache write, gates, token-shift state.  One workgroup per token; as above, the row's
// pieces, both norms' weights and the row that becomes the state leave together.
// A new latent may go to a second place as well, where a prompt's latents lie side by side for the product that expands them: read back out of the pages by a
// launch of their own they cost 4 - 6 us a layer (forwards of 8 layers, 1024 wide: 65 tokens 420 / 381 us, 4 prompts of 60 498 / 449, 16 of up to 128 1047 / 1025).
struct LatentRows { void* rows; const int32_t* base; int from; };      // token t >= from of batch row b: row base[b] + its position
template <typename E, bool SPLIT>
__global__ __launch_bounds__(DR_THREADS) void latent_write_kernel(const omni_latent_write a, const LatentRows side) {
    extern __shared__ __attribute__((aligned(16))) float sp[];     // the token's projections, partial sums added up
    __shared__ float red[2][DR_WAVES];
    const int t = blockIdx.x;
    const int row = a.row_of_tok[t], pos = a.positions[t];
    const bool live = !a.num_live || row < *a.num_live;
    const int blk = a.block_table[(size_t)row * a.bt_stride + pos / a.block_size];
    const bool last = a.state && (t == a.T - 1 || a.row_of_tok[t + 1] != row);
    const int slot = a.state ? a.state_slot[row] : 0;
    E* const also = side.rows && t >= side.from ? reinterpret_cast<E*>(side.rows) + (size_t)(side.base[row] + pos) * a.rp : nullptr;
    const float* y = a.proj + (size_t)t * a.ld;
    const E* qw = reinterpret_cast<const E*>(a.qw);
    const E* kw = reinterpret_cast<const E*>(a.kw);
    float sq = 0.f, sk = 0.f;
    slab_pieces<2, SPLIT> z;
    auto ask = [&](int k0) { z.load(y, a.slabs, a.slab_stride, [&](int c) { return min(k0 + (c * DR_THREADS + (int)threadIdx.x) * 4, a.ld - 4); }); };
    ask(0);
    raw4<E> wq, wk;                                                // the weights of this thread's next columns
    wq.load(qw + min((int)threadIdx.x * 4, a.qp - 4));
    wk.load(kw + min((int)threadIdx.x * 4, a.rp - 4));
    if (last && live)
        for (int k0 = threadIdx.x * 4; k0 < a.wp; k0 += 2 * DR_THREADS * 4) {
            const int k1 = min(k0 + DR_THREADS * 4, a.wp - 4);     // (past the row: its last piece, once more)
            const float4 x0 = *reinterpret_cast<const float4*>(a.x + (size_t)t * a.wp + k0), x1 = *reinterpret_cast<const float4*>(a.x + (size_t)t * a.wp + k1);
            *reinterpret_cast<float4*>(a.state + (size_t)slot * a.wp + k0) = x0;
            *reinterpret_cast<float4*>(a.state + (size_t)slot * a.wp + k1) = x1;
        }
    for (int k0 = 0; k0 < a.ld; k0 += 2 * DR_THREADS * 4) {
        if (k0 > 0) ask(k0);
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const int k = k0 + (c * DR_THREADS + (int)threadIdx.x) * 4;
            if (k >= a.ld) continue;
            float v[4];
            z.sum(c, a.slabs, v);
            st4<float>(sp + k, v);
            const float ss = sq4_sum(v[0], v[1], v[2], v[3]);      // (padded columns hold zeros; qp and rp are multiples of 4)
            if (k < a.qp) sq += ss;
            else if (k < a.qp + a.rp) sk += ss;
        }
    }
    sq = wave_sum(sq);
    sk = wave_sum(sk);
    if ((threadIdx.x & 63) == 0) { red[0][threadIdx.x >> 6] = sq; red[1][threadIdx.x >> 6] = sk; }
    __syncthreads();
    sq = sk = 0.f;
#pragma unroll
    for (int w = 0; w < DR_WAVES; ++w) { sq += red[0][w]; sk += red[1][w]; }
    const float rq = 1.0f / sqrtf(sq / (float)a.q_rank + a.eps), rk = 1.0f / sqrtf(sk / (float)a.kv_rank + a.eps);
    E* cq = reinterpret_cast<E*>(a.cq);
    for (int k = threadIdx.x * 4; k < a.qp; k += DR_THREADS * 4) {
        float v[4], w[4];
        wq.get(w);
        wq.load(qw + min(k + DR_THREADS * 4, a.qp - 4));
        ld4<float>(sp + k, v);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = v[e] * rq * w[e];
        st4<E>(cq + (a.frag ? frag_off(t, k, a.qp) : (size_t)t * a.qp + k), v);
    }
    if (a.gate)
        for (int h = threadIdx.x; h < a.heads; h += DR_THREADS) a.gate[(size_t)t * a.heads + h] = 1.0f / (1.0f + expf(-sp[a.qp + a.rp + h]));
    if (!live) return;
    E* dst = reinterpret_cast<E*>(a.cache) + ((size_t)blk * a.block_size + pos % a.block_size) * a.rp;
    for (int k = threadIdx.x * 4; k < a.rp; k += DR_THREADS * 4) {
        float v[4], w[4];
        wk.get(w);
        wk.load(kw + min(k + DR_THREADS * 4, a.rp - 4));
        ld4<float>(sp + a.qp + k, v);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = v[e] * rk * w[e];
        st4<E>(dst + k, v);
        if (also) st4<E>(also + k, v);
    }
}

int omni_latent_write_check(const omni_latent_write* p) {
    OMNI_CHECK_ARG(p && p->proj && p->qw && p->kw && p->cache && p->block_table && p->row_of_tok && p->positions, "omni_latent_write: null pointer");
    const omni_latent_write& a = *p;
    OMNI_CHECK_ARG(a.q_rank > 0 && a.kv_rank > 0 && a.qp >= a.q_rank && a.rp >= a.kv_rank && a.qp % 32 == 0 && a.rp % 32 == 0 && a.ld % 4 == 0 &&
                   a.ld >= a.qp + a.rp + (a.gate ? a.heads : 0), "omni_latent_write: q %d / %d, kv %d / %d, ld %d", a.q_rank, a.qp, a.kv_rank, a.rp, a.ld);
    OMNI_CHECK_ARG(a.block_size > 0 && a.bt_stride > 0 && a.heads > 0, "omni_latent_write: block_size=%d bt_stride=%d", a.block_size, a.bt_stride);
    OMNI_CHECK_ARG(!a.state || (a.x && a.state_slot && a.wp % 4 == 0), "omni_latent_write: state needs the stream rows and slots");
    OMNI_CHECK_ARG(a.elem == 1 || a.elem == 0, "omni_latent_write: elem=%d", a.elem);
    OMNI_CHECK_ARG(!a.frag || a.elem == 0, "omni_latent_write: fragment-major output is bf16");
    OMNI_CHECK_ARG(a.slabs <= OMNI_STREAM_MAX_SPLITS, "omni_latent_write: slabs=%d", a.slabs);
    return OMNI_OK;
}

static int latent_write(const omni_latent_write* p, const LatentRows& side, void* stream) {
    const int rc = omni_latent_write_check(p);
    if (rc != OMNI_OK) return rc;
    const omni_latent_write& a = *p;
    OMNI_CHECK_ARG(a.cq, "omni_latent_write: null pointer");
    OMNI_CHECK_ARG(a.ld <= 15 * 1024, "omni_latent_write: ld=%d (<= 15360: a token's projections are staged in LDS)", a.ld);
    if (a.T <= 0) return OMNI_OK;
    const size_t lds = (size_t)a.ld * sizeof(float);
    const dim3 grid(a.T), block(DR_THREADS);
    if (a.elem && a.slabs > 1) hipLaunchKernelGGL((latent_write_kernel<float, true>), grid, block, lds, (hipStream_t)stream, a, side);
    else if (a.elem) hipLaunchKernelGGL((latent_write_kernel<float, false>), grid, block, lds, (hipStream_t)stream, a, side);
    else if (a.slabs > 1) hipLaunchKernelGGL((latent_write_kernel<uint16_t, true>), grid, block, lds, (hipStream_t)stream, a, side);
    else hipLaunchKernelGGL((latent_write_kernel<uint16_t, false>), grid, block, lds, (hipStream_t)stream, a, side);
    OMNI_CHECK_LAUNCH("omni_latent_write");
    return OMNI_OK;
}

extern "C" int omni_latent_write_run(const omni_latent_write* p, void* stream) { return latent_write(p, LatentRows{}, stream); }

extern "C" int omni_latent_write_rows(const omni_latent_write* p, void* rows, const int32_t* row_base, int from, void* stream) {
    OMNI_CHECK_ARG(p && rows && row_base, "omni_latent_write_rows: null pointer");
    OMNI_CHECK_ARG(p->elem == 0 && from >= 0 && from <= p->T, "omni_latent_write_rows: elem=%d (bf16), rows from token %d of %d", p->elem, from, p->T);
    return latent_write(p, LatentRows{rows, row_base, from}, stream);
}

// ---- grouped attention: norms over whole projections, rotation, cache write, gate.  Three workgroups per token, by what they read: queries | keys and
// values | gate.  Queries and keys stay in LDS between the norm's sum and the rotation (a pair's other half belongs to another thread)
template <typename E, bool WIDE, bool SPLIT>           // WIDE: half a rotation is a multiple of 4, so 4 consecutive dimensions have 4 consecutive partners
__global__ __launch_bounds__(DR_THREADS) void qkv_write_kernel(const omni_qkv_write a) {
    extern __shared__ __attribute__((aligned(16))) float sp[];     // q or k of the token, partial sums added up
    __shared__ float red[DR_WAVES];
    const int t = blockIdx.x, part = blockIdx.y;
    const int nq = a.heads * a.dp, nk = a.kc ? a.kv_heads * a.dp : 0, nv = a.kc ? a.kv_heads * a.vp : 0, ng = a.heads * a.vp;
    const float* y = a.proj + (size_t)t * a.ld;
    auto ask = [&](slab_pieces<2, SPLIT>& z, const float* p, int k0, int n) {
        z.load(p, a.slabs, a.slab_stride, [&](int c) { return min(k0 + (c * DR_THREADS + (int)threadIdx.x) * 4, n - 4); });
    };
    if (part == 2) {
        for (int k0 = 0; k0 < ng; k0 += 2 * DR_THREADS * 4) {
            slab_pieces<2, SPLIT> z;
            ask(z, y + nq + nk + nv, k0, ng);
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                const int k = k0 + (c * DR_THREADS + (int)threadIdx.x) * 4;
                if (k >= ng) continue;
                float v[4];
                z.sum(c, a.slabs, v);
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = sigmoidf_(v[e]);
                st4<E>(reinterpret_cast<E*>(a.gate) + (size_t)t * ng + k, v);
            }
        }
        return;
    }
    const int row = a.row_of_tok[t], pos = a.positions[t];
    if (part == 1 && (!a.kc || (a.num_live && row >= *a.num_live))) return;
    // cache rows of this token: head g at base + g * block_size
    const size_t base = part ? (size_t)a.block_table[(size_t)row * a.bt_stride + pos / a.block_size] * a.kv_heads * a.block_size + pos % a.block_size : 0;
    const int n = part ? nk : nq, heads = part ? a.kv_heads : a.heads;
    const E* w = reinterpret_cast<const E*>(part ? a.kw : a.qw);
    if (part) y += nq;
    float ss = 0.f;
    slab_pieces<2, SPLIT> z;                           // the first pieces of q or k; v's leave behind them
    ask(z, y, 0, n);
    raw4<E> wn;                                        // the weights of this thread's next columns
    if (w) wn.load(w + min((int)threadIdx.x * 4, n - 4));
    if (part)
        for (int k0 = 0; k0 < nv; k0 += 2 * DR_THREADS * 4) {
            slab_pieces<2, SPLIT> zv;
            ask(zv, y + nk, k0, nv);
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                const int k = k0 + (c * DR_THREADS + (int)threadIdx.x) * 4;
                if (k >= nv) continue;
                float v[4];
                zv.sum(c, a.slabs, v);
                const int g = k / a.vp, d = k - g * a.vp;
                st4<E>(reinterpret_cast<E*>(a.vc) + (base + (size_t)g * a.block_size) * a.vp + d, v);
            }
        }
    for (int k0 = 0; k0 < n; k0 += 2 * DR_THREADS * 4) {
        if (k0 > 0) ask(z, y, k0, n);
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const int k = k0 + (c * DR_THREADS + (int)threadIdx.x) * 4;
            if (k >= n) continue;
            float v[4];
            z.sum(c, a.slabs, v);
            st4<float>(sp + k, v);
            ss += sq4_sum(v[0], v[1], v[2], v[3]);
        }
    }
    ss = wave_sum(ss);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
    __syncthreads();
    ss = 0.f;
#pragma unroll
    for (int i = 0; i < DR_WAVES; ++i) ss += red[i];
    const float r = w ? 1.0f / sqrtf(ss / (float)(heads * a.dim) + a.eps) : 1.0f;
    const int half = a.rot_dims >> 1;
    const float* cs = a.rot + (size_t)min(pos, a.rot_rows - 1) * a.rot_dims;
    for (int k = threadIdx.x * 4; k < n; k += DR_THREADS * 4) {
        const int hd = k / a.dp, d0 = k - hd * a.dp;
        float v[4], o[4] = {0.f, 0.f, 0.f, 0.f}, wv[4] = {1.f, 1.f, 1.f, 1.f};
        ld4<float>(sp + k, v);
        if (w) {
            wn.get(wv);
            wn.load(w + min(k + DR_THREADS * 4, n - 4));
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = v[e] * r * wv[e];
        if (d0 < a.rot_dims) {                         // (the vector may end past the rotated dimensions)
            float c[4] = {1.f, 1.f, 1.f, 1.f}, sn[4] = {0.f, 0.f, 0.f, 0.f};
            if constexpr (WIDE) {
                const bool lo = d0 < half;
                const int q = lo ? k + half : k - half;
                const float* p = cs + 2 * (lo ? d0 : d0 - half);
                ld4<float>(sp + q, o);
                float wo[4] = {1.f, 1.f, 1.f, 1.f}, z[4];
                if (w) ld4<E>(w + q, wo);
                ld4<float>(p, z);
                c[0] = z[0]; sn[0] = z[1]; c[1] = z[2]; sn[1] = z[3];
                ld4<float>(p + 4, z);
                c[2] = z[0]; sn[2] = z[1]; c[3] = z[2]; sn[3] = z[3];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    o[e] = o[e] * r * wo[e];
                    if (lo) o[e] = -o[e];
                }
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int d = d0 + e;
                    if (d >= a.rot_dims) continue;
                    const bool lo = d < half;
                    const int q = k + e + (lo ? half : -half);
                    float wo = 1.0f;
                    if (w) {
                        if constexpr (sizeof(E) == 4) wo = w[q];
                        else wo = bf2f(w[q]);
                    }
                    o[e] = sp[q] * r * wo;
                    if (lo) o[e] = -o[e];
                    const float2 f = *reinterpret_cast<const float2*>(cs + 2 * (lo ? d : d - half));
                    c[e] = f.x; sn[e] = f.y;
                }
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = fmaf(v[e], c[e], o[e] * sn[e]);
        }
        if (part) st4<E>(reinterpret_cast<E*>(a.kc) + (base + (size_t)hd * a.block_size) * a.dp + d0, v);
        else st4<E>(reinterpret_cast<E*>(a.q) + (size_t)t * nq + k, v);
    }
}

template <typename E, bool WIDE, bool SPLIT>
static int qkv_write_launch(const omni_qkv_write& a, size_t lds, hipStream_t st) {
    if (lds > 60 * 1024) {
        static const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(qkv_write_kernel<E, WIDE, SPLIT>), hipFuncAttributeMaxDynamicSharedMemorySize, 156 * 1024);
        if (e != hipSuccess) { omni_set_error("omni_qkv_write: LDS attribute: %s", hipGetErrorString(e)); return OMNI_EHIP; }
    }
    // parts in launch order: queries, (keys and values, of a layer with its own), (gate): a missing part in the middle starts and leaves
    const int parts = a.gate ? 3 : (a.kc ? 2 : 1);
    hipLaunchKernelGGL((qkv_write_kernel<E, WIDE, SPLIT>), dim3(a.T, parts), dim3(DR_THREADS), lds, st, a);
    OMNI_CHECK_LAUNCH("omni_qkv_write");
    return OMNI_OK;
}

extern "C" int omni_qkv_write_run(const omni_qkv_write* p, void* stream) {
    OMNI_CHECK_ARG(p && p->proj && p->q && p->row_of_tok && p->positions && (!p->kc == !p->vc), "omni_qkv_write: null pointer");
    const omni_qkv_write& a = *p;
    OMNI_CHECK_ARG(a.heads > 0 && a.kv_heads > 0 && a.heads % a.kv_heads == 0 && a.dim > 0 && a.dp >= a.dim && a.dp % 32 == 0 && a.vp > 0 && a.vp % 32 == 0,
                   "omni_qkv_write: heads %d / %d, dim %d / %d, vp %d", a.heads, a.kv_heads, a.dim, a.dp, a.vp);
    const int need = a.heads * a.dp + (a.kc ? a.kv_heads * (a.dp + a.vp) : 0) + (a.gate ? a.heads * a.vp : 0);
    OMNI_CHECK_ARG(a.ld >= need && a.ld % 4 == 0, "omni_qkv_write: ld=%d (>= %d)", a.ld, need);
    OMNI_CHECK_ARG(a.rot_dims >= 0 && a.rot_dims % 2 == 0 && a.rot_dims <= a.dim && (a.rot_dims == 0 || (a.rot && a.rot_rows > 0)), "omni_qkv_write: rot_dims=%d of %d", a.rot_dims, a.dim);
    OMNI_CHECK_ARG(!a.kc || (a.block_table && a.block_size > 0 && a.bt_stride > 0), "omni_qkv_write: block_size=%d bt_stride=%d", a.block_size, a.bt_stride);
    OMNI_CHECK_ARG(a.slabs <= OMNI_STREAM_MAX_SPLITS && (a.elem == 0 || a.elem == 1), "omni_qkv_write: slabs=%d elem=%d", a.slabs, a.elem);
    const size_t lds = (size_t)a.heads * a.dp * sizeof(float);      // (there are no more key heads than query heads)
    OMNI_CHECK_ARG(lds <= 156 * 1024, "omni_qkv_write: %d query heads of %d (a token's are staged in LDS)", a.heads, a.dp);
    if (a.T <= 0) return OMNI_OK;
    hipStream_t st = (hipStream_t)stream;
#define QKV(E_, W_) (a.slabs > 1 ? qkv_write_launch<E_, W_, true>(a, lds, st) : qkv_write_launch<E_, W_, false>(a, lds, st))
    if (a.rot_dims % 8 == 0) return a.elem ? QKV(float, true) : QKV(uint16_t, true);
    return a.elem ? QKV(float, false) : QKV(uint16_t, false);
#undef QKV
}

// ---- a recurrence's output: norm over all heads together, times the gate.  One workgroup per token
template <typename E, int MAXC>
__global__ __launch_bounds__(DR_THREADS) void gated_norm_kernel(const omni_gated_norm a) {
    __shared__ float red[2 * DR_WAVES];
    BlockSum bsum{red, 0};
    const int t = blockIdx.x;
    auto at = [&](int c) { return min((c * DR_THREADS + (int)threadIdx.x) * 4, a.n - 4); };
    auto in_row = [&](int c) { return (c * DR_THREADS + (int)threadIdx.x) * 4 < a.n; };
    raw4<float> o[MAXC];
    raw4<E> wr[MAXC];
#pragma unroll
    for (int c = 0; c < MAXC; ++c) {
        o[c].load(a.o + (size_t)t * a.n + at(c));
        wr[c].load(reinterpret_cast<const E*>(a.w) + at(c));
    }
    float v[MAXC][4], g[MAXC][4], ss = 0.f;
    if (a.slabs > 0) {
        slab_pieces<MAXC, true> z;
        z.load(reinterpret_cast<const float*>(a.gate) + (size_t)t * a.ld, a.slabs, a.slab_stride, at);
#pragma unroll
        for (int c = 0; c < MAXC; ++c) {
            z.sum(c, a.slabs, g[c]);
#pragma unroll
            for (int e = 0; e < 4; ++e) g[c][e] = 1.0f / (1.0f + expf(-g[c][e]));
        }
    } else {
        raw4<E> z[MAXC];
#pragma unroll
        for (int c = 0; c < MAXC; ++c) z[c].load(reinterpret_cast<const E*>(a.gate) + (size_t)t * a.ld + at(c));
#pragma unroll
        for (int c = 0; c < MAXC; ++c) z[c].get(g[c]);
    }
#pragma unroll
    for (int c = 0; c < MAXC; ++c) {
        o[c].get(v[c]);
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (!in_row(c)) v[c][e] = 0.f;
    }
#pragma unroll
    for (int c = 0; c < MAXC; ++c) ss += sq4_sum(v[c][0], v[c][1], v[c][2], v[c][3]);
    const float r = 1.0f / sqrtf(bsum(ss) / (float)a.count + a.eps);
#pragma unroll
    for (int c = 0; c < MAXC; ++c) {
        const int k = (c * DR_THREADS + threadIdx.x) * 4;
        if (k >= a.n) continue;
        float w[4];
        wr[c].get(w);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[c][e] = v[c][e] * r * w[e] * g[c][e];
        st4<E>(reinterpret_cast<E*>(a.out) + (a.frag ? frag_off(t, k, a.n) : (size_t)t * a.n + k), v[c]);
    }
}

template <typename E>
static void gated_norm_launch(const omni_gated_norm& a, hipStream_t st) {
    const int chunks = (a.n / 4 + DR_THREADS - 1) / DR_THREADS;
    const dim3 grid(a.T), block(DR_THREADS);
    if (chunks <= 1) hipLaunchKernelGGL((gated_norm_kernel<E, 1>), grid, block, 0, st, a);
    else if (chunks <= 2) hipLaunchKernelGGL((gated_norm_kernel<E, 2>), grid, block, 0, st, a);
    else if (chunks <= 4) hipLaunchKernelGGL((gated_norm_kernel<E, 4>), grid, block, 0, st, a);
    else hipLaunchKernelGGL((gated_norm_kernel<E, 8>), grid, block, 0, st, a);
}

extern "C" int omni_gated_norm_run(const omni_gated_norm* p, void* stream) {
    OMNI_CHECK_ARG(p && p->o && p->w && p->gate && p->out, "omni_gated_norm: null pointer");
    const omni_gated_norm& a = *p;
    OMNI_CHECK_ARG(a.n > 0 && a.n % 32 == 0 && a.n <= DR_THREADS * 4 * 8 && a.count > 0 && a.count <= a.n, "omni_gated_norm: n=%d (multiple of 32, <= 8192) count=%d", a.n, a.count);
    OMNI_CHECK_ARG(a.slabs >= 0 && a.slabs <= OMNI_STREAM_MAX_SPLITS && (a.elem == 0 || (a.elem == 1 && !a.frag)), "omni_gated_norm: slabs=%d elem=%d frag=%d", a.slabs, a.elem, a.frag);
    OMNI_CHECK_ARG(a.ld >= a.n && a.ld % 4 == 0, "omni_gated_norm: ld=%d", a.ld);
    if (a.T <= 0) return OMNI_OK;
    if (a.elem) gated_norm_launch<float>(a, (hipStream_t)stream);
    else gated_norm_launch<uint16_t>(a, (hipStream_t)stream);
    OMNI_CHECK_LAUNCH("omni_gated_norm");
    return OMNI_OK;
}
