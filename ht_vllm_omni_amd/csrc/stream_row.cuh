// One row of the residual stream of a decoder-only language model, by 256 threads (include/omni_decoder.h omni_stream_rows): decoder_rows.hip writes it out,
// gemm_stream.hip multiplies it.  One arithmetic, the same bits in both.
#pragma once
#include "row_io.cuh"

#define DR_THREADS 256
#define DR_WAVES (DR_THREADS / 64)

// arguments that the launches of decoder_rows.hip and the products of gemm_stream.hip take alike
int omni_stream_rows_check(const omni_stream_rows* p);
int omni_latent_write_check(const omni_latent_write* p);

// sum over the 256 threads, result in every thread; `buf` alternates between calls so that one barrier per sum is enough
struct BlockSum {
    float* lds;      // [2][DR_WAVES]
    int flip;
    __device__ __forceinline__ float operator()(float v) {
        v = wave_sum(v);
        float* b = lds + flip * DR_WAVES;
        flip ^= 1;
        if ((threadIdx.x & 63) == 0) b[(threadIdx.x >> 6) % DR_WAVES] = v;
        __syncthreads();
        float t = 0.f;
#pragma unroll
        for (int w = 0; w < DR_WAVES; ++w) t += b[w];
        return t;
    }
};

// A thread's pieces of a row: piece c holds 4 values from (c * DR_THREADS + tid) * 4 on; threads past the row's end read its last piece.
template <typename E, int MAXC, bool SPLIT>
struct StreamRow {
    const omni_stream_rows& a;
    const int tid;
    BlockSum bsum;
    raw4<E> ywr[MAXC], mur[MAXC];
    struct Pieces {
        raw4<float> x[MAXC];
        slab_pieces<MAXC, SPLIT> y;
    };
    __device__ __forceinline__ int at(int c) const { return min((c * DR_THREADS + tid) * 4, a.wp - 4); }
    __device__ __forceinline__ bool in_row(int c) const { return (c * DR_THREADS + tid) * 4 < a.wp; }
    __device__ __forceinline__ void fetch(int t, Pieces& r) const {        // (without y: x again, not used)
        const float* x = a.x_in + (size_t)t * a.wp;
#pragma unroll
        for (int c = 0; c < MAXC; ++c) r.x[c].load(x + at(c));
        r.y.load(a.y ? a.y + (size_t)t * a.wp : x, a.y_slabs, a.y_stride, [&](int c) { return at(c); });
    }
    __device__ __forceinline__ void weights(bool shift) {
        const E* yw = reinterpret_cast<const E*>(a.y_w);
#pragma unroll
        for (int c = 0; c < MAXC; ++c) {
            if (yw) ywr[c].load(yw + at(c));
            if (shift) mur[c].load(reinterpret_cast<const E*>(a.mu) + at(c));
        }
    }
    __device__ __forceinline__ void embed(int t, float (&v)[MAXC][4]) const {      // the stream row of token t: its table row
        const E* table = reinterpret_cast<const E*>(a.table);
        const int id = a.ids[t];
        const bool ok = id >= 0 && id < a.vocab;
        raw4<E> r[MAXC];
#pragma unroll
        for (int c = 0; c < MAXC; ++c) r[c].load(table + (size_t)(ok ? id : 0) * a.wp + at(c));
#pragma unroll
        for (int c = 0; c < MAXC; ++c) {
            r[c].get(v[c]);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if (!ok || !in_row(c)) v[c][e] = 0.f;
                if (a.table_scale != 0.f) v[c][e] *= a.table_scale;
            }
        }
    }
    __device__ __forceinline__ void join(const Pieces& r, float (&v)[MAXC][4]) {   // ... or its row behind the sublayer that just ran
        float y[MAXC][4], ss = 0.f;
#pragma unroll
        for (int c = 0; c < MAXC; ++c) {
            r.x[c].get(v[c]);
            r.y.sum(c, a.y_slabs, y[c]);
            if (!in_row(c)) {
#pragma unroll
                for (int e = 0; e < 4; ++e) v[c][e] = y[c][e] = 0.f;
            }
        }
        if (!a.y) return;
        if (a.post) {                                      // the norm takes the sum, not the sublayer's output
#pragma unroll
            for (int c = 0; c < MAXC; ++c)
#pragma unroll
                for (int e = 0; e < 4; ++e) { y[c][e] = fmaf(a.alpha, v[c][e], y[c][e]); v[c][e] = 0.f; }
        }
#pragma unroll
        for (int c = 0; c < MAXC; ++c) ss += sq4_sum(y[c][0], y[c][1], y[c][2], y[c][3]);
        ss = bsum(ss);
        const float g = (a.y_w ? 1.0f : a.gain) / sqrtf(ss / (float)a.width + a.eps);
#pragma unroll
        for (int c = 0; c < MAXC; ++c) {
            if (a.y_w) {
                float w[4];
                ywr[c].get(w);
#pragma unroll
                for (int e = 0; e < 4; ++e) y[c][e] *= in_row(c) ? w[e] : 0.f;
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) v[c][e] = fmaf(y[c][e], g, v[c][e]);
        }
    }
    __device__ __forceinline__ void shifted_in(int row, float (&prev)[MAXC][4]) const {    // the row before a batch's first token of a sequence
        const float* st = a.state + (size_t)a.state_slot[row] * a.wp;
        raw4<float> r[MAXC];
#pragma unroll
        for (int c = 0; c < MAXC; ++c) r[c].load(st + at(c));
#pragma unroll
        for (int c = 0; c < MAXC; ++c) {
            r[c].get(prev[c]);
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (!in_row(c)) prev[c][e] = 0.f;
        }
    }
    __device__ __forceinline__ float final_factor(const float (&v)[MAXC][4]) {
        float ss = 0.f;
#pragma unroll
        for (int c = 0; c < MAXC; ++c) ss += sq4_sum(v[c][0], v[c][1], v[c][2], v[c][3]);
        return (a.final_w ? 1.0f : a.final_gain) / sqrtf(bsum(ss) / (float)a.width + a.eps);
    }
    // piece c of h
    __device__ __forceinline__ void operand(bool shift, int c, const float (&cur)[4], const float (&prev)[4], float rf, float (&h)[4]) const {
        if (shift) {
            float m[4];
            mur[c].get(m);
#pragma unroll
            for (int e = 0; e < 4; ++e) h[e] = fmaf(prev[e] - cur[e], m[e], cur[e]);
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) h[e] = a.use_final ? cur[e] * rf : cur[e];
            if (a.use_final && a.final_w) {
                float w[4];
                ld4<E>(reinterpret_cast<const E*>(a.final_w) + at(c), w);
#pragma unroll
                for (int e = 0; e < 4; ++e) h[e] *= w[e];
            }
        }
    }
};
