// Causal grouped attention over a paged cache of keys and values, with an optional sliding window and an optional number per head in the softmax's
// denominator (include/omni_decoder.h omni_window_attn).  The heads that share a key / value head are query rows of one matrix problem, as all
// heads are in latent_attn.hip; the transposed-operand scheme and the three-term weights are the same (attn_tile.cuh):
//   S^T[key][row] = K . Q^T      A = K (lane (key, chunk qk): 8 dims), B = Q^T (registers for the whole kernel)
//   O^T[d][row]  += V^T . P^T    A = V^T: ds_read_b64_tr_b16 out of the row-major tile
// Scores, softmax statistics and weights are fp32.  Widths are run-time (dp, vp multiples of 32) below a compile-time bound WS; EX: both equal it.
//
//   window_decode_kernel   one token and one key / value head: up to 16 query heads fill the 16 rows.  Four waves score one 16-key tile each -- keys go
//                          from HBM straight into MFMA operands -- agree on the row maxima and share the second product by output columns.  Walks
//                          the window's tiles only; KV splits leave records a small kernel merges
//   window_prefill_kernel  up to wa_tile_rows() query rows (tokens x grouped heads) of one sequence, 16 per wave; the waves share each 32-key tile
//   window_plain_kernel    any width, bf16 or fp32: one wave per (token, head) on the vector units (the 32-bit mode)
#include "attn_tile.cuh"
#include "../../include/omni_decoder.h"

struct WinArgs {
    const uint16_t* q; const uint16_t* kc; const uint16_t* vc; const uint16_t* gate; const float* sink; uint16_t* out; int frag;
    const int32_t* block_table; int bt_stride, bs_shift, bs_mask;
    const int32_t* row_of_tok; const int32_t* positions; const int32_t* tiles;
    int heads, kv_heads, rep;       // rep = heads / kv_heads
    int ds, vs;                     // dp / 32, vp / 32
    float qs; int window;           // scale * log2(e); INT_MAX: no window
    float* partial; int nsplit;
    // prompt kernel: elements between blocks, rows of a block and key / value heads; rows of one array instead of pages; a gate per head
    int64_t k_block, v_block, k_head, v_head; int k_row, v_row;
    const int32_t* key_base; const float* head_gate;
};

// first key a token at `pos` sees
__device__ __forceinline__ int wa_first(int pos, int window) { return max(0, pos - window + 1); }

// 4 output columns [k, k + 4) of a token's row, times the gate
__device__ __forceinline__ void wa_store(const uint16_t* gate, uint16_t* out, int frag, size_t t, int k, int width, f32x4 v) {
    if (gate) {
        const uint2 g = *reinterpret_cast<const uint2*>(gate + t * width + k);
        v[0] *= bf_lo(g.x); v[1] *= bf_hi(g.x); v[2] *= bf_lo(g.y); v[3] *= bf_hi(g.y);
    }
    *reinterpret_cast<uint2*>(out + (frag ? frag_off((int)t, k, width) : t * width + k)) = make_uint2(pack_bf2(v[0], v[1]), pack_bf2(v[2], v[3]));
}

// The row's operand of q is asked for first and waited for before the loop, block ids ahead of the rows, and the next turn's pieces in the place of this
// turn's.  Us with the merge, 16 heads over 4 of 128, before / this: 64 rows of 1024 to 2048 keys 49.6 / 48.3, in windows of 1024 29.5 / 28.7; of 176 to 352
// 11.8 / 11.5; 48 of 352 to 704 18.8 / 18.3; one row of 352 8.4 either way; 8 heads over 2 of 64, 64 rows of up to 2048 18.1 / 17.8.  The same bits.
template <int WS, bool EX>
__global__ __launch_bounds__(64 * LA_DEC_WAVES, 2) void window_decode_kernel(const WinArgs a) {
    constexpr int DPW = (2 * WS + LA_DEC_WAVES - 1) / LA_DEC_WAVES;      // output column tiles of a wave: wave, wave + 4, ...
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];  // [wave] 16-key images of V | [pair][term][lane] weights
    __shared__ float sm[LA_DEC_WAVES][16], sl[LA_DEC_WAVES][16];
    const int ds = EX ? WS : a.ds, vs = EX ? WS : a.vs, dp = ds * 32, vp = vs * 32;
    const int pitch = vp * 2 + 32, himg = 16 * pitch;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int c = lane & 15, qk = lane >> 4;
    const int t = blockIdx.y, split = blockIdx.z;
    const int rt = (a.rep + 15) >> 4, g = blockIdx.x / rt;
    const int hr = (blockIdx.x - g * rt) * 16 + c, head = g * a.rep + min(hr, a.rep - 1);
    unsigned char* img = lds + wave * himg;
    u32x4* pw = reinterpret_cast<u32x4*>(lds + LA_DEC_WAVES * himg);
    const int pos = a.positions[t], len = pos + 1, lo = wa_first(pos, a.window);
    const int32_t* bt = a.block_table + (size_t)a.row_of_tok[t] * a.bt_stride;
    const int tl = lo >> 4, ntiles = (len + 15) / 16 - tl;
    const int nsplit = la_row_splits(ntiles, a.nsplit);
    if (split >= nsplit) return;
    const int t0 = tl + (int)((long long)ntiles * split / nsplit), t1 = tl + (int)((long long)ntiles * (split + 1) / nsplit);
    const int end = min(len, t1 * 16);                // keys of this split: [lo, end) from tile t0 on
    u32x4 Q[WS];
#pragma unroll
    for (int s = 0; s < WS; ++s)
        if (EX || s < ds) Q[s] = ld16(a.q + ((size_t)t * a.heads + head) * dp + 32 * s + 8 * qk);
    u32x4 K[WS], st[WS];                              // the wave's next tile: keys as operands, values on their way to LDS
    auto block_of = [&](int tile) { return bt[min(tile * 16 + c, len - 1) >> a.bs_shift]; };
    auto row_of = [&](int tile, int blk) {            // keys past the end: a valid row, masked below
        return ((size_t)(blk * a.kv_heads + g) << a.bs_shift) + (min(tile * 16 + c, len - 1) & a.bs_mask);
    };
    auto key_piece = [&](size_t row, int s) {         // lane (c, qk): 16-byte pieces qk, qk + 4, ... of key c's rows
        if (EX || s < ds) K[s] = ld16_nt(a.kc + row * dp + 32 * s + 8 * qk);
    };
    auto value_piece = [&](size_t row, int s) {
        if (EX || s < vs) st[s] = ld16_nt(a.vc + row * vp + 32 * s + 8 * qk);
    };
    const size_t row0 = row_of(t0 + wave, block_of(t0 + wave));
    int blk = block_of(t0 + wave + LA_DEC_WAVES);     // block ids are looked up a round ahead of the rows
#pragma unroll
    for (int s = 0; s < WS; ++s) key_piece(row0, s);
#pragma unroll
    for (int s = 0; s < WS; ++s) value_piece(row0, s);
    // waited for here: inside the loop the wait would be for what is in flight then
#pragma unroll
    for (int s = 0; s < WS; ++s)
        if (EX || s < ds) asm volatile("" : "+v"(Q[s]));
    f32x4 O[DPW];
#pragma unroll
    for (int i = 0; i < DPW; ++i) O[i] = (f32x4){0.f, 0.f, 0.f, 0.f};
    // m: common to the waves; l: this wave's keys.  The sink is a key without a value: it opens the first split's statistics
    const bool sink = a.sink && split == 0;
    float m = sink ? a.sink[head] * LA_LOG2E : LA_SENT, l = sink && wave == 0 ? 1.f : 0.f;
    for (int base = t0; base < t1; base += LA_DEC_WAVES) {
        const int key0 = (base + wave) * 16 + 4 * qk; // the lane's keys: key0 .. key0 + 3
        f32x4 S2[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
        auto score = [&](int s) { if (EX || s < ds) S2[s & 1] = mfma16(K[s], Q[s], S2[s & 1]); };
        auto keep = [&](int s) { if (EX || s < vs) *reinterpret_cast<u32x4*>(img + c * pitch + (32 * s + 8 * qk) * 2) = st[s]; };
        if (base + LA_DEC_WAVES < t1) {               // the next turn's pieces are asked for in the place of this one's
            const size_t row = row_of(base + wave + LA_DEC_WAVES, blk);
            blk = block_of(base + wave + 2 * LA_DEC_WAVES);      // (ahead of the rows: they are not waited for with it)
#pragma unroll
            for (int s = 0; s < WS; ++s) { score(s); key_piece(row, s); }
#pragma unroll
            for (int s = 0; s < WS; ++s) { keep(s); value_piece(row, s); }
        } else {
#pragma unroll
            for (int s = 0; s < WS; ++s) score(s);
#pragma unroll
            for (int s = 0; s < WS; ++s) keep(s);
        }
        const f32x4 S = S2[0] + S2[1];
        float sv[4], mx = LA_SENT;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            sv[j] = S[j] * a.qs;
            if (key0 + j >= lo && key0 + j < end) mx = fmaxf(mx, sv[j]);
        }
        mx = xor32_max(xor16_max(mx));
        if (qk == 0) sm[wave][c] = mx;
        __syncthreads();                              // maxima and images of this round
        float mn = m;
#pragma unroll
        for (int w = 0; w < LA_DEC_WAVES; ++w) mn = fmaxf(mn, sm[w][c]);
        const float alpha = exp2_w(m - mn);            // both the sentinel: 1, harmless (l = 0, O = 0)
        m = mn;
        float p[4], rs = 0.f;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            p[j] = key0 + j >= lo && key0 + j < end ? exp2_w(sv[j] - m) : 0.f;
            rs += p[j];
        }
        l = l * alpha + xor32_sum(xor16_sum(rs));
        u32x2 w3[3];                                  // three bf16 terms whose sum is the fp32 weight
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            uint32_t hi, mid, low;
            split3(p[2 * e], p[2 * e + 1], hi, mid, low);
            w3[0][e] = hi; w3[1][e] = mid; w3[2][e] = low;
        }
#pragma unroll
        for (int i = 0; i < 3; ++i) reinterpret_cast<u32x2*>(pw + ((wave >> 1) * 3 + i) * 64 + lane)[wave & 1] = w3[i];
#pragma unroll
        for (int i = 0; i < DPW; ++i) O[i] *= alpha;
        __syncthreads();                              // weights of this round
#pragma unroll
        for (int u = 0; u < LA_DEC_WAVES / 2; ++u) {
            if (base + 2 * u >= t1) break;            // (uniform; an image past t1 inside a pair holds valid rows with zero weights)
            u32x4 W[3], VT[DPW];
#pragma unroll
            for (int i = 0; i < 3; ++i) W[i] = pw[(u * 3 + i) * 64 + lane];
#pragma unroll
            for (int i = 0; i < DPW; ++i) VT[i] = la_transposed_at(lds + u * 2 * himg, pitch, min(wave + LA_DEC_WAVES * i, 2 * vs - 1), c, qk);
#pragma unroll
            for (int k = 2; k >= 0; --k)
#pragma unroll
                for (int i = 0; i < DPW; ++i) O[i] = mfma16(VT[i], W[k], O[i]);
        }
        if (base + LA_DEC_WAVES < t1) __syncthreads();      // the images are rewritten by the next round
    }
    if (qk == 0) sl[wave][c] = l;
    __syncthreads();
    float L = 0.f;
#pragma unroll
    for (int w = 0; w < LA_DEC_WAVES; ++w) L += sl[w][c];
    if (hr >= a.rep) return;
    float* rec = nsplit > 1 ? a.partial + (((size_t)t * a.heads + head) * a.nsplit + split) * (vp + 4) : nullptr;
    if (rec && wave == 0 && qk == 0) { rec[0] = m; rec[1] = L; }
    const float inv = L > 0.f ? 1.0f / L : 0.f;
#pragma unroll
    for (int i = 0; i < DPW; ++i) {
        const int d = wave + LA_DEC_WAVES * i;
        if (d >= 2 * vs) continue;
        if (rec) *reinterpret_cast<f32x4*>(rec + 4 + 16 * d + 4 * qk) = O[i];
        else wa_store(a.gate, a.out, a.frag, t, head * vp + 16 * d + 4 * qk, a.heads * vp, O[i] * inv);
    }
}

// KV splits of one (token, head): lane s holds split s's weight, every thread 4 columns
__global__ __launch_bounds__(64) void window_merge_kernel(const WinArgs a, int max_split) {
    const size_t rh = blockIdx.x;
    const int t = (int)(rh / a.heads), head = (int)(rh - (size_t)t * a.heads), vp = a.vs * 32;
    const int pos = a.positions[t];
    const int nsplit = la_row_splits((pos + 16) / 16 - (wa_first(pos, a.window) >> 4), max_split);
    if (nsplit == 1) return;                           // the decode kernel wrote the row
    const float* base = a.partial + rh * max_split * (vp + 4);
    const int lane = threadIdx.x, k = lane * 4;
    const float2 ml = lane < nsplit ? *reinterpret_cast<const float2*>(base + (size_t)lane * (vp + 4)) : make_float2(LA_SENT, 0.f);
    constexpr int S = 8;                               // that many records are asked for before the first is used: a step of 8 layers, 4 rows of 1000 keys 319 -> 308 us, 8 of 2048 358 -> 350
    f32x4 r[S];
#pragma unroll
    for (int s = 0; s < S; ++s) r[s] = *reinterpret_cast<const f32x4*>(base + (size_t)min(s, nsplit - 1) * (vp + 4) + 4 + min(k, vp - 4));
    const float M = wave_max(ml.x);
    const float w = lane < nsplit ? exp2_w(ml.x - M) : 0.f;
    const float L = wave_sum(ml.y * w);
    if (k >= vp) return;
    f32x4 v = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < S; ++s)
        if (s < nsplit) v += r[s] * __int_as_float(__builtin_amdgcn_readlane(__float_as_int(w), s));
#pragma unroll 4
    for (int s = S; s < nsplit; ++s)
        v += *reinterpret_cast<const f32x4*>(base + (size_t)s * (vp + 4) + 4 + k) * __int_as_float(__builtin_amdgcn_readlane(__float_as_int(w), s));
    wa_store(a.gate, a.out, a.frag, t, head * vp + k, a.heads * vp, v * (L > 0.f ? 1.0f / L : 0.f));
}

// Widths of exactly 32 WS (64, 128): keys and values go to LDS by LDS-DMA, and a wave owns TWO groups of 16 query rows.
// What bounds it: 16 rows x 32 keys of 128 dims are 8 + 24 MFMAs (512 cycles of the matrix pipe: the weights' three terms triple the second product), about
// as many cycles of softmax and splitting on the vector pipe, and 16 KB of LDS reads (128 cycles of the CU's, for each of four SIMDs).  Two
// groups share the LDS reads and are independent chains; without staging registers three waves of 168 fit a SIMD.
// A piece is 16 keys x 32 dims, row-major (a quad of lanes fetches 64 B of a key); three tiles in a ring, the one after the next in flight, one barrier a tile.
// The tiles of one key / value head run on one XCD: its keys and values come out of that L2.
// RG: groups of 16 rows a wave owns.  Two; one, with two workgroups to a tile, where the tiles are not more than the CUs: a wave's
// chain over the keys is then what a tile takes, and one group's is shorter.  Us, two groups / one, heads x keys' heads of 128: 16 x 4, 52 tiles of portions
// behind 512 tokens 30.4 / 19.9, 252 tiles (a prompt of 2000 in windows of 512) 30.5 / 27.7; 16 x 16, 256 tiles of 97 rows 11.2 / 9.9, 64 tiles behind 1000
// tokens 66 / 44.
// KT: teams of four waves that take the workgroup's 32-key steps in turn, each with a ring and running sums of its own; the first adds up.  Three, one
// workgroup to a CU, where the half tiles are no more than the CUs: a step is a chain of LDS reads, 8 + 24 MFMAs and the softmax between (0.85 us for one wave
// a SIMD, 1.6 for three in turn), and nothing else is there to fill its gaps.  Us, one team / three, heads x keys' heads of 128: 16 x 16, portions of 251 and 130
// tokens behind 512 26.3 / 18.8 (two: 19.9), 64 behind 1500 43.9 / 28.3 (31.7), a prompt of 1000 33.8 / 23.0 (24.6), of 300 12.8 / 11.0; 16 x 4, a prompt of 1000 31.3 /
// 22.3.  Up to WA_TEAM_KEYS keys the merge and the larger workgroups' start cost more: 16 x 4, 4 prompts of 96 7.7 / 8.3, of 128 8.5 / 9.2, of 160 9.7 / 10.2, of 176
// to 224 the same, of 256 12.7 / 12.2; where a batch's longest portion sees no more, one team is launched, and in other batches the first walks such a tile alone:
// the same sums either way.  Above 256 half tiles two workgroups of one team share a CU instead: 256 tiles of up to 128 tokens 9.4, by three teams in turns 15.8.
// Order.  An XCD deals its workgroups out in turn over its 32 CUs, three to a CU, and the tiles of a causal prompt are as long as the keys they see: by length
// the first CU gets the longest of each turn (one prompt of 6001 tokens, 47 tiles of 16 heads: 94 units of keys against 70 on average).  wa_deal orders the
// first turns so that what a CU gets adds up to the same (72).  Us a layer, that prompt, head after head 359, every head's tiles by length 312, dealt 304; one of 3000
// 147 / 139 / 136, of 2500 122 / 117 / 115; 16 x 4, by length / dealt, one of 6001 310 / 301, 24 of 128 15.6 / 14.0.
// The row's maximum is put together only where it moves: 312 -> 303 of that prompt, 16 x 4, 4 of up to 2048 99 -> 97.
// (Tried in the loop: blocks looked up by the scalar unit, 16 keys at a time -- 8 x 8 of 64, one of 3000, 66 -> 73 us, 16 x 4 of 128, one of 2048, 57 -> 60; the second product
// term by term over four column tiles: 0 to 3 % slower.)
// (The dealing is how an idle XCD was seen to go about it; another one costs time, never a result.)
__device__ __forceinline__ int wa_deal(int slot, int n) {                     // workgroup of an XCD -> rank by length among its n
    constexpr int C = 32;
    const int turn = slot / C, j = slot - turn * C, i = j >> 1;
    if (n <= C || turn >= 3) return slot;
    if (n <= 2 * C) return turn == 0 ? C - 1 - j : slot;                      // the shortest of the first turn get the longest of the second
    const int last = min(n - 2 * C, C);                                       // three turns: sums of three orders, 46 or 47 of 93 where all are full
    if (turn == 0) return j;
    if (turn == 1) return C + (j & 1 ? C - 1 - i : C / 2 - 1 - i);
    return 2 * C + (j & 1 ? last / 2 - 1 - i : last - 1 - i);
}

#define WA_TEAM_KEYS 160
template <int WS, int RG, int KT>
__global__ __launch_bounds__(256 * KT, KT == 1 ? 3 : KT) void window_prefill_dma_kernel(const WinArgs a, int n_tiles) {
    constexpr int WR = 16 * RG, PARTS = 2 / RG, HALF = WS * 1024, IMAGE = 4 * HALF, NB = 3, dp = 32 * WS;
    constexpr float LAZY = 8.0f;
    extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];     // [ring][keys 0-15 | keys 16-31 | values 0-15 | values 16-31][32-wide pieces]
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((threadIdx.x >> 6) & 3), team = KT == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
    const int c = lane & 15, qk = lane >> 4;
    int tile, g;
    {
        const int id = blockIdx.x, xcd = id & 7, slot = id >> 3, G = a.kv_heads;
        if (G % 8 == 0) { const int r = wa_deal(slot, n_tiles * (G / 8)); tile = r / (G / 8); g = (r - tile * (G / 8)) * 8 + xcd; }
        else if (8 % G == 0) { g = xcd % G; tile = wa_deal(slot, (int)gridDim.x >> 3) * (8 / G) + xcd / G; }
        else { g = id / n_tiles; tile = id - g * n_tiles; }
    }
    if (tile >= n_tiles || g >= a.kv_heads) return;
    const int part = tile % PARTS * 4 * WR;
    const int row0 = a.tiles[2 * (tile / PARTS)] + part, nrows = min(a.tiles[2 * (tile / PARTS) + 1] - part, 4 * WR);
    if (nrows <= 0) return;                                                  // (PARTS == 2: a tile of up to 64 rows)
    const int tok0 = row0 / a.rep, brow = a.row_of_tok[tok0];
    const int32_t* bt = a.block_table + (size_t)brow * a.bt_stride;
    const size_t first = a.key_base ? a.key_base[brow] : 0;                  // paged keys and values, or rows of one array
    int hi[RG], lo[RG];                                                      // keys a row sees: [lo, hi)
    u32x4 Q[RG][WS];
    f32x4 O[RG][2 * WS];
    float m[RG], l[RG];                                                      // l: this lane's share
#pragma unroll
    for (int rg = 0; rg < RG; ++rg) {
        const int r = wave * WR + 16 * rg + c, frow = row0 + min(r, nrows - 1), tok = frow / a.rep, head = g * a.rep + frow - tok * a.rep;
        const int pos = a.positions[tok];
        hi[rg] = r < nrows ? pos + 1 : 0;
        lo[rg] = wa_first(pos, a.window);
#pragma unroll
        for (int s = 0; s < WS; ++s) Q[rg][s] = ld16(a.q + ((size_t)tok * a.heads + head) * dp + 32 * s + 8 * qk);
#pragma unroll
        for (int d = 0; d < 2 * WS; ++d) O[rg][d] = (f32x4){0.f, 0.f, 0.f, 0.f};
        // a sink of -inf is none: the finite sentinel, against which a tile that holds no key of the row weighs nothing (of +inf: not a number, as its softmax)
        const float sink = a.sink && team == 0 ? a.sink[head] * LA_LOG2E : -INFINITY;
        m[rg] = sink < LA_SENT ? LA_SENT : (sink == INFINITY ? NAN : sink);
        l[rg] = sink < LA_SENT || qk != 0 ? 0.f : 1.f;
    }
    // keys the wave's rows see, the keys every one of them sees (no masks in a tile inside), and the tile's: positions grow along the rows
    const bool any = wave * WR < nrows;
    const int whi = any ? a.positions[(row0 + min(wave * WR + WR - 1, nrows - 1)) / a.rep] + 1 : 0;
    const int wfirst = any ? a.positions[(row0 + wave * WR) / a.rep] : 0;
    const int wlo = any ? wa_first(wfirst, a.window) : 0;
    const int fhi = wave * WR + WR <= nrows ? wfirst + 1 : 0, flo = wa_first(whi - 1, a.window);
    const int nkeys = a.positions[(row0 + nrows - 1) / a.rep] + 1;
    const int kbeg = wa_first(a.positions[tok0], a.window) & ~(LA_KEYS - 1);
    const int teams = KT == 1 || nkeys - kbeg <= WA_TEAM_KEYS ? 1 : KT, stride = LA_KEYS * teams;     // (uniform)
    if (team >= teams) return;
    // loader: wave -> keys 16 (wave & 1) ... of the keys (waves 0, 1) or the values (2, 3); lane -> key lane / 4, 16-byte quarter lane % 4 of every piece
    const bool vals = wave >= 2;
    const int lkey = 16 * (wave & 1) + (lane >> 2);
    const int lrow = vals ? a.v_row : a.k_row;
    const int64_t lblock = vals ? a.v_block : a.k_block;
    const uint16_t* src = (vals ? a.vc + first * a.v_row + (size_t)g * a.v_head : a.kc + first * a.k_row + (size_t)g * a.k_head) + 8 * (lane & 3);
    unsigned char* const ring = lds + team * (NB * IMAGE);
    unsigned char* const dst0 = ring + wave * HALF;
    // block ids: 64 of the sequence's table in the lanes of a register, looked up by a lane exchange (a load per tile would be waited for together with
    // the tiles in flight); read again when a tile leaves them
    int cached = 0, ids = 0;
    auto load_ids = [&](int k0) {
        cached = k0 >> a.bs_shift;
        const int b = min(cached + lane, (nkeys - 1) >> a.bs_shift);
        ids = b;
        if (!a.key_base) ids = bt[b];
        asm volatile("" : "+v"(ids));                  // waited for here, not where the lookups are
    };
    auto block_of = [&](int k0) {
        if (((k0 + LA_KEYS - 1) >> a.bs_shift) - cached > 63) load_ids(k0);
        return __shfl(ids, (min(k0 + lkey, nkeys - 1) >> a.bs_shift) - cached, 64);
    };
    auto stage = [&](int k0, int buf) {                                       // keys past the end: a valid row, masked below
        const int blk = block_of(min(k0, nkeys - 1));
        const uint16_t* p = src + (size_t)blk * lblock + (size_t)(min(k0 + lkey, nkeys - 1) & a.bs_mask) * lrow;
        unsigned char* d = dst0 + buf * IMAGE;
#pragma unroll
        for (int s = 0; s < WS; ++s)
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(p + 32 * s), (__attribute__((address_space(3))) void*)(d + s * 1024), 16, 0, 0);
    };
    load_ids(kbeg);
    stage(kbeg + LA_KEYS * team, 0);
    stage(kbeg + LA_KEYS * team + stride, 1);
    int buf = 0;
    for (int base = kbeg; base < nkeys; base += stride) {              // (as many turns for every team; one past the end stages a valid row and skips)
        const int k0 = base + LA_KEYS * team;
        asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(WS) : "memory");      // this tile is there; the one before is read by no wave any more
        stage(k0 + 2 * stride, buf >= 1 ? buf - 1 : NB - 1);                  // into the place that tile left
        const unsigned char* kimg = ring + buf * IMAGE + (c * 4 + qk) * 16;
        const unsigned char* vimg = ring + buf * IMAGE + 2 * HALF + (4 * qk + (c >> 2)) * 64 + (c & 3) * 8;
        buf = buf + 1 == NB ? 0 : buf + 1;
        if (k0 >= whi || k0 + LA_KEYS <= wlo) continue; // (wave-uniform; loads and barriers above stay common)
        f32x4 S[RG][2];
#pragma unroll
        for (int rg = 0; rg < RG; ++rg)
#pragma unroll
            for (int kt = 0; kt < 2; ++kt) S[rg][kt] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < WS; ++s)
#pragma unroll
            for (int kt = 0; kt < 2; ++kt) {
                const u32x4 A = *reinterpret_cast<const u32x4*>(kimg + kt * HALF + s * 1024);
#pragma unroll
                for (int rg = 0; rg < RG; ++rg) S[rg][kt] = mfma16(A, Q[rg][s], S[rg][kt]);
            }
        const bool inside = k0 >= flo && k0 + LA_KEYS <= fhi;      // (wave-uniform)
        u32x4 w3[RG][3];
#pragma unroll
        for (int rg = 0; rg < RG; ++rg) {
            float p[8], mx, rs = 0.f;
#pragma unroll
            for (int j = 0; j < 8; ++j) p[j] = S[rg][j >> 2][j & 3];
            if (!inside) {
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const int key = k0 + la_slot(qk, j);
                    if (key < lo[rg] || key >= hi[rg]) p[j] = -INFINITY;       // a weight of zero against any finite maximum (qs > 0)
                }
            }
            mx = p[0];
#pragma unroll
            for (int j = 1; j < 8; ++j) mx = fmaxf(mx, p[j]);
            // the maximum follows once a row has outgrown it by 2^LAZY (the conditional rescaling of FlashAttention-4): weights up to that size lose nothing
            // in fp32, nor in three terms.  The 16 rows of a group move together, so a row's last bits depend on the rows it shares a group with,
            // that is on where its portion was cut
            if (__any(mx * a.qs > m[rg] + LAZY)) {                 // (any lane's own keys: the row's maximum is put together only then)
                const float mn = fmaxf(m[rg], xor32_max(xor16_max(mx)) * a.qs), alpha = exp2_w(m[rg] - mn);      // (never below the finite sentinel: 1, harmless, where l = 0, O = 0)
                m[rg] = mn;
                l[rg] *= alpha;
#pragma unroll
                for (int d = 0; d < 2 * WS; ++d) O[rg][d] *= alpha;
            }
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                p[j] = exp2_w(fmaf(p[j], a.qs, -m[rg]));
                rs += p[j];
            }
            l[rg] += rs;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                uint32_t h0, m0, l0;
                split3(p[2 * e], p[2 * e + 1], h0, m0, l0);
                w3[rg][0][e] = h0; w3[rg][1][e] = m0; w3[rg][2][e] = l0;
            }
        }
        // V^T fragments of four column tiles at a time, waited for where they are read: as builtins they would wait for the tiles in flight too
        const unsigned vaddr = (unsigned)(size_t)(lds_s16x4*)vimg;
#pragma unroll
        for (int d0 = 0; d0 < 2 * WS; d0 += 4) {
            u32x2 x[4], y[4];
            asm volatile("ds_read_b64_tr_b16 %0, %8 offset:%9\n\tds_read_b64_tr_b16 %4, %8 offset:%13\n\t"
                         "ds_read_b64_tr_b16 %1, %8 offset:%10\n\tds_read_b64_tr_b16 %5, %8 offset:%14\n\t"
                         "ds_read_b64_tr_b16 %2, %8 offset:%11\n\tds_read_b64_tr_b16 %6, %8 offset:%15\n\t"
                         "ds_read_b64_tr_b16 %3, %8 offset:%12\n\tds_read_b64_tr_b16 %7, %8 offset:%16\n\ts_waitcnt lgkmcnt(0)"
                         : "=&v"(x[0]), "=&v"(x[1]), "=&v"(x[2]), "=&v"(x[3]), "=&v"(y[0]), "=&v"(y[1]), "=&v"(y[2]), "=&v"(y[3])
                         : "v"(vaddr), "n"(d0 * 512), "n"(d0 * 512 + 32), "n"(d0 * 512 + 1024), "n"(d0 * 512 + 1056), "n"(d0 * 512 + HALF), "n"(d0 * 512 + 32 + HALF),
                           "n"(d0 * 512 + 1024 + HALF), "n"(d0 * 512 + 1056 + HALF));
#pragma unroll
            for (int d = 0; d < 4; ++d) {
                const u32x4 VT = {x[d][0], x[d][1], y[d][0], y[d][1]};
#pragma unroll
                for (int k = 2; k >= 0; --k)
#pragma unroll
                    for (int rg = 0; rg < RG; ++rg) O[rg][d0 + d] = mfma16(VT, w3[rg][k], O[rg][d0 + d]);
            }
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the tiles behind the last one land before the LDS is another workgroup's
    if constexpr (KT > 1) if (teams > 1) {             // the other teams' rows into the first one's: [team][wave][row group][d tile | m, l][lane]
        constexpr int REC = RG * (2 * WS + 1) * 64;
        static_assert((KT - 1) * 4 * REC * 16 <= KT * NB * IMAGE, "the records lie in the rings");
        f32x4* const recs = reinterpret_cast<f32x4*>(lds) + (size_t)wave * REC + lane;
        __syncthreads();
        if (team) {
            f32x4* const rec = recs + (size_t)(team - 1) * (4 * REC);
#pragma unroll
            for (int rg = 0; rg < RG; ++rg) {
#pragma unroll
                for (int d = 0; d < 2 * WS; ++d) rec[(rg * (2 * WS + 1) + d) * 64] = O[rg][d];
                rec[(rg * (2 * WS + 1) + 2 * WS) * 64] = (f32x4){m[rg], l[rg], 0.f, 0.f};
            }
        }
        __syncthreads();
        if (team) return;
#pragma unroll
        for (int o = 0; o < KT - 1; ++o)
#pragma unroll
            for (int rg = 0; rg < RG; ++rg) {
                const f32x4* const rec = recs + (size_t)o * (4 * REC) + rg * (2 * WS + 1) * 64;
                const f32x4 ml = rec[2 * WS * 64];
                const float mn = fmaxf(m[rg], ml[0]), mine = exp2_w(m[rg] - mn), theirs = exp2_w(ml[0] - mn);      // (a team without a key of the row: the sentinel, l = 0, O = 0)
                m[rg] = mn;
                l[rg] = l[rg] * mine + ml[1] * theirs;
#pragma unroll
                for (int d = 0; d < 2 * WS; ++d) O[rg][d] = O[rg][d] * mine + rec[d * 64] * theirs;
            }
    }
#pragma unroll
    for (int rg = 0; rg < RG; ++rg) {
        const float L = xor32_sum(xor16_sum(l[rg]));
        const int r = wave * WR + 16 * rg + c;
        if (r >= nrows) continue;
        const int frow = row0 + r, tok = frow / a.rep, head = g * a.rep + frow - tok * a.rep;
        const float inv = (a.head_gate ? a.head_gate[(size_t)tok * a.heads + head] : 1.0f) / L;
#pragma unroll
        for (int d = 0; d < 2 * WS; ++d) wa_store(a.gate, a.out, a.frag, tok, head * dp + 16 * d + 4 * qk, a.heads * dp, O[rg][d] * inv);
    }
}

template <int WS, bool EX, int PW>
__global__ __launch_bounds__(64 * PW, 2) void window_prefill_kernel(const WinArgs a) {
    constexpr int SPT = PW / 2, LOADS = (WS + SPT - 1) / SPT;                // 32-wide pieces of a row the workgroup loads per pass, passes
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];      // two images of [32 keys | 32 values]
    const int ds = EX ? WS : a.ds, vs = EX ? WS : a.vs, dp = ds * 32, vp = vs * 32;
    const int kpitch = dp * 2 + 32, vpitch = vp * 2 + 32, image = LA_KEYS * (kpitch + vpitch);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int c = lane & 15, qk = lane >> 4;
    const int row0 = a.tiles[2 * blockIdx.x], nrows = a.tiles[2 * blockIdx.x + 1], g = blockIdx.y;
    const int tok0 = row0 / a.rep, brow = a.row_of_tok[tok0];
    const int32_t* bt = a.block_table + (size_t)brow * a.bt_stride;
    const size_t first = a.key_base ? a.key_base[brow] : 0;                  // paged keys and values, or rows of one array
    const uint16_t* kc = a.kc + first * a.k_row + (size_t)g * a.k_head;
    const uint16_t* vc = a.vc + first * a.v_row + (size_t)g * a.v_head;
    const int r = wave * 16 + c;
    const int frow = row0 + min(r, nrows - 1), tok = frow / a.rep, head = g * a.rep + frow - tok * a.rep;
    const int pos = a.positions[tok];
    const int hi = r < nrows ? pos + 1 : 0, lo = wa_first(pos, a.window);    // keys the row sees: [lo, hi)
    // keys the wave's rows see, and the tile's: positions grow along the rows
    const bool any = wave * 16 < nrows;
    const int whi = any ? a.positions[(row0 + min(wave * 16 + 15, nrows - 1)) / a.rep] + 1 : 0;
    const int wlo = any ? wa_first(a.positions[(row0 + wave * 16) / a.rep], a.window) : 0;
    // ... and the keys every one of the wave's rows sees: no masks in a tile inside
    const int fhi = wave * 16 + 16 <= nrows ? a.positions[(row0 + wave * 16) / a.rep] + 1 : 0, flo = wa_first(whi - 1, a.window);
    const int nkeys = a.positions[(row0 + nrows - 1) / a.rep] + 1;
    const int kbeg = wa_first(a.positions[tok0], a.window) & ~(LA_KEYS - 1);
    u32x4 Q[WS];
    f32x4 O[2 * WS];
#pragma unroll
    for (int s = 0; s < WS; ++s)
        if (EX || s < ds) Q[s] = ld16(a.q + ((size_t)tok * a.heads + head) * dp + 32 * s + 8 * qk);
#pragma unroll
    for (int d = 0; d < 2 * WS; ++d) O[d] = (f32x4){0.f, 0.f, 0.f, 0.f};
    float m = LA_SENT, l = 0.f;
    if (a.sink) { m = a.sink[head] * LA_LOG2E; l = 1.f; }
    // loader: thread -> key (tid / 4) % 32, 16-byte quarter tid % 4 of the 32-wide pieces tid / 128, + SPT, ...
    const int lkey = (threadIdx.x >> 2) & 31, lq = threadIdx.x & 3, lp = threadIdx.x >> 7;
    u32x4 sk[LOADS], sv_[LOADS];
    auto block_of = [&](int k0) { const int b = min(k0 + lkey, nkeys - 1) >> a.bs_shift; return a.key_base ? b : bt[b]; };
    auto fetch = [&](int k0, int blk) {
        const int off = min(k0 + lkey, nkeys - 1) & a.bs_mask;
        const size_t kofs = (size_t)blk * a.k_block + (size_t)off * a.k_row, vofs = (size_t)blk * a.v_block + (size_t)off * a.v_row;
#pragma unroll
        for (int j = 0; j < LOADS; ++j) {
            const int s = lp + SPT * j;
            if (s < ds) sk[j] = ld16(kc + kofs + 32 * s + 8 * lq);
            if (s < vs) sv_[j] = ld16(vc + vofs + 32 * s + 8 * lq);
        }
    };
    int blk = block_of(kbeg);                         // block ids are looked up a tile ahead of the rows
    fetch(kbeg, blk);
    blk = block_of(kbeg + LA_KEYS);
    int buf = 0;
    for (int k0 = kbeg; k0 < nkeys; k0 += LA_KEYS, buf ^= 1) {
        unsigned char* kimg = lds + buf * image;
        unsigned char* vimg = kimg + LA_KEYS * kpitch;
#pragma unroll
        for (int j = 0; j < LOADS; ++j) {
            const int s = lp + SPT * j;
            if (s < ds) *reinterpret_cast<u32x4*>(kimg + lkey * kpitch + (32 * s + 8 * lq) * 2) = sk[j];
            if (s < vs) *reinterpret_cast<u32x4*>(vimg + lkey * vpitch + (32 * s + 8 * lq) * 2) = sv_[j];
        }
        if (k0 + LA_KEYS < nkeys) {
            fetch(k0 + LA_KEYS, blk);
            blk = block_of(k0 + 2 * LA_KEYS);
        }
        __syncthreads();                                // image `buf` complete; image `buf ^ 1` is rewritten only behind the NEXT barrier's arrivals
        if (k0 >= whi || k0 + LA_KEYS <= wlo) continue; // (wave-uniform; the barriers above stay common)
        f32x4 S[2], T[2];
#pragma unroll
        for (int kt = 0; kt < 2; ++kt) S[kt] = T[kt] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < WS; ++s) {
            if (!EX && s >= ds) continue;
#pragma unroll
            for (int kt = 0; kt < 2; ++kt) {
                const u32x4 A = *reinterpret_cast<const u32x4*>(kimg + (16 * kt + c) * kpitch + (32 * s + 8 * qk) * 2);
                if (s & 1) T[kt] = mfma16(A, Q[s], T[kt]);
                else S[kt] = mfma16(A, Q[s], S[kt]);
            }
        }
        float p[8], mx = LA_SENT, rs = 0.f;
        const bool inside = k0 >= flo && k0 + LA_KEYS <= fhi;      // (wave-uniform)
#pragma unroll
        for (int j = 0; j < 8; ++j) p[j] = (S[j >> 2][j & 3] + T[j >> 2][j & 3]) * a.qs;
        if (!inside) {
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const int key = k0 + la_slot(qk, j);
                if (key < lo || key >= hi) p[j] = -INFINITY;       // a weight of zero against any finite maximum
            }
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) mx = fmaxf(mx, p[j]);
        const float mn = fmaxf(m, xor32_max(xor16_max(mx)));       // (never below the finite sentinel)
        const float alpha = exp2_w(m - mn);              // both the sentinel: 1, harmless (l = 0, O = 0)
        m = mn;
        u32x4 w3[3];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            p[j] = exp2_w(p[j] - mn);
            rs += p[j];
        }
        l = l * alpha + xor32_sum(xor16_sum(rs));
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            uint32_t h0, m0, l0;
            split3(p[2 * e], p[2 * e + 1], h0, m0, l0);
            w3[0][e] = h0; w3[1][e] = m0; w3[2][e] = l0;
        }
        if (__any(alpha != 1.0f)) {
#pragma unroll
            for (int d = 0; d < 2 * WS; ++d) O[d] *= alpha;
        }
#pragma unroll
        for (int d0 = 0; d0 < 2 * WS; d0 += 2) {        // pairs of column tiles: independent chains between dependent MFMAs
            if (!EX && d0 >= 2 * vs) continue;
            u32x4 VT[2];
#pragma unroll
            for (int d = 0; d < 2; ++d) VT[d] = la_transposed_at(vimg, vpitch, d0 + d, c, qk);
#pragma unroll
            for (int k = 2; k >= 0; --k)
#pragma unroll
                for (int d = 0; d < 2; ++d) O[d0 + d] = mfma16(VT[d], w3[k], O[d0 + d]);
        }
    }
    if (r >= nrows) return;
    const float inv = (a.head_gate ? a.head_gate[(size_t)tok * a.heads + head] : 1.0f) / l;
#pragma unroll
    for (int d = 0; d < 2 * WS; ++d)
        if (EX || d < 2 * vs) wa_store(a.gate, a.out, a.frag, tok, head * vp + 16 * d + 4 * qk, a.heads * vp, O[d] * inv);
}

// ---- any width, bf16 or fp32 elements: one wave per (token, head), 64 keys per pass (lane = key for the scores, lane = dims for the sum)
template <typename E>
__device__ __forceinline__ float wa_ld(const E* p, size_t i) {
    if constexpr (sizeof(E) == 4) return p[i];
    else return bf2f(p[i]);
}

#define WA_PLAIN_MAX 1024
template <typename E>
__global__ __launch_bounds__(64) void window_plain_kernel(const omni_window_attn a, int window) {
    __shared__ float sq[WA_PLAIN_MAX], sp[64];
    __shared__ size_t srow[64];
    constexpr int NI = WA_PLAIN_MAX / 64;
    const E* q = (const E*)a.q;
    const E* kc = (const E*)a.kc;
    const E* vc = (const E*)a.vc;
    const int lane = threadIdx.x, rep = a.heads / a.kv_heads;
    const size_t rh = blockIdx.x;
    const int t = (int)(rh / a.heads), head = (int)(rh - (size_t)t * a.heads), g = head / rep;
    for (int k = lane; k < a.dp; k += 64) sq[k] = wa_ld(q, rh * a.dp + k);
    const int pos = a.positions[t], len = pos + 1, lo = wa_first(pos, window);
    const int32_t* bt = a.block_table + (size_t)a.row_of_tok[t] * a.bt_stride;
    float m = LA_SENT, l = 0.f, acc[NI];
    if (a.sink) { m = a.sink[head]; l = 1.f; }
#pragma unroll
    for (int i = 0; i < NI; ++i) acc[i] = 0.f;
    for (int k0 = lo; k0 < len; k0 += 64) {
        __syncthreads();                               // one wave per workgroup: orders the LDS traffic of the passes
        const int key = k0 + lane, kk = min(key, len - 1);
        const size_t row = ((size_t)bt[kk / a.block_size] * a.kv_heads + g) * a.block_size + kk % a.block_size;
        float s = 0.f;
        for (int k = 0; k < a.dp; ++k) s = fmaf(sq[k], wa_ld(kc, row * a.dp + k), s);
        s *= a.scale;
        const bool ok = key < len;
        const float mn = fmaxf(m, wave_max(ok ? s : LA_SENT));
        const float alpha = expf(m - mn), p = ok ? expf(s - mn) : 0.f;
        l = l * alpha + wave_sum(p);
        m = mn;
        sp[lane] = p;
        srow[lane] = row;
        __syncthreads();
        const int nk = min(64, len - k0);
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const int d = lane + 64 * i;
            if (d >= a.vp) continue;
            float v = acc[i] * alpha;
            for (int u = 0; u < nk; ++u) v = fmaf(sp[u], wa_ld(vc, srow[u] * a.vp + d), v);
            acc[i] = v;
        }
    }
    const float inv = 1.0f / l;
    const int width = a.heads * a.vp;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        const int d = lane + 64 * i;
        if (d >= a.vp) continue;
        const int k = head * a.vp + d;
        const float v = acc[i] * inv * (a.gate ? wa_ld((const E*)a.gate, (size_t)t * width + k) : 1.0f);
        E* o = (E*)a.out + (a.frag ? frag_off(t, k, width) : (size_t)t * width + k);
        if constexpr (sizeof(E) == 4) *o = v;
        else *o = f2bf(v);
    }
}

// ---- host side
// compile-time width bound of the matrix-core kernels: 2, 4 or 8 (times 32); 0: too wide, the plain kernel runs
static int wa_bound(int dp, int vp) {
    const int w = (dp > vp ? dp : vp) / 32;
    return w <= 2 ? 2 : (w <= 4 ? 4 : (w <= 8 ? 8 : 0));
}
// (measured, 16 heads over 4 of 128, window 1024, 4 x 2048 tokens: 128 rows 174 us, 64 rows 191; 1 x 2048: 60 / 61)
static constexpr int wa_rows_of(int ws) { return ws <= 4 ? 128 : 64; }
extern "C" int omni_window_attn_tile_rows(int dp, int vp) {
    const int w = wa_bound(dp, vp);
    return w ? wa_rows_of(w) : 64;
}

extern "C" int64_t omni_window_attn_workspace_bytes(int n_decode, int heads, int vp) {
    return (int64_t)n_decode * heads * LA_MAX_SPLIT * (vp + 4) * (int64_t)sizeof(float);
}

template <typename K>
static int wa_lds(K kernel, int bytes) {
    if (bytes <= 60 * 1024) return OMNI_OK;         // (static shared memory comes on top)
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (e != hipSuccess) { omni_set_error("omni_window_attn: LDS attribute: %s", hipGetErrorString(e)); return OMNI_EHIP; }
    return OMNI_OK;
}

template <int WS, bool EX>
static int wa_run(const omni_window_attn& p, WinArgs a, hipStream_t st) {
    if (p.n_decode > 0) {
        constexpr int MAXLDS = LA_DEC_WAVES * 16 * (WS * 64 + 32) + LA_DEC_WAVES / 2 * 3 * 1024;
        static const int rc = wa_lds(window_decode_kernel<WS, EX>, MAXLDS);
        if (rc != OMNI_OK) return rc;
        const int lds = LA_DEC_WAVES * 16 * (p.vp * 2 + 32) + LA_DEC_WAVES / 2 * 3 * 1024;
        const int wgs = p.kv_heads * ((a.rep + 15) / 16);
        // One workgroup per CU.  A second to each halves no walk that two CUs' worth of keys in flight do not already fill, and its records cost their writing and a
        // merge.  Us with the merge, by two / one, 16 heads over 4 of 128, window 1024, contexts of up to 352 | 700 | 2048: 8 rows 10.0 / 10.0 | 11.2 / 11.1 |
        // 14.7 / 12.3, 16 rows 10.7 / 10.5 | 13.5 / 12.3 | 16.4 / 15.2, 32 rows 13.0 / 11.9 | 17.0 / 16.3 | 22.6 / 22.7, 64 rows -- which then leave no records -- 16.5 / 13.4 |
        // 25.2 / 22.0 | 37.5 / 35.2.  (By one per two CUs: 32 rows of up to 2048 29.8.  Eight waves a workgroup: 64 rows 14.1 | 23.8 | 37.4.)  What it costs: one row of
        // 8192 keys beside 31 of 100, no window, 47.9 / 49.9.
        // Heads of up to 64 are half the bytes a key, and one workgroup's walk no longer fills a CU: two per CU, as ever (8 heads over 2 of 64, two / one: 64 rows of up to
        // 2048 20.3 / 22.4, in windows of 1024 14.5 / 15.4, one of 8192 beside 63 of 100 44.0 / 60.2; 32 rows 14.6 / 15.0, 12.5 / 11.5, 26.6 / 33.9).
        a.nsplit = p.workspace ? la_split_count(wgs * p.n_decode, p.window > 0 && p.window < p.max_keys ? p.window + 15 : p.max_keys, WS <= 2 ? 512 : 256) : 1;
        hipLaunchKernelGGL((window_decode_kernel<WS, EX>), dim3(wgs, p.n_decode, a.nsplit), dim3(64 * LA_DEC_WAVES), lds, st, a);
        OMNI_CHECK_LAUNCH("omni_window_attn(decode)");
        if (a.nsplit > 1) {
            hipLaunchKernelGGL(window_merge_kernel, dim3(p.n_decode * p.heads), dim3(64), 0, st, a, a.nsplit);
            OMNI_CHECK_LAUNCH("omni_window_attn(merge)");
        }
    }
    if (p.n_tiles > 0) {
        if constexpr (EX && WS <= 4) if (a.qs > 0.f) {
            constexpr int LDS = 3 * 4 * WS * 1024;
            static const int rc = wa_lds(window_prefill_dma_kernel<WS, 2, 1>, LDS), rc1 = wa_lds(window_prefill_dma_kernel<WS, 1, 1>, LDS), rc3 = wa_lds(window_prefill_dma_kernel<WS, 1, 3>, 3 * LDS);
            if (rc != OMNI_OK) return rc;
            if (rc1 != OMNI_OK) return rc1;
            if (rc3 != OMNI_OK) return rc3;
            const int G = p.kv_heads, per = 8 % G == 0 ? 8 / G : 1;           // workgroups in whole groups of 8 where an XCD takes part of one head's tiles
            const bool halves = (int64_t)p.n_tiles * G <= 256;
            const int n = halves ? 2 * p.n_tiles : p.n_tiles;
            const int64_t wgs = 8 % G == 0 ? (int64_t)(n + per - 1) / per * 8 : (int64_t)n * G;
            const bool one_team = p.prompt_keys > 0 && p.prompt_keys <= WA_TEAM_KEYS;
            if (halves && (int64_t)n * G <= 256 && !one_team) hipLaunchKernelGGL((window_prefill_dma_kernel<WS, 1, 3>), dim3((unsigned)wgs), dim3(768), 3 * LDS, st, a, n);
            else if (halves) hipLaunchKernelGGL((window_prefill_dma_kernel<WS, 1, 1>), dim3((unsigned)wgs), dim3(256), LDS, st, a, n);
            else hipLaunchKernelGGL((window_prefill_dma_kernel<WS, 2, 1>), dim3((unsigned)wgs), dim3(256), LDS, st, a, n);
            OMNI_CHECK_LAUNCH("omni_window_attn(prefill)");
            return OMNI_OK;
        }
        {
            constexpr int PW = wa_rows_of(WS) / 16, MAXLDS = 2 * LA_KEYS * 2 * (WS * 64 + 32);
            static const int rc = wa_lds(window_prefill_kernel<WS, EX, PW>, MAXLDS);
            if (rc != OMNI_OK) return rc;
            hipLaunchKernelGGL((window_prefill_kernel<WS, EX, PW>), dim3(p.n_tiles, p.kv_heads), dim3(64 * PW), 2 * LA_KEYS * (p.dp * 2 + p.vp * 2 + 64), st, a);
        }
        OMNI_CHECK_LAUNCH("omni_window_attn(prefill)");
    }
    return OMNI_OK;
}

extern "C" int omni_window_attn_run(const omni_window_attn* pp, void* stream) {
    OMNI_CHECK_ARG(pp && pp->q && pp->kc && pp->vc && pp->out && pp->block_table && pp->row_of_tok && pp->positions, "omni_window_attn: null pointer");
    const omni_window_attn& p = *pp;
    OMNI_CHECK_ARG(p.heads > 0 && p.kv_heads > 0 && p.heads % p.kv_heads == 0 && p.kv_heads <= 65535, "omni_window_attn: %d heads over %d key / value heads", p.heads, p.kv_heads);
    OMNI_CHECK_ARG(p.dp > 0 && p.dp % 32 == 0 && p.dp <= WA_PLAIN_MAX && p.vp > 0 && p.vp % 32 == 0 && p.vp <= WA_PLAIN_MAX, "omni_window_attn: dp=%d vp=%d (multiples of 32, <= %d)", p.dp, p.vp, WA_PLAIN_MAX);
    OMNI_CHECK_ARG(p.block_size > 0 && (p.block_size & (p.block_size - 1)) == 0 && p.bt_stride > 0, "omni_window_attn: block_size=%d (a power of two)", p.block_size);
    OMNI_CHECK_ARG(p.n_decode >= 0 && p.n_decode <= p.T && p.n_decode <= 65535 && p.n_tiles >= 0 && (p.n_tiles == 0 || p.tiles) && (p.n_decode == p.T || p.n_tiles > 0 || p.elem == 1),
                   "omni_window_attn: T=%d n_decode=%d n_tiles=%d", p.T, p.n_decode, p.n_tiles);
    OMNI_CHECK_ARG(p.n_tiles == 0 || p.tile_rows == omni_window_attn_tile_rows(p.dp, p.vp), "omni_window_attn: tile_rows=%d (omni_window_attn_tile_rows(%d, %d) = %d)", p.tile_rows, p.dp, p.vp,
                   omni_window_attn_tile_rows(p.dp, p.vp));
    OMNI_CHECK_ARG((p.elem == 0 || (p.elem == 1 && !p.frag)) && p.window >= 0, "omni_window_attn: elem=%d frag=%d window=%d", p.elem, p.frag, p.window);
    OMNI_CHECK_ARG(!p.workspace || p.workspace_bytes >= omni_window_attn_workspace_bytes(p.n_decode, p.heads, p.vp), "omni_window_attn: workspace of %lld bytes", (long long)p.workspace_bytes);
    OMNI_CHECK_ARG(!p.key_base || (p.elem == 0 && p.n_decode == 0 && wa_bound(p.dp, p.vp) && p.k_row >= p.kv_heads * p.dp && p.k_row % 8 == 0 && p.v_row >= p.kv_heads * p.vp && p.v_row % 8 == 0),
                   "omni_window_attn: keys in one array take prompt tiles in bf16, widths the matrix-core kernel has, k_row=%d v_row=%d (heads * width, %% 8)", p.k_row, p.v_row);
    OMNI_CHECK_ARG(!p.head_gate || (p.elem == 0 && p.n_decode == 0 && !p.gate && wa_bound(p.dp, p.vp)), "omni_window_attn: a gate per head takes prompt tiles in bf16 and no other gate");
    if (p.T <= 0) return OMNI_OK;
    hipStream_t st = (hipStream_t)stream;
    const int window = p.window > 0 ? p.window : 0x7fffffff, bound = wa_bound(p.dp, p.vp);
    if (p.elem == 1 || !bound) {
        const dim3 grid((unsigned)((int64_t)p.T * p.heads)), block(64);
        if (p.elem == 1) hipLaunchKernelGGL(window_plain_kernel<float>, grid, block, 0, st, p, window);
        else hipLaunchKernelGGL(window_plain_kernel<uint16_t>, grid, block, 0, st, p, window);
        OMNI_CHECK_LAUNCH("omni_window_attn(plain)");
        return OMNI_OK;
    }
    WinArgs a{};
    a.q = (const uint16_t*)p.q; a.kc = (const uint16_t*)p.kc; a.vc = (const uint16_t*)p.vc; a.gate = (const uint16_t*)p.gate; a.sink = p.sink;
    a.out = (uint16_t*)p.out; a.frag = p.frag;
    a.block_table = p.block_table; a.bt_stride = p.bt_stride; a.bs_shift = __builtin_ctz((unsigned)p.block_size); a.bs_mask = p.block_size - 1;
    a.row_of_tok = p.row_of_tok; a.positions = p.positions; a.tiles = p.tiles;
    a.heads = p.heads; a.kv_heads = p.kv_heads; a.rep = p.heads / p.kv_heads; a.ds = p.dp / 32; a.vs = p.vp / 32;
    a.qs = p.scale * LA_LOG2E; a.window = window; a.partial = p.workspace; a.nsplit = 1;
    a.key_base = p.key_base; a.head_gate = p.head_gate;
    a.k_row = p.key_base ? p.k_row : p.dp; a.v_row = p.key_base ? p.v_row : p.vp;
    a.k_head = p.key_base ? p.dp : (int64_t)p.block_size * p.dp; a.v_head = p.key_base ? p.vp : (int64_t)p.block_size * p.vp;
    a.k_block = (p.key_base ? 1 : p.kv_heads) * (int64_t)p.block_size * a.k_row; a.v_block = (p.key_base ? 1 : p.kv_heads) * (int64_t)p.block_size * a.v_row;
    const bool ex = a.ds == bound && a.vs == bound;
    if (bound == 2) return ex ? wa_run<2, true>(p, a, st) : wa_run<2, false>(p, a, st);
    if (bound == 4) return ex ? wa_run<4, true>(p, a, st) : wa_run<4, false>(p, a, st);
    return ex ? wa_run<8, true>(p, a, st) : wa_run<8, false>(p, a, st);
}
