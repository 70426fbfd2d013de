// Large-M bf16 GEMM on the matrix cores: out[M, N] = epilogue(x[M, K] . W[N, K]^T), fp32 accumulate.
//
// The prefill-side counterpart of gemm.hip's weight-streaming skinny kernel: at M = 512 ... 600 k rows the op is MFMA-bound, so a
// workgroup owns a 256-row x BN-column output tile, stages 64-deep slices of both operands in LDS and reuses every fragment
// 4 - 8 times from registers.  Built for two callers:
//   * talker prefill (engine.prefill_native): the four per-layer GEMMs on the SAME fragment-major weights the decode step
//     streams (OMNI_LAYOUT_W_FRAG; gate_up in its 8-row interleave with SiLU(gate) * up fused) -- weights are stored once;
//   * Code2Wav decoder (codec.hip / code2wav.py): activations are TIME-major [T, C], so a causal dilated conv1d is this GEMM
//     over overlapping row windows of x -- K = taps x C_in split into `seg_len`-wide segments, segment s of output row m
//     reading x row m + row_off + s * seg_rows -- with no im2col buffer, and a transposed conv of stride s / kernel 2s is
//     the GEMM [T, 2 C_in] x [2 C_in, s * C_out] whose row-major output IS the up-sampled [T * s, C_out] signal.
//
// Data movement.  Both operands reach LDS by LDS-DMA (buffer_load_dwordx4 ... lds, 1 KB per wave instruction, no VGPR
// staging): W fragments are contiguous 1 KB runs of the fragment-major matrix; of x a wave instruction fetches 16 rows x 64 B, FOUR
// NEIGHBOURING LANES PER ROW: the address unit takes a quad of lanes per cycle if they share a line (51 B / clock and CU of contiguous
// pieces, 34 of such rows), and a lane per cycle if each has a row of its own (15 B / clock; the 256 x 256 tile's slices were bound by it:
// 3200 x 9216 x 2048 103.4 -> 96.8 us with the gather alone changed).  The image is row-major inside a fragment: lane (c, q) reads it at c * 64 + q * 16,
// as free of bank conflicts as the lane-linear reads of W (117 B / clock both).  Rows outside [0, x_rows) (the causal left padding, the
// M tail) and k-steps past K are out of range of the buffer descriptor and read as zero.  Two LDS buffers; the loads of
// slice t + 1 are issued before the MFMAs of slice t, one counted wait + barrier per slice.
// MFMA v_mfma_f32_16x16x32_bf16 with W as the A operand: D[n][m], lane holds m = l & 15, n = 4 (l >> 4) + reg.
// Epilogue: y = (acc + bias) -> GELU -> * scale (+ fp32 residual) in fp32, transposed through LDS (one m-tile per pass) so that global
// stores are whole row pieces; on the way out SiLU(gate) * up for the interleaved gate_up layout, and up to three stores of y: fp32 (a residual
// STREAM kept in fp32: snake's sin(alpha x) turns a bf16 ulp of x ~ 16 into a phase error of 0.1 rad), bf16 (the next GEMM's
// operand) and bf16(snake(y)) = y + inv_beta * sin^2(alpha * y) -- the activation in front of the NEXT conv, so that no
// stand-alone activation pass runs over the 24 kHz-rate tensors.
// Workgroups are dealt to the 8 XCDs in contiguous chunks of the (n block, m block) order, m fastest: the workgroups that
// share an L2 share a W panel.
#include "common.cuh"
#include "kernels.h"

#define TG_WAVES 8
#define TG_THREADS (TG_WAVES * 64)
#define TG_OOB 0x80000000u           // byte offset beyond any descriptor (num_records < 2^31): reads as zero
#define TG_LDS_MAX (160 * 1024)

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void lds_void_t;

struct TileArgs {
    const uint16_t* x; int64_t x_rows; int ldx, x_bytes;      // x_bytes: what the descriptor of x covers
    int seg_len, seg_rows, row_off;
    const uint16_t* W; const float* bias; const float* scale;
    const float* resid; int ldr;
    float* out_f32; int ldf;
    uint16_t* out; int ldo;
    uint16_t* out2; int ldo2; const float* snake_alpha; const float* snake_inv_beta;
    int M, N, K;
    int act;                         // OMNI_TILE_ACT_*
    int mblocks, nblocks, band;
    // grouped (batched) launch: blockIdx.y = group; group g reads x rows [g * gx_rows, + its row count), the matrix
    // W + g * gw_elems, and writes output rows from g * gout_rows.  group_rows (device, optional) = live rows per group:
    // tiles past it leave at once, rows past it read as zero and are not stored
    long long gx_rows, gw_elems, gout_rows;
    const int32_t* group_rows;
    float act_p, act_n;              // OMNI_TILE_ACT_XIELU
    int act_cols;                    // OMNI_TILE_ACT_SILU_SIGMOID
    const uint16_t* mul_table; const int32_t* mul_ids; int mul_rows, mul_ld;      // OMNI_TILE_ACT_GELU_MUL
    int splits; long long slab_stride;      // k-splits: split z's partial sums go to out_f32 + z * slab_stride (elements)
    long long gx_cols, gout_cols;    // grouped launch: column offset of a group in x and in the outputs (per-head products of one token array)
};

__device__ __forceinline__ f32x4 tg_mfma(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

__device__ __forceinline__ float tg_gelu(float v) { return 0.5f * v * (1.0f + erff(v * 0.70710678118654752f)); }

// Epilogues, each a body of its own: one that held every activation outgrew the compiler's unrolling of its passes at 256 rows, and accumulators
// indexed by a run-time pass live in scratch memory (+ 25 us per launch).
//   EPI_PLAIN  bf16 out        EPI_F32  fp32 out        EPI_ACT  XIELU, RELU2, SILU_SIGMOID, GELU_MUL or none -> bf16 and / or fp32 out
//   EPI_FULL   bias, scale, GELU or none, residual, any outputs
enum { EPI_PLAIN = 0, EPI_ACT = 1, EPI_FULL = 2, EPI_F32 = 3 };
__host__ __device__ __forceinline__ int tile_epi(const TileArgs& a) {
    if (a.bias || a.scale || a.act == OMNI_TILE_ACT_GELU || a.resid || a.out2) return EPI_FULL;
    if (a.out_f32 && !a.out && a.act == OMNI_TILE_ACT_NONE) return EPI_F32;
    return a.out_f32 || a.act >= OMNI_TILE_ACT_XIELU ? EPI_ACT : EPI_PLAIN;
}

// Epilogue of a tile kernel: `acc[j][i]` = this wave's WN n-tiles x WM m-tiles (D[n][m] fragments), first row mw0, first column nw0; `lds` is dead.
// EPI_PLAIN (the talker prefill's four GEMMs): the same values as EPI_FULL (acc + 0 and * 1 change nothing) without ~20 wave-uniform branches per
// pass -- they, not the stores, were most of an 11 k-cycle epilogue (profiles/r05_gemm_pp_stamps.txt).
template <int WN, int WM, bool GU8, int EPI>
__device__ __forceinline__ void tile_epilogue(const TileArgs& a, f32x4 (&acc)[WN][WM], uint8_t* lds, int wave, int lane, int mw0, int nw0) {
    asm volatile("" : "+v"(lane));                        // addresses are this body's own: shared ones would be computed, and held, before the branch
    const int c = lane & 15, q = lane >> 4;
    // ---- epilogue.  Register side: y = act(acc + bias) * scale in fp32, transposed through this wave's LDS image in fp32, ONE m-tile
    // (16 rows x the wave's WN * 16 columns) per pass.  Row side: 8 columns per lane, a row's lanes cover WN * 64 contiguous bytes
    // of an fp32 output (whole 128-byte lines); + fp32 residual (the pass's residual loads are issued before its image is written:
    // the epilogue of a residual GEMM is an HBM phase, not a chain of load -> add -> store round trips), then up to three stores of
    // the SAME fp32 value: fp32 (the residual stream), bf16 (the next GEMM's operand), bf16(snake(y)) (the next conv's operand).
    // fp32 alone (EPI_F32, the products that a row kernel reads): 4 columns per lane, so that a wave's store is whole rows of 256 contiguous bytes; two stores of 16 of every
    // 32 bytes, as behind the other outputs, write at 3 - 4 TB/s.  Us, before / now: 1547 x 1024 x 2048 in two partial sums 13.8 / 12.5, 1000 x 2048 x 2048 in two 16.3 / 14.9,
    // 6001 x 2048 x 2048 48.8 / 46.2, 70 x 2048 x 2048 in four 6.4 / 6.2; straight from the registers, 64 bytes a row, 13.6, 15.4 and 46.6.  With a residual or a second output
    // it is the other way round (twice the instructions: 6001 x 2048 x 2048 58.2 / 59.1, with GELU 56.7 / 58.8).
    // (Two images per wave, pass p + 1's written before pass p's is read back, measured SLOWER: 5.9 k -> 8.5 k cycles per epilogue.)
    constexpr int IPITCH = WN * 64 + 16;                  // bytes per image row
    constexpr int PER_ROW = GU8 ? WN : EPI == EPI_F32 ? WN * 4 : WN * 2;      // lane items per image row: a [8 gate | 8 up] tile, 4 columns, or 8
    constexpr int RIT = (16 * PER_ROW + 63) / 64;         // row-side iterations per pass
    uint8_t* img = lds + wave * (16 * IPITCH);
    auto bias_scale = [&](int j, f32x4& b, f32x4& s) {
        const int n = nw0 + j * 16 + 4 * q;
        b = f32x4{0.f, 0.f, 0.f, 0.f};
        s = f32x4{1.f, 1.f, 1.f, 1.f};
        if (EPI == EPI_FULL && n < a.N) {
            if (a.bias) b = *reinterpret_cast<const f32x4*>(a.bias + n);
            if (a.scale) s = *reinterpret_cast<const f32x4*>(a.scale + n);
        }
    };
    constexpr bool HELD = WN < 8;                         // wider waves read them once per pass: their registers are full
    f32x4 bq[WN], sq[WN];
    if (HELD) {
#pragma unroll
        for (int j = 0; j < WN; ++j) bias_scale(j, bq[j], sq[j]);
    }
    const bool gelu = EPI == EPI_FULL && a.act == OMNI_TILE_ACT_GELU, mul = EPI == EPI_ACT && a.act == OMNI_TILE_ACT_GELU_MUL;
    auto write_as = [&](const int pass, auto f) {         // f(value, n-tile, bias, scale)
#pragma unroll
        for (int j = 0; j < WN; ++j) {
            f32x4 v, b = bq[j], s = sq[j];
            if (!HELD) bias_scale(j, b, s);
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = f(acc[j][pass][e], j, b[e], s[e]);
            *reinterpret_cast<f32x4*>(img + c * IPITCH + (j * 16 + 4 * q) * 4) = v;
        }
    };
    auto write_image = [&](const int pass) {
        if (EPI == EPI_ACT && a.act == OMNI_TILE_ACT_XIELU) write_as(pass, [&](float z, int, float, float) { return xielu(z, a.act_p, a.act_n); });
        else if (EPI == EPI_ACT && a.act == OMNI_TILE_ACT_RELU2) write_as(pass, [&](float z, int, float, float) { return relu2(z); });
        else if (EPI == EPI_ACT && a.act == OMNI_TILE_ACT_SILU_SIGMOID)
            write_as(pass, [&](float z, int j, float, float) { return (nw0 + j * 16 + 4 * q < a.act_cols ? z : 1.0f) * sigmoid_w(z); });
        else if (mul) write_as(pass, [&](float z, int, float, float) { return gelu_tanh(z); });
        else if (gelu) write_as(pass, [&](float z, int, float b, float s) { return tg_gelu(z + b) * s; });
        else if (EPI == EPI_FULL) write_as(pass, [&](float z, int, float b, float s) { return (z + b) * s; });
        else write_as(pass, [&](float z, int, float, float) { return z; });
    };
    f32x4 rv[RIT][2];
#pragma unroll
    for (int pass = 0; pass < WM; ++pass) {
        const int mp0 = mw0 + pass * 16;
        if (EPI == EPI_FULL && !GU8 && a.resid) {
#pragma unroll
            for (int it = 0; it < RIT; ++it) {
                const int idx = lane + 64 * it;
                const int row = idx / PER_ROW, ch = idx - row * PER_ROW;
                const int m = mp0 + row, n = nw0 + ch * 8;
                rv[it][0] = rv[it][1] = f32x4{0.f, 0.f, 0.f, 0.f};
                if (idx < 16 * PER_ROW && m < a.M && n < a.N) {
                    const float* rp = a.resid + (size_t)m * a.ldr + n;
                    rv[it][0] = *reinterpret_cast<const f32x4*>(rp);
                    rv[it][1] = *reinterpret_cast<const f32x4*>(rp + 4);
                }
            }
        }
        write_image(pass);
        __builtin_amdgcn_wave_barrier();
        if (GU8) {
            // tile j of a row = [8 gate | 8 up] -> 8 act columns at n / 2: bf16(bf16(SiLU(bf16 gate)) * bf16 up), the rounding points of
            // torch's F.silu(g) * u on bf16 tensors (omni_silu_mul, oracle silu_mul)
#pragma unroll
            for (int it = 0; it < RIT; ++it) {
                const int idx = lane + 64 * it;
                const int row = idx / PER_ROW, j = idx - row * PER_ROW;
                const int m = mp0 + row, n = nw0 + j * 16;
                if (idx >= 16 * PER_ROW || m >= a.M || n >= a.N) continue;
                const float* gp = reinterpret_cast<const float*>(img + row * IPITCH + j * 64);
                u32x4 o;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float g0 = bfround(gp[2 * e]), g1 = bfround(gp[2 * e + 1]);
                    const float u0 = bfround(gp[8 + 2 * e]), u1 = bfround(gp[8 + 2 * e + 1]);
                    const float s0 = bfround(silu_b(g0)), s1 = bfround(silu_b(g1));   // torch: F.silu(bf16) is bf16
                    o[e] = pack_bf2(s0 * u0, s1 * u1);
                }
                *reinterpret_cast<u32x4*>(a.out + (size_t)m * a.ldo + (n >> 1)) = o;
            }
        } else if (EPI == EPI_F32) {
#pragma unroll
            for (int it = 0; it < RIT; ++it) {
                const int idx = lane + 64 * it;
                const int row = idx / PER_ROW, ch = idx - row * PER_ROW;
                const int m = mp0 + row, n = nw0 + ch * 4;
                if (m < a.M && n < a.N) *reinterpret_cast<f32x4*>(a.out_f32 + (size_t)m * a.ldf + n) = *reinterpret_cast<const f32x4*>(img + row * IPITCH + ch * 16);
            }
        } else {
#pragma unroll
            for (int it = 0; it < RIT; ++it) {
                const int idx = lane + 64 * it;
                const int row = idx / PER_ROW, ch = idx - row * PER_ROW;
                const int m = mp0 + row, n = nw0 + ch * 8;
                if (idx >= 16 * PER_ROW || m >= a.M || n >= a.N) continue;
                f32x4 y0 = *reinterpret_cast<const f32x4*>(img + row * IPITCH + ch * 32);
                f32x4 y1 = *reinterpret_cast<const f32x4*>(img + row * IPITCH + ch * 32 + 16);
                if (EPI == EPI_PLAIN) {
                    u32x4 o;
                    o[0] = pack_bf2(y0[0], y0[1]); o[1] = pack_bf2(y0[2], y0[3]);
                    o[2] = pack_bf2(y1[0], y1[1]); o[3] = pack_bf2(y1[2], y1[3]);
                    *reinterpret_cast<u32x4*>(a.out + (size_t)m * a.ldo + n) = o;
                    continue;
                }
                if (mul) {
                    const int id = a.mul_ids[m];
                    u32x4 z = {0, 0, 0, 0};
                    if (id >= 0 && id < a.mul_rows) z = *reinterpret_cast<const u32x4*>(a.mul_table + (size_t)id * a.mul_ld + n);
#pragma unroll
                    for (int e = 0; e < 2; ++e) {
                        y0[2 * e] *= bf_lo(z[e]); y0[2 * e + 1] *= bf_hi(z[e]);
                        y1[2 * e] *= bf_lo(z[2 + e]); y1[2 * e + 1] *= bf_hi(z[2 + e]);
                    }
                }
                if (EPI == EPI_FULL && a.resid) {
                    y0 += rv[it][0];
                    y1 += rv[it][1];
                }
                if (a.out_f32) {
                    float* op = a.out_f32 + (size_t)m * a.ldf + n;
                    *reinterpret_cast<f32x4*>(op) = y0;
                    *reinterpret_cast<f32x4*>(op + 4) = y1;
                }
                if (a.out) {
                    u32x4 o;
                    o[0] = pack_bf2(y0[0], y0[1]); o[1] = pack_bf2(y0[2], y0[3]);
                    o[2] = pack_bf2(y1[0], y1[1]); o[3] = pack_bf2(y1[2], y1[3]);
                    *reinterpret_cast<u32x4*>(a.out + (size_t)m * a.ldo + n) = o;
                }
                if (EPI == EPI_FULL && a.out2) {
                    const f32x4 al0 = *reinterpret_cast<const f32x4*>(a.snake_alpha + n), al1 = *reinterpret_cast<const f32x4*>(a.snake_alpha + n + 4);
                    const f32x4 ib0 = *reinterpret_cast<const f32x4*>(a.snake_inv_beta + n), ib1 = *reinterpret_cast<const f32x4*>(a.snake_inv_beta + n + 4);
                    f32x4 z0, z1;
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float s0 = __sinf(y0[e] * al0[e]), s1 = __sinf(y1[e] * al1[e]);
                        z0[e] = y0[e] + ib0[e] * s0 * s0;
                        z1[e] = y1[e] + ib1[e] * s1 * s1;
                    }
                    u32x4 o;
                    o[0] = pack_bf2(z0[0], z0[1]); o[1] = pack_bf2(z0[2], z0[3]);
                    o[2] = pack_bf2(z1[0], z1[1]); o[3] = pack_bf2(z1[2], z1[3]);
                    *reinterpret_cast<u32x4*>(a.out2 + (size_t)m * a.ldo2 + n) = o;
                }
            }
        }
        __builtin_amdgcn_wave_barrier();
    }
}

template <int WN, int WM, bool GU8>
__device__ __forceinline__ void tile_epilogue_of(const TileArgs& a, f32x4 (&acc)[WN][WM], uint8_t* lds, int wave, int lane, int mw0, int nw0) {
    const int epi = tile_epi(a);
    if (epi == EPI_PLAIN) tile_epilogue<WN, WM, GU8, EPI_PLAIN>(a, acc, lds, wave, lane, mw0, nw0);
    else if (!GU8 && epi == EPI_F32) tile_epilogue<WN, WM, GU8, EPI_F32>(a, acc, lds, wave, lane, mw0, nw0);
    else if (!GU8 && epi == EPI_ACT) tile_epilogue<WN, WM, GU8, EPI_ACT>(a, acc, lds, wave, lane, mw0, nw0);
    else tile_epilogue<WN, WM, GU8, EPI_FULL>(a, acc, lds, wave, lane, mw0, nw0);
}

// Geometry of one instantiation: 8 waves (two per SIMD: while one issues its LDS-DMA pieces -- 60 - 180 cycles each -- or waits
// for fragments, the other feeds the matrix pipe) as WAVES_N x (8 / WAVES_N); a wave owns WN n-tiles x WM m-tiles of 16 x 16
// (acc = WN * WM * 4 of its 256 registers); BN = WAVES_N * WN * 16, BM = (8 / WAVES_N) * WM * 16.
template <int WAVES_N, int WN, int WM>
struct TileGeom {
    static constexpr int WAVES_M = TG_WAVES / WAVES_N;
    static constexpr int NTILES = WAVES_N * WN, MTILES = WAVES_M * WM;
    static constexpr int BN = NTILES * 16, BM = MTILES * 16;
    static constexpr int SLICE = (NTILES + MTILES) * 1024;                   // one 32-deep slice of both operands
    static constexpr int NLW = (NTILES + TG_WAVES - 1) / TG_WAVES, NLX = (MTILES + TG_WAVES - 1) / TG_WAVES;   // LDS-DMA per wave and slice
    static constexpr bool W_RAGGED = NTILES % TG_WAVES != 0;                 // some waves issue a dummy W load (uniform counts)
    static constexpr bool X_RAGGED = MTILES % TG_WAVES != 0;                 // likewise for x (the 64-row tile of the small-M geometry)
    static constexpr bool RAGGED = W_RAGGED || X_RAGGED;
    static constexpr int NBUF = (TG_LDS_MAX - (RAGGED ? TG_WAVES * 1024 : 0)) / SLICE >= 4 ? 4 : 3;
    static constexpr int EPI_BYTES = TG_WAVES * 16 * (WN * 64 + 16);           // fp32 image of one m-tile x the wave's columns
    static constexpr int RING_BYTES = NBUF * SLICE + (RAGGED ? TG_WAVES * 1024 : 0);
    static constexpr int LDS_BYTES = RING_BYTES > EPI_BYTES ? RING_BYTES : EPI_BYTES;
    static_assert(WN % 2 == 0 && LDS_BYTES <= TG_LDS_MAX, "geometry");
};

template <int WAVES_N, int WN, int WM, bool GU8>
__global__ __launch_bounds__(TG_THREADS) void gemm_tile_kernel(const TileArgs a_in) {
    using G = TileGeom<WAVES_N, WN, WM>;
    TileArgs a = a_in;
    long long x_lo = 0, x_hi = a.x_rows, x_skip = 0;                          // rows of x this launch may read; elements ahead of the group's first column
    if (gridDim.y > 1 || a.group_rows) {
        const int grp = blockIdx.y;
        if (a.group_rows) a.M = min(a.M, a.group_rows[grp]);
        x_lo = grp * a.gx_rows;
        x_hi = min(x_lo + a.M, a.x_rows);
        a.W += (size_t)grp * a.gw_elems;
        const size_t orow = (size_t)grp * a.gout_rows;
        if (a.out) a.out += orow * a.ldo;
        if (a.out2) a.out2 += orow * a.ldo2;
        if (a.out_f32) a.out_f32 += orow * a.ldf;
        if (a.resid) a.resid += orow * a.ldr;
        x_skip = grp * a.gx_cols;
        a.x += x_skip;
        const size_t ocol = (size_t)grp * a.gout_cols;
        if (a.out) a.out += ocol;
        if (a.out_f32) a.out_f32 += ocol;
    }
    constexpr int NTILES = G::NTILES, SLICE = G::SLICE, NLW = G::NLW, NLX = G::NLX, NBUF = G::NBUF;
    constexpr int INFLIGHT = NBUF - 2;                                        // slices still landing when slice t + 1 is awaited
    extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wn = wave % WAVES_N, wm = wave / WAVES_N;
    const int c = lane & 15, q = lane >> 4;

    // XCD-aware tile order (bijective for any grid size): the hardware deals workgroup ids round-robin over the 8 XCDs
    int tile;
    {
        const int nwg = gridDim.x, id = blockIdx.x;
        const int xcd = id & 7, slot = id >> 3, per = nwg >> 3, rem = nwg & 7;
        tile = (xcd < rem ? xcd * (per + 1) : rem * (per + 1) + (xcd - rem) * per) + slot;
    }
    // tile order: bands of `band` m blocks, n-major inside a band, so that an XCD's contiguous chunk of ~nwg / 8 tiles is a compact
    // 2-D block (~sqrt x sqrt) of the tile grid: it touches the fewest distinct W and x panels (L2 misses go to the MALL / HBM)
    int n_blk, m_blk;
    {
        const int per_band = a.band * a.nblocks;
        const int b = tile / per_band, r = tile - b * per_band;
        const int h = min(a.band, a.mblocks - b * a.band);            // rows of this (possibly last, shorter) band
        n_blk = r / h;
        m_blk = b * a.band + (r - n_blk * h);
    }
    const int m0 = m_blk * G::BM, n0 = n_blk * G::BN;
    if (m0 >= a.M) return;                                                    // a group with fewer rows than the launch's M (uniform)
    const int nsteps = a.K >> 5;                                              // 32-deep slices

    const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc((void*)a.W, 0, (int)((size_t)a.N * a.K * 2), 0x00020000);
    const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc((void*)a.x, 0, a.x_bytes - (int)(x_skip * 2), 0x00020000);

    // ---- staging.  Slice image: W tile f at f KB, x tile g at (NTILES + g) KB.  Wave w issues W tiles w + 8 i (i < NLW; a wave
    // without an i-th tile loads zeros into a spare KB so that every wave has the same count in flight) and x tiles w + 8 i.
    unsigned wbase[NLW];
    int xrow[NLX], xbyte[NLX];
#pragma unroll
    for (int i = 0; i < NLW; ++i) {
        const int f = wave + TG_WAVES * i;
        const int n16 = (n0 >> 4) + f;
        wbase[i] = (f < NTILES && n16 * 16 < a.N) ? (unsigned)((size_t)n16 * nsteps * 1024 + lane * 16) : TG_OOB;
    }
#pragma unroll
    for (int i = 0; i < NLX; ++i) {
        const int g = wave + TG_WAVES * i;
        xrow[i] = (int)x_lo + m0 + g * 16 + (lane >> 2) + a.row_off;
        xbyte[i] = (xrow[i] * a.ldx + 8 * (lane & 3)) * 2;        // wraps out of the descriptor for rows < 0 (never used then)
    }
    int seg = 0, cs = 0;                                  // segment walk of the NEXT slice to stage: k = seg * seg_len + cs
    const int seg_row_bytes = a.seg_rows * a.ldx * 2;
    auto stage = [&](int slice) {                         // slices are staged in order, one call each
        const int buf = slice % NBUF;
        const bool live = slice < nsteps;
        const int shift = seg * a.seg_rows, add = seg * seg_row_bytes + cs * 2;
        uint8_t* base = lds + buf * SLICE + wave * 1024;
#pragma unroll
        for (int i = 0; i < NLW; ++i) {
            const bool mine = !G::W_RAGGED || wave + TG_WAVES * i < NTILES;
            const unsigned off = (live && mine && wbase[i] != TG_OOB) ? wbase[i] + (unsigned)slice * 1024u : TG_OOB;
            uint8_t* dst = mine ? base + i * (TG_WAVES * 1024) : lds + NBUF * SLICE + wave * 1024;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rw, (lds_void_t*)dst, 16, off, 0, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < NLX; ++i) {
            const bool mine = !G::X_RAGGED || wave + TG_WAVES * i < G::MTILES;
            const int r = xrow[i] + shift;
            const unsigned off = (live && mine && r >= (int)x_lo && r < (int)x_hi) ? (unsigned)(xbyte[i] + add) : TG_OOB;
            uint8_t* dst = mine ? base + (NTILES + i * TG_WAVES) * 1024 : lds + NBUF * SLICE + wave * 1024;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (lds_void_t*)dst, 16, off, 0, 0, 0);
        }
        cs += 32;
        if (cs >= a.seg_len) { cs = 0; ++seg; }
    };

    f32x4 acc[WN][WM];
#pragma unroll
    for (int j = 0; j < WN; ++j)
#pragma unroll
        for (int i = 0; i < WM; ++i) acc[j][i] = f32x4{0.f, 0.f, 0.f, 0.f};

    // ---- main loop.  Per slice a wave reads WM x fragments + WN W fragments and issues WN * WM MFMAs, in two halves of the W
    // tiles.  The wait for slice t + 1 and the workgroup barrier sit BETWEEN the halves of slice t; right after it the wave
    // reads the x fragments and the first W half of slice t + 1 into the other register set, so that LDS latency hides behind
    // the second half's MFMAs, and the second W half is read at the top of the next slice behind the first half's MFMAs.
    // NBUF-deep ring, slice t + NBUF - 1 staged at the top of slice t: NBUF - 2 slices stay in flight across every barrier
    // (counted vmcnt, never 0 inside the loop).  lgkmcnt(0) before the barrier retires this wave's reads of the buffer that
    // the next top-of-slice staging overwrites.
    constexpr int HW = WN / 2;
    auto lds_w = [&](int slice, int j) {
        return *reinterpret_cast<const u32x4*>(lds + (slice % NBUF) * SLICE + (wn * WN + j) * 1024 + lane * 16);
    };
    auto lds_x = [&](int slice, int i) {
        return *reinterpret_cast<const u32x4*>(lds + (slice % NBUF) * SLICE + (NTILES + wm * WM + i) * 1024 + (c * 4 + q) * 16);
    };
    u32x4 xa[WM], xb[WM], w0[HW], w1[HW];
#pragma unroll
    for (int s = 0; s < NBUF - 1; ++s) stage(s);
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(INFLIGHT * (NLW + NLX)) : "memory");
#pragma unroll
    for (int i = 0; i < WM; ++i) xa[i] = lds_x(0, i);
#pragma unroll
    for (int j = 0; j < HW; ++j) w0[j] = lds_w(0, j);

#define TG_SLICE(T, XCUR, XNEXT)                                                                             \
    {                                                                                                        \
        _Pragma("unroll") for (int j = 0; j < HW; ++j) w1[j] = lds_w((T), HW + j);                           \
        stage((T) + NBUF - 1);                                                                               \
        __builtin_amdgcn_s_setprio(1);                                                                       \
        _Pragma("unroll") for (int j = 0; j < HW; ++j)                                                       \
            _Pragma("unroll") for (int i = 0; i < WM; ++i) acc[j][i] = tg_mfma(w0[j], XCUR[i], acc[j][i]);   \
        __builtin_amdgcn_s_setprio(0);                                                                       \
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(INFLIGHT * (NLW + NLX)) : "memory"); \
        _Pragma("unroll") for (int i = 0; i < WM; ++i) XNEXT[i] = lds_x((T) + 1, i);                         \
        _Pragma("unroll") for (int j = 0; j < HW; ++j) w0[j] = lds_w((T) + 1, j);                            \
        __builtin_amdgcn_s_setprio(1);                                                                       \
        _Pragma("unroll") for (int j = 0; j < HW; ++j)                                                       \
            _Pragma("unroll") for (int i = 0; i < WM; ++i) acc[HW + j][i] = tg_mfma(w1[j], XCUR[i], acc[HW + j][i]); \
        __builtin_amdgcn_s_setprio(0);                                                                       \
    }
    for (int t = 0; t < nsteps; t += 2) {                // an odd slice count runs one slice of zeros (staged out of range)
        TG_SLICE(t, xa, xb)
        TG_SLICE(t + 1, xb, xa)
    }
#undef TG_SLICE
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");   // the ring is dead: its tail loads (zeros) landed

    tile_epilogue_of<WN, WM, GU8>(a, acc, lds, wave, lane, m0 + wm * WM * 16, n0 + wn * WN * 16);
}

// ---- the two-group ("ping-pong") form of the 256-column tile.  Same images, same MFMA, same accumulation order as gemm_tile_kernel
// (bit-identical output); what differs is WHEN a wave does what.  The eight waves are two groups of four, one wave of each group per SIMD:
// group g owns the tile's m-tiles [MW g, + MW) (16 rows each; BM = 32 MW), wave column wc = wave & 3 owns n-tiles [4 wc, + 4).  A K-tile
// (64 deep: two 32-deep steps) is two phases of [12 LDS reads + 4 LDS-DMA pieces | barrier | 24 - 32 MFMAs | barrier], and group 1 runs ONE
// barrier interval behind group 0: while one wave of a SIMD issues its loads (an LDS-DMA piece costs its issuer 60 - 180 cycles) and waits
// for its fragments, the other one owns the matrix pipe.  In gemm_tile_kernel both waves of a SIMD load at the same time and then want the
// pipe at the same time.  Phase 2 t: [x low (t), W high (t) | x low (t) x all four n-tiles]; phase 2 t + 1: [x high (t), W low (t + 1) |
// x high (t) x all four] (the low W fragments live in two register sets).
// Staging: a K-tile's image is four 16 KB half-tiles (x: the low m-tiles of both groups | W: n-tiles 0-1 of every wave column | W: n-tiles
// 2-3 | x: the high m-tiles; a wave without a real piece loads zeros into a spare KB: uniform vmcnt), two 64 KB buffers.  Each phase stages
// the two half-tiles that the phase after the next one reads, and waits -- vmcnt(4) behind its own four pieces, in front of its first
// barrier -- for the two that the NEXT phase reads.  Order of a region's life: read in phase p (the reads retire at that wave's lgkmcnt(0)
// behind the phase's first barrier) -> re-staged in phase p + 2 -> waited for in p + 3 -> read in p + 4.  With the groups one interval
// apart every one of these edges still has a barrier that BOTH parties passed in between.
// Measured (scripts/probes/gemm_pp_stamps.hip, profiles/r05_gemm_pp_stamps.txt): 2 400 - 2 600 cycles per K-tile against 2 048 of MFMA at
// full rate (gemm_tile_kernel: ~2 900); four phases of 12 - 16 MFMAs: +1.5 %; the closing barrier 4 or 8 MFMAs before a section's end
// (both groups on the pipe for a moment): +9 %; unequal groups (240 / 208 rows): slower than the next taller equal pair.
//
// -DPP_STAMPS (the probe only): 1 / 2 = the shader clock at the section boundaries of K-tiles 8 ... 23 of one workgroup (first wave of each
// group; 2 adds a stamp between the loads and the first barrier), kept in LDS behind the ring (a global store would count in vmcnt);
// 3 = shader clock and the 100 MHz clock at kernel entry, loop start, loop end, kernel end, nothing inside the loop.
#ifdef PP_STAMPS
__device__ unsigned long long g_pp_stamps[2][1024];
__device__ int g_pp_stamp_wg;
#if PP_STAMPS == 3
#define PP_T()
#define PP_C(k) do { if (st_wave) { g_pp_stamps[grp][1 + 2 * (k)] = __builtin_amdgcn_s_memtime(); g_pp_stamps[grp][2 + 2 * (k)] = __builtin_amdgcn_s_memrealtime(); } } while (0)
#else
#define PP_T() do { if (st_on) { st_buf[st_n] = __builtin_amdgcn_s_memtime(); ++st_n; } } while (0)
#define PP_C(k)
#endif
#if PP_STAMPS == 2
#define PP_T1() PP_T()
#else
#define PP_T1()
#endif
#else
#define PP_T()
#define PP_T1()
#define PP_C(k)
#endif

template <int MW, bool GU8>
__global__ __launch_bounds__(TG_THREADS) void gemm_tile_pp_kernel(const TileArgs a_in) {
    TileArgs a = a_in;
    constexpr int KT_BYTES = 64 * 1024, HALF = 16 * 1024, SPARE = 2 * KT_BYTES;
    constexpr int LO = (MW + 1) / 2, HI = MW - LO;            // low / high m-tiles of a wave
    static_assert(MW >= 2 && MW <= 8, "geometry");
    extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int grp = wave >> 2, wc = wave & 3;
    const int c = lane & 15, q = lane >> 4;
#ifdef PP_STAMPS
    const bool st_wave = (int)blockIdx.x == g_pp_stamp_wg && wc == 0 && lane == 0;
#endif
    PP_C(0);
    int tile;
    {
        const int nwg = gridDim.x, id = blockIdx.x;
        const int xcd = id & 7, slot = id >> 3, per = nwg >> 3, rem = nwg & 7;
        tile = (xcd < rem ? xcd * (per + 1) : rem * (per + 1) + (xcd - rem) * per) + slot;
    }
    int n_blk, m_blk;
    {
        const int per_band = a.band * a.nblocks;
        const int b = tile / per_band, r = tile - b * per_band;
        const int h = min(a.band, a.mblocks - b * a.band);
        n_blk = r / h;
        m_blk = b * a.band + (r - n_blk * h);
    }
    const int m0 = m_blk * (32 * MW), n0 = n_blk * 256;
    // this workgroup's 32-deep steps [s0, s0 + nsteps): all of them, or one of a.splits runs (its partial sums go to a slab of their own)
    const int all = a.K >> 5;
    int s0 = 0, nsteps = all;
    float* slab = a_in.out_f32;
    if (a_in.splits > 1) {
        s0 = (int)blockIdx.y * all / a_in.splits;
        nsteps = ((int)blockIdx.y + 1) * all / a_in.splits - s0;
        slab += (size_t)blockIdx.y * a_in.slab_stride;
    }
    const int nkt = (nsteps + 1) >> 1;
    const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc((void*)a.W, 0, (int)((size_t)a.N * a.K * 2), 0x00020000);
    const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc((void*)a.x, 0, a.x_bytes, 0x00020000);

    // staging: piece e (0 / 1) of a half-tile = fragment f = wave + 8 e of its 16 = (slot t = f >> 1, k-step f & 1).  Slot t of an x half is
    // the t-th m-tile of [group 0's half | group 1's half]; slot t of a W half is n-tile 4 (t >> 1) + (t & 1) (+ 2 in the high half).
    unsigned wofs[2][2], xofs[2][2];
    bool xreal[2][2];
#pragma unroll
    for (int hi = 0; hi < 2; ++hi)
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const int f = wave + 8 * e, t = f >> 1, ks = f & 1;
            const int n16 = (n0 >> 4) + 4 * (t >> 1) + (t & 1) + 2 * hi;
            wofs[hi][e] = n16 * 16 < a.N ? (unsigned)(((size_t)n16 * all + s0 + ks) * 1024 + lane * 16) : TG_OOB;
            const int cnt = hi ? HI : LO;                     // per group
            const int mt = (t < cnt ? 0 : MW) + (hi ? LO : 0) + (t < cnt ? t : t - cnt);
            const int row = m0 + mt * 16 + (lane >> 2);
            xreal[hi][e] = t < 2 * cnt;
            xofs[hi][e] = (t < 2 * cnt && row < a.M && row < a.x_rows) ? (unsigned)(((size_t)row * a.ldx + (s0 + ks) * 32 + 8 * (lane & 3)) * 2) : TG_OOB;
        }
    auto stage = [&](int kt, int h, int buf) {                // h: 0 x low, 1 W low, 2 W high, 3 x high
        const bool live = kt < nkt;
        const bool is_w = h == 1 || h == 2;
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const unsigned base = is_w ? wofs[h == 2][e] : xofs[h == 3][e];
            // an odd count of 32-deep steps: the last K-tile's second step lies past the row's K (x: the next row's data; W: the next n-tile's)
            const bool tail = ((wave + 8 * e) & 1) && 2 * kt + 1 >= nsteps;
            const unsigned off = (live && !tail && base != TG_OOB) ? base + (unsigned)kt * (is_w ? 2048u : 128u) : TG_OOB;
            const bool real = is_w || xreal[h == 3][e];
            uint8_t* dst = real ? lds + buf * KT_BYTES + h * HALF + (wave + 8 * e) * 1024 : lds + SPARE + wave * 1024;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(is_w ? rw : rx, (lds_void_t*)dst, 16, off, 0, 0, 0);
        }
    };
    const int t_lo = grp ? LO : 0, t_hi = grp ? HI : 0;       // this group's first slot in the x halves
    auto lds_x = [&](int buf, int hi, int i, int ks) {
        return *reinterpret_cast<const u32x4*>(lds + buf * KT_BYTES + (hi ? 3 : 0) * HALF + ((((hi ? t_hi : t_lo) + i) * 2 + ks) * 1024) + (c * 4 + q) * 16);
    };
    auto lds_w = [&](int buf, int hi, int j, int ks) {
        return *reinterpret_cast<const u32x4*>(lds + buf * KT_BYTES + (hi ? 2 : 1) * HALF + (((wc * 2 + j) * 2 + ks) * 1024) + lane * 16);
    };

    // prologue: K-tile 0 whole and K-tile 1's low W -- what phase 0 expects to be in flight behind what it reads
    stage(0, 1, 0); stage(0, 0, 0); stage(0, 2, 0); stage(0, 3, 0); stage(1, 1, 1);
    asm volatile("s_waitcnt vmcnt(4)\n\ts_barrier" ::: "memory");
    if (grp) asm volatile("s_barrier" ::: "memory");          // group 1 starts one interval late

    f32x4 acc[4][MW];
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int i = 0; i < MW; ++i) acc[j][i] = f32x4{0.f, 0.f, 0.f, 0.f};
    u32x4 xr[LO][2], wl[2][2], wl2[2][2], wh[2][2];
#ifdef PP_STAMPS
    unsigned long long* st_buf = reinterpret_cast<unsigned long long*>(lds + SPARE + 8192 + grp * 4096);
    int st_n = 0;
    bool st_on = false;
#endif

#define PP_MFMA(WL, XCNT, XHI)                                                                                           \
    PP_T1();                                                                                                             \
    asm volatile("s_barrier\n\ts_waitcnt lgkmcnt(0)" ::: "memory");                                                      \
    PP_T();                                                                                                              \
    __builtin_amdgcn_sched_barrier(0);                                                                                   \
    __builtin_amdgcn_s_setprio(1);                                                                                       \
    _Pragma("unroll") for (int ks = 0; ks < 2; ++ks)                                                                     \
        _Pragma("unroll") for (int i = 0; i < (XCNT); ++i) {                                                             \
            _Pragma("unroll") for (int j = 0; j < 2; ++j)                                                                \
                acc[j][(XHI) * LO + i] = tg_mfma(WL[j][ks], xr[i][ks], acc[j][(XHI) * LO + i]);                          \
            _Pragma("unroll") for (int j = 0; j < 2; ++j)                                                                \
                acc[2 + j][(XHI) * LO + i] = tg_mfma(wh[j][ks], xr[i][ks], acc[2 + j][(XHI) * LO + i]);                  \
        }                                                                                                                \
    __builtin_amdgcn_s_setprio(0);                                                                                       \
    __builtin_amdgcn_sched_barrier(0);                                                                                   \
    PP_T();                                                                                                              \
    asm volatile("s_barrier" ::: "memory");                                                                              \
    PP_T();
#define PP_KTILE(KT, BUF, WL, WLNEXT)                                                                                    \
    {                                                                                                                    \
        _Pragma("unroll") for (int i = 0; i < LO; ++i)                                                                   \
            _Pragma("unroll") for (int ks = 0; ks < 2; ++ks) xr[i][ks] = lds_x(BUF, 0, i, ks);                           \
        _Pragma("unroll") for (int j = 0; j < 2; ++j)                                                                    \
            _Pragma("unroll") for (int ks = 0; ks < 2; ++ks) wh[j][ks] = lds_w(BUF, 1, j, ks);                           \
        stage((KT) + 1, 0, (BUF) ^ 1);                                                                                   \
        stage((KT) + 1, 2, (BUF) ^ 1);                                                                                   \
        asm volatile("s_waitcnt vmcnt(4)" ::: "memory");                                                                 \
        __builtin_amdgcn_sched_barrier(0);                                                                               \
        PP_MFMA(WL, LO, 0)                                                                                               \
        _Pragma("unroll") for (int i = 0; i < HI; ++i)                                                                   \
            _Pragma("unroll") for (int ks = 0; ks < 2; ++ks) xr[i][ks] = lds_x(BUF, 1, i, ks);                           \
        _Pragma("unroll") for (int j = 0; j < 2; ++j)                                                                    \
            _Pragma("unroll") for (int ks = 0; ks < 2; ++ks) WLNEXT[j][ks] = lds_w((BUF) ^ 1, 0, j, ks);                 \
        stage((KT) + 1, 3, (BUF) ^ 1);                                                                                   \
        stage((KT) + 2, 1, BUF);                                                                                         \
        asm volatile("s_waitcnt vmcnt(4)" ::: "memory");                                                                 \
        __builtin_amdgcn_sched_barrier(0);                                                                               \
        PP_MFMA(WL, HI, 1)                                                                                               \
    }
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) wl[j][ks] = lds_w(0, 0, j, ks);
    PP_C(1);
    for (int u = 0; u < nkt; u += 2) {                        // an odd K-tile count runs one K-tile of zeros (staged out of range)
#ifdef PP_STAMPS
        st_on = st_wave && u >= 8 && u < 24;
        if (u == 8) PP_T();
#endif
        PP_KTILE(u, 0, wl, wl2)
        PP_KTILE(u + 1, 1, wl2, wl)
    }
#undef PP_KTILE
#undef PP_MFMA
    PP_C(2);
    if (!grp) asm volatile("s_barrier" ::: "memory");
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
#if defined(PP_STAMPS) && PP_STAMPS != 3
    if (st_wave)
        for (int i = 0; i < st_n && i < 1023; ++i) g_pp_stamps[grp][1 + i] = st_buf[i];
    if (st_wave) g_pp_stamps[grp][0] = st_n;
#endif
    a.out_f32 = slab;
    tile_epilogue_of<4, MW, GU8>(a, acc, lds, wave, lane, m0 + grp * MW * 16, n0 + wc * 64);
#if defined(PP_STAMPS) && PP_STAMPS == 3
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    PP_C(3);
#endif
}

template <int MW, bool GU8>
static int launch_tile_pp(TileArgs a, hipStream_t st) {
    constexpr int BM = 32 * MW;
    a.mblocks = (a.M + BM - 1) / BM;
    a.nblocks = (a.N + 255) / 256;
    {
        const int per_xcd = (a.mblocks * a.nblocks + 7) / 8;
        int band = 1;
        while (band * band < per_xcd) ++band;
        a.band = band > a.mblocks ? a.mblocks : band;
    }
#ifdef PP_STAMPS
    constexpr int LDS_BYTES = 128 * 1024 + TG_WAVES * 1024 + 8192 + 8192;
#else
    constexpr int LDS_BYTES = 128 * 1024 + TG_WAVES * 1024;
#endif
    static bool attr_set = false;
    if (!attr_set) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_tile_pp_kernel<MW, GU8>), hipFuncAttributeMaxDynamicSharedMemorySize, LDS_BYTES);
        if (e != hipSuccess) { omni_set_error("omni_gemm_tile: LDS attribute: %s", hipGetErrorString(e)); return OMNI_EHIP; }
        attr_set = true;
    }
    hipLaunchKernelGGL((gemm_tile_pp_kernel<MW, GU8>), dim3(a.mblocks * a.nblocks, a.splits), dim3(TG_THREADS), LDS_BYTES, st, a);
    OMNI_CHECK_LAUNCH("omni_gemm_tile");
    return OMNI_OK;
}

template <bool GU8>
static int launch_tile_pp_rows(int bm, const TileArgs& a, hipStream_t st) {
    if (bm == 256) return launch_tile_pp<8, GU8>(a, st);
    if (bm == 224) return launch_tile_pp<7, GU8>(a, st);
    return launch_tile_pp<6, GU8>(a, st);
}

template <int WAVES_N, int WN, int WM, bool GU8>
static int launch_tile(TileArgs a, hipStream_t st, int groups = 1) {
    using G = TileGeom<WAVES_N, WN, WM>;
    a.mblocks = (a.M + G::BM - 1) / G::BM;
    a.nblocks = (a.N + G::BN - 1) / G::BN;
    {
        const int per_xcd = (a.mblocks * a.nblocks + 7) / 8;
        int band = 1;
        while (band * band < per_xcd) ++band;                         // ~sqrt(tiles per XCD)
        a.band = band < 1 ? 1 : (band > a.mblocks ? a.mblocks : band);
    }
    static bool attr_set = false;
    if (!attr_set) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_tile_kernel<WAVES_N, WN, WM, GU8>),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, G::LDS_BYTES);
        if (e != hipSuccess) { omni_set_error("omni_gemm_tile: LDS attribute: %s", hipGetErrorString(e)); return OMNI_EHIP; }
        attr_set = true;
    }
    hipLaunchKernelGGL((gemm_tile_kernel<WAVES_N, WN, WM, GU8>), dim3(a.mblocks * a.nblocks, groups), dim3(TG_THREADS), G::LDS_BYTES, st, a);
    OMNI_CHECK_LAUNCH("omni_gemm_tile");
    return OMNI_OK;
}

// ---- the mid-size form: the same images, MFMA and accumulation order (bit-identical output) for problems of a few rounds of small tiles or less.
// Slices are 64 deep (two 32-deep steps behind one barrier); the ring holds NB of them, and the fragments of the next step are read while the current
// step's MFMAs run: two register sets, one per step parity.  With one wave per SIMD what a slice costs is the instructions around its few MFMAs, so the
// loop is unrolled over the ring (every LDS address an immediate), a piece of a plain product is one load with a scalar offset, and conv windows,
// whose rows move with the segment, are an instantiation of their own.
template <int WAVES, int WAVES_N, int WN, int WM, int NB>
struct MidGeom {
    static constexpr int WAVES_M = WAVES / WAVES_N, NT = WAVES_N * WN, MT = WAVES_M * WM, BN = NT * 16, BM = MT * 16;
    static constexpr int SLICE = (NT + MT) * 2048;
    static constexpr int PW = NT * 2 / WAVES, PX = MT * 2 / WAVES;           // LDS-DMA pieces (1 KB) per wave and slice
    static constexpr int EPI_BYTES = WAVES * 16 * (WN * 64 + 16);
    static constexpr int LDS_BYTES = NB * SLICE > EPI_BYTES ? NB * SLICE : EPI_BYTES;
    static_assert(NT * 2 % WAVES == 0 && MT * 2 % WAVES == 0 && WAVES % 2 == 0 && NB >= 3 && LDS_BYTES <= TG_LDS_MAX && (NB - 2) * (PW + PX) < 64, "geometry");
};

template <int WAVES, int WAVES_N, int WN, int WM, int NB, bool GU8, bool WINDOW>
__global__ __launch_bounds__(WAVES * 64, 2) void gemm_mid_kernel(const TileArgs a_in) {
    using G = MidGeom<WAVES, WAVES_N, WN, WM, NB>;
    TileArgs a = a_in;
    long long x_lo = 0, x_hi = a.x_rows, x_skip = 0;
    if (gridDim.y > 1 || a.group_rows) {
        const int grp = blockIdx.y;
        if (a.group_rows) a.M = min(a.M, a.group_rows[grp]);
        x_lo = grp * a.gx_rows;
        x_hi = min(x_lo + a.M, a.x_rows);
        a.W += (size_t)grp * a.gw_elems;
        const size_t orow = (size_t)grp * a.gout_rows, ocol = (size_t)grp * a.gout_cols;
        if (a.out) a.out += orow * a.ldo + ocol;
        if (a.out2) a.out2 += orow * a.ldo2;
        if (a.out_f32) a.out_f32 += orow * a.ldf + ocol;
        if (a.resid) a.resid += orow * a.ldr;
        x_skip = grp * a.gx_cols;
        a.x += x_skip;
    }
    extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wn = wave % WAVES_N, wm = wave / WAVES_N;
    const int c = lane & 15, q = lane >> 4;
    int n_blk, m_blk;
    {
        const int nwg = gridDim.x, id = blockIdx.x;
        const int xcd = id & 7, slot = id >> 3, per = nwg >> 3, rem = nwg & 7;
        const int tile = (xcd < rem ? xcd * (per + 1) : rem * (per + 1) + (xcd - rem) * per) + slot;
        const int per_band = a.band * a.nblocks;
        const int b = tile / per_band, r = tile - b * per_band;
        const int h = min(a.band, a.mblocks - b * a.band);
        n_blk = r / h;
        m_blk = b * a.band + (r - n_blk * h);
    }
    const int m0 = m_blk * G::BM, n0 = n_blk * G::BN;
    if (m0 >= a.M) return;
    // this workgroup's 32-deep steps [s0, s0 + nsteps): all of them, or one of a.splits runs (its partial sums go to a slab of their own)
    const int all = a.K >> 5;
    const int s0 = a.splits > 1 ? (int)blockIdx.z * all / a.splits : 0, nsteps = (a.splits > 1 ? ((int)blockIdx.z + 1) * all / a.splits : all) - s0;
    if (a.splits > 1) a.out_f32 += (size_t)blockIdx.z * a.slab_stride;

    // staging: piece p = wave + WAVES i of an operand is (tile p >> 1, step p & 1): a wave's pieces are all of ONE step parity.  A piece's address is a
    // per-lane constant (out of the descriptor, i.e. zeros, for rows that are not there) plus the step's scalar offset; the pieces behind the last
    // step fetch the first one's bytes again, for the count: nothing reads them.
    const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc((void*)a.W, 0, (int)((size_t)a.N * a.K * 2), 0x00020000);
    const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc((void*)a.x, 0, a.x_bytes - (int)(x_skip * 2), 0x00020000);
    const int ks = wave & 1;
    unsigned wofs[G::PW], xofs[G::PX];
    int xrow[G::PX];
#pragma unroll
    for (int i = 0; i < G::PW; ++i) {
        const int n16 = (n0 >> 4) + ((wave + WAVES * i) >> 1);
        wofs[i] = n16 * 16 < a.N ? (unsigned)(((size_t)n16 * all + s0 + ks) * 1024 + lane * 16) : TG_OOB;
    }
#pragma unroll
    for (int i = 0; i < G::PX; ++i) {
        xrow[i] = (int)x_lo + m0 + ((wave + WAVES * i) >> 1) * 16 + (lane >> 2) + a.row_off;
        xofs[i] = (unsigned)((xrow[i] * a.ldx + 8 * (lane & 3)) * 2);
        if (!WINDOW) xofs[i] = xrow[i] >= (int)x_lo && xrow[i] < (int)x_hi ? xofs[i] + (unsigned)(s0 + ks) * 64u : TG_OOB;
    }
    int step = ks;                                         // of the next slice to stage
    int seg = WINDOW ? (s0 + ks) * 32 / a.seg_len : 0, cs = (s0 + ks) * 32 - seg * a.seg_len;
    const int seg_row_bytes = a.seg_rows * a.ldx * 2;
    auto piece = [&](int i, int buf) {                     // the wave's i-th piece of that slice into ring place buf
        const int at = step < nsteps ? step - ks : 0;
        uint8_t* dst = lds + wave * 1024 + buf * G::SLICE + (i < G::PW ? i : G::NT * 2 / WAVES + i - G::PW) * (WAVES * 1024);
        if (i < G::PW) {
            const unsigned off = wofs[i < G::PW ? i : 0];
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rw, (lds_void_t*)dst, 16, off, at * 1024, 0, 0);
        } else {
            const int j = i - G::PW;
            const unsigned fixed = xofs[j];
            if (!WINDOW) {
                __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (lds_void_t*)dst, 16, fixed, at * 64, 0, 0);
            } else {
                const int r = xrow[j] + seg * a.seg_rows;
                const unsigned off = r >= (int)x_lo && r < (int)x_hi ? fixed + (unsigned)(seg * seg_row_bytes + cs * 2) : TG_OOB;
                __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (lds_void_t*)dst, 16, off, 0, 0, 0);
            }
        }
    };
    auto staged = [&]() {
        step += 2;
        if (WINDOW) {
            cs += 64;
            while (cs >= a.seg_len) { cs -= a.seg_len; ++seg; }
            if (step >= nsteps) seg = cs = 0;
        }
    };
    f32x4 acc[WN][WM];
#pragma unroll
    for (int j = 0; j < WN; ++j)
#pragma unroll
        for (int i = 0; i < WM; ++i) acc[j][i] = f32x4{0.f, 0.f, 0.f, 0.f};
    u32x4 x0[WM], w0[WN], x1[WM], w1[WN];
    const uint8_t* wp = lds + wn * WN * 2048 + lane * 16;
    const uint8_t* xp = lds + (G::NT + wm * WM) * 2048 + (c * 4 + q) * 16;
    constexpr int P = G::PW + G::PX, HALF = (P + 1) / 2;
#define MID_READ(X, W, BUF, KS)                                                                                          \
    _Pragma("unroll") for (int j = 0; j < WN; ++j) W[j] = *reinterpret_cast<const u32x4*>(wp + (BUF) * G::SLICE + j * 2048 + (KS) * 1024); \
    _Pragma("unroll") for (int i = 0; i < WM; ++i) X[i] = *reinterpret_cast<const u32x4*>(xp + (BUF) * G::SLICE + i * 2048 + (KS) * 1024);
    // one step's MFMAs with pieces [FROM, TO) of the slice being staged dealt out between them
#define MID_MFMA(X, W, FROM, TO, BUF)                                                                                    \
    _Pragma("unroll") for (int j = 0; j < WN; ++j) {                                                                     \
        _Pragma("unroll") for (int p = (FROM) + ((TO) - (FROM)) * j / WN; p < (FROM) + ((TO) - (FROM)) * (j + 1) / WN; ++p) piece(p, BUF); \
        __builtin_amdgcn_sched_barrier(0);                                                                               \
        _Pragma("unroll") for (int i = 0; i < WM; ++i) acc[j][i] = tg_mfma(W[j], X[i], acc[j][i]);                       \
        __builtin_amdgcn_sched_barrier(0);                                                                               \
    }
#pragma unroll
    for (int i = 0; i < NB - 1; ++i) {
#pragma unroll
        for (int p = 0; p < P; ++p) piece(p, i);
        staged();
    }
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((NB - 2) * P) : "memory");
    MID_READ(x0, w0, 0, 0)
    // slice t: its second step's fragments | first step's MFMAs, the first half of slice t + NB - 1 between them (into the place that slice t - 1 left:
    // its last reads retired in front of t - 1's barrier) | slice t + 1 has landed on every wave | its first step's fragments | second step's MFMAs
    // (none where the step count ends on the first) and the other half
    for (int t = 0; t < nsteps;) {
#pragma unroll
        for (int u = 0; u < NB; ++u) {
            MID_READ(x1, w1, u, 1)
            __builtin_amdgcn_sched_barrier(0);
            MID_MFMA(x0, w0, 0, HALF, (u + NB - 1) % NB)
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((NB - 3) * P + HALF) : "memory");
            MID_READ(x0, w0, (u + 1) % NB, 0)
            __builtin_amdgcn_sched_barrier(0);
            if (t + 1 >= nsteps) { t = nsteps; break; }
            MID_MFMA(x1, w1, HALF, P, (u + NB - 1) % NB)
            staged();
            t += 2;
            if (t >= nsteps) break;
        }
    }
#undef MID_READ
#undef MID_MFMA
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");      // the ring is dead: its tail loads landed
    tile_epilogue_of<WN, WM, GU8>(a, acc, lds, wave, lane, m0 + wm * WM * 16, n0 + wn * WN * 16);
}

template <int WAVES, int WAVES_N, int WN, int WM, int NB, bool GU8, bool WINDOW>
static int launch_mid(TileArgs a, hipStream_t st, int groups) {
    using G = MidGeom<WAVES, WAVES_N, WN, WM, NB>;
    a.mblocks = (a.M + G::BM - 1) / G::BM;
    a.nblocks = (a.N + G::BN - 1) / G::BN;
    {
        const int per_xcd = (a.mblocks * a.nblocks + 7) / 8;
        int band = 1;
        while (band * band < per_xcd) ++band;
        // Row blocks of up to 5 stay together: a panel of W, which comes out of HBM, is fetched by one XCD then, and the rows of so few blocks fit its L2; more in
        // bands of equal height, not 6 and 1.  The same products in a whole forward, us (in launches of one product in turn x stays in the L2s and the
        // difference is another): one prompt of 130 tokens 459 / 447, 2 of 251 1101 / 1076, 48 decoded tokens beside two portions 1477 / 1454; the mean of forty
        // forwards 0.5 % less (up to 8 blocks together 0.6, with products of 16 rows in two runs of K slower).  W fetched past the caches where only one XCD reads
        // it is up to 20 % faster in such launches, and up to 7 % slower in forwards of a model whose weights the last-level cache holds.
        const int bands = (a.mblocks + band - 1) / band;
        a.band = a.mblocks <= 5 ? a.mblocks : (a.mblocks + bands - 1) / bands;
    }
    static bool attr_set = false;
    if (!attr_set) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_mid_kernel<WAVES, WAVES_N, WN, WM, NB, GU8, WINDOW>), hipFuncAttributeMaxDynamicSharedMemorySize, G::LDS_BYTES);
        if (e != hipSuccess) { omni_set_error("omni_gemm_tile: LDS attribute: %s", hipGetErrorString(e)); return OMNI_EHIP; }
        attr_set = true;
    }
    hipLaunchKernelGGL((gemm_mid_kernel<WAVES, WAVES_N, WN, WM, NB, GU8, WINDOW>), dim3(a.mblocks * a.nblocks, groups, a.splits), dim3(WAVES * 64), G::LDS_BYTES, st, a);
    OMNI_CHECK_LAUNCH("omni_gemm_tile");
    return OMNI_OK;
}

// waves, waves along n, n-tiles x m-tiles per wave, ring: 32 x 32 | 32 x 64 | 64 x 64 | 64 x 128 (rows x columns; two workgroups fit a CU) |
// 128 x 128 | 256 x 128 | 128 x 256 (one) | 96 x 64 (two) | 192 x 128 | 96 x 128 (one)
#define MID_LIST(X) X(0, 4, 2, 1, 1, 9) X(1, 4, 2, 2, 1, 6) X(2, 4, 2, 2, 2, 4) X(3, 8, 4, 2, 2, 3) X(4, 8, 4, 2, 4, 4) X(5, 8, 2, 4, 4, 3) X(6, 8, 4, 4, 4, 3) \
                    X(7, 4, 2, 2, 3, 4) X(8, 8, 2, 4, 3, 4) X(9, 4, 2, 4, 3, 4)
template <bool GU8, bool WINDOW>
static int launch_mid_of(int geom, const TileArgs& a, hipStream_t st, int groups) {
    switch (geom) {
#define MID_CASE(I, A, B, C, D, E) case I: return launch_mid<A, B, C, D, E, GU8, WINDOW>(a, st, groups);
        MID_LIST(MID_CASE)
#undef MID_CASE
    }
    return OMNI_EINVAL;
}

// ---- up to 64 rows of a plain product (tile_hint 17): a wave alone owns 16 rows x 16 columns of one run of K and takes both operands straight into registers, P steps in flight.  One
// chain of MFMAs over K as in every tile: the same bits.  What bounds it: trips to memory, 24 KB of W a wave in flight (8 steps 5.1 of the first, 16 4.4, 32 4.3), and the rows, which
// every wave of a column reads for itself.  Us, weights out of HBM, the rule's tile / this, rows x columns x K: 12 x 3072 x 1024 5.6 / 4.0, 12 x 1024 x 1024 in four runs of K 4.0 / 2.7,
// 12 x 1024 x 3072 in four 5.1 / 3.8; 25 rows 5.6 / 5.1, 4.1 / 3.0, 5.3 / 4.6; 33 5.7 / 5.7, 4.1 / 3.2, 5.3 / 5.3; 64 5.8 / 6.6, 4.4 / 3.8, 5.5 / 6.9.
template <bool F32>
__global__ __launch_bounds__(64) void gemm_few_kernel(const TileArgs a) {
    constexpr int P = 24;
    const int lane = threadIdx.x, c = lane & 15, q = lane >> 4, all = a.K >> 5;
    const int s0 = (int)blockIdx.z * all / a.splits, n = ((int)blockIdx.z + 1) * all / a.splits - s0;
    const int m = blockIdx.y * 16 + c, col = blockIdx.x * 16 + 4 * q;
    const u32x4* wp = reinterpret_cast<const u32x4*>(a.W + ((size_t)blockIdx.x * all + s0) * 512 + lane * 8);
    const u32x4* xp = reinterpret_cast<const u32x4*>(a.x + (size_t)min(m, a.M - 1) * a.ldx + s0 * 32 + 8 * q);      // rows past M: the last one again, not stored
    u32x4 W[P], X[P];
    auto load = [&](int d, int s) {
        W[d] = __builtin_nontemporal_load(wp + s * 64);
        X[d] = xp[s * 4];
    };
#pragma unroll
    for (int d = 0; d < P; ++d)
        if (d < n) load(d, d);
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    for (int s = 0; s < n; s += P)
#pragma unroll
        for (int d = 0; d < P; ++d) {
            if (s + d >= n) break;
            acc = tg_mfma(W[d], X[d], acc);
            if (s + d + P < n) load(d, s + d + P);
        }
    if (m >= a.M) return;
    if (F32) *reinterpret_cast<f32x4*>(a.out_f32 + blockIdx.z * a.slab_stride + (size_t)m * a.ldf + col) = acc;
    else *reinterpret_cast<uint2*>(a.out + (size_t)m * a.ldo + col) = make_uint2(pack_bf2(acc[0], acc[1]), pack_bf2(acc[2], acc[3]));
}

static int launch_few(const TileArgs& a, bool f32, hipStream_t st) {
    const dim3 grid(a.N / 16, (a.M + 15) / 16, a.splits), block(64);
    if (f32) hipLaunchKernelGGL((gemm_few_kernel<true>), grid, block, 0, st, a);
    else hipLaunchKernelGGL((gemm_few_kernel<false>), grid, block, 0, st, a);
    OMNI_CHECK_LAUNCH("omni_gemm_tile");
    return OMNI_OK;
}

// ---- which tile.  Every geometry accumulates in the same order, so the choice moves time only.  A grid costs its rounds: 256 workgroups run at a time,
// one per CU (512 where two fit), and a round costs a prologue and an epilogue (`round`) and the slices of K (`slice`, per 64-deep slice).  What a slice
// costs is what a CU takes in -- 60 - 90 GB/s of operands in every geometry (a slice of the 32 x 64 tile is 12 KB in 0.17 us, of the 256 x 256 tile
// 64 KB in 1.1 - 1.3 us) -- so small grids want small tiles on all 256 CUs and large ones tall tiles.  Two workgroups on a CU share that rate
// but hide each other's barriers: 0.44 us for a slice of each of two 64 x 64 tiles, 0.27 alone.
// Numbers: ns above what every launch costs, least squares over M 13 ... 6300 x the weight shapes of the language models, talkers and the vocoder by every tile and count
// of partial sums; some were then moved by a few per cent, with those of omni_gemm_tile_splits, to where the fp32 products' counts are the better ones and no other product of
// 1400 takes a slower tile.  What the rule picks is 0.8 % behind the best on average, 1.0 % over 398 rows and sizes it was not found on (before: 0.9 %, of the fp32 products
// 1.2 %); 38 of 1323 take more than 3 % longer than under the rule of fewer tiles before it, all together 4 % less.  Table: profiles/gemm_tile_sweep.txt.  Every weight
// comes out of HBM there, 700 MB of them in turn, as in a step: weights that are in the last-level cache want fewer, larger tiles (50 x 1024 x 3072 by 32 x 32 9.8, by 32 x 64
// 11.7; the other way round from 150 MB in turn), and numbers searched on those cost the vocoder 2 %.
// The heights between the powers of two are there for the rounds: a product of 500 rows by 9216 columns is 288 tiles of 128 x 128 on 256 CUs (two rounds,
// 36 us), 144 of 256 x 128 (33.2) and 216 of 192 x 128 (24.7); 200 x 4608 x 1024 9.1 -> 8.0 by 96 x 64, 251 x 5120 x 2048 18.7 -> 13.1, 800 x 5120 x 2048 32 -> 22 by
// 192 x 128, 502 x 5120 x 2048 20.6 -> 16.5 by 96 x 128.  On average over those products the three are worth 3.3 %.
enum { KIND_MID, KIND_PP, KIND_LARGE };
struct TileChoice {
    int kind, geom, bm, bn;          // geom: MID_LIST index, or rows of the two-group / lockstep tile
    int round1, slice1, round2, slice2;      // alone on a CU; two per CU (0: one fits)
};
#define MID_SIZE_CASE(I, A, B, C, D, E) if (I == i) return rows ? MidGeom<A, B, C, D, E>::BM : MidGeom<A, B, C, D, E>::BN;
static constexpr int mid_size(int i, bool rows) { MID_LIST(MID_SIZE_CASE) return 0; }
#undef MID_SIZE_CASE
#define MID(I) KIND_MID, I, mid_size(I, true), mid_size(I, false)
static const TileChoice TILE_CHOICES[] = {
    {MID(0), 2484, 140, 2750, 249}, {MID(1), 2402, 196, 2909, 316}, {MID(2), 2563, 280, 3110, 432}, {MID(3), 3100, 466, 4990, 650},
    {MID(4), 4400, 447},            {MID(5), 5450, 871},            {MID(6), 5800, 912},
    {MID(7), 3010, 306, 4090, 542}, {MID(8), 5178, 572},            {MID(9), 3999, 425},
    {KIND_PP, 192, 192, 256, 8570, 996},     {KIND_PP, 224, 224, 256, 9350, 1044},    {KIND_PP, 256, 256, 256, 10300, 1088},
    {KIND_LARGE, 192, 192, 256, 9600, 1015}, {KIND_LARGE, 224, 224, 256, 10300, 1090}, {KIND_LARGE, 256, 256, 256, 11800, 1150},
    {KIND_LARGE, 0, 256, 192, 9600, 1040},   {KIND_LARGE, 0, 512, 128, 11800, 1450},  {KIND_LARGE, 0, 512, 96, 11300, 1320},
};
#undef MID
static const TileChoice& pick_tile(int M, int N, int K, int groups, int splits, bool plain, bool gu8, long long* ns) {
    const TileChoice* best = nullptr;
    long long least = 0;
    const long long slices = (K / 32 / splits + 1) / 2;
    const int large_bn = N % 256 == 0 ? 256 : gu8 ? 128 : N % 192 == 0 ? 192 : N % 128 == 0 ? 128 : N % 96 == 0 ? 96 : 0;
    for (const TileChoice& c : TILE_CHOICES) {
        if (c.kind == KIND_PP && !plain) continue;                            // the two-group tile takes a plain product, the lockstep ones the others
        if (c.kind == KIND_LARGE && (c.bn != large_bn || (plain && c.bn == 256) || splits > 1)) continue;
        // 96 x 128 is four waves: where it makes as many row blocks as 128 x 128 (rows 257 ... 288; below, its blocks are the fuller ones) eight are faster, 284 x 7936 x 2048 19.5 / 18.0 us
        if (c.kind == KIND_MID && c.geom == 9 && M > 256 && (M + 95) / 96 == (M + 127) / 128) continue;
        const long long tiles = (long long)((M + c.bm - 1) / c.bm) * ((N + c.bn - 1) / c.bn) * groups * splits;
        long long t;
        // (a CU that gets a third small tile while the first two run does not wait for a round of two)
        if (c.slice2 && tiles > 256) t = (c.round2 + slices * c.slice2) * ((tiles + 255) / 256) / 2;
        else t = (c.round1 + slices * c.slice1) * ((tiles + 255) / 256);
        // 192 x 128 in runs of K costs 80 ns a slice more than whole: 700 x 2048 x 9216 in four runs 43 us, by 96 x 128 in two 35
        if (c.kind == KIND_MID && c.geom == 8 && splits > 1) t += 80 * slices * ((tiles + 255) / 256);
        if (!best || t < least) { best = &c; least = t; }
    }
    if (ns) *ns = least;
    return *best;
}

// Partial sums for the reader of an fp32 product to add up: as many as make the product and their extra traffic (written here, read there) cheapest; at
// most 4, what the readers take (OMNI_STREAM_MAX_SPLITS).  The traffic at 3.5 TB/s and 124 ns, found with the tiles' numbers: over 325 fp32 products of up to 1100 rows
// product and reader (a slab read at 8 TB/s and 30 ns) are 0.6 % behind the best tile and count on average.  At 3.8 TB/s and 100 ns, from before the tiles' numbers moved,
// 1.2 %: 66 x 2080 x 2048 in four took 7.6 us, in two 6.4, 800 x 2048 x 7936 in three 40 to 43, in two 34.
extern "C" int omni_gemm_tile_splits(int M, int N, int K) {
    int best = 1;
    long long least = -1;
    for (int s = 1; s <= 4; ++s) {
        if (s > 1 && (K / 32 < 8 * s || N % 16)) break;
        long long t;
        pick_tile(M, N, K, 1, s, true, false, &t);
        t += (long long)(s - 1) * M * N * 8 / 3500 + (s > 1 ? 124 : 0);
        if (least < 0 || t < least) { least = t; best = s; }
    }
    return best;
}

extern "C" int omni_gemm_tile(const omni_tile_gemm* g, void* stream) {
    OMNI_CHECK_ARG(g && g->x && g->w && (g->out || g->out2 || g->out_f32), "omni_gemm_tile: null argument");
    OMNI_CHECK_ARG(g->M > 0 && g->N > 0 && g->N % 16 == 0 && g->K > 0 && g->K % 32 == 0, "omni_gemm_tile: M=%d N=%d K=%d (N %% 16, K %% 32)", g->M, g->N, g->K);
    const int seg_len = g->seg_len > 0 ? g->seg_len : g->K;
    OMNI_CHECK_ARG(seg_len % 32 == 0 && g->K % seg_len == 0, "omni_gemm_tile: seg_len=%d must divide K=%d and be a multiple of 32", seg_len, g->K);
    OMNI_CHECK_ARG(g->ldx % 8 == 0 && g->ldx >= seg_len, "omni_gemm_tile: ldx=%d (>= seg_len, multiple of 8)", g->ldx);
    OMNI_CHECK_ARG(g->x_rows > 0 && g->x_rows * (int64_t)g->ldx * 2 < (int64_t)TG_OOB, "omni_gemm_tile: x of %lld rows x %d exceeds the 2 GB descriptor", (long long)g->x_rows, g->ldx);
    OMNI_CHECK_ARG((int64_t)g->N * g->K * 2 < (int64_t)TG_OOB, "omni_gemm_tile: W exceeds the 2 GB descriptor");
    const bool gu8 = g->act == OMNI_TILE_ACT_SILU_MUL_GU8;
    OMNI_CHECK_ARG(g->act >= OMNI_TILE_ACT_NONE && g->act <= OMNI_TILE_ACT_GELU_MUL, "omni_gemm_tile: act=%d", g->act);
    OMNI_CHECK_ARG(g->act < OMNI_TILE_ACT_XIELU || (!g->bias && !g->scale && !g->resid && !g->out2), "omni_gemm_tile: act=%d takes no bias, scale, residual or second output", g->act);
    OMNI_CHECK_ARG(g->act != OMNI_TILE_ACT_SILU_SIGMOID || (g->act_cols >= 0 && g->act_cols % 4 == 0), "omni_gemm_tile: act_cols=%d (%% 4)", g->act_cols);
    OMNI_CHECK_ARG(g->act != OMNI_TILE_ACT_GELU_MUL || (g->mul_table && g->mul_ids && g->mul_rows > 0 && g->mul_ld >= g->N && g->mul_ld % 8 == 0 && g->out && !g->out2 && !g->resid &&
                                                        g->groups <= 1), "omni_gemm_tile: the row table takes ids, mul_ld >= N (%% 8), a bf16 output and one group");
    OMNI_CHECK_ARG(g->tile_hint >= 0 && g->tile_hint <= 17, "omni_gemm_tile: tile_hint=%d", g->tile_hint);
    OMNI_CHECK_ARG(g->tile_hint < 3 || g->tile_hint > 7 || g->N % 256 == 0, "omni_gemm_tile: tile_hint=%d needs N %% 256 == 0", g->tile_hint);
    OMNI_CHECK_ARG(!gu8 || (g->out && !g->resid && !g->out2 && !g->out_f32), "omni_gemm_tile: SiLU-mul takes out only");
    OMNI_CHECK_ARG(!g->out2 || (g->snake_alpha && g->snake_inv_beta), "omni_gemm_tile: out2 needs the snake parameters");
    const int nout = gu8 ? g->N / 2 : g->N;
    OMNI_CHECK_ARG((!g->out || (g->ldo >= nout && g->ldo % 8 == 0)) && (!g->resid || (g->ldr >= nout && g->ldr % 4 == 0)) &&
                   (!g->out2 || (g->ldo2 >= nout && g->ldo2 % 8 == 0)) && (!g->out_f32 || (g->ldf >= nout && g->ldf % 4 == 0)),
                   "omni_gemm_tile: ldo / ldr / ldo2 / ldf (>= N; multiples of 8 (bf16) / 4 (fp32))");
    TileArgs a;
    a.x = (const uint16_t*)g->x; a.x_rows = g->x_rows; a.ldx = g->ldx;
    a.seg_len = seg_len; a.seg_rows = g->seg_rows; a.row_off = g->row_off;
    a.W = (const uint16_t*)g->w; a.bias = g->bias; a.scale = g->scale;
    a.resid = g->resid; a.ldr = g->ldr;
    a.out_f32 = g->out_f32; a.ldf = g->ldf;
    a.out = (uint16_t*)g->out; a.ldo = g->ldo;
    a.out2 = (uint16_t*)g->out2; a.ldo2 = g->ldo2; a.snake_alpha = g->snake_alpha; a.snake_inv_beta = g->snake_inv_beta;
    a.M = g->M; a.N = g->N; a.K = g->K; a.act = g->act;
    const int groups = g->groups > 1 ? g->groups : 1;
    OMNI_CHECK_ARG(groups <= 65535, "omni_gemm_tile: groups=%d", g->groups);
    OMNI_CHECK_ARG(groups == 1 || (seg_len == g->K && g->row_off == 0 && g->x_group_rows >= 0 && g->w_group_elems >= 0 && g->out_group_rows >= 0),
                   "omni_gemm_tile: a grouped launch is a plain GEMM per group (no conv window) with non-negative group strides");
    OMNI_CHECK_ARG(groups == 1 || (int64_t)groups * g->w_group_elems * 2 + (int64_t)g->N * g->K * 2 < ((int64_t)1 << 40), "omni_gemm_tile: W groups");
    a.gx_rows = groups > 1 ? g->x_group_rows : 0; a.gw_elems = groups > 1 ? g->w_group_elems : 0; a.gout_rows = groups > 1 ? g->out_group_rows : 0;
    a.group_rows = g->group_rows;
    a.act_p = g->act_p; a.act_n = g->act_n; a.act_cols = g->act_cols;
    a.mul_table = (const uint16_t*)g->mul_table; a.mul_ids = g->mul_ids; a.mul_rows = g->mul_rows; a.mul_ld = g->mul_ld;
    // groups as column ranges of one token array: group g reads x columns [g * x_group_cols, + K) and writes columns [g * out_group_cols, + N)
    OMNI_CHECK_ARG(groups == 1 || (g->x_group_cols >= 0 && g->out_group_cols >= 0 && g->x_group_cols % 8 == 0 && g->out_group_cols % 8 == 0 &&
                                   (groups - 1) * g->x_group_cols + seg_len <= g->ldx &&
                                   (!g->out || (groups - 1) * g->out_group_cols + nout <= g->ldo) &&
                                   (!g->out_f32 || (groups - 1) * g->out_group_cols + nout <= g->ldf) &&
                                   (g->out_group_cols == 0 || (!g->out2 && !g->resid))),
                   "omni_gemm_tile: group columns leave the rows of x / out");
    a.gx_cols = groups > 1 ? g->x_group_cols : 0; a.gout_cols = groups > 1 ? g->out_group_cols : 0;
    // up to the end of the last row's last column: rows of a wider array need not be followed by anything
    a.x_bytes = (int)(((g->x_rows - 1) * g->ldx + (groups - 1) * a.gx_cols + seg_len) * 2);
    hipStream_t st = (hipStream_t)stream;
    const int N = g->N;
    OMNI_CHECK_ARG(g->k_splits >= 0 && g->k_splits <= 4 && (g->k_splits <= 1 || (tile_epi(a) == EPI_F32 && groups == 1 && g->k_splits <= g->K / 32 &&
                   g->slab_stride >= (int64_t)(g->M - 1) * g->ldf + N && g->slab_stride % 4 == 0)), "omni_gemm_tile: k_splits=%d (<= K / 32; one group, fp32 output alone)", g->k_splits);
    a.splits = g->k_splits > 1 ? g->k_splits : 1; a.slab_stride = g->slab_stride;
    // tile_hint: 1 the large lockstep tiles, 2 and 8 ... 16 the mid-size ones, 17 a wave per 16 x 16, 3 / 4 lockstep and 5 / 6 / 7 two-group at 224 / 192 and 256 / 224 / 192 rows
    const bool plain = groups == 1 && !g->group_rows && seg_len == g->K && g->row_off == 0;
    OMNI_CHECK_ARG(g->tile_hint < 5 || g->tile_hint > 7 || plain, "omni_gemm_tile: tile_hint=%d (two-group tile) takes a plain GEMM", g->tile_hint);
    OMNI_CHECK_ARG(a.splits == 1 || g->tile_hint == 0 || g->tile_hint == 2 || g->tile_hint >= 5, "omni_gemm_tile: tile_hint=%d takes no k_splits", g->tile_hint);
    if (g->tile_hint == 17) {
        const int epi = tile_epi(a);
        OMNI_CHECK_ARG(plain && !gu8 && (epi == EPI_PLAIN || epi == EPI_F32) && g->M <= 64 && g->M <= g->x_rows && ((uintptr_t)g->x & 15) == 0,
                       "omni_gemm_tile: tile_hint=17 takes a plain product of up to 64 rows, x aligned to 16 bytes, bf16 or fp32 output alone (M=%d)", g->M);
        return launch_few(a, epi == EPI_F32, st);
    }
    int kind = KIND_LARGE, geom = 256;
    switch (g->tile_hint) {
        case 0: {
            const TileChoice& c = pick_tile(g->M, N, g->K, groups, a.splits, plain, gu8, nullptr);
            kind = c.kind; geom = c.geom;
            break;
        }
        case 1: break;
        case 2: kind = KIND_MID; geom = 3; break;
        case 3: geom = 224; break;
        case 4: geom = 192; break;
        case 5: case 6: case 7: kind = KIND_PP; geom = 256 - 32 * (g->tile_hint - 5); break;
        default: kind = KIND_MID; geom = g->tile_hint - 8; if (geom >= 3) ++geom;
    }
    const bool window = seg_len != g->K;
    if (kind == KIND_MID && !(gu8 && window))
        return gu8 ? launch_mid_of<true, false>(geom, a, st, groups) : window ? launch_mid_of<false, true>(geom, a, st, groups) : launch_mid_of<false, false>(geom, a, st, groups);
    if (kind == KIND_PP) return gu8 ? launch_tile_pp_rows<true>(geom, a, st) : launch_tile_pp_rows<false>(geom, a, st);
    // <waves along n, n tiles per wave, m tiles per wave>: 256 x 256 (224, 192 rows) | 256 x 192 | 512 x 128 | 512 x 96 output tiles
    if (N % 256 == 0) {
        if (geom == 224) return gu8 ? launch_tile<4, 4, 7, true>(a, st, groups) : launch_tile<4, 4, 7, false>(a, st, groups);
        if (geom == 192) return gu8 ? launch_tile<4, 4, 6, true>(a, st, groups) : launch_tile<4, 4, 6, false>(a, st, groups);
        return gu8 ? launch_tile<2, 8, 4, true>(a, st, groups) : launch_tile<2, 8, 4, false>(a, st, groups);
    }
    if (gu8) return launch_tile<1, 8, 4, true>(a, st, groups);
    if (N % 192 == 0) return launch_tile<2, 6, 4, false>(a, st, groups);
    if (N % 128 == 0) return launch_tile<1, 8, 4, false>(a, st, groups);
    if (N % 96 == 0) return launch_tile<1, 6, 4, false>(a, st, groups);
    return N > 128 ? launch_tile<2, 8, 4, false>(a, st, groups) : launch_tile<1, 8, 4, false>(a, st, groups);
}
