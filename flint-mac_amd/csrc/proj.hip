// Attention projections in the engine's GGUF weight formats, for gfx950:
//   * get_rows_kernel: rows dequantised to fp32 (Engine::debug_get_row,
//     /root/reference/src/engine.mm:1370-1383, kernel k_get_row, fused.metal:589-600; and
//     the prefill's embedding, k_embed_rows, prefill.metal:272, engine.mm:1067-1069);
//   * matvec_kernel: y = W x with 2048- or 4096-element rows, optionally on RMSNorm(x) * g
//     (the q/k/v projections, engine.mm:728-732) or added to y (o_proj with the residual,
//     engine.mm:811);
//   * matvec_tokens_kernel: the same for a few tokens.
//
// Formats: ggml's block layouts (/root/reference/third_party/ggml/ggml-common.h), type ids
// from /root/reference/src/gguf.h:14-19. Every row is cut into 32-element sub-blocks, the
// unit all formats share: a q8_0 block, a half of a q5_K/iq4_xs 64-element pair, two q6_K
// 16-element groups. Lane l of a wave owns sub-blocks l, l + 64, ..., so the 32 x values it
// multiplies stay in its registers. Dequantisation repeats ggml's float operations in order
// with contraction off, so get_row is bit-identical to dequantize_row_*
// (/root/reference/src/ref/dequant_gen.c).
//
// Matvec layout (HBM-bound on the weight bytes): a wave takes R consecutive rows. It requests
// their bytes at kernel start (16-byte loads, coalesced) while the workgroup reads x once
// into LDS (normalised there when the RMSNorm is fused). The rows' bytes then go into an
// LDS area of the wave's own; each lane reads the bytes of its sub-block from LDS at the
// alignment the format gives (q8_0 and q6_K blocks are only 2-byte aligned: q8_0 as aligned
// words realigned in registers), decodes 32 weights and accumulates their products with x in
// fp32; a wave-wide sum gives y[row].
// f32/f16/bf16 rows are read straight from HBM (64- or 128-byte sub-blocks, aligned).
#include <hip/hip_runtime.h>

#include <type_traits>

#include "common.h"
#include "dequant.h"
#include "flint_attn_internal.h"

namespace flint {



// ---------------------------------------------------------------------------
// get_rows: workgroup (c, i) dequantises sub-blocks 64c .. 64c+63 of row rows[i] into
// out + i * out_stride, so one launch serves every token of a prefill's embedding (the
// reference's k_embed_rows, prefill.metal:272). The row's bytes start on a block boundary;
// they are staged through LDS with 2-byte loads (any row alignment the block size allows).
constexpr int GR_STAGE = 64 * 32 * 4;  // bytes of 64 f32 sub-blocks, the largest chunk
__global__ __launch_bounds__(64) void get_rows_kernel(const RowsParams P) {
    __shared__ __align__(16) uint8_t stage[GR_STAGE];
    const int lane = threadIdx.x, c = blockIdx.x, i = blockIdx.y;
    const int type = P.type, n_sub = P.n_sub;
    const uint8_t *__restrict__ row = P.w + (size_t)P.rows[i] * (size_t)P.row_bytes;
    float *__restrict__ out = P.out + (size_t)i * (size_t)P.out_stride;
    const int sub0 = 64 * c, nsub = min(64, n_sub - sub0);
    const int be = w_block_elems(type), bb = w_block_bytes(type);
    const size_t off = (size_t)sub0 * 32 / be * bb;
    const int nbytes = nsub * 32 / be * bb;  // chunks are whole blocks (64 is a multiple of 8)
    const uint16_t *src = (const uint16_t *)(row + off);
    uint16_t *dst = (uint16_t *)stage;
    for (int j = lane; j < nbytes / 2; j += 64) dst[j] = src[j];
    __syncthreads();
    if (lane < nsub) {
        float w[32];
        deq32(type, stage, lane, w);
        f32x4 *o = (f32x4 *)(out + 32 * (size_t)(sub0 + lane));
#pragma unroll
        for (int k = 0; k < 8; k++) o[k] = f32x4{w[4 * k], w[4 * k + 1], w[4 * k + 2], w[4 * k + 3]};
    }
}

// ---------------------------------------------------------------------------
// matvec: one token. A workgroup of MV_WAVES waves serves MV_WAVES * R consecutive rows.
// x (times the RMSNorm gains, when norm_w is given; the norm's scale multiplies the row sums)
// is read from HBM once per workgroup into LDS; each wave then takes R rows, whose bytes it
// requested at kernel start, and reads its lanes' 32-element slices of x from LDS. The arguments are plain
// words, 14 of them, so that they are preloaded into SGPRs: with them in a struct every wave's first loads
// waited for the arguments' round trip (q8_0 weights from HBM: q/k/v 5.74 -> 5.31 us, o 4.88 -> 4.45; a step
// of Flint's 49 layers at 6001 tokens 878 -> 831).
constexpr int MV_WAVES = 4;

// x in LDS: float4 column c (elements 4c .. 4c+3) of sub-block s at s * 32 + 4 (c ^ ((s >> 1) & 7)).
// Lane l reads its own sub-block's eight columns one instruction at a time; unswizzled, the
// 64 lanes' addresses 128 bytes apart fell on two groups of 4 banks (32-way conflicts), and
// with the swizzle any 8 consecutive lanes read 8 different columns.
__device__ inline int xs_index(int e) {
    const int s = e >> 5, c = (e >> 2) & 7;
    return s * 32 + 4 * (c ^ ((s >> 1) & 7)) + (e & 3);
}

// Sum over the 64 lanes in double, on VALU lane permutes (each 32-bit half moved by DPP within
// rows of 16, then v_permlane16/32_swap across rows): no LDS round trips (a __shfl_xor chain
// costs six dependent ds_bpermute pairs).
template <int CTRL>
__device__ inline double dpp_f64(double v) {
    const uint64_t b = __builtin_bit_cast(uint64_t, v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)b, CTRL, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)(b >> 32), CTRL, 0xf, 0xf, false);
    return __builtin_bit_cast(double, ((uint64_t)(uint32_t)hi << 32) | (uint32_t)lo);
}
__device__ inline double wave_sum_f64(double v) {
    v += dpp_f64<DPP_ROR8>(v);
    v += dpp_f64<DPP_ROR4>(v);
    v += dpp_f64<DPP_ROR2>(v);
    v += dpp_f64<DPP_ROR1>(v);  // every lane of a row of 16 holds the row's sum
    uint64_t b = __builtin_bit_cast(uint64_t, v);
    const auto l16 = __builtin_amdgcn_permlane16_swap((uint32_t)b, (uint32_t)b, false, false);
    const auto h16 = __builtin_amdgcn_permlane16_swap((uint32_t)(b >> 32), (uint32_t)(b >> 32), false, false);
    v = __builtin_bit_cast(double, ((uint64_t)h16[0] << 32) | l16[0]) + __builtin_bit_cast(double, ((uint64_t)h16[1] << 32) | l16[1]);
    b = __builtin_bit_cast(uint64_t, v);
    const auto l32 = __builtin_amdgcn_permlane32_swap((uint32_t)b, (uint32_t)b, false, false);
    const auto h32 = __builtin_amdgcn_permlane32_swap((uint32_t)(b >> 32), (uint32_t)(b >> 32), false, false);
    return __builtin_bit_cast(double, ((uint64_t)h32[0] << 32) | l32[0]) + __builtin_bit_cast(double, ((uint64_t)h32[1] << 32) | l32[1]);
}

template <int K, int R>
__global__ __launch_bounds__(64 * MV_WAVES) void matvec_kernel(const uint8_t *w0, const uint8_t *w1, const uint8_t *w2,
                                                               const float *xt, const float *norm_w, float *yt,
                                                               const uint32_t types, const float eps) {
    constexpr int SUBS = K / 32 / 64;               // sub-blocks per lane
    constexpr int QBYTES = K / 32 * 34;             // largest quantised row (q8_0)
    constexpr int UNITS = (QBYTES / 16 + 63) / 64;  // 16-byte loads per lane for it
    constexpr int XPT = K / (64 * MV_WAVES);        // x elements per thread in the shared pass
    constexpr bool QKV = K == N_EMBD, add = !QKV;   // three segments of normed inputs, or one added to y
    __shared__ __align__(16) float xs[K];           // the (normalised) x row
    constexpr int QROW = (QBYTES + 4 + 15) / 16 * 16;  // a staged row, + 4 bytes read past a q8_0 row's end
    __shared__ __align__(16) uint8_t stage[MV_WAVES][R][QROW];
    __shared__ double part[MV_WAVES];
    // wave index made scalar: the row segment, its type and its row pointer are then known
    // to be wave-uniform (scalar branches for the format, scalar load bases)
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int row0 = (blockIdx.x * MV_WAVES + wave) * R;  // R rows, all in one segment
    const bool in2 = QKV && row0 >= Q_DIM + KV_DIM, in1 = QKV && !in2 && row0 >= Q_DIM;
    MatvecSeg S;
    S.w = in2 ? w2 : in1 ? w1 : w0;
    S.type = (types >> (in2 ? 16 : in1 ? 8 : 0)) & 0xff;
    S.row0 = in2 ? Q_DIM + KV_DIM : in1 ? Q_DIM : 0;
    S.row_bytes = K / w_block_elems(S.type) * w_block_bytes(S.type);
    const uint8_t *wrow = S.w + (size_t)(row0 - S.row0) * S.row_bytes;
    const bool fl = w_is_float(S.type);

    // x and the gains: XPT consecutive elements per thread, 16-byte loads
    f32x4 xv[XPT / 4], gv[XPT / 4];
#pragma unroll
    for (int k = 0; k < XPT / 4; k++) xv[k] = *(const f32x4 *)(xt + XPT * tid + 4 * k);
    if (QKV) {
#pragma unroll
        for (int k = 0; k < XPT / 4; k++) gv[k] = *(const f32x4 *)(norm_w + XPT * tid + 4 * k);
    }
    // this wave's rows, as quantised-row units (float rows are read again in the dot loop;
    // the units loaded here are within their rows and go unused). Every lane loads (lanes
    // past the row's end re-read its last unit and do not store it), so the loads are
    // unconditional and the RMSNorm below waits for x and the gains only.
    u32x4 u[R][UNITS];
    const int n_units = S.row_bytes >> 4;
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
        for (int k = 0; k < UNITS; k++) {
            const int idx = min(lane + 64 * k, n_units - 1);
            u[r][k] = ((const u32x4 *)(wrow + (size_t)r * S.row_bytes))[idx];
        }
    if (QKV) {
        // RMSNorm as the CPU reference (ref_model.cpp:45-50): double sum of squares, float
        // scale = 1 / sqrt(ss / K + eps). The scale is one number per token, so W (x scale g) =
        // scale (W (x g)): x g goes to LDS at once and the scale multiplies each row's sum at the
        // end (within a few ulp of scaling x first), so the reduction and its barrier are off the
        // path to the dots (one workgroup barrier instead of two).
        double ss = 0;
#pragma unroll
        for (int k = 0; k < XPT / 4; k++)
#pragma unroll
            for (int e = 0; e < 4; e++) ss += (double)xv[k][e] * xv[k][e];
        ss = wave_sum_f64(ss);
        if (lane == 0) part[wave] = ss;
#pragma unroll
        for (int k = 0; k < XPT / 4; k++)
#pragma unroll
            for (int e = 0; e < 4; e++) xv[k][e] = xv[k][e] * gv[k][e];
    }
#pragma unroll
    for (int k = 0; k < XPT / 4; k++) *(f32x4 *)&xs[xs_index(XPT * tid + 4 * k)] = xv[k];
    __syncthreads();
    float scale = 1.f;
    if (QKV) {
        double ss = 0;
#pragma unroll
        for (int w = 0; w < MV_WAVES; w++) ss += part[w];
        scale = 1.0f / sqrtf((float)(ss / K) + eps);
    }

    // this lane's slices of x: sub-blocks lane + 64 i
    float xl[SUBS][32];
#pragma unroll
    for (int i = 0; i < SUBS; i++)
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const f32x4 v = *(const f32x4 *)&xs[xs_index(32 * (lane + 64 * i) + 4 * k)];
            xl[i][4 * k] = v[0], xl[i][4 * k + 1] = v[1], xl[i][4 * k + 2] = v[2], xl[i][4 * k + 3] = v[3];
        }
    // The two row sources take separate code paths, so that each dequantiser's reads have a
    // known address space: LDS reads for the staged quantised rows, global reads for float
    // rows (one pointer that may be either compiles to generic flat loads, several times slower).
    float acc[R];
    if (!fl) {
        // every row of the wave staged at once, then the dots
#pragma unroll
        for (int r = 0; r < R; r++)
#pragma unroll
            for (int k = 0; k < UNITS; k++) {
                const int idx = lane + 64 * k;
                if (idx < n_units) ((u32x4 *)stage[wave][r])[idx] = u[r][k];
            }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        if (S.type == W_Q8_0) {
            // d * sum(q x) per block. The block (2-byte scale, 32 int8) sits at 34 L bytes, 2-byte
            // aligned: it is read as 9 aligned words and realigned (alignbit); each int8 weight is one
            // sign-extending byte convert (SDWA) and an FMA, in two interleaved chains. (Converting
            // unsigned bytes after a sign flip, with 128 sum(x) subtracted per block, measured slower
            // and loses exactness on blocks of small quantised values.)
#pragma unroll
            for (int r = 0; r < R; r++) acc[r] = 0.f;
#pragma unroll
            for (int i = 0; i < SUBS; i++) {
                const int base = 34 * (lane + 64 * i);
                const bool odd = base & 2;  // the block starts 2 bytes into a word
#pragma unroll
                for (int r = 0; r < R; r++) {
                    const uint32_t *dw = (const uint32_t *)(stage[wave][r] + (base & ~3));
                    uint32_t d[9];
#pragma unroll
                    for (int j = 0; j < 9; j++) d[j] = dw[j];
                    const uint32_t sc = odd ? d[0] >> 16 : d[0] & 0xffffu;
                    float b0 = 0.f, b1 = 0.f;
#pragma unroll
                    for (int j = 0; j < 8; j++) {
                        const uint32_t q = odd ? d[j + 1] : __builtin_amdgcn_alignbit(d[j + 1], d[j], 16);
                        b0 = fmaf((float)(int8_t)(q & 0xffu), xl[i][4 * j], b0);
                        b1 = fmaf((float)(int8_t)((q >> 8) & 0xffu), xl[i][4 * j + 1], b1);
                        b0 = fmaf((float)(int8_t)((q >> 16) & 0xffu), xl[i][4 * j + 2], b0);
                        b1 = fmaf((float)(int8_t)(q >> 24), xl[i][4 * j + 3], b1);
                    }
                    acc[r] = fmaf(h2f(sc), b0 + b1, acc[r]);
                }
            }
        } else {
#pragma unroll
            for (int r = 0; r < R; r++) {
                float a = 0.f;
#pragma unroll
                for (int i = 0; i < SUBS; i++) {
                    float w[32];
                    deq32(S.type, stage[wave][r], lane + 64 * i, w);
#pragma unroll
                    for (int e = 0; e < 32; e++) a = fmaf(w[e], xl[i][e], a);
                }
                acc[r] = a;
            }
        }
    } else {
#pragma unroll
        for (int r = 0; r < R; r++) {
            const uint8_t *__restrict__ src = wrow + (size_t)r * S.row_bytes;
            float a = 0.f;
#pragma unroll
            for (int i = 0; i < SUBS; i++) {
                float w[32];
                deq32(S.type, src, lane + 64 * i, w);
#pragma unroll
                for (int e = 0; e < 32; e++) a = fmaf(w[e], xl[i][e], a);
            }
            acc[r] = a;
        }
    }
#pragma unroll
    for (int r = 0; r < R; r++) acc[r] = wave_sum(acc[r]);
    if (lane < R) {
        float a = acc[0];
#pragma unroll
        for (int r = 1; r < R; r++) a = lane == r ? acc[r] : a;
        a *= scale;
        const int row = row0 + lane;
        yt[row] = add ? yt[row] + a : a;
    }
}

// ---------------------------------------------------------------------------
// matvec_tokens: 2 .. 15 tokens (and longer batches whose output rows the GEMM cannot store) through the
// same rows. Bound by instruction issue and LDS reads: a token's 64 products a lane need its 8 KB of x.
// With a workgroup a token, as in matvec_kernel, every token decoded the rows again. Here a wave decodes
// its rows once into registers (64 weights a lane: two rows of 2048 elements or one of 4096), the workgroup
// puts the x rows of up to TOKENS tokens into LDS (times the gains) and a wave takes the tokens one after
// another. Token t's sum goes to lane t: a pass ends with one store a row (and one load, when
// adding). Every sum has matvec_kernel's terms in its order, so a token has the single-token call's
// bits. 256 workgroups of 10 (q/k/v) or 8 (o) waves: one round of the CUs; half the waves with twice the
// rows each, which halves the LDS reads, measured slower (9 tokens 31 us, 15 tokens 39): too few waves to
// cover the reads' latency. q/k/v + o, a workgroup a token -> here: 9 tokens of q5_K 59.2 -> 24.3 us, of q8_0
// 35.1 -> 21.2, of bf16 62.3 -> 23.2; 15 tokens of q8_0 52.7 -> 29.4; 2 tokens (kernel times, trace medians) of
// q8_0 7.5 + 6.3 -> 6.9 + 6.1, of q5_K 11.0 + 9.1 -> 8.8 + 7.5; 2000 tokens into unaligned rows (q5_K o
// alone) 4817 -> 1281.
template <int K>
struct MtShape;
template <>
struct MtShape<2048> {
    static constexpr int WAVES = 10, R = 2, TOKENS = 15;
};
template <>
struct MtShape<4096> {
    static constexpr int WAVES = 8, R = 1, TOKENS = 7;
};

template <int K>
__global__ __launch_bounds__(64 * MtShape<K>::WAVES) void matvec_tokens_kernel(const MatvecParams P) {
    constexpr int WAVES = MtShape<K>::WAVES, R = MtShape<K>::R, TOKENS = MtShape<K>::TOKENS;
    constexpr int SUBS = K / 32 / 64;                  // sub-blocks per lane and row
    constexpr int QBYTES = K / 32 * 34;                // largest quantised row (q8_0)
    constexpr int UNITS = (QBYTES / 16 + 63) / 64;     // 16-byte loads per lane for it
    constexpr int QROW = (QBYTES + 4 + 15) / 16 * 16;  // a staged row, + 4 bytes read past a q8_0 row's end
    constexpr int XPT = K / 256;                       // x elements per thread: 256 threads a token, as matvec_kernel's
    constexpr int N_ROWS = K == N_EMBD ? QKV_DIM : N_EMBD;
    static_assert(N_ROWS % (WAVES * R) == 0 && KV_DIM % R == 0, "every workgroup is whole, a wave's rows in one segment");
    static_assert(SUBS * R == 2 && WAVES * R * QROW <= TOKENS * K * 4 && WAVES * 64 >= 512, "shape");
    __shared__ __align__(16) uint8_t lds[TOKENS * K * 4];  // the rows' bytes, then the x rows
    __shared__ double part[TOKENS][4];
    float *const xs = (float *)lds;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int row0 = (blockIdx.x * WAVES + wave) * R;  // R rows, all in one segment
    // always so: the workgroups are whole (N_ROWS). Without this use of n_rows the compiler loads n_seg behind a
    // wait of its own (9 tokens of q5_K 24.66 us, with it 24.43)
    const bool rows_ok = row0 < P.n_rows;
    const MatvecSeg s0 = P.seg[0], s1 = P.seg[1], s2 = P.seg[2];
    const bool in2 = P.n_seg > 2 && row0 >= s2.row0, in1 = !in2 && P.n_seg > 1 && row0 >= s1.row0;
    const MatvecSeg S = in2 ? s2 : in1 ? s1 : s0;
    const uint8_t *wrow = S.w + (size_t)((rows_ok ? row0 : S.row0) - S.row0) * S.row_bytes;
    const bool q8 = S.type == W_Q8_0;
    // this lane's weights: sub-block lane + 64 i of row r at w[r * SUBS + i] (q8_0: the quants, d their scale)
    float w[2][32], d[2] = {1.f, 1.f};
    if (w_is_float(S.type)) {
#pragma unroll
        for (int k = 0; k < 2; k++) deq32(S.type, wrow + (size_t)(k / SUBS) * S.row_bytes, lane + 64 * (k % SUBS), w[k]);
    } else {
        uint8_t *const stage = lds + wave * (R * QROW);
        const int n_units = S.row_bytes >> 4;
        u32x4 u[R][UNITS];
#pragma unroll
        for (int r = 0; r < R; r++)
#pragma unroll
            for (int k = 0; k < UNITS; k++)
                u[r][k] = ((const u32x4 *)(wrow + (size_t)r * S.row_bytes))[min(lane + 64 * k, n_units - 1)];
#pragma unroll
        for (int r = 0; r < R; r++)
#pragma unroll
            for (int k = 0; k < UNITS; k++)
                if (lane + 64 * k < n_units) ((u32x4 *)(stage + r * QROW))[lane + 64 * k] = u[r][k];
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        if (q8) {
#pragma unroll
            for (int k = 0; k < 2; k++) {
                const int base = 34 * (lane + 64 * (k % SUBS));
                const bool odd = base & 2;  // the block starts 2 bytes into a word
                const uint32_t *dw = (const uint32_t *)(stage + (k / SUBS) * QROW + (base & ~3));
                uint32_t v[9];
#pragma unroll
                for (int j = 0; j < 9; j++) v[j] = dw[j];
                d[k] = h2f(odd ? v[0] >> 16 : v[0] & 0xffffu);
#pragma unroll
                for (int j = 0; j < 8; j++) {
                    const uint32_t q = odd ? v[j + 1] : __builtin_amdgcn_alignbit(v[j + 1], v[j], 16);
                    w[k][4 * j] = (float)(int8_t)(q & 0xffu);
                    w[k][4 * j + 1] = (float)(int8_t)((q >> 8) & 0xffu);
                    w[k][4 * j + 2] = (float)(int8_t)((q >> 16) & 0xffu);
                    w[k][4 * j + 3] = (float)(int8_t)(q >> 24);
                }
            }
        } else {
#pragma unroll
            for (int k = 0; k < 2; k++) deq32(S.type, stage + (k / SUBS) * QROW, lane + 64 * (k % SUBS), w[k]);
        }
    }
#pragma unroll
    for (int k = 0; k < 2; k++)
#pragma unroll
        for (int e = 0; e < 32; e++) asm volatile("" : "+v"(w[k][e]));  // decoded here, not once a token

    for (int t0 = 0; t0 < P.n_tok; t0 += TOKENS) {
        const int n = min(TOKENS, P.n_tok - t0);
        __syncthreads();  // the rows' bytes, or the pass before's x, have been read
        // x of tokens t0 .. t0 + n - 1: two at a time, 256 threads each
        if (tid < 512) {
            const int u = tid & 255;
            for (int t = tid >> 8; t < n; t += 2) {
                const float *xt = P.x + (size_t)(t0 + t) * P.x_stride + XPT * u;
                f32x4 xv[XPT / 4];
#pragma unroll
                for (int k = 0; k < XPT / 4; k++) xv[k] = *(const f32x4 *)(xt + 4 * k);
                if (P.norm_w) {
                    double ss = 0;
#pragma unroll
                    for (int k = 0; k < XPT / 4; k++)
#pragma unroll
                        for (int e = 0; e < 4; e++) ss += (double)xv[k][e] * xv[k][e];
                    ss = wave_sum_f64(ss);
                    if (lane == 0) part[t][(tid >> 6) & 3] = ss;
#pragma unroll
                    for (int k = 0; k < XPT / 4; k++) {
                        const f32x4 gv = *(const f32x4 *)(P.norm_w + XPT * u + 4 * k);
#pragma unroll
                        for (int e = 0; e < 4; e++) xv[k][e] = xv[k][e] * gv[e];
                    }
                }
#pragma unroll
                for (int k = 0; k < XPT / 4; k++) *(f32x4 *)&xs[t * K + xs_index(XPT * u + 4 * k)] = xv[k];
            }
        }
        // lane t: token t0 + t's row of y
        const bool mine = lane < n && rows_ok;
        float *const y = P.y + (size_t)(t0 + (mine ? lane : 0)) * P.y_stride + row0;
        float yin[R], out[R];
#pragma unroll
        for (int r = 0; r < R; r++) yin[r] = P.add && mine ? y[r] : 0.f, out[r] = 0.f;
        __syncthreads();
        float scale = 1.f;
        if (P.norm_w && lane < n) {
            double ss = 0;
#pragma unroll
            for (int i = 0; i < 4; i++) ss += part[lane][i];
            scale = 1.0f / sqrtf((float)(ss / K) + P.eps);
        }
        auto dots = [&](auto is_q8) {
            for (int t = 0; t < n; t++) {
                float acc[R];
#pragma unroll
                for (int r = 0; r < R; r++) acc[r] = 0.f;
#pragma unroll
                for (int i = 0; i < SUBS; i++) {
                    float xl[32];
#pragma unroll
                    for (int k = 0; k < 8; k++) {
                        const f32x4 v = *(const f32x4 *)&xs[t * K + xs_index(32 * (lane + 64 * i) + 4 * k)];
                        xl[4 * k] = v[0], xl[4 * k + 1] = v[1], xl[4 * k + 2] = v[2], xl[4 * k + 3] = v[3];
                    }
#pragma unroll
                    for (int r = 0; r < R; r++) {
                        const int k = r * SUBS + i;
                        if constexpr (decltype(is_q8)::value) {
                            float b0 = 0.f, b1 = 0.f;
#pragma unroll
                            for (int j = 0; j < 32; j += 2) b0 = fmaf(w[k][j], xl[j], b0), b1 = fmaf(w[k][j + 1], xl[j + 1], b1);
                            acc[r] = fmaf(d[k], b0 + b1, acc[r]);
                        } else {
#pragma unroll
                            for (int e = 0; e < 32; e++) acc[r] = fmaf(w[k][e], xl[e], acc[r]);
                        }
                    }
                }
#pragma unroll
                for (int r = 0; r < R; r++) {
                    const float a = wave_sum(acc[r]);
                    out[r] = lane == t ? a : out[r];
                }
            }
        };
        if (q8)
            dots(std::true_type{});
        else
            dots(std::false_type{});
        if (mine)
#pragma unroll
            for (int r = 0; r < R; r++) {
                const float a = out[r] * scale;
                y[r] = P.add ? yin[r] + a : a;
            }
    }
}

hipError_t launch_get_rows(const RowsParams &P, hipStream_t stream) {
    hipLaunchKernelGGL(get_rows_kernel, dim3((P.n_sub + 63) / 64, P.n), dim3(64), 0, stream, P);
    return hipGetLastError();
}

// Rows per wave: 2 for the 2048-element rows (q/k/v: 640 workgroups) and 1 for the
// 4096-element rows (o: 512 workgroups, two waves per SIMD: with one, each row's LDS reads and
// FMA chain were exposed); measured best of 1, 2, 4 and 8 for either.
constexpr int MV_ROWS_2048 = 2, MV_ROWS_4096 = 1;
constexpr int MT_MIN_TOKENS = 2;  // at 2 tokens matvec_tokens_kernel is ahead of a workgroup a token (figures above it)

int matvec_row_multiple(int k) { return MV_WAVES * (k == 2048 ? MV_ROWS_2048 : MV_ROWS_4096); }

hipError_t launch_matvec(const MatvecParams &P, int k, hipStream_t stream) {
    // a layer's two projections: matvec_kernel has the segments, the norm and the sum into y of each built in
    const bool qkv = k == N_EMBD && P.n_seg == 3 && P.seg[1].row0 == Q_DIM && P.seg[2].row0 == Q_DIM + KV_DIM &&
                     P.n_rows == QKV_DIM && P.norm_w && !P.add;
    const bool o = k == Q_DIM && P.n_seg == 1 && P.n_rows == N_EMBD && !P.norm_w && P.add;
    if (P.n_tok < 1 || P.seg[0].row0 != 0 || !(qkv || o)) return hipErrorInvalidValue;
    if (P.n_tok >= MT_MIN_TOKENS) {
        if (k == 2048) {
            constexpr int ROWS = MtShape<2048>::WAVES * MtShape<2048>::R;
            hipLaunchKernelGGL(matvec_tokens_kernel<2048>, dim3(P.n_rows / ROWS), dim3(64 * MtShape<2048>::WAVES), 0, stream, P);
        } else {
            constexpr int ROWS = MtShape<4096>::WAVES * MtShape<4096>::R;
            hipLaunchKernelGGL(matvec_tokens_kernel<4096>, dim3(P.n_rows / ROWS), dim3(64 * MtShape<4096>::WAVES), 0, stream, P);
        }
        return hipGetLastError();
    }
    const dim3 grid(P.n_rows / matvec_row_multiple(k)), block(64 * MV_WAVES);
    const uint32_t types = P.seg[0].type | P.seg[1].type << 8 | P.seg[2].type << 16;
    if (k == 2048)
        hipLaunchKernelGGL((matvec_kernel<2048, MV_ROWS_2048>), grid, block, 0, stream, P.seg[0].w, P.seg[1].w, P.seg[2].w, P.x,
                           P.norm_w, P.y, types, P.eps);
    else
        hipLaunchKernelGGL((matvec_kernel<4096, MV_ROWS_4096>), grid, block, 0, stream, P.seg[0].w, nullptr, nullptr, P.x, nullptr,
                           P.y, types, 0.f);
    return hipGetLastError();
}

}  // namespace flint
