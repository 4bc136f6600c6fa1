// The attention projections of a prefill batch on the matrix cores (gfx950).
//
// Y[t][n] = sum_k W[n][k] X[t][k] for T tokens at once: the q/k/v projection of the RMSNorm'd
// hidden rows and the o projection (added to the residual) of a layer-major prefill step
// (/root/reference/src/engine.mm:1083-1086, 1105-1111). The reference's CPU path sums in double
// (ref_model.cpp:74-93); the one-token kernels here sum fp32 FMAs. The batch reaches the same
// fp32-level accuracy on v_mfma_f32_32x32x16_f16 by splitting both operands into f16 hi/lo
// pairs:
//   * every weight row (dequantised as in proj.hip) and every activation row is scaled by a
//     power of two that puts its largest magnitude in [2^14, 2^15), then split as
//     v = hi + lo with hi = f16(v), lo = f16(v - hi): 22 significant bits, and no value
//     overflows f16 whatever the row's range;
//   * the GEMM accumulates hi*hi + hi*lo + lo*hi in fp32 (the lo*lo term is below 2^-22 of
//     the product) and scales each output by 2^(e_t + f_n), which is exact.
// Three launches: wprep (weights -> planes), xprep (activations -> planes, the RMSNorm fused
// for q/k/v) and gemm3 or gemm_int. The stage-level calls rebuild the weight planes from the GGUF
// rows each time (18-20 us for a layer's 19M weights in q8_0); a model keeps every layer's planes after
// building them once, and its calls launch only xprep and the GEMM. Batches of up to
// GEMM_RAW_TOKENS tokens (GEMM_RAW_TOKENS_KEPT with kept planes) in the integer form take gemm_raw instead,
// which reads the GGUF rows itself.
#include "common.h"
#include "dequant.h"
#include "flint_attn_internal.h"

namespace flint {

namespace {

// exponent that puts a row's largest magnitude mx in [2^14, 2^15): x * 2^-e fits f16 with its
// full 11 bits at the top of the row (0 for an all-zero row, inf / nan left as they are)
__device__ inline int row_exp(float mx) {
    if (!(mx > 0.f) || !__builtin_isfinite(mx)) return 0;
    return __builtin_amdgcn_frexp_expf(mx) - 15;  // mx in [2^(f-1), 2^f)
}

__device__ inline void split_store(float v, int e, _Float16 *hi, _Float16 *lo) {
    const float s = __builtin_amdgcn_ldexpf(v, -e);
    const _Float16 h = (_Float16)s;
    *hi = h;
    *lo = (_Float16)(s - (float)h);
}

// Planes are stored in the order the GEMMs keep them in LDS, so that a workgroup's chunk of a plane
// (128 rows x 32 k) is one contiguous 8 KiB block that it copies into LDS unchanged: blocks
// [row tile n >> 7][chunk k >> 5], and in a block the 16-byte unit of row r (n & 127), k group
// k8 ((k >> 3) & 3) at unit ((r >> 5) * 2 + (k8 >> 1)) * 64 + (r & 31) + 32 (k8 & 1). The element
// offset of the unit that holds elements 8 g .. 8 g + 7 of row n:
__device__ inline size_t plane_unit(int n, int g, int K) {
    const int r = n & 127, k8 = g & 3;
    const int q = ((r >> 5) * 2 + (k8 >> 1)) * 64 + (r & 31) + 32 * (k8 & 1);
    return (((size_t)(n >> 7) * (K / 32) + (g >> 2)) * 512 + q) * 8;
}

}  // namespace

// ---------------------------------------------------------------------------
// wprep: one 512-thread workgroup per 8 weight rows n0 .. n0 + 7, wave w on row n0 + w: the row's
// bytes staged through its LDS area (2-byte copies: q8_0 and q6_K blocks are only 2-byte aligned),
// dequantised 32 elements per lane per sub-block (lane l owns sub-blocks l, l + 64, ...), the
// row's exponent f_n from its largest magnitude, then its hi/lo values written over the staged
// bytes. After the workgroup's barrier every store writes 8 whole 128-byte lines of the planes'
// chunk order: lane (row rho = lane & 7, group lane gl = lane >> 3) of wave w takes the 16-byte
// units of groups gl + 8 (w + 8 j) of row n0 + rho. The wave areas are 16 bytes longer than a
// row's values, so the 8 rows' reads of one group fall on different banks.
template <int K>
__global__ __launch_bounds__(512) void wprep_kernel(const GemmWeightParams P) {
    constexpr int SUBS = K / 32 / 64;
    constexpr int AREA = K * 4 + 16;  // a staged row (at most K floats), later its hi|lo values
    static_assert(K / 32 * 34 <= K * 4, "a quantised row fits its area");
    __shared__ __align__(16) uint8_t areas[8 * AREA];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int n = 8 * blockIdx.x + wave;  // this wave's plane row
    uint8_t *const stage = areas + wave * AREA;
    const int in2 = P.n_seg > 2 && n >= P.seg[2].row0, in1 = !in2 && P.n_seg > 1 && n >= P.seg[1].row0;
    const MatvecSeg S = in2 ? P.seg[2] : in1 ? P.seg[1] : P.seg[0];
    const uint8_t *row = S.w + (size_t)(n - S.row0) * S.row_bytes;
    const uint16_t *src = (const uint16_t *)row;
    uint16_t *dst = (uint16_t *)stage;
    for (int i = lane; i < S.row_bytes / 2; i += 64) dst[i] = src[i];
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    float w[SUBS][32];
    float mx = 0.f;
#pragma unroll
    for (int i = 0; i < SUBS; i++) {
        deq32(S.type, stage, lane + 64 * i, w[i]);
#pragma unroll
        for (int e = 0; e < 32; e++) mx = fmaxf(mx, fabsf(w[i][e]));
    }
    const int f = row_exp(wave_max(mx));
    // every lane has read the staged bytes before any lane overwrites them
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    _Float16 *const hi = (_Float16 *)stage, *const lo = hi + K;
#pragma unroll
    for (int i = 0; i < SUBS; i++) {
        const int k0 = 32 * (lane + 64 * i);
        f16x8 h8[4], l8[4];
#pragma unroll
        for (int e = 0; e < 32; e++) {
            _Float16 h, l;
            split_store(w[i][e], f, &h, &l);
            h8[e >> 3][e & 7] = h;
            l8[e >> 3][e & 7] = l;
        }
#pragma unroll
        for (int q = 0; q < 4; q++) {
            *(f16x8 *)(hi + k0 + 8 * q) = h8[q];
            *(f16x8 *)(lo + k0 + 8 * q) = l8[q];
        }
    }
    if (lane == 0) P.fexp[n] = f;
    __syncthreads();
    const int rho = lane & 7, gl = lane >> 3, nr = 8 * blockIdx.x + rho;
    const _Float16 *const rh = (const _Float16 *)(areas + rho * AREA), *const rl = rh + K;
#pragma unroll
    for (int j = 0; j < K / 512; j++) {
        const int g = gl + 8 * (wave + 8 * j);
        const size_t o = plane_unit(nr, g, K);
        *(f16x8 *)(P.wh + o) = *(const f16x8 *)(rh + 8 * g);
        *(f16x8 *)(P.wl + o) = *(const f16x8 *)(rl + 8 * g);
    }
}


// ---------------------------------------------------------------------------
// The integer form. A q8_0, iq4_xs, q5_K or q6_K weight is s v (- m for q5_K), with v an integer
// of magnitude at most 127 (exact in f16), s the scale of its 32 (q8_0, iq4_xs, q5_K) or 16 (q6_K)
// elements and m the min of its 32, and a 32-k chunk of the GEMM is one 32-element sub-block. So
// a chunk's products are sum_k (xh + xl) v on the matrix cores, two products per pair instead of
// gemm3's three and no weight lo plane, and the scale joins in fp32: acc += s T, one s per weight
// row and chunk (SUB = 32) or k-step of 16 (SUB = 16); the min as acc -= m S with S = sum_k
// (xh + xl) over the block, which xprep writes per row and block. The x planes are gemm3's.
// The rows' bytes are decoded the same way for the planes (wprep_int) and by gemm_raw: a wave stages 32 rows'
// bytes of a group of blocks in LDS with 16-byte loads along the rows, and a lane decodes the 16 weights
// of a block that the MFMA takes from it.

// 4 bytes u (0 .. 255) as f16, less `bias` (exact): 0x6400 | u is 1024 + u
__device__ inline void bytes_f16(uint32_t u, int bias, f16x8 &w, int at) {
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    const h2 off = {(_Float16)(float)(1024 + bias), (_Float16)(float)(1024 + bias)};
    const h2 a = __builtin_bit_cast(h2, __builtin_amdgcn_perm(0x64646464u, u, 0x04010400u)) - off;
    const h2 b = __builtin_bit_cast(h2, __builtin_amdgcn_perm(0x64646464u, u, 0x04030402u)) - off;
    w[at] = a[0], w[at + 1] = a[1], w[at + 2] = b[0], w[at + 3] = b[1];
}

// 8 bytes at p + odd (p 4-byte aligned, odd 0 or 2)
__device__ inline uint2 lds8(const uint8_t *p, int odd) {
    const uint32_t *w = (const uint32_t *)p;
    if (!odd) return make_uint2(w[0], w[1]);
    return make_uint2(__builtin_amdgcn_alignbit(w[1], w[0], 16), __builtin_amdgcn_alignbit(w[2], w[1], 16));
}

// The GGUF rows in groups of G chunks: UNITS 16-byte units of a row a group, the last of them at byte
// LAST of the group's BYTES (whole units but for q6_K, whose last unit overlaps the one before), in LDS
// rows of STRIDE bytes (an odd number of units, so that the 32 rows' reads of one place spread over the
// banks). get: lane (row, half h)'s elements 8 h .. 8 h + 7 and 16 + 8 h .. 16 + 8 h + 7 of the group's
// block j (a constant once unrolled), from its row in LDS: the values, the scales of elements
// 0-15 and 16-31, and the min, in ggml's float order, so that scale * value - min is deq32's weight
// (f16: scale 1; bf16: 8 significant bits, exact in f16 once the block's largest magnitude is scaled into
// [2^14, 2^15): values below 2^-28 of it, beneath f16's normal range, round to f16's subnormal steps).
template <int TYPE>
struct RawRows;

template <>
struct RawRows<W_Q8_0> {
    static constexpr int G = 8, BYTES = 272, UNITS = 17, LAST = 256, STRIDE = 272;
    __device__ static inline void get(const uint8_t *row, int j, int h, f16x8 (&w)[2], float (&sc)[2], float &) {
        const int odd = j & 1 ? 0 : 2;  // the block's values start at + 2
#pragma unroll
        for (int s = 0; s < 2; s++) {
            const uint2 v = lds8(row + 34 * j + 2 - odd + 16 * s + 8 * h, odd);
            bytes_f16(v.x ^ 0x80808080u, 128, w[s], 0);
            bytes_f16(v.y ^ 0x80808080u, 128, w[s], 4);
        }
        sc[0] = sc[1] = h2f(*(const uint16_t *)(row + 34 * j));
    }
};
template <>
struct RawRows<W_Q5_K> {
    static constexpr int G = 8, BYTES = 176, UNITS = 11, LAST = 160, STRIDE = 176;
    __device__ static inline void get(const uint8_t *row, int j, int h, f16x8 (&w)[2], float (&sc)[2], float &m) {
#pragma clang fp contract(off)
        const u32x4 hdr = *(const u32x4 *)row;
        const int ls = 4 * (j & 1);
#pragma unroll
        for (int s = 0; s < 2; s++) {
            const uint2 qh = *(const uint2 *)(row + 16 + 16 * s + 8 * h);
            const uint2 ql = *(const uint2 *)(row + 48 + 32 * (j >> 1) + 16 * s + 8 * h);
            bytes_f16(((ql.x >> ls) & 0x0f0f0f0fu) | (((qh.x >> j) & 0x01010101u) << 4), 0, w[s], 0);
            bytes_f16(((ql.y >> ls) & 0x0f0f0f0fu) | (((qh.y >> j) & 0x01010101u) << 4), 0, w[s], 4);
        }
        // 6-bit scale and min of block j (deq32's)
        const uint32_t s[3] = {hdr[1], hdr[2], hdr[3]};
        const uint32_t q = j < 4 ? byte_of(s, j) & 63 : (byte_of(s, j + 4) & 15) | ((byte_of(s, j - 4) >> 6) << 4);
        const uint32_t mn = j < 4 ? byte_of(s, j + 4) & 63 : (byte_of(s, j + 4) >> 4) | ((byte_of(s, j) >> 6) << 4);
        sc[0] = sc[1] = h2f(hdr[0] & 0xffff) * (float)q;
        m = h2f(hdr[0] >> 16) * (float)mn;
    }
};
template <>
struct RawRows<W_Q6_K> {
    static constexpr int G = 16, BYTES = 420, UNITS = 27, LAST = 404, STRIDE = 432;
    __device__ static inline void get(const uint8_t *row, int j, int h, f16x8 (&w)[2], float (&sc)[2], float &) {
        const int r = j >> 3, n = (j >> 2) & 1, b = j & 3, odd = r ? 2 : 0;  // blocks of 210 bytes
        const int ls = 4 * (b >> 1), hs = 2 * b;
        const uint8_t *blk = row + 210 * r - odd;
#pragma unroll
        for (int s = 0; s < 2; s++) {
            const uint2 ql = lds8(blk + 64 * n + 32 * (b & 1) + 16 * s + 8 * h, odd);
            const uint2 qh = lds8(blk + 128 + 32 * n + 16 * s + 8 * h, odd);
            bytes_f16(((ql.x >> ls) & 0x0f0f0f0fu) | (((qh.x >> hs) & 0x03030303u) << 4), 32, w[s], 0);
            bytes_f16(((ql.y >> ls) & 0x0f0f0f0fu) | (((qh.y >> hs) & 0x03030303u) << 4), 32, w[s], 4);
        }
        // the group's last 4 bytes lie at the end of the overlapping unit
        const int so = 210 * r + 192 + 2 * (j & 7), end = 16 * UNITS - BYTES;
        const uint32_t s = *(const uint16_t *)(row + so + (so >= BYTES - 4 ? end : 0));
        const float d = h2f(*(const uint16_t *)(row + 210 * r + 208 + (r ? end : 0)));
        sc[0] = d * (float)(int8_t)(s & 0xff), sc[1] = d * (float)(int8_t)(s >> 8);
    }
};
template <>
struct RawRows<W_IQ4_XS> {
    static constexpr int G = 16, BYTES = 272, UNITS = 17, LAST = 256, STRIDE = 272;
    __device__ static inline void get(const uint8_t *row, int j, int h, f16x8 (&w)[2], float (&sc)[2], float &) {
        const int b = j & 7;
        const uint2 *blk = (const uint2 *)(row + 136 * (j >> 3)), hdr = blk[0];
        const uint2 q = blk[1 + 2 * b + h];  // bytes 8 h ..: low nibbles elements 8 h .., high 16 + 8 h ..
        // the code book + 128 as unsigned bytes
        constexpr uint32_t X = 0x80808080u, T0 = IQ4_T0 ^ X, T1 = IQ4_T1 ^ X, T2 = IQ4_T2 ^ X, T3 = IQ4_T3 ^ X;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t v = (i & 1 ? q.y : q.x) >> (4 * (i >> 1)), sel = v & 0x07070707u;
            const uint32_t lo = __builtin_amdgcn_perm(T1, T0, sel), hi = __builtin_amdgcn_perm(T3, T2, sel);
            const uint32_t m = __builtin_amdgcn_perm(0u, 0u, ((v >> 3) & 0x01010101u) | 0x0c0c0c0cu);  // 0xff where bit 3 is set
            bytes_f16((lo & ~m) | (hi & m), 128, w[i >> 1], 4 * (i & 1));
        }
        const uint32_t ls = ((hdr.y >> (8 * (b >> 1) + 4 * (b & 1))) & 15) | (((hdr.x >> (16 + 2 * b)) & 3) << 4);
        sc[0] = sc[1] = h2f(hdr.x & 0xffff) * (float)((int)ls - 32);
    }
};
template <>
struct RawRows<W_F16> {
    static constexpr int G = 4, BYTES = 256, UNITS = 16, LAST = 240, STRIDE = 272;
    __device__ static inline void get(const uint8_t *row, int j, int h, f16x8 (&w)[2], float (&sc)[2], float &) {
#pragma unroll
        for (int s = 0; s < 2; s++) w[s] = *(const f16x8 *)(row + 64 * j + 32 * s + 16 * h);
        sc[0] = sc[1] = 1.f;
    }
};
template <>
struct RawRows<W_BF16> {
    static constexpr int G = 4, BYTES = 256, UNITS = 16, LAST = 240, STRIDE = 272;
    __device__ static inline void get(const uint8_t *row, int j, int h, f16x8 (&w)[2], float (&sc)[2], float &) {
        u32x4 q[2];
        float mx = 0.f;
#pragma unroll
        for (int s = 0; s < 2; s++) {
            q[s] = *(const u32x4 *)(row + 64 * j + 32 * s + 16 * h);
#pragma unroll
            for (int i = 0; i < 4; i++)
                mx = fmaxf(mx, fmaxf(fabsf(__uint_as_float(q[s][i] << 16)), fabsf(__uint_as_float(q[s][i] & 0xffff0000u))));
        }
        mx = xor32_max(mx);  // the block's largest magnitude: both lane halves
        const int e = mx > 0.f && __builtin_isfinite(mx) ? __builtin_amdgcn_frexp_expf(mx) - 15 : 0;
#pragma unroll
        for (int s = 0; s < 2; s++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                w[s][2 * i] = (_Float16)__builtin_amdgcn_ldexpf(__uint_as_float(q[s][i] << 16), -e);
                w[s][2 * i + 1] = (_Float16)__builtin_amdgcn_ldexpf(__uint_as_float(q[s][i] & 0xffff0000u), -e);
            }
        sc[0] = sc[1] = __builtin_amdgcn_ldexpf(1.f, e);
    }
};

constexpr int GR_TILE = 32;  // weight rows of a wave (and tokens of a gemm_raw workgroup)

// A wave's copy of its rows' group bytes into LDS: unit u = 64 i + lane is unit u % UNITS of row u / UNITS
// of the 32 rows from seg (the first row's byte of the group).
template <int TYPE>
struct RawCopy {
    typedef RawRows<TYPE> RR;
    static constexpr int NU = GR_TILE * RR::UNITS, WL = (NU + 63) / 64;
    struct __attribute__((packed, aligned(4))) Unit {
        u32x4 v;
    };
    uint32_t go[WL], lo[WL];
    u32x4 w[WL];
    __device__ inline void init(int row_bytes, int lane) {
#pragma unroll
        for (int i = 0; i < WL; i++) {
            const int u = min(64 * i + lane, NU - 1), row = u / RR::UNITS, c = u % RR::UNITS;
            go[i] = row * row_bytes + (c == RR::UNITS - 1 ? RR::LAST : 16 * c);
            lo[i] = row * RR::STRIDE + 16 * c;
        }
    }
    __device__ inline void load(const uint8_t *seg) {
#pragma unroll
        for (int i = 0; i < WL; i++) w[i] = ((const Unit *)(seg + go[i]))->v;
    }
    __device__ inline void store(uint8_t *area, int lane) const {
#pragma unroll
        for (int i = 0; i < WL; i++)
            if (NU % 64 == 0 || i < WL - 1 || 64 * i + lane < NU) *(u32x4 *)(area + lo[i]) = w[i];
    }
};
__device__ inline void wave_lds_fence() {  // the wave's LDS accesses so far stay ahead of those to come
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// wprep_int: a wave writes 32 rows x 256 elements (512 for the types whose groups are 16 blocks): the values as
// f16 into the plane's chunk order (plane_unit: lane's k-step s of a block is unit 64 s + lane, so a
// store writes 1 KiB), the scales into wd[n / 128][b][32 / SUB][n % 128] and, with mins, its min into
// wm[n / 128][b][n % 128]. HBM-bound: 11.1 MB in and 21.6 MB out for q/k/v in q8_0. (A thread a block, its
// row bytes read 2 at a time and its 16-byte units written to lines of their own: 12.2 + 12.5 us for a layer's
// q/k/v and o, q6_K 14.5 + 16.0; now 9.4 + 9.1 and 9.3 + 9.7.)
constexpr int WP_WAVES = 4;
template <int SUB, int TYPE>
__device__ __forceinline__ void wprep_int_wave(const GemmWeightParams &P, const MatvecSeg &S, uint8_t *area, int n0, int item, int K) {
    typedef RawRows<TYPE> RR;
    constexpr int G = RR::G, GROUPS = G < 8 ? 8 / G : 1;
    if (G == 16 && (item & 1)) return;  // the even items take 512 elements
    const int lane = threadIdx.x & 63, h = lane >> 5, r32 = lane & 31, NB = K / 32;
    const uint8_t *const row0 = S.w + (size_t)(n0 - S.row0) * S.row_bytes;
    RawCopy<TYPE> C;
    C.init(S.row_bytes, lane);
#pragma unroll
    for (int q = 0; q < GROUPS; q++) {
        const int b0 = 8 * item + G * q;  // first block
        C.load(row0 + (size_t)(b0 / G) * RR::BYTES);
        if (q > 0) wave_lds_fence();
        C.store(area, lane);
        wave_lds_fence();
#pragma unroll
        for (int j = 0; j < G; j++) {
            f16x8 w[2];
            float sc[2], m = 0.f;
            RR::get(area + r32 * RR::STRIDE, j, h, w, sc, m);
            const int b = b0 + j;
            _Float16 *const o = P.wh + (((size_t)(n0 >> 7) * NB + b) * 512 + ((n0 >> 5) & 3) * 128 + lane) * 8;
            *(f16x8 *)o = w[0];
            *(f16x8 *)(o + 512) = w[1];
            float *const d = P.wd + ((size_t)(n0 >> 7) * NB + b) * (32 / SUB) * GEMM_TILE + (n0 & 127) + r32;
            if (SUB == 16 || h == 0) d[SUB == 16 ? GEMM_TILE * h : 0] = h == 0 ? sc[0] : sc[1];  // SUB = 32: they are one
            if (P.imin && h == 0) P.wm[((size_t)(n0 >> 7) * NB + b) * GEMM_TILE + (n0 & 127) + r32] = m;
        }
    }
}
template <int SUB>
__global__ __launch_bounds__(64 * WP_WAVES) void wprep_int_kernel(const GemmWeightParams P, int K) {
    constexpr int AREA = GR_TILE * (SUB == 16 ? RawRows<W_Q6_K>::STRIDE : RawRows<W_Q8_0>::STRIDE);
    __shared__ __align__(16) uint8_t lds[WP_WAVES][AREA];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n0 = blockIdx.y * GR_TILE, item = blockIdx.x * WP_WAVES + wave;
    const MatvecSeg s0 = P.seg[0], s1 = P.seg[1], s2 = P.seg[2];
    const bool in2 = P.n_seg > 2 && n0 >= s2.row0, in1 = !in2 && P.n_seg > 1 && n0 >= s1.row0;
    const MatvecSeg S = in2 ? s2 : in1 ? s1 : s0;
    switch (S.type) {
        case W_Q8_0: wprep_int_wave<SUB, W_Q8_0>(P, S, lds[wave], n0, item, K); break;
        case W_Q5_K: wprep_int_wave<SUB, W_Q5_K>(P, S, lds[wave], n0, item, K); break;
        case W_IQ4_XS: wprep_int_wave<SUB, W_IQ4_XS>(P, S, lds[wave], n0, item, K); break;
        case W_F16: wprep_int_wave<SUB, W_F16>(P, S, lds[wave], n0, item, K); break;
        case W_BF16: wprep_int_wave<SUB, W_BF16>(P, S, lds[wave], n0, item, K); break;
        default:
            if constexpr (SUB == 16) wprep_int_wave<SUB, W_Q6_K>(P, S, lds[wave], n0, item, K);
    }
}

__device__ inline double group_ss(const float (&v)[8]) {
    double ss = 0;
#pragma unroll
    for (int e = 0; e < 8; e++) ss += (double)v[e] * v[e];
    return ss;
}

// ---------------------------------------------------------------------------
// xprep: one 512-thread workgroup per 8 activation rows t0 .. t0 + 7 (rows T .. T_pad - 1 are
// written as zeros). Lane (row rho = lane & 7, group lane gl = lane >> 3) of wave w holds the
// row's 8-element groups gl + 8 (w + 8 j) in registers, read once. The RMSNorm is computed as
// matvec_kernel computes it (double sum of squares, float scale, xn = (x * scale) * g; the sum
// runs in another order), then the row's exponent from the largest |xn|, then the hi/lo planes.
// In the planes' chunk order the 8 rows' units of one group are one 128-byte line, so every
// store instruction writes 8 whole lines.
template <int K>
__global__ __launch_bounds__(512) void xprep_kernel(const GemmActParams P) {
    constexpr int GPJ = K / 8 / 64;  // groups per lane
    __shared__ double red_ss[8][8];  // [wave][row]
    __shared__ float red_mx[8][8];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, rho = lane & 7, gl = lane >> 3;
    const int t = 8 * blockIdx.x + rho;
    const bool live = t < P.T;
    const float *xt = P.x + (size_t)(live ? t : 0) * P.x_stride;
    float v[GPJ][8];
#pragma unroll
    for (int j = 0; j < GPJ; j++) {
        const int g = gl + 8 * (wave + 8 * j);
        const f32x4 a = *(const f32x4 *)(xt + 8 * g), b = *(const f32x4 *)(xt + 8 * g + 4);
        v[j][0] = a[0], v[j][1] = a[1], v[j][2] = a[2], v[j][3] = a[3];
        v[j][4] = b[0], v[j][5] = b[1], v[j][6] = b[2], v[j][7] = b[3];
    }
    if (P.norm_w) {
        double ss = 0;
#pragma unroll
        for (int j = 0; j < GPJ; j++) ss += group_ss(v[j]);
#pragma unroll
        for (int m = 8; m < 64; m <<= 1) ss += __shfl_xor(ss, m, 64);
        if (gl == 0) red_ss[wave][rho] = ss;
        __syncthreads();
        ss = 0;
#pragma unroll
        for (int w = 0; w < 8; w++) ss += red_ss[w][rho];
        const float scale = 1.0f / sqrtf((float)(ss / K) + P.eps);
#pragma unroll
        for (int j = 0; j < GPJ; j++) {
            const int g = gl + 8 * (wave + 8 * j);
            const f32x4 a = *(const f32x4 *)(P.norm_w + 8 * g), b = *(const f32x4 *)(P.norm_w + 8 * g + 4);
            const float gg[8] = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
#pragma unroll
            for (int e = 0; e < 8; e++) v[j][e] = v[j][e] * scale * gg[e];
        }
    }
    float mx = 0.f;
#pragma unroll
    for (int j = 0; j < GPJ; j++)
#pragma unroll
        for (int e = 0; e < 8; e++) mx = fmaxf(mx, fabsf(v[j][e]));
#pragma unroll
    for (int m = 8; m < 64; m <<= 1) mx = fmaxf(mx, __shfl_xor(mx, m, 64));
    if (gl == 0) red_mx[wave][rho] = mx;
    __syncthreads();
    mx = red_mx[0][rho];
#pragma unroll
    for (int w = 1; w < 8; w++) mx = fmaxf(mx, red_mx[w][rho]);
    const int e = live ? row_exp(mx) : 0;
#pragma unroll
    for (int j = 0; j < GPJ; j++) {
        f16x8 h8, l8;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            _Float16 h, l;
            split_store(live ? v[j][i] : 0.f, e, &h, &l);
            h8[i] = h;
            l8[i] = l;
        }
        const size_t o = plane_unit(t, gl + 8 * (wave + 8 * j), K);
        *(f16x8 *)(P.xh + o) = h8;
        *(f16x8 *)(P.xl + o) = l8;
        if (P.xs) {  // the block sums: a 32-element block's 4 groups are lanes gl ^ 1, ^ 2, ^ 3
            float gs = 0.f;
#pragma unroll
            for (int i = 0; i < 8; i++) gs += (float)h8[i] + (float)l8[i];
            gs += __shfl_xor(gs, 8, 64);
            gs += __shfl_xor(gs, 16, 64);
            const int b = (gl + 8 * (wave + 8 * j)) >> 2;
            if ((gl & 3) == 0) P.xs[((size_t)(t >> 7) * (K / 32) + b) * GEMM_TILE + (t & 127)] = gs;
        }
    }
    if (tid < 8) P.eexp[t] = e;  // lanes 0..7 of wave 0: rows rho = tid
}

// xprep for a few rows: one workgroup per row, a thread per 8-element group, so that a row takes one load
// and one pass of 8 elements instead of 4 or 8 (trace medians, 32 rows: 3.8 against 5.6 us for K = 2048, 3.8
// against 7.6 for K = 4096; 512 rows 6.8 and 9.6 against 7.4 and 10.9). The row sum's terms are added in
// xprep_kernel's order (group_ss, then a lane's groups, the 8 lanes by pairs, the 8 waves), so a row's planes
// have the same bits. A row's units are 16-byte pieces of lines it shares with 7 others, which long batches
// pay for (4000 rows: 31 and 62 us for a row a workgroup, 12 and 26 for 8): they keep the 8-row form.
template <int K>
__global__ __launch_bounds__(K / 8) void xprep_row_kernel(const GemmActParams P) {
    constexpr int NG = K / 8, WAVES = NG / 64;
    __shared__ double sg[NG];
    __shared__ float red_mx[WAVES];
    const int g = threadIdx.x, lane = g & 63, wave = g >> 6, t = blockIdx.x;
    const bool live = t < P.T;
    const float *xt = P.x + (size_t)(live ? t : 0) * P.x_stride + 8 * g;
    const f32x4 a = *(const f32x4 *)xt, b = *(const f32x4 *)(xt + 4);
    float v[8] = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
    if (P.norm_w) {
        const f32x4 wa = *(const f32x4 *)(P.norm_w + 8 * g), wb = *(const f32x4 *)(P.norm_w + 8 * g + 4);
        sg[g] = group_ss(v);
        __syncthreads();
        // lane (w, gl) of xprep_kernel: groups gl + 8 (w + 8 j); every wave sums the row for itself
        const int gl = lane & 7, w = lane >> 3;
        double ss = 0;
#pragma unroll
        for (int j = 0; j < NG / 64; j++) ss += sg[gl + 8 * (w + 8 * j)];
#pragma unroll
        for (int m = 1; m < 8; m <<= 1) ss += __shfl_xor(ss, m, 64);
        double tot = 0;
#pragma unroll
        for (int i = 0; i < 8; i++) tot += __shfl(ss, 8 * i, 64);
        const float scale = 1.0f / sqrtf((float)(tot / K) + P.eps);
        const float gg[8] = {wa[0], wa[1], wa[2], wa[3], wb[0], wb[1], wb[2], wb[3]};
#pragma unroll
        for (int e = 0; e < 8; e++) v[e] = v[e] * scale * gg[e];
    }
    float mx = 0.f;
#pragma unroll
    for (int e = 0; e < 8; e++) mx = fmaxf(mx, fabsf(v[e]));
    mx = wave_max(mx);
    if (lane == 0) red_mx[wave] = mx;
    __syncthreads();
    mx = red_mx[0];
#pragma unroll
    for (int w = 1; w < WAVES; w++) mx = fmaxf(mx, red_mx[w]);
    const int e = live ? row_exp(mx) : 0;
    f16x8 h8, l8;
#pragma unroll
    for (int i = 0; i < 8; i++) {
        _Float16 h, l;
        split_store(live ? v[i] : 0.f, e, &h, &l);
        h8[i] = h;
        l8[i] = l;
    }
    const size_t o = plane_unit(t, g, K);
    *(f16x8 *)(P.xh + o) = h8;
    *(f16x8 *)(P.xl + o) = l8;
    if (P.xs) {  // the block sums: a 32-element block's 4 groups are 4 lanes
        float gs = 0.f;
#pragma unroll
        for (int i = 0; i < 8; i++) gs += (float)h8[i] + (float)l8[i];
        gs += __shfl_xor(gs, 1, 64);
        gs += __shfl_xor(gs, 2, 64);
        if ((g & 3) == 0) P.xs[((size_t)(t >> 7) * (K / 32) + (g >> 2)) * GEMM_TILE + (t & 127)] = gs;
    }
    if (g == 0) P.eexp[t] = e;
}

// ---------------------------------------------------------------------------
// gemm3: workgroup tile 128 weight rows (n) x 128 tokens (t), 4 waves in a 2 x 2 grid of
// 64 x 64, each four 32 x 32 MFMA blocks. K runs in chunks of 32 (two MFMA k-steps of 16). A
// chunk of each operand (hi and lo planes, 128 rows x 32 k) goes into LDS in the MFMA operand
// order: per plane, 32-row block and k-step, 1 KiB in which lane l's 16 bytes hold row l & 31,
// k 8 (l >> 5) .. +7 (the same order for the weight rows, operand A, and for the tokens,
// operand B), so every fragment read is one conflict-free ds_read_b128 per lane. The planes
// are stored in that order already (plane_unit), so the chunk's copy into LDS is contiguous on
// both sides. While a chunk is computed from LDS, the next one is stored there and the two
// after it are in flight.
constexpr int GM_TILE = GEMM_TILE, GM_KC = 32, GM_THREADS = 256;
constexpr int GM_PLANE_CHUNK = GM_TILE * GM_KC * 2;  // bytes of one plane's chunk (8 KiB)

__global__ __launch_bounds__(GM_THREADS, 2) void gemm3_kernel(const GemmParams P) {
    // [buffer][operand (A = weights, B = tokens)][plane (hi, lo)]: 8 KiB each
    __shared__ __align__(16) uint8_t lds[2][2][2][GM_PLANE_CHUNK];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wn = wave & 1, wt = wave >> 1;
    // Tile of this workgroup. The hardware deals workgroups to the 8 XCDs in id order (id % 8),
    // each XCD with its own L2: XCD x takes the stripe of weight-row tiles [x w, x w + w) and
    // walks it token-tile-major, so the workgroups resident on one XCD share their weight and
    // token chunks in that L2 (a row-major deal spreads them over the whole output grid).
    const int NT = P.N / GM_TILE, id = blockIdx.x;
    int nt, tt;
    if (NT % 8 == 0) {
        const int w = NT / 8, j = id >> 3;
        nt = (id & 7) * w + j % w;
        tt = j / w;
    } else {
        nt = id % NT;
        tt = id / NT;
    }
    const int n0 = nt * GM_TILE, t0 = tt * GM_TILE;
    const int K = P.K;
    // global -> LDS: a plane's chunk is 512 contiguous units of 16 bytes already in the LDS
    // order (plane_unit); thread tid copies units tid and tid + 256, so a wave's load and its
    // LDS store each cover 1 KiB contiguously (whole cache lines, no bank conflicts)
    const _Float16 *srcA[2] = {P.wh + (size_t)n0 * K, P.wl + (size_t)n0 * K};
    const _Float16 *srcB[2] = {P.xh + (size_t)t0 * K, P.xl + (size_t)t0 * K};
    int goff[2], loff[2];
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const int u = tid + GM_THREADS * i;
        goff[i] = 8 * u;
        loff[i] = 16 * u;
    }
    // two register sets of loaded chunks, so two chunks are in flight while one is computed
    u32x4 ga[2][2][2], gb[2][2][2];  // [operand][plane][unit]
    auto gload = [&](u32x4 (&g)[2][2][2], int kc) {
#pragma unroll
        for (int p = 0; p < 2; p++)
#pragma unroll
            for (int i = 0; i < 2; i++) {
                g[0][p][i] = *(const u32x4 *)(srcA[p] + goff[i] + (size_t)kc * GM_TILE);
                g[1][p][i] = *(const u32x4 *)(srcB[p] + goff[i] + (size_t)kc * GM_TILE);
            }
    };
    auto lstore = [&](const u32x4 (&g)[2][2][2], int buf) {
#pragma unroll
        for (int o = 0; o < 2; o++)
#pragma unroll
            for (int p = 0; p < 2; p++)
#pragma unroll
                for (int i = 0; i < 2; i++) *(u32x4 *)(lds[buf][o][p] + loff[i]) = g[o][p][i];
    };
    f32x16 acc[2][2];
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
        for (int b = 0; b < 2; b++) acc[a][b] = f32x16{};
    auto compute = [&](int buf) {
#pragma unroll
        for (int s = 0; s < 2; s++) {  // k-steps of 16
            f16x8 ah[2], al[2], bh[2], bl[2];
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const int ob = ((2 * wn + j) * 2 + s) * 1024 + lane * 16;  // A block 2wn + j
                const int tb = ((2 * wt + j) * 2 + s) * 1024 + lane * 16;  // B block 2wt + j
                ah[j] = *(const f16x8 *)(lds[buf][0][0] + ob);
                al[j] = *(const f16x8 *)(lds[buf][0][1] + ob);
                bh[j] = *(const f16x8 *)(lds[buf][1][0] + tb);
                bl[j] = *(const f16x8 *)(lds[buf][1][1] + tb);
            }
#pragma unroll
            for (int a = 0; a < 2; a++)
#pragma unroll
                for (int b = 0; b < 2; b++) {
                    acc[a][b] = mfma32_f16(ah[a], bh[b], acc[a][b]);
                    acc[a][b] = mfma32_f16(ah[a], bl[b], acc[a][b]);
                    acc[a][b] = mfma32_f16(al[a], bh[b], acc[a][b]);
                }
        }
    };
    // chunk c lives in LDS buffer c & 1; chunks c + 1 and c + 2 are in registers (set gb holds
    // the odd chunks, ga the even ones) while chunk c is computed. K is a multiple of 64, so
    // the chunk count is even. The barriers order LDS only (lds_barrier): a full __syncthreads
    // would also wait for the chunk loads in flight.
    const int n_chunks = K / GM_KC;
    gload(ga, 0);
    gload(gb, GM_KC);
    lstore(ga, 0);
    gload(ga, 2 * GM_KC);
    lds_barrier();
    // Loads and stores are unconditional (past the last chunk they re-read it and store it into
    // a buffer no one reads again), so the compiler's wait counts are static: a store waits for
    // its own register set only, with the other set's loads still in flight.
    const int last = (n_chunks - 1) * GM_KC;
    for (int c = 0; c < n_chunks; c += 2) {
        // chunk c + 1 into buffer 1 (its chunk c - 1 was finished before the last barrier)
        lstore(gb, 1);
        gload(gb, min((c + 3) * GM_KC, last));
        compute(0);
        lds_barrier();
        lstore(ga, 0);
        gload(ga, min((c + 4) * GM_KC, last));
        compute(1);
        lds_barrier();
    }
    // epilogue: block (a, b) element e is weight row n0 + 64 wn + 32 a + 8 (e >> 2) + 4 (lane >> 5) + (e & 3)
    // and token t0 + 64 wt + 32 b + (lane & 31)
#pragma unroll
    for (int b = 0; b < 2; b++) {
        const int t = t0 + 64 * wt + 32 * b + (lane & 31);
        if (t >= P.T) continue;
        const int et = P.eexp[t];
        float *yt = P.y + (size_t)t * P.y_stride;
        // the exponents and the residual (add) first: a load after a store to y that may alias it
        // waits for that store
        int4 f[2][4];
        f32x4 yin[2][4];
#pragma unroll
        for (int a = 0; a < 2; a++)
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int n = n0 + 64 * wn + 32 * a + 8 * q + 4 * (lane >> 5);
                f[a][q] = *(const int4 *)(P.fexp + n);
                if (P.add) yin[a][q] = *(const f32x4 *)(yt + n);
            }
#pragma unroll
        for (int a = 0; a < 2; a++)
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int n = n0 + 64 * wn + 32 * a + 8 * q + 4 * (lane >> 5);
                f32x4 v = {__builtin_amdgcn_ldexpf(acc[a][b][4 * q], et + f[a][q].x),
                           __builtin_amdgcn_ldexpf(acc[a][b][4 * q + 1], et + f[a][q].y),
                           __builtin_amdgcn_ldexpf(acc[a][b][4 * q + 2], et + f[a][q].z),
                           __builtin_amdgcn_ldexpf(acc[a][b][4 * q + 3], et + f[a][q].w)};
                if (P.add) v += yin[a][q];
                *(f32x4 *)(yt + n) = v;
            }
    }
}


// gemm_int: gemm3's tiles, deal and LDS order with the tokens as operand A and the weights'
// values as operand B, so that an MFMA output lane holds one weight row (16 tokens of it) and
// takes one scale per chunk (SUB = 32) or k-step (SUB = 16). The chunks go straight from memory
// into LDS (global_load_lds_dwordx4: each wave-wide load writes 1 KiB, lane l's 16 bytes at
// l * 16 from the wave's LDS address), STAGES deep: while chunk c is computed, the STAGES - 1 after it
// are in flight, and no register holds them. A chunk's 128 (SUB = 32) or 256 scales ride along
// (lanes 0-7 or 0-15 of each wave load 128 or 256 bytes), and with mins (MIN) the chunk's block sums of
// its tokens and mins of its 128 rows (a few lanes again, two loads).
// Each step makes the products T = sum (xh + xl) v of one chunk (SUB = 32: chains of four MFMAs) or
// k-step (SUB = 16: chains of two), token block by token block, and scales the other block's
// (acc += s T) in between, so that those FMAs run beside MFMAs that do not feed them (against one
// chunk's MFMAs and FMAs in the same step, q8_0: 4000 tokens through 49 Flint blocks 23.2 against
// 24.0 ms). K is summed in segments of GEMM_SEG elements, so that gemm_raw, whose waves take a
// segment each, gives the same bits; the segments' registers come from T in two half sets instead of
// two whole ones.
// What bounds it: at 4000 tokens (q8_0, trace medians) q/k/v 194 and o 152 us, 0.87 and 0.88 PF of MFMA
// work; counters: the matrix pipes are busy 47-48 % of the launch's cycles (53-56 % of those in which a CU has
// waves), LDS indexed operations 22 % without bank conflicts, and a wave spends 21 % of its time at waits
// and barriers and 35 % ready but not issued. At 1000 tokens (64-token tiles) the pipes are busy 29 and
// 26 %. (With whole T sets, no segments and
// loads of 64-bit lane addresses: 195 and 158.)

// 16 bytes a lane from base + voff (base wave-uniform) into LDS at dst + 16 lane. Inline asm: the builtin
// takes a 64-bit address a lane (2 VALU adds per load: a chunk's 7 loads had more of them than the
// scaling has FMAs per MFMA), and the compiler makes LDS reads wait for every load that it tracks.
__device__ inline void lds_load16(uint32_t dst, const void *base, uint32_t voff) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(dst), "v"(voff), "s"(base) : "m0", "memory");
}

template <int SUB>
constexpr int gq_scales() { return (32 / SUB) * GM_TILE; }  // a chunk's scales, per row tile
// a stage: x hi, x lo (64 TB tokens), values, scales, then with mins the token sums and the mins
template <int SUB, int TB>
constexpr int gq_stage() { return (TB + 1) * GM_PLANE_CHUNK + gq_scales<SUB>() * 4; }
template <int SUB, bool MIN, int TB>
constexpr int gq_bytes() { return gq_stage<SUB, TB>() + (MIN ? (64 * TB + GM_TILE) * 4 : 0); }

// TB token blocks a wave: 128 rows x 64 TB tokens a workgroup. STAGES chunks in LDS, so STAGES - 1
// in flight. EU: waves per SIMD that the registers are held to.
template <int SUB, bool MIN, int TB, int STAGES, int EU>
__global__ __launch_bounds__(GM_THREADS, EU) void gemm_int_kernel(const GemmParams P) {
    constexpr int SCB = gq_scales<SUB>(), SCL = SCB / 16;  // scales per chunk; lanes that load them
    constexpr int STAGE = gq_stage<SUB, TB>(), LOADS = 2 * TB + 2 + 1 + (MIN ? 2 : 0);  // direct loads per wave per chunk
    constexpr int TT = 64 * TB, XP = TT * GM_KC * 2;  // tokens; bytes of an x plane's chunk
    static_assert(LOADS * (STAGES - 1) < 64, "the loads in flight fit vmcnt");
    __shared__ __align__(16) uint8_t lds[STAGES][gq_bytes<SUB, MIN, TB>()];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wn = wave & 1, wt = wave >> 1;
    const int NT = P.N / GM_TILE, id = blockIdx.x;
    int nt, tt;
    if (NT % 8 == 0) {  // the XCD deal of gemm3
        const int w = NT / 8, j = id >> 3;
        nt = (id & 7) * w + j % w;
        tt = j / w;
    } else {
        nt = id % NT;
        tt = id / NT;
    }
    const int n0 = nt * GM_TILE, t0 = tt * TT;
    const int K = P.K;
    // wave-uniform starts of the tile's planes (the x planes' blocks hold 128 tokens), its scales, and with mins
    // its block sums and mins; a lane's offset in a wave's 1 KiB load, and in its part of the small ones
    const size_t xo = (size_t)(t0 >> 7) * GM_TILE * K + (t0 & 127) * GM_KC;
    const uint8_t *const srcx[2] = {(const uint8_t *)(P.xh + xo), (const uint8_t *)(P.xl + xo)};
    const uint8_t *const srcw = (const uint8_t *)(P.wh + (size_t)n0 * K);
    const uint8_t *const srcd = (const uint8_t *)(P.wd + (size_t)nt * (K / GM_KC) * SCB);
    const uint8_t *const srcs = MIN ? (const uint8_t *)(P.xs + (size_t)(t0 >> 7) * (K / GM_KC) * GM_TILE + (t0 & 127)) : nullptr;
    const uint8_t *const srcm = MIN ? (const uint8_t *)(P.wm + (size_t)nt * (K / GM_KC) * GM_TILE) : nullptr;
    constexpr int SL = TT / 16;  // lanes of a wave that load 16 bytes of the block sums
    const uint32_t lo16 = 16 * tid, lod = SCB * wave + 16 * (lane & (SCL - 1)), los = TT * wave + 16 * (lane & (SL - 1)), lom = 128 * wave + 16 * (lane & 7);
    const uint32_t l0 = (uint32_t)(uintptr_t)(lds_void *)lds;
    const int n_chunks = K / GM_KC;
    auto issue = [&](int c, int st) {  // chunk c into stage st
        const uint32_t base = l0 + st * sizeof(lds[0]), mine = base + 1024 * wave;
        const size_t cb = (size_t)c * GM_PLANE_CHUNK;
#pragma unroll
        for (int p = 0; p < 2; p++)
#pragma unroll
            for (int i = 0; i < TB; i++) lds_load16(mine + p * XP + 4096 * i, srcx[p] + cb + 4096 * i, lo16);
#pragma unroll
        for (int i = 0; i < 2; i++) lds_load16(mine + 2 * XP + 4096 * i, srcw + cb + 4096 * i, lo16);
        if (lane < SCL) lds_load16(base + STAGE - 4 * SCB + SCB * wave, srcd + (size_t)c * (4 * SCB), lod);
        if constexpr (MIN) {
            if (lane < SL) lds_load16(base + STAGE + TT * wave, srcs + (size_t)c * (4 * GM_TILE), los);
            if (lane < 8) lds_load16(base + STAGE + 4 * TT + 128 * wave, srcm + (size_t)c * (4 * GM_TILE), lom);
        }
    };
    // tot: the sums of the finished segments; acc: the running segment's [token block][weight block]
    f32x16 tot[TB][2], acc[TB][2];
#pragma unroll
    for (int a = 0; a < TB; a++)
#pragma unroll
        for (int b = 0; b < 2; b++) tot[a][b] = acc[a][b] = f32x16{};
    // Products in flight, two sets that take turns: one token block's MFMAs into a set run beside the FMAs
    // that scale the other's. A turn is a chunk's (SUB = 16: a k-step's) token block.
    f32x16 T[2][2];      // [set][weight block]
    float d[2][2];       // their scales
    f16x8 wq[2][2];      // [k-step][weight block]
#pragma unroll
    for (int b = 0; b < 2; b++) T[1][b] = f32x16{}, d[1][b] = 0.f;
    auto scale = [&](int set, int a) {
#pragma unroll
        for (int b = 0; b < 2; b++)
#pragma unroll
            for (int e = 0; e < 16; e++) acc[a][b][e] = fmaf(d[set][b], T[set][b][e], acc[a][b][e]);
    };
    auto flush = [&](int a) {
#pragma unroll
        for (int b = 0; b < 2; b++) tot[a][b] += acc[a][b], acc[a][b] = f32x16{};
    };
    // token block a's products of k-steps s0 .. s1 - 1 of the chunk at base: x hi over the steps' k,
    // then x lo (gemm_raw's order: the MFMA adds its k in groups of 8, in order)
    auto mul = [&](const uint8_t *base, int set, int a, int s0, int s1) {
#pragma unroll
        for (int p = 0; p < 2; p++)
#pragma unroll
            for (int s = s0; s < s1; s++) {
                const f16x8 x = *(const f16x8 *)(base + p * XP + ((TB * wt + a) * 2 + s) * 1024 + lane * 16);
#pragma unroll
                for (int b = 0; b < 2; b++) T[set][b] = mfma32_f16(x, wq[s][b], p == 0 && s == s0 ? f32x16{} : T[set][b]);
            }
    };
    auto mins = [&](const uint8_t *base, int a) {  // acc -= m S, S of element e's token
        const float *const sl = (const float *)(base + STAGE), *const ml = sl + TT;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const f32x4 S4 = *(const f32x4 *)(sl + 32 * (TB * wt + a) + 8 * q + 4 * (lane >> 5));
#pragma unroll
            for (int b = 0; b < 2; b++) {
                const float m = ml[64 * wn + 32 * b + (lane & 31)];
#pragma unroll
                for (int i = 0; i < 4; i++) acc[a][b][4 * q + i] = fmaf(-m, S4[i], acc[a][b][4 * q + i]);
            }
        }
    };
    // One step: k-steps s0 .. s1 - 1 of the chunk in stage st; set: the one its first token block takes.
    // first: the step begins a segment, so the one before is complete once its last products are scaled.
    auto step = [&](int st, int set, int s0, int s1, bool first) {
        const uint8_t *const base = lds[st];
#pragma unroll
        for (int s = s0; s < s1; s++)
#pragma unroll
            for (int b = 0; b < 2; b++)
                wq[s][b] = *(const f16x8 *)(base + 2 * XP + ((2 * wn + b) * 2 + s) * 1024 + lane * 16);
        const float *const sc = (const float *)(base + STAGE - 4 * SCB) + (SUB == 16 ? GM_TILE * s0 : 0);
#pragma unroll
        for (int b = 0; b < 2; b++) d[set][b] = sc[64 * wn + 32 * b + (lane & 31)];
        mul(base, set, 0, s0, s1);
        scale(set ^ 1, TB - 1);
        if (first)
#pragma unroll
            for (int a = 0; a < TB; a++) flush(a);
        if (MIN && s0 == 0)
#pragma unroll
            for (int a = 0; a < TB; a++) mins(base, a);
        if constexpr (TB == 2) {
#pragma unroll
            for (int b = 0; b < 2; b++) d[set ^ 1][b] = d[set][b];
            mul(base, set ^ 1, 1, s0, s1);
            scale(set, 0);
        }
    };
    // Chunk c lives in stage c % STAGES. Every wave issues the same LOADS loads per chunk (past the
    // last chunk it re-reads the last one into a stage no one reads again), so "chunk c has
    // landed" is vmcnt(LOADS (STAGES - 2)) with the chunks after it still in flight; the barrier then
    // makes every wave's part of it visible, and it also ends every wave's reads of the stage of chunk
    // c - 1, which chunk c + STAGES - 1 overwrites after it. Those reads are waited for too: the ones that feed
    // FMAs (scales, token sums, mins) are otherwise still on their way here, since the FMAs that use them
    // follow the barrier. The wait is asm with a memory clobber, so that no LDS access moves past it
    // or across the barrier. No fence: a workgroup-scope fence would wait for every load in flight (vmcnt(0)).
    int st = 0;
    auto sync = [&](int c) {
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(LOADS *(STAGES - 2)) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        const int at = st;
        issue(min(c + STAGES - 1, n_chunks - 1), at == 0 ? STAGES - 1 : at - 1);
        st = at == STAGES - 1 ? 0 : at + 1;
        return at;
    };
    auto begins = [&](int c) { return (c & (GEMM_SEG / GM_KC - 1)) == 0; };
#pragma unroll
    for (int c = 0; c < STAGES - 1; c++) issue(c, c);
    // (TB = 2 and SUB = 16 end a chunk on the set they began it with; else the chunks alternate)
    constexpr int TURN = TB == 2 || SUB == 16 ? 1 : 2;
    for (int c = 0; c < n_chunks; c += TURN) {  // K is a multiple of 64: the chunk count is even
#pragma unroll
        for (int i = 0; i < TURN; i++) {
            const int at = sync(c + i);
            if constexpr (SUB == 32) {
                step(at, TB == 2 ? 0 : i, 0, 2, i == 0 && begins(c));
            } else {
                step(at, 0, 0, 1, i == 0 && begins(c));
                step(at, TB == 2 ? 0 : 1, 1, 2, false);
            }
        }
    }
    scale(1, TB - 1);
#pragma unroll
    for (int a = 0; a < TB; a++) flush(a);
    wait_vmcnt<0>();  // the re-reads past the last chunk land before the workgroup's LDS goes
    // epilogue: block (a, b) element e is token t0 + 32 (TB wt + a) + 8 (e >> 2) + 4 (lane >> 5) + (e & 3)
    // and weight row n0 + 64 wn + 32 b + (lane & 31): a store instruction writes 32 consecutive
    // floats of each of two token rows. Token block a by token block a, its row exponents and
    // its residual (add) are all read before its first store (rows past T re-read row T - 1): a
    // load after a store that may alias it waits for the store, so loads between the stores cost
    // a round trip each (36 us per o launch at T = 4000).
    auto token = [&](int a, int e) { return t0 + 32 * (TB * wt + a) + 8 * (e >> 2) + 4 * (lane >> 5) + (e & 3); };
    float *const y0 = P.y + n0 + 64 * wn + (lane & 31);
#pragma unroll
    for (int a = 0; a < TB; a++) {
        int ex[16];
        float yin[16][2];
#pragma unroll
        for (int e = 0; e < 16; e++) ex[e] = P.eexp[min(token(a, e), P.T - 1)];
        if (P.add) {
#pragma unroll
            for (int e = 0; e < 16; e++)
#pragma unroll
                for (int b = 0; b < 2; b++) yin[e][b] = y0[(size_t)min(token(a, e), P.T - 1) * P.y_stride + 32 * b];
        }
#pragma unroll
        for (int e = 0; e < 16; e++) {
            const int t = token(a, e);
            if (t >= P.T) continue;
#pragma unroll
            for (int b = 0; b < 2; b++) {
                float v = __builtin_amdgcn_ldexpf(tot[a][b][e], ex[e]);
                if (P.add) v += yin[e][b];
                y0[(size_t)t * P.y_stride + 32 * b] = v;
            }
        }
    }
}

template <int TB, int STAGES, int EU>
static void launch_gemm_int(const GemmParams &G, hipStream_t stream) {
    void (*gk)(GemmParams) = G.imin ? (G.isub == 32 ? gemm_int_kernel<32, true, TB, STAGES, EU> : gemm_int_kernel<16, true, TB, STAGES, EU>)
                                    : (G.isub == 32 ? gemm_int_kernel<32, false, TB, STAGES, EU> : gemm_int_kernel<16, false, TB, STAGES, EU>);
    hipLaunchKernelGGL(gk, dim3(G.N / GM_TILE * ((G.T + 64 * TB - 1) / (64 * TB))), dim3(GM_THREADS), 0, stream, G);
}

// ---------------------------------------------------------------------------
// gemm_raw: the integer form's GEMM for short batches, straight from the GGUF rows.
//
// A short batch has too few 128 x 128 tiles to fill the GPU (16 tokens: 40 workgroups for q/k/v, 16
// for o, each walking K alone at a memory round trip every two chunks), and the weight planes cost
// more than the products. Here a workgroup takes 32 weight rows x 32 tokens (160 and 64 row tiles),
// and its waves one segment of K each (GEMM_SEG: 4 waves for q/k/v, 8 for o) with nothing shared until
// the segments' sums meet in LDS at the end. A wave requests its row bytes a group of chunks ahead
// (16-byte loads along the rows, staged in its own LDS area) and its
// tokens' units from the x planes straight into the MFMA operands, XD chunks ahead; per chunk it
// decodes 16 weights a lane, makes the products T on four MFMAs and adds acc += s T (- m S). T's groups
// of 8, the chunks of a segment and the segments are added in gemm_int_kernel's order, so a
// token's output has the same bits in a batch of any size.
// The row bytes go through LDS because lanes that each read their own row's 8-32 bytes of a block
// fetched whole lines for a quarter of their bytes and evicted each other's from the L1 (an unsegmented
// form of this kernel at 512 tokens 121 us against 71 without those loads).

static_assert(GEMM_RAW_TOKENS <= 512, "xprep_row_kernel is the faster one up to 512 rows");
constexpr int GR_CHUNKS = GEMM_SEG / 32;    // chunks of a segment
static_assert(GR_TILE == GEMM_RAW_TILE, "the x planes hold whole token tiles");

// LDS of one wave: a group of its rows, and with mins its segment's token sums; later its sums
template <int TYPE>
constexpr int raw_area() {
    return 32 * RawRows<TYPE>::STRIDE + (TYPE == W_Q5_K ? GR_CHUNKS * GR_TILE * 4 : 0);
}
template <int SUB>
constexpr int raw_area_max() {  // q8_0, iq4_xs and the 2-byte types have one size
    return SUB == 16 ? raw_area<W_Q6_K>() : raw_area<W_Q8_0>() > raw_area<W_Q5_K>() ? raw_area<W_Q8_0>() : raw_area<W_Q5_K>();
}

// A wave's segment of the tile's sums (the caller's acc): seg is the tile's first row at the segment's
// first byte, chunk0 its first chunk.
template <int SUB, int TYPE>
__device__ __forceinline__ void gemm_raw_segment(const GemmParams &P, const uint8_t *seg, int row_bytes, uint8_t *area, int t0,
                                                 int chunk0, f32x16 &acc) {
    typedef RawRows<TYPE> RR;
    constexpr int NS = 32 / SUB, G = RR::G, NG = GR_CHUNKS / G, XD = 4;
    constexpr bool MIN = TYPE == W_Q5_K;
    const int lane = threadIdx.x & 63, h = lane >> 5, r32 = lane & 31;
    RawCopy<TYPE> C;  // the group after the one in LDS
    C.init(row_bytes, lane);
    // x: the tile's units of a chunk are 2 KiB of each plane (plane_unit), lane's k-step s at 64 s + lane
    const size_t xo = ((size_t)(t0 >> 7) * (P.K / 32) + chunk0) * (512 * 16) + ((t0 >> 5) & 3) * 2048;
    const uint8_t *const xp[2] = {(const uint8_t *)P.xh + xo, (const uint8_t *)P.xl + xo};
    f16x8 X[XD][2][2];  // [chunk][plane][k-step]
    auto xload = [&](int c) {
#pragma unroll
        for (int p = 0; p < 2; p++) {
            const uint8_t *xr = xp[p] + c * (512 * 16);
            asm volatile("" : "+s"(xr));  // a scalar base, no vector address to keep
#pragma unroll
            for (int s = 0; s < 2; s++) X[c % XD][p][s] = *(const f16x8 *)(xr + (16 * lane + 1024 * s));
        }
    };
    f32x16 T[2][NS];  // the products of the even / odd chunks
    float sc[2][2];
    auto scale = [&](int c) {
#pragma unroll
        for (int k = 0; k < NS; k++)
#pragma unroll
            for (int e = 0; e < 16; e++) acc[e] = fmaf(sc[c & 1][k], T[c & 1][k][e], acc[e]);
    };
    f32x4 S0, S1;
    uint8_t *const sums = area + 32 * RR::STRIDE;  // [chunk][token]
    C.load(seg);
    if (MIN) {
        const float *const sp = P.xs + ((size_t)(t0 >> 7) * (P.K / 32) + chunk0 + (lane >> 3)) * GEMM_TILE + (t0 & 127) + 4 * (lane & 7);
        S0 = *(const f32x4 *)sp, S1 = *(const f32x4 *)(sp + 8 * GEMM_TILE);
    }
#pragma unroll
    for (int c = 0; c < XD; c++) xload(c);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int c = 0; c < GR_CHUNKS; c++) {
        const int q = c / G, j = c % G;
        if (j == 0) {
            if (q > 0) wave_lds_fence();  // the group before's reads, of other types, stay ahead of these stores
            C.store(area, lane);
            if (MIN && q == 0) *(f32x4 *)(sums + 16 * lane) = S0, *(f32x4 *)(sums + 1024 + 16 * lane) = S1;
            wave_lds_fence();
            if (q + 1 < NG) C.load(seg + (q + 1) * RR::BYTES);
        }
        f16x8 w[2];
        float m = 0.f;
        uint32_t ro = r32 * RR::STRIDE;  // opaque per chunk: the compiler would merge reads of several chunks
        asm volatile("" : "+v"(ro));
        RR::get(area + ro, j, h, w, sc[c & 1], m);
#pragma unroll
        for (int k = 0; k < NS; k++)
#pragma unroll
            for (int p = 0; p < 2; p++)
#pragma unroll
                for (int s = k; s < (NS == 1 ? 2 : k + 1); s++)
                    T[c & 1][k] = mfma32_f16(X[c % XD][p][s], w[s], p == 0 && s == k ? f32x16{} : T[c & 1][k]);
        if (c + XD < GR_CHUNKS) xload(c + XD);
        if (c > 0) scale(c - 1);  // the chunk before, while this one's MFMAs run
        if (MIN)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const f32x4 S = *(const f32x4 *)(sums + 128 * c + 32 * i + 16 * h);
#pragma unroll
                for (int e = 0; e < 4; e++) acc[4 * i + e] = fmaf(-m, S[e], acc[4 * i + e]);
            }
        asm volatile("" : "+v"(acc));  // or the compiler keeps many chunks' T and scales them at the end
        __builtin_amdgcn_sched_barrier(0);
    }
    scale(GR_CHUNKS - 1);
}

// SUB as gemm_int_kernel's; WAVES = K / GEMM_SEG segments
template <int SUB, int WAVES>
__global__ __launch_bounds__(64 * WAVES, 2) void gemm_raw_kernel(const GemmParams P, const GemmWeightParams W, int n_tt) {
    constexpr int AREA = raw_area_max<SUB>();
    static_assert(AREA >= 4096, "a wave's sums fit its area");
    __shared__ __align__(16) uint8_t lds[WAVES][AREA];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // workgroup ids go to the 8 XCDs in turn: the token tiles of a row tile follow each other on one
    // XCD, whose L2 then holds the rows
    const int id = blockIdx.x, j = id >> 3, n0 = ((id & 7) + 8 * (j / n_tt)) * GR_TILE, t0 = (j % n_tt) * GR_TILE;
    const MatvecSeg s0 = W.seg[0], s1 = W.seg[1], s2 = W.seg[2];
    const bool in2 = W.n_seg > 2 && n0 >= s2.row0, in1 = !in2 && W.n_seg > 1 && n0 >= s1.row0;
    const MatvecSeg S = in2 ? s2 : in1 ? s1 : s0;
    const uint8_t *const row0 = S.w + (size_t)(n0 - S.row0) * S.row_bytes;  // the tile's first row
    const uint8_t *const seg = row0 + wave * (S.row_bytes / WAVES);
    f32x16 acc = f32x16{};
    switch (S.type) {
        case W_Q8_0: gemm_raw_segment<SUB, W_Q8_0>(P, seg, S.row_bytes, lds[wave], t0, wave * GR_CHUNKS, acc); break;
        case W_Q5_K: gemm_raw_segment<SUB, W_Q5_K>(P, seg, S.row_bytes, lds[wave], t0, wave * GR_CHUNKS, acc); break;
        case W_IQ4_XS: gemm_raw_segment<SUB, W_IQ4_XS>(P, seg, S.row_bytes, lds[wave], t0, wave * GR_CHUNKS, acc); break;
        case W_F16: gemm_raw_segment<SUB, W_F16>(P, seg, S.row_bytes, lds[wave], t0, wave * GR_CHUNKS, acc); break;
        case W_BF16: gemm_raw_segment<SUB, W_BF16>(P, seg, S.row_bytes, lds[wave], t0, wave * GR_CHUNKS, acc); break;
        default:
            if constexpr (SUB == 16) gemm_raw_segment<SUB, W_Q6_K>(P, seg, S.row_bytes, lds[wave], t0, wave * GR_CHUNKS, acc);
    }
    // the segments' sums, in order: thread (wave, lane) takes EPT elements e0 .. of lane's 16
    constexpr int EPT = 16 / WAVES;
    float *const mine = (float *)lds[wave];  // read by no other wave until the barrier: [e / 4][lane][e % 4]
#pragma unroll
    for (int q = 0; q < 4; q++) *(f32x4 *)(mine + 256 * q + 4 * lane) = f32x4{acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]};
    __syncthreads();
    const int e0 = EPT * wave, h = lane >> 5;
    float tot[EPT];
#pragma unroll
    for (int e = 0; e < EPT; e++) tot[e] = 0.f;
#pragma unroll
    for (int w = 0; w < WAVES; w++) {
        typedef float vec __attribute__((ext_vector_type(EPT)));
        const vec v = *(const vec *)((const float *)lds[w] + 256 * (e0 >> 2) + 4 * lane + (e0 & 3));
#pragma unroll
        for (int e = 0; e < EPT; e++) tot[e] += v[e];
    }
    // element e is token t0 + 8 (e >> 2) + 4 h + (e & 3), row n0 + lane % 32
    const int t = t0 + 8 * (e0 >> 2) + 4 * h + (e0 & 3);
    float *const y = P.y + (size_t)t * P.y_stride + n0 + (lane & 31);
    float yin[EPT];
    int ex[EPT];
#pragma unroll
    for (int e = 0; e < EPT; e++) {
        ex[e] = P.eexp[t + e];  // has entries up to the padded token count
        if (P.add) yin[e] = t + e < P.T ? y[e * P.y_stride] : 0.f;
    }
#pragma unroll
    for (int e = 0; e < EPT; e++) {
        float v = __builtin_amdgcn_ldexpf(tot[e], ex[e]);
        if (P.add) v += yin[e];
        if (t + e < P.T) y[e * P.y_stride] = v;
    }
}

hipError_t launch_proj_gemm(const GemmWeightParams &W, const GemmActParams &X, const GemmParams &G, bool prep_weights,
                            hipStream_t stream) {
    // the planes' chunk order and the GEMM's tiles need whole 128-row tiles of both operands
    if (G.N % GM_TILE != 0 || (G.K != 2048 && G.K != 4096)) return hipErrorInvalidValue;
    if (G.raw) {  // the integer form from the GGUF rows
        if (X.T_pad % GR_TILE != 0 || X.T_pad < G.T || G.T <= 0 || G.N % (8 * GR_TILE) != 0 || (G.isub != 32 && G.isub != 16))
            return hipErrorInvalidValue;
        hipLaunchKernelGGL(G.K == 2048 ? xprep_row_kernel<2048> : xprep_row_kernel<4096>, dim3(X.T_pad), dim3(G.K / 8), 0, stream, X);
        const int n_tt = X.T_pad / GR_TILE;
        void (*gk)(GemmParams, GemmWeightParams, int) =
            G.K == 2048 ? (G.isub == 32 ? gemm_raw_kernel<32, 2048 / GEMM_SEG> : gemm_raw_kernel<16, 2048 / GEMM_SEG>)
                        : (G.isub == 32 ? gemm_raw_kernel<32, 4096 / GEMM_SEG> : gemm_raw_kernel<16, 4096 / GEMM_SEG>);
        hipLaunchKernelGGL(gk, dim3(G.N / GR_TILE * n_tt), dim3(64 * (G.K / GEMM_SEG)), 0, stream, G, W, n_tt);
        return hipGetLastError();
    }
    if (X.T_pad % GM_TILE != 0) return hipErrorInvalidValue;
    if (G.isub == 32 || G.isub == 16) {
        if (prep_weights)
            hipLaunchKernelGGL(G.isub == 32 ? wprep_int_kernel<32> : wprep_int_kernel<16>, dim3(G.K / 256 / WP_WAVES, G.N / GR_TILE),
                               dim3(64 * WP_WAVES), 0, stream, W, G.K);
        if (X.T_pad > 0) {
            if (G.K == 2048)
                hipLaunchKernelGGL(xprep_kernel<2048>, dim3(X.T_pad / 8), dim3(512), 0, stream, X);
            else
                hipLaunchKernelGGL(xprep_kernel<4096>, dim3(X.T_pad / 8), dim3(512), 0, stream, X);
            if (G.T <= GEMM_INT_64)
                launch_gemm_int<1, 4, 2>(G, stream);
            else
                launch_gemm_int<2, 3, 2>(G, stream);
        }
        return hipGetLastError();
    }
    if (G.K == 2048) {
        if (prep_weights) hipLaunchKernelGGL(wprep_kernel<2048>, dim3(G.N / 8), dim3(512), 0, stream, W);
        if (X.T_pad > 0) hipLaunchKernelGGL(xprep_kernel<2048>, dim3(X.T_pad / 8), dim3(512), 0, stream, X);
    } else {
        if (prep_weights) hipLaunchKernelGGL(wprep_kernel<4096>, dim3(G.N / 8), dim3(512), 0, stream, W);
        if (X.T_pad > 0) hipLaunchKernelGGL(xprep_kernel<4096>, dim3(X.T_pad / 8), dim3(512), 0, stream, X);
    }
    if (X.T_pad > 0)
        hipLaunchKernelGGL(gemm3_kernel, dim3(G.N / GM_TILE * (X.T_pad / GM_TILE)), dim3(GM_THREADS), 0, stream, G);
    return hipGetLastError();
}

}  // namespace flint
