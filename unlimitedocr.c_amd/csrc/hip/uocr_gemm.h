/*
 * uocr_gemm.h - what the prefill GEMM kernels share: operand types, the
 * dequantisation of .uocr weights into MFMA operands, epilogue functions and
 * the kernels' argument block.
 */
#ifndef UOCR_GEMM_H
#define UOCR_GEMM_H

#include "uocr_kernels.h"

#include <type_traits>

typedef _Float16 h16;
typedef _Float16 h16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32;

__device__ __forceinline__ float silu_p(float g) {
    return g / (1.0f + expf(-g));
}

union U4H8 {
    uint4 u;
    h16x8 v;
    h16 h[8];
};

/* exact fp16 of bytes b0,b1 (each < 256) + 1024 */
__device__ __forceinline__ u32 magic2(u32 v, u32 sel) {
    return __builtin_amdgcn_perm(0x64646464u, v, sel);
}

typedef _Float16 h16x2 __attribute__((ext_vector_type(2)));

/* Eight weights as fp16(q * scale), the product of two fp16 values rounded
 * once, as half(float(q) * scale) in gemm_q4.metal:55 (the integer q is exact
 * after the bias subtraction); sc holds the scale's fp16 bits.
 * Q4: the low (or high) nibbles of the bytes of w0 and w1. */
__device__ __forceinline__ h16x8 dequant_q4(u32 w0, u32 w1, bool high, u32 sc) {
    const h16 sv = __builtin_bit_cast(h16, (unsigned short)sc);
    const h16x2 sc2 = {sv, sv}, bb = __builtin_bit_cast(h16x2, 0x64086408u); /* (1032, 1032) */
    union {
        h16x8 v;
        u32 d[4];
    } o;
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const u32 x = q == 0 ? w0 : w1;
        const u32 nb = high ? (x >> 4) & 0x0F0F0F0Fu : x & 0x0F0F0F0Fu;
        o.d[2 * q] = __builtin_bit_cast(u32, (__builtin_bit_cast(h16x2, magic2(nb, 0x04010400u)) - bb) * sc2);
        o.d[2 * q + 1] = __builtin_bit_cast(u32, (__builtin_bit_cast(h16x2, magic2(nb, 0x04030402u)) - bb) * sc2);
    }
    return o.v;
}

/* Q8: the bytes of w0 and w1. */
__device__ __forceinline__ h16x8 dequant_q8(u32 w0, u32 w1, u32 sc) {
    const h16 sv = __builtin_bit_cast(h16, (unsigned short)sc);
    const h16x2 sc2 = {sv, sv}, bb = __builtin_bit_cast(h16x2, 0x64806480u); /* (1152, 1152) */
    union {
        h16x8 v;
        u32 d[4];
    } o;
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const u32 u = (q == 0 ? w0 : w1) ^ 0x80808080u;
        o.d[2 * q] = __builtin_bit_cast(u32, (__builtin_bit_cast(h16x2, magic2(u, 0x04010400u)) - bb) * sc2);
        o.d[2 * q + 1] = __builtin_bit_cast(u32, (__builtin_bit_cast(h16x2, magic2(u, 0x04030402u)) - bb) * sc2);
    }
    return o.v;
}

__device__ __forceinline__ h16x8 operand_f16(u32 a, u32 b, u32 c, u32 d) {
    U4H8 o;
    o.u = make_uint4(a, b, c, d);
    return o.v;
}

/* f(integral_constant<int, i>) for i = 0..N-1, in order, unrolled at compile
 * time (register-ring slots need constant indices). */
template <int N, typename F>
__device__ __forceinline__ void static_for(F &&f) {
    if constexpr (N > 0) {
        static_for<N - 1>(f);
        f(std::integral_constant<int, N - 1>{});
    }
}

enum { GE_F16 = 0, GE_F32 = 1, GE_SWIGLU = 2, GE_VISION = 3, GE_PART = 4, GE_ROPE = 5 };

/* QuickGELU of the CLIP MLP: x * sigmoid(1.702 x) (dense.metal:63-66). */
__device__ __forceinline__ float quick_gelu(float x) {
    /* hardware exp2 and reciprocal (about 1 ulp each in fp32; the result is
     * rounded to fp16) instead of the full-precision expf and divide */
    return x * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.702f * 1.4426950408889634f * x));
}

/* GELU of the SAM MLP, 0.5 x (1 + erf(x / sqrt 2)), with erf from
 * Abramowitz & Stegun 7.1.26 (|error| <= 1.5e-7), the approximation the
 * reference's SAM kernels use (sam.metal:78-91). */
__device__ __forceinline__ float gelu_erf_as(float x) {
    const float z = x * 0.70710678118654752f;
    const float az = fabsf(z);
    const float t = __builtin_amdgcn_rcpf(1.0f + 0.3275911f * az);
    const float poly = ((((1.061405429f * t - 1.453152027f) * t + 1.421413741f) * t - 0.284496736f) * t + 0.254829592f) * t;
    const float e = 1.0f - poly * __builtin_amdgcn_exp2f(-1.4426950408889634f * az * az);
    return 0.5f * x * (1.0f + (z < 0.0f ? -e : e));
}

template <int QT>
__device__ __forceinline__ u32 b_koff(u32 i, u32 h) {
    return QT == 4 ? ((i & 2u) << 4) + 16u * h + ((i & 1u) << 3) : 32u * h + 8u * i;
}

struct RopeTabP {
    float f[UOCR_K_HEAD_DIM / 2];
};

/* GE_ROPE destinations: q rows [P][1280], the layer's K / V caches
 * [head][cap][128]; cs holds (cos, sin) of token t's angle t * f[d] at
 * cs[64 t + d]. */
struct RopeDst {
    const float2 *cs;
    h16 *q, *k, *v;
    u32 cap;
};

struct GemmArgs {
    const h16 *A;        /* activations, row stride lda (halves) */
    u32 lda;
    const int32_t *a_idx;  /* grouped: A row of each slot */
    const int32_t *o_idx;  /* grouped: output row of each slot */
    u32 M, N, K;
    uocr_qmat W[3];      /* W[0] (and W[1] for SwiGLU; W[seg] when nseg) */
    u32 nseg;            /* when nonzero, columns [s*nseg, (s+1)*nseg) use W[s] */
    uint64_t w_stride, s_stride; /* grouped: per-expert strides (bytes / halves) */
    const int32_t *tile_e, *tile_s0, *tile_s1, *ntiles; /* grouped tile table */
    void *out;
    u32 ldo;
    const h16 *res;      /* GE_F16: optional residual, row stride ldr */
    u32 ldr;
    const h16 *bias;     /* GE_VISION: per-column bias */
    u32 act;             /* GE_VISION: UOCR_VISION_ACT_* */
    u32 split;           /* GE_VISION: 0, or the width of each of out/out1/out2 */
    void *out1, *out2;
    u32 kst;             /* split-K: K steps per blockIdx.z (0: all of K in one block) */
    u32 sc_lds;          /* the block's scale rows are preloaded into dynamic LDS */
    u32 packed;          /* Q4/Q8 payloads in the GEMM-packed layout */
    u32 vec;             /* rows of the outputs, the residual and the bias are whole 16-byte pieces */
    u32 nx, ny, by_row;  /* row tiles, column tiles; each XCD takes a run of row (else column) tiles */
};

/* The kernels of uocr_gemm_tile.hip: whether a GEMM's operands and sizes fit
 * them (16-byte aligned rows, 32-bit offsets), whether a plain one takes them
 * (fits, and the general kernel is not the faster one), and its launch. */
bool uocr_gemm_tile_fits(int epi, u32 qt, const GemmArgs &a);
bool uocr_gemm_tile_takes(int epi, u32 qt, const GemmArgs &a);
/* Whether a plain fp16 GEMM with fp32 output can take the router's half of uocr_gemm_tile_router. */
bool uocr_gemm_router_fits(const GemmArgs &a);
hipError_t uocr_gemm_tile_plain(hipStream_t st, int epi, u32 qt, const GemmArgs &a);
/* The Q | K | V projection (N = 3 nseg) with RoPE and the cache scatter. */
hipError_t uocr_gemm_tile_rope(hipStream_t st, u32 qt, GemmArgs a, const RopeDst &rd);
/* Rows per tile (32 or 128) of the grouped GEMMs over `pairs` (token,
 * rank) pairs whose tile table holds `table` entries; their launch; a plain
 * GE_F16 GEMM a beside a grouped one of the same weight type and layout (eb:
 * GE_F16 or GE_F32); and a plain SwiGLU GEMM a beside fp16 router logits b. */
u32 uocr_gemm_grouped_rows(u32 pairs, u32 table);
hipError_t uocr_gemm_tile_grouped(hipStream_t st, int epi, u32 qt, const GemmArgs &a, u32 pairs, u32 rows);
hipError_t uocr_gemm_tile_pair(hipStream_t st, int eb, u32 qt, const GemmArgs &a, const GemmArgs &b, u32 pairs, u32 rows);
hipError_t uocr_gemm_tile_router(hipStream_t st, u32 qt, const GemmArgs &a, const GemmArgs &b);

#endif /* UOCR_GEMM_H */
