/*
 * uocr_prefill.hip - MFMA prompt prefill for the UnlimitedOCR decoder on
 * gfx950 (replaces the reference's prefill path, uocr_metal.m:14550-14908,
 * with its tiled GEMMs gemm_q4.metal / gemm_q8.metal).
 *
 * All P prompt rows go through each layer together, so the projections are
 * real GEMMs [P x K] x [K x N]; the tiled kernels (uocr_gemm_tile.hip) and the
 * attention (uocr_attn_prefill.hip) have files of their own.  Here:
 *  - the launchers, which check a GEMM and choose its kernel;
 *  - k_gemm, the general GEMM: for operands off 16-byte pieces (the operators
 *    accept them, the engine has none), and where it is the faster one (K split
 *    over blocks, some vision linears and Q4 projections).  64 x 128 output
 *    tiles, K in 64-column steps (one quantisation group), activations staged
 *    in LDS as fp16, each wavefront dequantising its own 32 weight rows straight into
 *    MFMA operand registers as fp16(q * scale), the reference's prefill
 *    staging (gemm_q4.metal:48-55: half(float(q) * scale)), with fp32
 *    accumulation by v_mfma_f32_32x32x16_f16.  Epilogues: fp16 store with
 *    optional residual, fp32 store, and SwiGLU over two weight matrices.  In
 *    grouped mode a tile table maps each block to an expert's bucket of
 *    (token, rank) pairs: rows are gathered through an index list and the
 *    expert's weights are addressed by slab stride;
 *  - routing (top-6 per token, expert buckets), RoPE table, MoE combine and
 *    row RMSNorm kernels.
 * fp16 rounding happens where the decode path rounds (norm, q/k/v, RoPE,
 * attention output, O + residual, SwiGLU mids, shared output, layer output).
 */
#include "uocr_gemm.h"

#include <math.h>

#define PB 256 /* threads per prefill block */
#define TM 64  /* GEMM tile rows */
#define TN 128 /* GEMM tile columns */
#define TK 64  /* one quantisation group */
#define LDA (TK + 8) /* padded LDS row of the activation tile (halves) */
#ifndef GDEPTH
#define GDEPTH 2 /* K steps in flight per GEMM block (2, 3 and 5 measured: 2 best on the SAM shapes, equal on the prefill) */
#endif
/* The SwiGLU GEMMs (two weight matrices; here only off 16-byte pieces) keep one
 * K step in flight: 16 fewer registers take them from 2 to 3 wavefronts per SIMD
 * (932 rows on this kernel: routed gate/up 66.8 -> 62.4 us, dense gate/up 62.9 ->
 * 60.8); the one-matrix GEMMs run 4 per SIMD either way and lose with one step
 * (dense down, unsplit, 44.4 -> 48.7). */
#ifndef GDEPTH_SWIGLU
#define GDEPTH_SWIGLU 1
#endif

/* ------------------------------------------------------------------------ */
/* GEMM                                                                      */
/* ------------------------------------------------------------------------ */

/* Weight piece of one K step (one 64-column quantisation group) for the
 * weight row n = the output column of this lane, lane half h = lane / 32:
 *   Q4: bytes 16h..16h+15 of the group (one uint4); f16 / Q8: columns
 *   32h..32h+31 (Q8 two uint4, f16 four), plus the row's group scale.
 * A K step is four 16-deep MFMA substeps; substep i takes 8 of these
 * weights, at the group columns b_koff(i, h)..+7 (any order of the K sum
 * works as long as the activation operand is read at the same columns):
 *   Q4: i = 0, 1: low nibbles of bytes 8i..8i+7 (columns 16h + 8i ..);
 *       i = 2, 3: high nibbles of the same bytes (columns + 32);
 *   Q8 / f16: columns 32h + 8i ... */
template <int QT>
struct BPiece {
    static constexpr int NV = QT == 4 ? 1 : (QT == 3 ? 2 : 4); /* uint4 loads */
    static constexpr int NW = 4 * NV;                          /* words */
};

/* The piece is kept as plain words (no struct or vector copies), so the
 * register ring stays in registers. */
template <int QT>
__device__ __forceinline__ void b_load(u32 (&w)[BPiece<QT>::NW], u32 &sc, const uint8_t *W, const h16 *S, u32 K,
                                       u32 n, u32 g, u32 h, bool with_scale = true, bool packed = false) {
    /* packed (Q4/Q8): the 32-row block's step is one run, half h of row r at
     * (32h + r) * RB/2 */
    constexpr u32 RB = QT == 4 ? 32u : 64u;
    const uint4 *src =
        packed && QT != 1
            ? (const uint4 *)(W + ((size_t)(n / 32u) * (K / 64u) + g) * (32u * RB) + (32u * h + n % 32u) * (RB / 2u))
            : (QT == 4 ? (const uint4 *)(W + (size_t)n * (K / 2u) + g * 32u + 16u * h)
                       : (QT == 3 ? (const uint4 *)(W + (size_t)n * K + g * 64u + 32u * h)
                                  : (const uint4 *)((const h16 *)W + (size_t)n * K + g * 64u + 32u * h)));
#pragma unroll
    for (int v = 0; v < BPiece<QT>::NV; ++v) {
        const uint4 x = src[v];
        w[4 * v] = x.x;
        w[4 * v + 1] = x.y;
        w[4 * v + 2] = x.z;
        w[4 * v + 3] = x.w;
    }
    if (QT != 1 && with_scale) sc = ((const unsigned short *)S)[(size_t)n * (K / 64u) + g];
}

/* The four B operands (8 fp16 each) of a loaded piece: fp16(q * scale). */
template <int QT>
__device__ __forceinline__ void b_dequant(const u32 (&w)[BPiece<QT>::NW], u32 sc, h16x8 (&b)[4]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        if (QT == 4) b[i] = dequant_q4(w[2 * (i & 1)], w[2 * (i & 1) + 1], (i & 2) != 0, sc);
        else if (QT == 3) b[i] = dequant_q8(w[2 * i], w[2 * i + 1], sc);
        else b[i] = operand_f16(w[4 * i], w[4 * i + 1], w[4 * i + 2], w[4 * i + 3]);
    }
}

/* Scale rows in LDS: a block's 128 weight rows x K/64 groups are one
 * contiguous region of the scale tensor, loaded once with wide loads instead
 * of one 2-byte load per row per K step (each of which touches a separate
 * cache line).  Used while NMAT x K/64 <= SC_LDS_STEPS (28 KB). */
#define SC_LDS_STEPS 112u

/* C[m][n] = sum_k A[m][k] W[n][k] over one 64 x 128 tile per block.  Wave
 * w owns output columns 32w..32w+31 (its weight rows, dequantised straight
 * into MFMA B operands in registers) for all 64 rows (two 32x32 MFMA
 * tiles); only the activation tile goes through LDS, double-buffered, so a
 * K step has one barrier and LDS carries one activation read per MFMA. */
#ifndef UOCR_GEMM_BLDS
#define UOCR_GEMM_BLDS 1
#endif

template <int QT, int EPI, bool GROUPED>
__device__ __forceinline__ void gemm_body(GemmArgs p, u32 bx, u32 by, u32 bz) {
    constexpr int AQ4 = TM * (TK / 8) / PB; /* activation pieces (8 halves) per thread per K step */
    static_assert(TM % 32 == 0 && TM <= PB && AQ4 * PB == TM * (TK / 8), "tile rows");
    constexpr int NMAT = EPI == GE_SWIGLU ? 2 : 1;
    constexpr int GD = EPI == GE_SWIGLU ? GDEPTH_SWIGLU : GDEPTH; /* K steps in flight */
    /* (the SAM and CLIP figures are of this kernel at shapes that the tiled
     * kernels run now) f16 with one weight matrix: the block loads each K step's raw weight
     * tile with eight lanes per row (whole 128-byte row pieces) into LDS, and
     * each wavefront reads its 32 rows back in the MFMA operand layout; loads
     * of one row per lane touched a cache line per lane (SAM lin1 with fp16
     * weights 58.4 -> 48.5 us).  The same for Q8 (four lanes per 64-byte
     * piece) measured -4.6% to +3.6% across the SAM / CLIP shapes, the extra
     * 20 KB of LDS costing occupancy at long K, so Q8 keeps the per-lane
     * loads; Q4 rows are 32 bytes per K step. */
    constexpr bool BL = UOCR_GEMM_BLDS && QT == 1 && NMAT == 1;
    constexpr u32 RB = QT == 3 ? 64u : 128u; /* raw bytes per row per K step */
    constexpr u32 LDB = RB + 16u;            /* padded LDS row (bytes) */
    constexpr u32 CPR = RB / 16u;            /* 16-byte pieces per row */
    __shared__ __attribute__((aligned(16))) uint8_t bsm[BL ? 2u * TN * LDB : 16u];
    __shared__ __attribute__((aligned(16))) h16 as[2][TM * LDA];
    __shared__ int32_t arow[TM], orow[TM];
    const u32 t = threadIdx.x, lane = t & 63u, wave = t >> 6, hf = lane >> 5;
    u32 n0 = by * TN, rows = p.M, e = 0, s0 = 0;
    if (GROUPED) {
        if ((int)bx >= *p.ntiles) return;
        e = (u32)p.tile_e[bx];
        s0 = (u32)p.tile_s0[bx];
        rows = (u32)p.tile_s1[bx] - s0;
        if (t < TM) {
            const u32 s = s0 + min(t, rows - 1u);
            arow[t] = p.a_idx[s];
            orow[t] = p.o_idx[s];
        }
    } else {
        s0 = bx * TM;
        rows = min((u32)TM, p.M - s0);
        if (t < TM) {
            arow[t] = (int32_t)(s0 + min(t, rows - 1u));
            orow[t] = arow[t];
        }
    }
    const uocr_qmat W0 = p.W[0], W1 = p.W[1];
    const uint8_t *wp[2] = {(const uint8_t *)W0.w + (GROUPED ? e * p.w_stride : 0),
                            NMAT == 2 ? (const uint8_t *)W1.w + (GROUPED ? e * p.w_stride : 0) : nullptr};
    const h16 *sp[2] = {(const h16 *)W0.s + (GROUPED ? e * p.s_stride : 0),
                        NMAT == 2 ? (const h16 *)W1.s + (GROUPED ? e * p.s_stride : 0) : nullptr};
    /* this lane's weight row (clamped; columns past N are not stored) */
    const u32 nrow = min(n0 + 32u * wave + (lane & 31u), p.N - 1u);
    __syncthreads();

    f32x16 acc[NMAT][TM / 32];
#pragma unroll
    for (int m = 0; m < NMAT; ++m)
#pragma unroll
        for (int j = 0; j < TM / 32; ++j)
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[m][j][i] = 0.0f;

    /* K steps run GD deep: step s's loads were issued GD steps
     * earlier into a register ring (constant indices only, so the ring stays
     * in registers) */
    /* the lambdas below see plain locals: a reference to the kernel
     * argument struct would copy it to private memory */
    const h16 *Ap = p.A;
    const u32 lda = p.lda, Kd = p.K;
    const bool pk = p.packed != 0u;
    const u32 NT = Kd / TK, kb0 = p.kst != 0u ? bz * p.kst : 0u;
    const u32 NS = p.kst != 0u ? min(p.kst, NT - kb0) : NT;
    u32 ka[GD][AQ4][4]; /* words, not uint4: no struct copies, so they stay in registers */
    u32 kb[GD][NMAT][BPiece<QT>::NW], ks[GD][NMAT];
    extern __shared__ __attribute__((aligned(16))) unsigned short ssc[];
    const bool scl = QT != 1 && p.sc_lds != 0u;
    const u32 nvalid = min((u32)TN, p.N - n0);
    const u32 lrow = nrow - n0; /* this lane's row within the block's scale rows */
    /* this thread's two activation rows, resolved once */
    const h16 *arp[AQ4];
#pragma unroll
    for (int q = 0; q < AQ4; ++q) {
        const u32 idx = t + q * PB;
        arp[q] = Ap + (size_t)arow[idx >> 3] * lda + (size_t)kb0 * TK + 8u * (idx & 7u);
    }
    const uint8_t *bsrc[BPiece<QT>::NV];
    if constexpr (BL) {
        const u32 rowbytes = QT == 3 ? Kd : 2u * Kd;
#pragma unroll
        for (int v = 0; v < BPiece<QT>::NV; ++v) {
            const u32 pidx = t + v * PB, r = pidx / CPR, c = pidx % CPR;
            bsrc[v] = wp[0] + (size_t)min(n0 + r, p.N - 1u) * rowbytes + 16u * c;
        }
    }
    auto issue = [&](auto D, u32 st) {
        constexpr int d = decltype(D)::value;
#pragma unroll
        for (int q = 0; q < AQ4; ++q) {
            const uint4 v = *(const uint4 *)(arp[q] + st * TK);
            ka[d][q][0] = v.x;
            ka[d][q][1] = v.y;
            ka[d][q][2] = v.z;
            ka[d][q][3] = v.w;
        }
        if constexpr (BL) {
            /* piece v of this thread: row (t + v PB) / CPR of the block's
             * rows, 16-byte piece (t + v PB) % CPR of its K step */
#pragma unroll
            for (int v = 0; v < BPiece<QT>::NV; ++v) {
                const uint4 x = *(const uint4 *)(bsrc[v] + (size_t)(kb0 + st) * RB);
                kb[d][0][4 * v] = x.x;
                kb[d][0][4 * v + 1] = x.y;
                kb[d][0][4 * v + 2] = x.z;
                kb[d][0][4 * v + 3] = x.w;
            }
            if (!scl) ks[d][0] = ((const unsigned short *)sp[0])[(size_t)nrow * (Kd / 64u) + kb0 + st];
        } else {
#pragma unroll
            for (int m = 0; m < NMAT; ++m) b_load<QT>(kb[d][m], ks[d][m], wp[m], sp[m], Kd, nrow, kb0 + st, hf, !scl, pk);
        }
    };
    auto step = [&](auto D, u32 st) {
        constexpr int d = decltype(D)::value;
        /* keeps the scheduler from hoisting a later step's dequantisation
         * (which waits for that step's loads) into this one */
        __builtin_amdgcn_sched_barrier(0);
        h16 *ab = as[st & 1u];
#pragma unroll
        for (int q = 0; q < AQ4; ++q) {
            const u32 idx = t + q * PB, r = idx >> 3, c8 = idx & 7u;
            *(uint4 *)(ab + r * LDA + 8u * c8) = make_uint4(ka[d][q][0], ka[d][q][1], ka[d][q][2], ka[d][q][3]);
        }
        h16x8 bop[NMAT][4];
        if (scl) {
#pragma unroll
            for (int m = 0; m < NMAT; ++m) ks[d][m] = ssc[(m * TN + lrow) * NT + kb0 + st];
        }
        uint8_t *bb = bsm + (st & 1u) * (BL ? TN * LDB : 0u);
        if constexpr (BL) {
#pragma unroll
            for (int v = 0; v < BPiece<QT>::NV; ++v) {
                const u32 pidx = t + v * PB;
                *(uint4 *)(bb + (pidx / CPR) * LDB + 16u * (pidx % CPR)) =
                    make_uint4(kb[d][0][4 * v], kb[d][0][4 * v + 1], kb[d][0][4 * v + 2], kb[d][0][4 * v + 3]);
            }
        } else {
#pragma unroll
            for (int m = 0; m < NMAT; ++m) b_dequant<QT>(kb[d][m], ks[d][m], bop[m]);
        }
        /* the other buffer's readers (step st - 1) all passed this barrier
         * before anyone writes it again at step st + 1 */
        __syncthreads();
        if constexpr (BL) {
            /* this lane's MFMA piece of its row: bytes RB / 2 * h .. + RB / 2 */
            u32 w[BPiece<QT>::NW];
            const uint8_t *src = bb + (32u * wave + (lane & 31u)) * LDB + (RB / 2u) * hf;
#pragma unroll
            for (int v = 0; v < BPiece<QT>::NV; ++v) {
                const uint4 x = *(const uint4 *)(src + 16u * v);
                w[4 * v] = x.x;
                w[4 * v + 1] = x.y;
                w[4 * v + 2] = x.z;
                w[4 * v + 3] = x.w;
            }
            b_dequant<QT>(w, ks[d][0], bop[0]);
        }
        /* unconditional (past the end it re-reads the last step into a slot
         * no later step consumes): loads issued on every path keep the
         * compiler's load counting exact, so the wait before a step covers
         * only that step's loads and the later steps' stay in flight */
        issue(D, min(st + GD, NS - 1u));
#pragma unroll
        for (u32 i = 0; i < 4; ++i) {
#pragma unroll
            for (int j = 0; j < TM / 32; ++j) {
                U4H8 a;
                a.u = *(const uint4 *)(ab + (32u * j + (lane & 31u)) * LDA + b_koff<QT>(i, hf));
#pragma unroll
                for (int m = 0; m < NMAT; ++m) {
                    acc[m][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a.v, bop[m][i], acc[m][j], 0, 0, 0);
                }
            }
        }
    };
    static_for<GD>([&](auto D) { issue(D, min((u32)decltype(D)::value, NS - 1u)); });
    if (scl) {
        /* after the first steps' loads are in flight; rows past p.N are not
         * loaded (their lanes read the last valid row, nrow is clamped) */
#pragma unroll
        for (int m = 0; m < NMAT; ++m) {
            const unsigned short *src = (const unsigned short *)sp[m] + (size_t)n0 * NT;
            unsigned short *dst = ssc + m * TN * NT;
            const u32 cnt = nvalid * NT;
            if ((((uintptr_t)src) & 15u) == 0u && cnt % 8u == 0u) {
                for (u32 i = t; i < cnt / 8u; i += PB) ((uint4 *)dst)[i] = ((const uint4 *)src)[i];
            } else {
                for (u32 i = t; i < cnt; i += PB) dst[i] = src[i];
            }
        }
        __syncthreads();
    }
    u32 st = 0;
    for (; st + GD <= NS; st += GD) {
        static_for<GD>([&](auto D) { step(D, st + (u32)decltype(D)::value); });
    }
    static_for<GD>([&](auto D) {
        if (st + (u32)decltype(D)::value < NS) step(D, st + (u32)decltype(D)::value);
    });

    /* C layout of a 32x32 MFMA tile: lane l, element i -> row 8*(i/4) +
     * 4*(l/32) + i%4, column l%32.  Everything that depends only on the
     * column (output pointer, split routing, bias) is resolved once per lane;
     * rows of a plain GEMM are s0 + r (the row list is only read when
     * grouped). */
    const u32 col = n0 + 32u * wave + (lane & 31u);
    if (col >= p.N) return;
    auto out_row = [&](u32 r) -> size_t { return GROUPED ? (size_t)orow[r] : (size_t)(s0 + r); };
    h16 *vdst = (h16 *)p.out + col;
    size_t vld = p.ldo;
    float bcol = 0.0f;
    if (EPI == GE_VISION) {
        bcol = (float)p.bias[col];
        if (p.split != 0u) {
            const u32 pj = col / p.split;
            vdst = (h16 *)(pj == 0u ? p.out : (pj == 1u ? p.out1 : p.out2)) + (col - pj * p.split);
            vld = p.split;
        }
    }
    const u32 act = p.act;
#pragma unroll
    for (int j = 0; j < TM / 32; ++j) {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const u32 r = 32u * j + 8u * (i / 4) + 4u * hf + (i % 4);
            if (r >= rows) continue;
            const size_t orw = out_row(r);
            if (EPI == GE_F32) {
                ((float *)p.out)[orw * p.ldo + col] = acc[0][j][i];
            } else if (EPI == GE_PART) {
                ((float *)p.out)[((size_t)bz * p.M + orw) * p.ldo + col] = acc[0][j][i];
            } else if (EPI == GE_SWIGLU) {
                ((h16 *)p.out)[orw * p.ldo + col] = (h16)(silu_p(acc[0][j][i]) * acc[NMAT - 1][j][i]);
            } else if (EPI == GE_VISION) {
                float v = acc[0][j][i] + bcol;
                if (act == UOCR_VISION_ACT_QUICKGELU) v = quick_gelu(v);
                else if (act == UOCR_VISION_ACT_GELU_ERF) v = gelu_erf_as(v);
                vdst[orw * vld] = (h16)v;
            } else {
                float v = acc[0][j][i];
                if (p.res != nullptr) v += (float)p.res[orw * p.ldr + col];
                ((h16 *)p.out)[orw * p.ldo + col] = (h16)v;
            }
        }
    }
}

template <int QT, int EPI, bool GROUPED>
__global__ __launch_bounds__(PB) void k_gemm(GemmArgs p) {
    gemm_body<QT, EPI, GROUPED>(p, blockIdx.x, blockIdx.y, blockIdx.z);
}

/* cs[64 t + d] = (cos, sin)(t * f[d]) for the P prompt tokens. */
__global__ __launch_bounds__(PB) void k_rope_table(RopeTabP rope, u32 P, float2 *__restrict__ cs) {
    const u32 idx = blockIdx.x * PB + threadIdx.x;
    if (idx >= P * 64u) return;
    const float ang = (float)(idx / 64u) * rope.f[idx % 64u];
    cs[idx] = make_float2(cosf(ang), sinf(ang));
}

/* Split-K epilogue of the vision GEMM: the z partials summed in order (the
 * result does not depend on block timing), out = f16(act(sum + bias)), split
 * into o0/o1/o2 when split. */
__global__ __launch_bounds__(PB) void k_split_reduce(const float *__restrict__ part, u32 S, u32 M, u32 N,
                                                     const h16 *__restrict__ bias, u32 act, u32 split,
                                                     h16 *__restrict__ o0, h16 *__restrict__ o1, h16 *__restrict__ o2) {
    /* four consecutive columns per thread (N and split are
     * multiples of 4, checked by the launcher), so every load is 16 bytes */
    const size_t i = 4u * ((size_t)blockIdx.x * PB + threadIdx.x), MN = (size_t)M * N;
    if (i >= MN) return;
    /* all planes' loads issued before the (ordered) sum; S <= 8 */
    float4 w[8];
#pragma unroll
    for (u32 z = 0; z < 8u; ++z) {
        if (z < S) w[z] = *(const float4 *)(part + z * MN + i);
    }
    float4 v = w[0];
#pragma unroll
    for (u32 z = 1; z < 8u; ++z) {
        if (z < S) {
            v.x += w[z].x;
            v.y += w[z].y;
            v.z += w[z].z;
            v.w += w[z].w;
        }
    }
    const u32 row = (u32)(i / N), col = (u32)(i - (size_t)row * N);
    float r[4] = {v.x, v.y, v.z, v.w};
    union {
        h16 h[4];
        uint2 u;
    } o;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        float x = r[c] + (float)bias[col + c];
        if (act == UOCR_VISION_ACT_QUICKGELU) x = quick_gelu(x);
        else if (act == UOCR_VISION_ACT_GELU_ERF) x = gelu_erf_as(x);
        o.h[c] = (h16)x;
    }
    if (split == 0u) {
        *(uint2 *)(o0 + (size_t)row * N + col) = o.u;
    } else {
        const u32 pj = col / split, lc = col - pj * split;
        *(uint2 *)((pj == 0u ? o0 : (pj == 1u ? o1 : o2)) + (size_t)row * split + lc) = o.u;
    }
}

/* ------------------------------------------------------------------------ */
/* row RMSNorm, RoPE + KV scatter                                            */
/* ------------------------------------------------------------------------ */

/* RMSNorm of one row of 1280 held by a wavefront: lane l holds the 8-half
 * pieces l, l + 64, l + 128 (< 160) in v.  Writes yr = f16(x * inv_rms * w)
 * (norm.metal:12-40), the sum of squares in fp32 in a fixed order (lane
 * pieces in order, then the butterfly), so every caller rounds alike. */
/* The norm weights' pieces of a lane (i = lane + 64q, clamped to the row),
 * loaded at a kernel's start so the tail waits on no further load round. */
__device__ __forceinline__ void norm_w_load(const h16 *__restrict__ w, u32 lane, U4H8 (&wv)[3]) {
#pragma unroll
    for (int q = 0; q < 3; ++q) wv[q].u = ((const uint4 *)w)[min(lane + 64u * q, UOCR_K_HIDDEN / 8u - 1u)];
}

__device__ __forceinline__ void row_norm_tail(U4H8 (&v)[3], u32 lane, const U4H8 (&wv)[3], h16 *__restrict__ yr) {
    float ss = 0.0f;
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        if (lane + 64u * q < UOCR_K_HIDDEN / 8u) {
#pragma unroll
            for (int j = 0; j < 8; ++j) ss = fmaf((float)v[q].h[j], (float)v[q].h[j], ss);
        }
    }
    for (int o = 32; o > 0; o >>= 1) ss += __shfl_xor(ss, o);
    const float inv = 1.0f / sqrtf(ss / (float)UOCR_K_HIDDEN + 1.0e-6f);
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        const u32 i = lane + 64u * q;
        if (i < UOCR_K_HIDDEN / 8u) {
            U4H8 y;
#pragma unroll
            for (int j = 0; j < 8; ++j) y.h[j] = (h16)(((float)v[q].h[j] * inv) * (float)wv[q].h[j]);
            ((uint4 *)yr)[i] = y.u;
        }
    }
}

/* One wavefront per row of 1280: y = f16(x * inv_rms * w). */
__global__ __launch_bounds__(PB) void k_rows_rmsnorm(const h16 *__restrict__ x, const h16 *__restrict__ w, u32 P,
                                                     h16 *__restrict__ y) {
    const u32 row = blockIdx.x * (PB / 64) + (threadIdx.x >> 6), lane = threadIdx.x & 63u;
    if (row >= P) return;
    const h16 *xr = x + (size_t)row * UOCR_K_HIDDEN;
    U4H8 wv[3];
    norm_w_load(w, lane, wv);
    U4H8 v[3];
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        const u32 i = lane + 64u * q;
        if (i < UOCR_K_HIDDEN / 8u) v[q].u = ((const uint4 *)xr)[i];
    }
    row_norm_tail(v, lane, wv, y + (size_t)row * UOCR_K_HIDDEN);
}

/* Split-K reduce of a 1280-column fp16 GEMM output with its residual, fused
 * with the RMSNorm that reads it: per row (one wavefront), out = f16(sum of
 * the S planes in order + res), then y = rmsnorm(out) * w as k_rows_rmsnorm
 * rounds it. */
__global__ __launch_bounds__(PB) void k_reduce_norm(const float *__restrict__ part, u32 S, u32 M,
                                                    const h16 *__restrict__ res, u32 ldr, h16 *__restrict__ out,
                                                    u32 ldo, const h16 *__restrict__ w, h16 *__restrict__ y) {
    const u32 row = blockIdx.x * (PB / 64) + (threadIdx.x >> 6), lane = threadIdx.x & 63u;
    if (row >= M) return;
    const size_t MN = (size_t)M * UOCR_K_HIDDEN;
    /* the first two planes of the row's pieces (and the residual), all in
     * flight before any sum; planes beyond the second are added in order
     * after them */
    float4 pa[3][2], pb2[3][2];
    U4H8 rr[3], wv[3];
    norm_w_load(w, lane, wv);
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        const u32 i = min(lane + 64u * q, UOCR_K_HIDDEN / 8u - 1u);
        const float *p0 = part + (size_t)row * UOCR_K_HIDDEN + 8u * i;
#pragma unroll
        for (u32 z = 0; z < 2u; ++z) {
            if (z < S) {
                pa[q][z] = *(const float4 *)(p0 + z * MN);
                pb2[q][z] = *(const float4 *)(p0 + z * MN + 4);
            }
        }
        if (res != nullptr) rr[q].u = *(const uint4 *)(res + (size_t)row * ldr + 8u * i);
    }
    U4H8 v[3];
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        const u32 i = lane + 64u * q;
        if (i >= UOCR_K_HIDDEN / 8u) continue;
        const float *p0 = part + (size_t)row * UOCR_K_HIDDEN + 8u * i;
        float4 a = pa[q][0], b = pb2[q][0];
        if (S > 1u) {
            const float4 c = pa[q][1], d = pb2[q][1];
            a.x += c.x;
            a.y += c.y;
            a.z += c.z;
            a.w += c.w;
            b.x += d.x;
            b.y += d.y;
            b.z += d.z;
            b.w += d.w;
        }
        for (u32 z = 2; z < S; ++z) {
            const float4 c = *(const float4 *)(p0 + z * MN), d = *(const float4 *)(p0 + z * MN + 4);
            a.x += c.x;
            a.y += c.y;
            a.z += c.z;
            a.w += c.w;
            b.x += d.x;
            b.y += d.y;
            b.z += d.z;
            b.w += d.w;
        }
        const float r[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
        for (int j = 0; j < 8; ++j) v[q].h[j] = (h16)(res != nullptr ? r[j] + (float)rr[q].h[j] : r[j]);
        *(uint4 *)(out + (size_t)row * ldo + 8u * i) = v[q].u;
    }
    row_norm_tail(v, lane, wv, y + (size_t)row * UOCR_K_HIDDEN);
}

/* ------------------------------------------------------------------------ */
/* MoE routing, buckets, combine                                             */
/* ------------------------------------------------------------------------ */

__device__ __forceinline__ float lane_fp(float v, int l) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}

/* One wavefront per token: softmax over its 64 logits, greedy top-6 (ties to
 * the lower id; same key order as the decode router), raw probabilities
 * unless norm_topk. */
__global__ __launch_bounds__(PB) void k_route_rows(const float *__restrict__ logits, u32 P, int norm_topk,
                                                   int32_t *__restrict__ ids, float *__restrict__ wts) {
    const u32 tok = blockIdx.x * (PB / 64) + (threadIdx.x >> 6), lane = threadIdx.x & 63u;
    if (tok >= P) return;
    const float lg = logits[(size_t)tok * 64u + lane];
    float mx = lg;
    for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
    const float pe = expf(lg - mx);
    float sum = pe;
    for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o);
    const float prob = pe / sum;
    const u32 pb = __float_as_uint(prob);
    const unsigned long long key = ((unsigned long long)pb << 32) | (0xffffffffu - lane);
    u32 rank = 0;
#pragma unroll
    for (int j = 0; j < 64; ++j) {
        const unsigned long long kj =
            ((unsigned long long)(u32)__builtin_amdgcn_readlane((int)pb, j) << 32) | (0xffffffffu - (u32)j);
        rank += kj > key ? 1u : 0u;
    }
    float tot = 0.0f;
    float sel[UOCR_K_TOPK];
#pragma unroll
    for (int r = 0; r < UOCR_K_TOPK; ++r) {
        const unsigned long long m = __ballot(rank == (u32)r);
        const u32 l = m != 0ull ? (u32)__builtin_ctzll(m) : 0u;
        sel[r] = __uint_as_float((u32)__builtin_amdgcn_readlane((int)pb, (int)l));
        tot += sel[r];
    }
    if (rank < (u32)UOCR_K_TOPK) {
        ids[tok * UOCR_K_TOPK + rank] = (int32_t)lane;
        wts[tok * UOCR_K_TOPK + rank] = norm_topk ? prob / tot : prob;
    }
}

/* The routing's outputs for the grouped GEMMs. */
struct BucketOut {
    int32_t *offsets, *tile_e, *tile_s0, *tile_s1, *ntiles, *list_tok, *list_pair;
    int32_t tile_rows;
};

#define BUCKET_THREADS 1024

/* Exclusive scans of the 64 bucket sizes and tile counts (one wavefront, a
 * lane per expert) and the tile table of the grouped GEMMs. */
__device__ __forceinline__ void bucket_tables(const int32_t *cnt, int32_t *off, const BucketOut &o) {
    const u32 t = threadIdx.x;
    if (t < 64u) {
        const int32_t c = cnt[t], tl = (c + o.tile_rows - 1) / o.tile_rows;
        int32_t a = c, b = tl;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int32_t x = __shfl_up(a, d), y = __shfl_up(b, d);
            if ((int)t >= d) {
                a += x;
                b += y;
            }
        }
        off[t] = a - c;
        o.offsets[t] = a - c;
        if (t == 63u) *o.ntiles = b;
        for (int32_t k = 0; k * o.tile_rows < c; ++k) {
            const int32_t ti = b - tl + k;
            o.tile_e[ti] = (int32_t)t;
            o.tile_s0[ti] = a - c + k * o.tile_rows;
            o.tile_s1[ti] = a - c + min(c, (k + 1) * o.tile_rows);
        }
    }
    __syncthreads();
}

/* One block builds the expert buckets of all P*6 (token, rank) pairs in LDS:
 * the bucket sizes (LDS atomics, which also give each pair its place in its
 * bucket), their scan, the tile table and the slot lists.  The order of pairs
 * inside a bucket does not matter: each pair's row is computed on its own and
 * the combine reads it by pair index.  Nothing is left in global memory that
 * the next routing has to find cleared.  One CU does all of it, so what
 * bounds it are its dependent loads and its scattered stores: a thread's R pairs
 * are loaded together and stay in registers with their places, and the lists
 * are put in order in LDS and leave as whole lines: 4,001 rows 28 us with 8
 * pairs in registers and loops above, 25 with 24, 9.5 with the lists in LDS;
 * 932 rows 4.4 us.
 * More than R per thread take two passes in batches with direct stores. */
template <u32 R>
__global__ __launch_bounds__(BUCKET_THREADS) void k_bucket_build(const int32_t *__restrict__ ids, u32 P, BucketOut o) {
    __shared__ int32_t cnt[64], off[64], cur[64];
    __shared__ uint16_t list[R * BUCKET_THREADS];
    const u32 t = threadIdx.x, n = P * UOCR_K_TOPK;
    if (t < 64u) {
        cnt[t] = 0;
        cur[t] = 0;
    }
    int32_t id[R], place[R];
    auto load = [&](u32 base) {
#pragma unroll
        for (u32 k = 0; k < R; ++k) {
            const u32 pr = base + t + k * BUCKET_THREADS;
            id[k] = pr < n ? ids[pr] : -1;
        }
    };
    auto count = [&](int32_t *c) {
#pragma unroll
        for (u32 k = 0; k < R; ++k)
            if (id[k] >= 0) place[k] = atomicAdd(&c[id[k]], 1);
    };
    auto store = [&](u32 base) {
#pragma unroll
        for (u32 k = 0; k < R; ++k) {
            const u32 pr = base + t + k * BUCKET_THREADS;
            if (id[k] >= 0) {
                const int32_t slot = off[id[k]] + place[k];
                o.list_tok[slot] = (int32_t)(pr / UOCR_K_TOPK);
                o.list_pair[slot] = (int32_t)pr;
            }
        }
    };
    load(0u);
    __syncthreads();
    count(cnt);
    const bool once = n <= R * BUCKET_THREADS;
    for (u32 base = R * BUCKET_THREADS; base < n; base += R * BUCKET_THREADS) {
        load(base);
        count(cnt);
    }
    __syncthreads();
    bucket_tables(cnt, off, o);
    if (once) {
#pragma unroll
        for (u32 k = 0; k < R; ++k)
            if (id[k] >= 0) list[off[id[k]] + place[k]] = (uint16_t)(t + k * BUCKET_THREADS);
        __syncthreads();
#pragma unroll
        for (u32 k = 0; k < R; ++k) {
            const u32 s = t + k * BUCKET_THREADS;
            if (s < n) {
                const u32 pr = list[s];
                o.list_tok[s] = (int32_t)(pr / UOCR_K_TOPK);
                o.list_pair[s] = (int32_t)pr;
            }
        }
        return;
    }
    for (u32 base = 0; base < n; base += R * BUCKET_THREADS) {
        load(base);
        count(cur);
        store(base);
    }
}

/* h[t] = f16(sum_r w[t][r] * Y[t*6+r] + shared[t] + res[t]) (decode_gemv_q4.
 * metal:185-224 order: routed sum in fp32, shared already fp16). */
/* the per-pair expert outputs as fp32 (operator API) or fp16 (the prefill,
 * rounded as the reference keeps them) */
__device__ __forceinline__ void y_load8(const float *yr, float (&e)[8]) {
    const float4 a = *(const float4 *)yr, b = *(const float4 *)(yr + 4);
    e[0] = a.x; e[1] = a.y; e[2] = a.z; e[3] = a.w; e[4] = b.x; e[5] = b.y; e[6] = b.z; e[7] = b.w;
}
__device__ __forceinline__ void y_load8(const h16 *yr, float (&e)[8]) {
    U4H8 v;
    v.u = *(const uint4 *)yr;
#pragma unroll
    for (int j = 0; j < 8; ++j) e[j] = (float)v.h[j];
}

template <typename YT>
__global__ __launch_bounds__(PB) void k_moe_combine(const YT *__restrict__ Y, const float *__restrict__ wts,
                                                    const h16 *__restrict__ shared, const h16 *__restrict__ res, u32 P,
                                                    h16 *__restrict__ out) {
    const u32 idx = blockIdx.x * PB + threadIdx.x;
    if (idx >= P * UOCR_K_HIDDEN) return;
    const u32 t = idx / UOCR_K_HIDDEN, c = idx % UOCR_K_HIDDEN;
    float acc = 0.0f;
#pragma unroll
    for (int r = 0; r < UOCR_K_TOPK; ++r) {
        acc = fmaf(wts[t * UOCR_K_TOPK + r], (float)Y[((size_t)t * UOCR_K_TOPK + r) * UOCR_K_HIDDEN + c], acc);
    }
    out[idx] = (h16)(acc + (float)shared[idx] + (float)res[idx]);
}

/* k_moe_combine fused with the next layer's input RMSNorm: one wavefront
 * per token row, the same per-element arithmetic, then y = rmsnorm(out) * w
 * as k_rows_rmsnorm rounds it. */
template <typename YT>
__global__ __launch_bounds__(PB) void k_moe_combine_norm(const YT *__restrict__ Y, const float *__restrict__ wts,
                                                         const h16 *__restrict__ shared, const h16 *__restrict__ res,
                                                         u32 P, h16 *__restrict__ out, const h16 *__restrict__ w,
                                                         h16 *__restrict__ y) {
    const u32 t = blockIdx.x * (PB / 64) + (threadIdx.x >> 6), lane = threadIdx.x & 63u;
    if (t >= P) return;
    float wr[UOCR_K_TOPK];
#pragma unroll
    for (int r = 0; r < UOCR_K_TOPK; ++r) wr[r] = wts[t * UOCR_K_TOPK + r];
    U4H8 wv[3], v[3];
    norm_w_load(w, lane, wv);
    if constexpr (sizeof(YT) == 2) {
        /* fp16 pair rows: every load of the row issued before any sum */
        U4H8 ey[3][UOCR_K_TOPK], sh[3], rs[3];
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            const u32 i = min(lane + 64u * q, UOCR_K_HIDDEN / 8u - 1u);
            const size_t base = (size_t)t * UOCR_K_HIDDEN + 8u * i;
#pragma unroll
            for (int r = 0; r < UOCR_K_TOPK; ++r)
                ey[q][r].u = *(const uint4 *)(Y + ((size_t)t * UOCR_K_TOPK + r) * UOCR_K_HIDDEN + 8u * i);
            sh[q].u = *(const uint4 *)(shared + base);
            rs[q].u = *(const uint4 *)(res + base);
        }
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            const u32 i = lane + 64u * q;
            if (i >= UOCR_K_HIDDEN / 8u) continue;
            float acc[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int r = 0; r < UOCR_K_TOPK; ++r) {
#pragma unroll
                for (int j = 0; j < 8; ++j) acc[j] = fmaf(wr[r], (float)ey[q][r].h[j], acc[j]);
            }
#pragma unroll
            for (int j = 0; j < 8; ++j) v[q].h[j] = (h16)(acc[j] + (float)sh[q].h[j] + (float)rs[q].h[j]);
            *(uint4 *)(out + (size_t)t * UOCR_K_HIDDEN + 8u * i) = v[q].u;
        }
    } else {
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            const u32 i = lane + 64u * q;
            if (i >= UOCR_K_HIDDEN / 8u) continue;
            const size_t base = (size_t)t * UOCR_K_HIDDEN + 8u * i;
            float acc[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int r = 0; r < UOCR_K_TOPK; ++r) {
                float e[8];
                y_load8(Y + ((size_t)t * UOCR_K_TOPK + r) * UOCR_K_HIDDEN + 8u * i, e);
#pragma unroll
                for (int j = 0; j < 8; ++j) acc[j] = fmaf(wr[r], e[j], acc[j]);
            }
            U4H8 sh, rs;
            sh.u = *(const uint4 *)(shared + base);
            rs.u = *(const uint4 *)(res + base);
#pragma unroll
            for (int j = 0; j < 8; ++j) v[q].h[j] = (h16)(acc[j] + (float)sh.h[j] + (float)rs.h[j]);
            *(uint4 *)(out + base) = v[q].u;
        }
    }
    row_norm_tail(v, lane, wv, y + (size_t)t * UOCR_K_HIDDEN);
}

/* ------------------------------------------------------------------------ */
/* launchers                                                                 */
/* ------------------------------------------------------------------------ */

static bool pq_ok(u32 q) {
    return q == UOCR_QT_F16 || q == UOCR_QT_Q8 || q == UOCR_QT_Q4;
}

static bool pmat_ok(uocr_qmat m) {
    return m.w != nullptr && pq_ok(m.qtype) && (m.qtype == UOCR_QT_F16 || m.s != nullptr);
}

template <int EPI, bool GROUPED>
static void gemm_dispatch(hipStream_t st, u32 qt, GemmArgs a, dim3 grid) {
    const u32 nm = EPI == GE_SWIGLU ? 2u : 1u, nt = a.K / TK;
    a.sc_lds = qt != UOCR_QT_F16 && nm * nt <= SC_LDS_STEPS ? 1u : 0u;
    const size_t shm = a.sc_lds ? (size_t)nm * TN * nt * sizeof(unsigned short) : 0;
    switch (qt) {
        case UOCR_QT_F16: hipLaunchKernelGGL((k_gemm<1, EPI, GROUPED>), grid, dim3(PB), 0, st, a); break;
        case UOCR_QT_Q8: hipLaunchKernelGGL((k_gemm<3, EPI, GROUPED>), grid, dim3(PB), shm, st, a); break;
        default: hipLaunchKernelGGL((k_gemm<4, EPI, GROUPED>), grid, dim3(PB), shm, st, a); break;
    }
}

/* Splits of K over blocks for the prompt's O projection (K = 1280) and layer 0's
 * dense down (6848), N = 1280 both, summed by k_reduce_norm together with the
 * residual and the next norm; 1: the tiled kernel and a norm launch.  A split
 * grid fills the chip where the tiles' grids do not: with quantised weights from
 * one round of 32 x 64 tiles up to 190 tiles of 64 x 128, with fp16 weights
 * also below (each 32-row tile fetches all of the weights, four times the bytes
 * of Q4) and up to a tile per CU.  Measured in a prompt's first layer (us, GEMM + reduce or norm, split / tiled):
 *   rows                      64          384         400         932        1200        1600
 *   O projection, Q8     13.8 / 13.4  15.2 / 13.8 16.4 / 19.6 19.4 / 20.2 20.8 / 20.7 23.7 / 21.9
 *   O projection, F16    13.0 / 16.6  14.1 / 16.4 16.7 / 22.0 19.9 / 23.5 21.6 / 24.1 23.0 / 23.7
 *   dense down, Q4       28.1 / 28.1  30.1 / 29.6 32.3 / 44.8 43.4 / 48.3 46.1 / 49.4 62.3 / 53.1
 *   dense down, Q8       28.9 / 30.1  30.2 / 30.9 32.8 / 47.3 46.1 / 51.5 49.9 / 51.9 66.4 / 52.9
 *   dense down, F16      23.3 / 38.3  29.6 / 37.2 40.6 / 60.8 55.9 / 64.5 56.5 / 66.1 65.9 / 66.5
 * The split count: doubling while the grid stays within 512 blocks and a split
 * keeps 5 K steps, or a split keeps 16. */
extern "C" uint32_t uocr_gemm_ksplit(uint32_t qtype, uint32_t M, uint32_t N, uint32_t K) {
    const u32 blocks = ((M + TM - 1u) / TM) * ((N + TN - 1u) / TN), narrow = ((M + 31u) / 32u) * ((N + 63u) / 64u), steps = K / TK;
    if (qtype == UOCR_QT_F16 ? blocks >= 256u : narrow <= 256u || blocks > 190u) return 1u;
    u32 s = 1u;
    while (s < UOCR_KSPLIT_MAX && ((blocks * 2u * s <= 512u && steps / (2u * s) >= 5u) || steps / (2u * s) >= 16u)) s *= 2u;
    return s;
}

static bool gemm_desc_ok(int epi, const uocr_gemm_desc *d) {
    if (d == nullptr || d->A == nullptr || d->out == nullptr || d->N == 0u || d->K == 0u || d->K % 64u != 0u ||
        d->lda % 8u != 0u || !pmat_ok(d->W[0]) || (epi == UOCR_GEMM_SWIGLU && (!pmat_ok(d->W[1]) || d->W[1].qtype != d->W[0].qtype)) ||
        (d->nseg != 0u && (d->nseg % TN != 0u || d->N % d->nseg != 0u || d->N / d->nseg > 3u))) {
        return false;
    }
    for (u32 s = 1; d->nseg != 0u && s < d->N / d->nseg; ++s) {
        if (!pmat_ok(d->W[s]) || d->W[s].qtype != d->W[0].qtype) return false;
    }
    const bool grouped = d->tile_e != nullptr;
    if (grouped ? (d->a_idx == nullptr || d->o_idx == nullptr || d->tile_s0 == nullptr || d->tile_s1 == nullptr ||
                   d->ntiles == nullptr || d->max_tiles == 0u)
                : d->M == 0u) {
        return false;
    }
    return true;
}

/* 16-byte accesses of the epilogues: every row of the outputs, the residual
 * and the bias starts on such a boundary. */
static bool gemm_vec(const uocr_gemm_desc *d) {
    const uintptr_t p = (uintptr_t)d->out | (uintptr_t)d->out1 | (uintptr_t)d->out2 | (uintptr_t)d->bias | (uintptr_t)d->res;
    return d->N % 8u == 0u && d->ldo % 8u == 0u && d->split % 8u == 0u && (d->res == nullptr || d->ldr % 8u == 0u) && p % 16u == 0u;
}

static GemmArgs gemm_args(const uocr_gemm_desc *d) {
    GemmArgs a;
    a.A = (const h16 *)d->A;
    a.lda = d->lda;
    a.a_idx = d->a_idx;
    a.o_idx = d->o_idx;
    a.M = d->tile_e != nullptr ? d->a_rows : d->M;
    a.N = d->N;
    a.K = d->K;
    for (int i = 0; i < 3; ++i) a.W[i] = d->W[i];
    a.nseg = d->nseg;
    a.w_stride = d->w_stride;
    a.s_stride = d->s_stride;
    a.tile_e = d->tile_e;
    a.tile_s0 = d->tile_s0;
    a.tile_s1 = d->tile_s1;
    a.ntiles = d->ntiles;
    a.out = d->out;
    a.ldo = d->ldo;
    a.res = (const h16 *)d->res;
    a.ldr = d->ldr;
    a.bias = (const h16 *)d->bias;
    a.act = d->act;
    a.split = d->split;
    a.out1 = d->out1;
    a.out2 = d->out2;
    a.kst = 0u;
    a.packed = d->packed != 0u && d->W[0].qtype != UOCR_QT_F16 ? 1u : 0u;
    a.sc_lds = 0u;
    a.vec = gemm_vec(d) ? 1u : 0u;
    return a;
}

extern "C" int uocr_gemm_splits_itself(int epi, const uocr_gemm_desc *d) {
    return d->tile_e == nullptr && uocr_gemm_tile_takes(epi, d->W[0].qtype, gemm_args(d));
}

extern "C" hipError_t uocr_launch_gemm(hipStream_t st, int epi, const uocr_gemm_desc *d) {
    if (!gemm_desc_ok(epi, d) || d->nseg != 0u) return hipErrorInvalidValue;
    const bool grouped = d->tile_e != nullptr;
    GemmArgs a = gemm_args(d);
    const dim3 grid(grouped ? d->max_tiles : (d->M + TM - 1u) / TM, (d->N + TN - 1u) / TN);
    const u32 qt = d->W[0].qtype;
    if (epi == UOCR_GEMM_VISION && (grouped || d->bias == nullptr || d->act > UOCR_VISION_ACT_GELU_ERF ||
                                    (d->split != 0u && (d->N != 3u * d->split || d->out1 == nullptr ||
                                                        d->out2 == nullptr)))) {
        return hipErrorInvalidValue;
    }
    const bool split = !grouped && d->ksplit > 1u && d->part != nullptr;
    /* norm_w: the F16 output rows also go through the RMSNorm into norm_out
     * (fused into the split-K reduce, else a row-norm launch after the GEMM) */
    const bool want_norm = d->norm_w != nullptr;
    if (want_norm && (epi != UOCR_GEMM_F16 || grouped || d->norm_out == nullptr || d->N != UOCR_K_HIDDEN ||
                      d->ldo != UOCR_K_HIDDEN || (d->res != nullptr && d->ldr % 8u != 0u))) {
        return hipErrorInvalidValue;
    }
    if (grouped && d->tile_rows != 0u) return uocr_gemm_tile_grouped(st, epi, qt, a, d->pairs, d->tile_rows);
    const bool fused = split && want_norm, splittable = fused || (split && epi == UOCR_GEMM_VISION && d->N % 4u == 0u && d->split % 4u == 0u);
    if (!grouped && !fused && uocr_gemm_tile_takes(epi, qt, a)) {
        const hipError_t e = uocr_gemm_tile_plain(st, epi, qt, a);
        if (e != hipSuccess) return e;
    } else if (splittable) {
        /* split-K: blockIdx.z takes K steps [z*kst, (z+1)*kst) into an fp32
         * partial plane of part, then one ordered reduce applies the
         * epilogue */
        const u32 nt = d->K / TK;
        const u32 kst = (nt + min(d->ksplit, 8u) - 1u) / min(d->ksplit, 8u), S = (nt + kst - 1u) / kst;
        a.kst = kst;
        a.out = d->part;
        a.ldo = d->N;
        gemm_dispatch<GE_PART, false>(st, qt, a, dim3(grid.x, grid.y, S));
        if (fused) {
            hipLaunchKernelGGL(k_reduce_norm, dim3((d->M + 3u) / 4u), dim3(PB), 0, st, (const float *)d->part, S, d->M, (const h16 *)d->res, d->ldr,
                               (h16 *)d->out, d->ldo, (const h16 *)d->norm_w, (h16 *)d->norm_out);
            return hipGetLastError();
        }
        const size_t mn = (size_t)d->M * d->N;
        hipLaunchKernelGGL(k_split_reduce, dim3((unsigned)((mn / 4u + PB - 1u) / PB)), dim3(PB), 0, st,
                           (const float *)d->part, S, d->M, d->N, (const h16 *)d->bias, d->act, d->split, (h16 *)d->out,
                           (h16 *)d->out1, (h16 *)d->out2);
    } else if (epi == UOCR_GEMM_VISION) {
        gemm_dispatch<GE_VISION, false>(st, qt, a, grid);
    } else if (epi == UOCR_GEMM_F32) {
        if (grouped) gemm_dispatch<GE_F32, true>(st, qt, a, grid);
        else gemm_dispatch<GE_F32, false>(st, qt, a, grid);
    } else if (epi == UOCR_GEMM_SWIGLU) {
        if (grouped) gemm_dispatch<GE_SWIGLU, true>(st, qt, a, grid);
        else gemm_dispatch<GE_SWIGLU, false>(st, qt, a, grid);
    } else {
        if (grouped) gemm_dispatch<GE_F16, true>(st, qt, a, grid);
        else gemm_dispatch<GE_F16, false>(st, qt, a, grid);
    }
    if (want_norm) {
        hipLaunchKernelGGL(k_rows_rmsnorm, dim3((d->M + 3u) / 4u), dim3(PB), 0, st, (const h16 *)d->out,
                           (const h16 *)d->norm_w, d->M, (h16 *)d->norm_out);
    }
    return hipGetLastError();
}

extern "C" uint32_t uocr_moe_tile_rows(int epi_dn, const uocr_gemm_desc *gu, const uocr_gemm_desc *dn, uint32_t P) {
    const bool strides = (gu->w_stride | dn->w_stride) % 16u == 0u;
    if (!strides || !uocr_gemm_tile_fits(UOCR_GEMM_SWIGLU, gu->W[0].qtype, gemm_args(gu)) ||
        !uocr_gemm_tile_fits(epi_dn, dn->W[0].qtype, gemm_args(dn))) {
        return 0u;
    }
    return uocr_gemm_grouped_rows(P * UOCR_K_TOPK, gu->max_tiles);
}

extern "C" hipError_t uocr_launch_gemm_pair(hipStream_t st, int epi_a, const uocr_gemm_desc *da, int epi_b,
                                            const uocr_gemm_desc *db) {
    if (!gemm_desc_ok(epi_a, da) || !gemm_desc_ok(epi_b, db)) return hipErrorInvalidValue;
    const u32 q = da->W[0].qtype;
    const GemmArgs a = gemm_args(da), b = gemm_args(db);
    if (da->tile_e == nullptr && da->norm_w == nullptr && uocr_gemm_tile_fits(epi_a, q, a)) {
        if (epi_a == UOCR_GEMM_F16 && (epi_b == UOCR_GEMM_F16 || epi_b == UOCR_GEMM_F32) && db->tile_rows != 0u &&
            q == db->W[0].qtype && a.packed == b.packed) {
            return uocr_gemm_tile_pair(st, epi_b, q, a, b, db->pairs, db->tile_rows);
        }
        if (epi_a == UOCR_GEMM_SWIGLU && epi_b == UOCR_GEMM_F32 && db->W[0].qtype == UOCR_QT_F16 && uocr_gemm_router_fits(b)) {
            return uocr_gemm_tile_router(st, q, a, b);
        }
    }
    const hipError_t e = uocr_launch_gemm(st, epi_a, da);
    return e != hipSuccess ? e : uocr_launch_gemm(st, epi_b, db);
}

extern "C" hipError_t uocr_launch_rows_rmsnorm(hipStream_t st, const uint16_t *x, const uint16_t *w, uint32_t P,
                                               uint16_t *y) {
    if (x == nullptr || w == nullptr || y == nullptr || P == 0u) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_rows_rmsnorm, dim3((P + 3u) / 4u), dim3(PB), 0, st, (const h16 *)x, (const h16 *)w, P, (h16 *)y);
    return hipGetLastError();
}

extern "C" hipError_t uocr_launch_rope_table(hipStream_t st, const float *inv_freq, uint32_t P, float *cs) {
    if (inv_freq == nullptr || cs == nullptr || P == 0u) return hipErrorInvalidValue;
    RopeTabP tab;
    for (int i = 0; i < UOCR_K_HEAD_DIM / 2; ++i) tab.f[i] = inv_freq[i];
    hipLaunchKernelGGL(k_rope_table, dim3((P * 64u + PB - 1u) / PB), dim3(PB), 0, st, tab, P, (float2 *)cs);
    return hipGetLastError();
}

extern "C" hipError_t uocr_launch_gemm_qkv_rope(hipStream_t st, const uocr_gemm_desc *d, const float *cs,
                                                uint16_t *qout, uint16_t *kcache, uint16_t *vcache, uint32_t cap) {
    if (!gemm_desc_ok(UOCR_GEMM_F16, d) || d->tile_e != nullptr || d->nseg != UOCR_K_HIDDEN ||
        d->N != 3u * UOCR_K_HIDDEN || d->M > cap || cs == nullptr || qout == nullptr || kcache == nullptr ||
        vcache == nullptr) {
        return hipErrorInvalidValue;
    }
    GemmArgs a = gemm_args(d);
    a.nseg = 0u;
    uintptr_t al = 0;
    for (int i = 0; i < 3; ++i) al |= (uintptr_t)d->W[i].w;
    a.vec = 1u; /* the epilogue writes q and the cache slots only */
    if (al % 16u != 0u || (((uintptr_t)qout | (uintptr_t)kcache | (uintptr_t)vcache | (uintptr_t)cs) % 16u) != 0u ||
        !uocr_gemm_tile_fits(UOCR_GEMM_F16, d->W[0].qtype, a)) {
        return hipErrorInvalidValue;
    }
    a.nseg = d->nseg;
    return uocr_gemm_tile_rope(st, d->W[0].qtype, a, RopeDst{(const float2 *)cs, (h16 *)qout, (h16 *)kcache, (h16 *)vcache, cap});
}

extern "C" hipError_t uocr_launch_route_rows(hipStream_t st, const float *logits, uint32_t P, int norm_topk,
                                             int32_t *ids, float *wts, int32_t *offsets, int32_t *tile_e,
                                             int32_t *tile_s0, int32_t *tile_s1, int32_t *ntiles, int32_t *list_tok,
                                             int32_t *list_pair, uint32_t tile_rows) {
    if (logits == nullptr || P == 0u || ids == nullptr || wts == nullptr || offsets == nullptr || tile_e == nullptr || tile_s0 == nullptr || tile_s1 == nullptr || ntiles == nullptr ||
        list_tok == nullptr || list_pair == nullptr) {
        return hipErrorInvalidValue;
    }
    const BucketOut o = {offsets, tile_e, tile_s0, tile_s1, ntiles, list_tok, list_pair, (int32_t)(tile_rows != 0u ? tile_rows : TM)};
    hipLaunchKernelGGL(k_route_rows, dim3((P + 3u) / 4u), dim3(PB), 0, st, logits, P, norm_topk, ids, wts);
    if (P * UOCR_K_TOPK <= 8u * BUCKET_THREADS)
        hipLaunchKernelGGL(k_bucket_build<8u>, dim3(1), dim3(BUCKET_THREADS), 0, st, (const int32_t *)ids, P, o);
    else
        hipLaunchKernelGGL(k_bucket_build<24u>, dim3(1), dim3(BUCKET_THREADS), 0, st, (const int32_t *)ids, P, o);
    return hipGetLastError();
}

extern "C" hipError_t uocr_launch_moe_combine_norm(hipStream_t st, const float *Y, const float *wts,
                                                   const uint16_t *shared, const uint16_t *res, uint32_t P,
                                                   uint16_t *out, const uint16_t *norm_w, uint16_t *norm_out) {
    if (Y == nullptr || wts == nullptr || shared == nullptr || res == nullptr || out == nullptr || norm_w == nullptr ||
        norm_out == nullptr || P == 0u) {
        return hipErrorInvalidValue;
    }
    hipLaunchKernelGGL(k_moe_combine_norm<float>, dim3((P + 3u) / 4u), dim3(PB), 0, st, Y, wts, (const h16 *)shared,
                       (const h16 *)res, P, (h16 *)out, (const h16 *)norm_w, (h16 *)norm_out);
    return hipGetLastError();
}

extern "C" hipError_t uocr_launch_moe_combine_norm_h(hipStream_t st, const uint16_t *Y, const float *wts,
                                                     const uint16_t *shared, const uint16_t *res, uint32_t P,
                                                     uint16_t *out, const uint16_t *norm_w, uint16_t *norm_out) {
    if (Y == nullptr || wts == nullptr || shared == nullptr || res == nullptr || out == nullptr || norm_w == nullptr ||
        norm_out == nullptr || P == 0u) {
        return hipErrorInvalidValue;
    }
    hipLaunchKernelGGL(k_moe_combine_norm<h16>, dim3((P + 3u) / 4u), dim3(PB), 0, st, (const h16 *)Y, wts,
                       (const h16 *)shared, (const h16 *)res, P, (h16 *)out, (const h16 *)norm_w, (h16 *)norm_out);
    return hipGetLastError();
}

extern "C" hipError_t uocr_launch_moe_combine(hipStream_t st, const float *Y, const float *wts, const uint16_t *shared,
                                              const uint16_t *res, uint32_t P, uint16_t *out) {
    if (Y == nullptr || wts == nullptr || shared == nullptr || res == nullptr || out == nullptr || P == 0u) {
        return hipErrorInvalidValue;
    }
    const u32 n = P * UOCR_K_HIDDEN;
    hipLaunchKernelGGL(k_moe_combine<float>, dim3((n + PB - 1u) / PB), dim3(PB), 0, st, Y, wts, (const h16 *)shared,
                       (const h16 *)res, P, (h16 *)out);
    return hipGetLastError();
}

extern "C" hipError_t uocr_launch_moe_combine_h(hipStream_t st, const uint16_t *Y, const float *wts,
                                                const uint16_t *shared, const uint16_t *res, uint32_t P,
                                                uint16_t *out) {
    if (Y == nullptr || wts == nullptr || shared == nullptr || res == nullptr || out == nullptr || P == 0u) {
        return hipErrorInvalidValue;
    }
    const u32 n = P * UOCR_K_HIDDEN;
    hipLaunchKernelGGL(k_moe_combine<h16>, dim3((n + PB - 1u) / PB), dim3(PB), 0, st, (const h16 *)Y, wts,
                       (const h16 *)shared, (const h16 *)res, P, (h16 *)out);
    return hipGetLastError();
}

/* ---- GEMM-packed weight copies -------------------------------------------- */

/* One 16-byte piece per thread: destination piece i of matrix blockIdx.y. */
template <u32 RB>
__global__ __launch_bounds__(PB) void k_pack_gemm_rows(const uint8_t *__restrict__ src, uint8_t *__restrict__ dst,
                                                       u32 rows, u32 K, uint64_t stride) {
    const u32 steps = K / 64u, per = 32u * RB / 16u; /* pieces per (32-row block, step) */
    const size_t i = (size_t)blockIdx.x * PB + threadIdx.x, total = (size_t)rows / 32u * steps * per;
    if (i >= total) return;
    const size_t blk = i / per;
    const u32 in = (u32)(i % per), rb = (u32)(blk / steps), g = (u32)(blk % steps);
    const u32 lanes = RB / 2u / 16u;                       /* pieces per lane */
    const u32 l = in / lanes, v = in % lanes, h = l / 32u, r = l % 32u;
    const size_t so = (size_t)(rb * 32u + r) * (K / 64u * RB) + (size_t)g * RB + h * (RB / 2u) + 16u * v;
    const size_t m = (size_t)blockIdx.y * stride;
    *(uint4 *)(dst + m + i * 16u) = *(const uint4 *)(src + m + so);
}

extern "C" hipError_t uocr_launch_pack_gemm_rows(hipStream_t st, uint32_t qtype, const void *src, void *dst,
                                                 uint32_t rows, uint32_t K, uint32_t count, uint64_t stride) {
    if (src == nullptr || dst == nullptr || rows == 0u || rows % 32u != 0u || K == 0u || K % 64u != 0u || count == 0u ||
        (qtype != UOCR_QT_Q4 && qtype != UOCR_QT_Q8)) {
        return hipErrorInvalidValue;
    }
    const size_t pieces = (size_t)rows * (qtype == UOCR_QT_Q4 ? K / 2u : K) / 16u;
    const dim3 grid((unsigned)((pieces + PB - 1u) / PB), count);
    if (qtype == UOCR_QT_Q4) {
        hipLaunchKernelGGL(k_pack_gemm_rows<32u>, grid, dim3(PB), 0, st, (const uint8_t *)src, (uint8_t *)dst, rows, K,
                           stride);
    } else {
        hipLaunchKernelGGL(k_pack_gemm_rows<64u>, grid, dim3(PB), 0, st, (const uint8_t *)src, (uint8_t *)dst, rows, K,
                           stride);
    }
    return hipGetLastError();
}
