/*
 * uocr_attn_prefill.hip - causal flash attention of the prompt prefill on
 * gfx950 (replaces uocr_prefill_attention_flash_staged_f16_to_f16,
 * attention_prefill.metal:105; attention_decode.metal arithmetic per query).
 */
#include "uocr_async.h"

#include <math.h>

#define HD UOCR_K_HEAD_DIM

namespace {

/* Four keys of one dim per lane from a row-major V tile: in each group of 16
 * lanes, lane 4 i + j points at dims 4 j .. 4 j + 3 of key i and receives the
 * keys' values of dim (lane % 16). */
__device__ __forceinline__ uint2 lds_read_tr(const uint8_t *p) {
    typedef short s16x4 __attribute__((ext_vector_type(4)));
    const s16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4 *)p);
    return __builtin_bit_cast(uint2, v);
}

/* Bound by the matrix and vector pipes (per 32 x 32 scores 512 cycles of MFMA,
 * about 450 of exponentials, maxima and conversions); at 4,001 queries 72 us,
 * 570 TFLOP/s, against 186 us for 16-query wavefronts, each of which read
 * every K and V tile from LDS for half as many MFMAs, behind two barriers per
 * tile and a register transpose of V.
 *
 * Block: WQ x 32 queries of a head; its wavefronts are WG key groups of WQ
 * wavefronts, group g takes the key tiles g, g + WG, .. of the causal range
 * and the groups' softmax states are merged through LDS at the end.
 *
 * A wavefront keeps its 32 queries' state in registers (32x32x16 MFMAs):
 *   S^T = K Q^T: lane l holds query l % 32 and keys 8 q + 4 (l / 32) + i
 *   (i, q < 4) of the tile;
 *   the fp32 online softmax per query over the two lanes l, l ^ 32;
 *   O^T += V^T P^T: the probabilities stay where S^T left them, the B
 *   operand's 8 K slots of a lane are keys 16 s + 4 (l / 32) + i and + 8, and
 *   the A operand (V^T) is read at the same keys.
 * K and V tiles go straight to LDS, row-major; V is transposed by the LDS
 * read.  Both are swizzled by 16-byte pieces so that the reads touch all
 * banks: K by key % 16 (32 keys at one piece), V by pairs of pieces (4 keys,
 * 32 bytes each).  NB tiles of each group are in LDS, NB - 1 in flight.
 * DMA = false (caches off a 16-byte boundary): through registers. */
template <int WQ, int WG, int KT, int NB, bool DMA>
__global__ __launch_bounds__(64 * WQ * WG, 2) void k_flash_attn(const uint16_t *__restrict__ Q, const uint16_t *__restrict__ kc,
                                                               const uint16_t *__restrict__ vc, u32 cap, u32 P,
                                                               uint16_t *__restrict__ ctx, u32 nq) {
    constexpr u32 FA_TILE = KT * HD * 2u; /* bytes of a K or V tile in LDS */
    constexpr u32 GB = NB * 2u * FA_TILE; /* LDS of a key group */
    constexpr int LD = (int)(2u * FA_TILE / 1024u) / WQ; /* loads of a wavefront per tile (K, then V) */
    constexpr u32 MERGE = (WG - 1u) * WQ * (32u * HD * 4u + 512u), STAGE = WQ * 32u * HD * 2u;
    constexpr u32 LDS = WG * GB > MERGE ? WG * GB : MERGE;
    static_assert(LDS >= STAGE, "output staging");
    __shared__ __attribute__((aligned(1024))) uint8_t sm[LDS];
    const u32 t = threadIdx.x, lane = t & 63u, r = lane & 31u, hf = lane >> 5;
    const u32 wave = uni(t >> 6), wq = wave % WQ, g = wave / WQ;
    /* longest query tiles first */
    const u32 qt = nq - 1u - blockIdx.x / UOCR_K_HEADS, h = blockIdx.x % UOCR_K_HEADS;
    const u32 q0 = qt * WQ * 32u, qw = q0 + 32u * wq, qr = qw + r; /* the block's, the wavefront's, the lane's query */
    const u32 qlast = min(q0 + WQ * 32u, P) - 1u, nt = qlast / KT + 1u, iters = (nt + WG - 1u) / WG;
    const u32 qmax = min(qr, P - 1u);
    const uint8_t *kh = (const uint8_t *)(kc + (size_t)h * cap * HD), *vh = (const uint8_t *)(vc + (size_t)h * cap * HD);
    uint8_t *gsm = sm + g * GB;
    const u32 lds0 = uni((u32)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)gsm);

    /* loads: 4 keys of 256 bytes each; load x of the tile (the first KT / 4:
     * K, else V) covers keys 4 (x % (KT / 4)) .. + 3 */
    const u32 lr = lane >> 4, lp = lane & 15u;
    auto issue = [&](u32 tile, u32 buf) {
#pragma unroll
        for (int y = 0; y < LD; ++y) {
            const u32 x = wq * LD + y, kr = 4u * (x % (KT / 4u)) + lr; /* key within the tile */
            const u32 key = min(tile * KT + kr, P - 1u);
            const u32 pc = x < KT / 4u ? lp ^ (kr & 15u) : lp ^ ((kr & 7u) << 1);
            if constexpr (DMA) lds_load16(x < KT / 4u ? kh : vh, key * (HD * 2u) + 16u * pc, lds0 + buf * 2u * FA_TILE + 1024u * x);
            else *(uint4 *)(gsm + buf * 2u * FA_TILE + 1024u * x + 16u * lane) = *(const uint4 *)((x < KT / 4u ? kh : vh) + key * (HD * 2u) + 16u * pc);
        }
    };

    U4H8 qreg[HD / 16];
#pragma unroll
    for (u32 s = 0; s < HD / 16; ++s) qreg[s].u = *(const uint4 *)(Q + (size_t)qmax * UOCR_K_HIDDEN + h * HD + 16u * s + 8u * hf);
    f32x16 o[HD / 32];
#pragma unroll
    for (int d = 0; d < HD / 32; ++d)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[d][i] = 0.0f;
    float m = -INFINITY, l = 0.0f; /* m in units of the raw scores; l: this lane's half of the sum */
    const float c = 0.08838834764831845f * 1.4426950408889634f; /* 1/sqrt(128) * log2(e) */

#pragma unroll
    for (u32 b = 0; b + 1u < NB; ++b) issue(min(b * WG + g, nt - 1u), b);
    u32 buf = 0;
    for (u32 it = 0; it < iters; ++it) {
        /* tile it has landed for all wavefronts; its predecessor's buffer is free */
        wait_barrier<LD * (NB - 2)>();
        issue(min((it + NB - 1u) * WG + g, nt - 1u), buf == 0u ? NB - 1u : buf - 1u);
        const u32 tile = it * WG + g, k0 = tile * KT;
        const uint8_t *kt = gsm + buf * 2u * FA_TILE, *vt = kt + FA_TILE;
        buf = buf + 1u == NB ? 0u : buf + 1u;
        if (tile >= nt || k0 > qw + 31u) continue; /* no key of the tile is visible to these queries */
        f32x16 s[KT / 32];
        float tm = -INFINITY;
#pragma unroll
        for (u32 n = 0; n < KT / 32; ++n) {
#pragma unroll
            for (int i = 0; i < 16; ++i) s[n][i] = 0.0f;
#pragma unroll
            for (u32 x = 0; x < HD / 16; ++x) {
                U4H8 a;
                a.u = *(const uint4 *)(kt + (32u * n + r) * 256u + 16u * ((2u * x + hf) ^ (r & 15u)));
                s[n] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a.v, qreg[x].v, s[n], 0, 0, 0);
            }
            if (k0 + 32u * n + 31u > qw) {
#pragma unroll
                for (u32 i = 0; i < 16; ++i) {
                    const u32 key = k0 + 32u * n + 8u * (i / 4u) + 4u * hf + i % 4u;
                    if (key > qmax) s[n][i] = -INFINITY;
                }
            }
#pragma unroll
            for (int i = 0; i < 16; ++i) tm = fmaxf(tm, s[n][i]);
        }
        tm = fmaxf(tm, __shfl_xor(tm, 32));
        /* Only when some query's maximum grew.  (Letting the reference lag by up
         * to 2^8 skips more rescaling, but then a row's largest probability is
         * no longer exactly 1 in fp16: 2.6e-4 from 64 bits against 2.5e-4.) */
        if (__any(tm > m)) {
            const float mn = fmaxf(m, tm), corr = m == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f((m - mn) * c);
            m = mn;
            l *= corr;
#pragma unroll
            for (int d = 0; d < HD / 32; ++d)
#pragma unroll
                for (int i = 0; i < 16; ++i) o[d][i] *= corr;
        }
        const float mc = m == -INFINITY ? 0.0f : m * c;
        U4H8 p[KT / 16];
#pragma unroll
        for (int i = 0; i < KT / 2; ++i) {
            const float e = __builtin_amdgcn_exp2f(fmaf(s[i >> 4][i & 15], c, -mc));
            l += e;
            p[i >> 3].h[i & 7] = (h16)e;
        }
#pragma unroll
        for (u32 y = 0; y < KT / 16; ++y) {
#pragma unroll
            for (u32 d = 0; d < HD / 32; ++d) {
                /* lane's key of the transposing read: 16 y + 4 hf + i (and + 8), i = lane % 16 / 4; dims 32 d + 16 (lane / 16 % 2) + 4 (lane % 4) */
                const u32 key = 16u * y + 4u * hf + ((lane >> 2) & 3u), byte = 64u * d + 32u * ((lane >> 4) & 1u) + 8u * (lane & 3u);
                const uint2 lo = lds_read_tr(vt + key * 256u + ((byte & ~15u) ^ ((key & 7u) << 5)) + (byte & 15u));
                const uint2 hi = lds_read_tr(vt + (key + 8u) * 256u + ((byte & ~15u) ^ (((key + 8u) & 7u) << 5)) + (byte & 15u));
                U4H8 a;
                a.u = make_uint4(lo.x, lo.y, hi.x, hi.y);
                o[d] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a.v, p[y].v, o[d], 0, 0, 0);
            }
        }
    }
    l += __shfl_xor(l, 32);
    wait_barrier<0>(); /* the tiles' LDS is free (loads past the last tile have landed) */
    if constexpr (WG > 1) {
        constexpr u32 SLOT = 32u * HD * 4u + 512u;
        if (g > 0u) {
            uint8_t *dst = sm + ((g - 1u) * WQ + wq) * SLOT;
#pragma unroll
            for (int d = 0; d < HD / 32; ++d)
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    *(float4 *)(dst + (4u * d + q) * 1024u + 16u * lane) = make_float4(o[d][4 * q], o[d][4 * q + 1], o[d][4 * q + 2], o[d][4 * q + 3]);
            *(float2 *)(dst + 32u * HD * 4u + 8u * lane) = make_float2(m, l);
        }
        __syncthreads();
        if (g == 0u) {
            float mg[WG], lg[WG];
            mg[0] = m;
            lg[0] = l;
            float M = m;
#pragma unroll
            for (u32 x = 1; x < WG; ++x) {
                const float2 v = *(const float2 *)(sm + ((x - 1u) * WQ + wq) * SLOT + 32u * HD * 4u + 8u * lane);
                mg[x] = v.x;
                lg[x] = v.y;
                M = fmaxf(M, v.x);
            }
            l = 0.0f;
#pragma unroll
            for (u32 x = 0; x < WG; ++x) {
                /* M is finite: group 0 holds key 0 */
                const float w = mg[x] == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f((mg[x] - M) * c);
                l += lg[x] * w;
#pragma unroll
                for (int d = 0; d < HD / 32; ++d)
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        if (x == 0u) {
#pragma unroll
                            for (int i = 0; i < 4; ++i) o[d][4 * q + i] *= w;
                        } else {
                            const float4 v = *(const float4 *)(sm + ((x - 1u) * WQ + wq) * SLOT + (4u * d + q) * 1024u + 16u * lane);
                            o[d][4 * q] = fmaf(v.x, w, o[d][4 * q]);
                            o[d][4 * q + 1] = fmaf(v.y, w, o[d][4 * q + 1]);
                            o[d][4 * q + 2] = fmaf(v.z, w, o[d][4 * q + 2]);
                            o[d][4 * q + 3] = fmaf(v.w, w, o[d][4 * q + 3]);
                        }
                    }
            }
        }
        __syncthreads();
    }
    if (g == 0u) {
        const float li = 1.0f / l;
#pragma unroll
        for (u32 d = 0; d < HD / 32; ++d)
#pragma unroll
            for (u32 q = 0; q < 4; ++q) {
                union {
                    h16 x[4];
                    uint2 u;
                } v;
#pragma unroll
                for (int i = 0; i < 4; ++i) v.x[i] = (h16)(o[d][4 * q + i] * li);
                *(uint2 *)(sm + (32u * wq + r) * 256u + 16u * ((4u * d + q) ^ (r & 15u)) + 8u * hf) = v.u;
            }
    }
    __syncthreads();
    for (u32 x = t; x < WQ * 32u * 16u; x += 64u * WQ * WG) {
        const u32 row = x >> 4, pc = x & 15u;
        if (q0 + row >= P) break;
        *(uint4 *)(ctx + (size_t)(q0 + row) * UOCR_K_HIDDEN + h * HD + 8u * pc) = *(const uint4 *)(sm + row * 256u + 16u * (pc ^ (row & 15u)));
    }
}

template <int WQ, int WG, int KT, int NB>
hipError_t launch(hipStream_t st, const uint16_t *q, const uint16_t *kc, const uint16_t *vc, u32 cap, u32 P, uint16_t *ctx) {
    const u32 nq = (P + WQ * 32u - 1u) / (WQ * 32u);
    if ((((uintptr_t)kc | (uintptr_t)vc) & 15u) == 0u)
        hipLaunchKernelGGL((k_flash_attn<WQ, WG, KT, NB, true>), dim3(nq * UOCR_K_HEADS), dim3(64 * WQ * WG), 0, st, q, kc, vc, cap, P, ctx, nq);
    else
        hipLaunchKernelGGL((k_flash_attn<WQ, WG, KT, NB, false>), dim3(nq * UOCR_K_HEADS), dim3(64 * WQ * WG), 0, st, q, kc, vc, cap, P, ctx, nq);
    return hipGetLastError();
}

}  // namespace

extern "C" hipError_t uocr_launch_flash_attn(hipStream_t st, const uint16_t *q, const uint16_t *kcache,
                                             const uint16_t *vcache, uint32_t cap, uint32_t P, uint16_t *ctx) {
    if (q == nullptr || kcache == nullptr || vcache == nullptr || ctx == nullptr || P == 0u || P > cap) {
        return hipErrorInvalidValue;
    }
    /* Measured (us; wavefronts along queries x along keys, keys per tile):
     *   P      4 x 1, 64   2 x 4, 32   4 x 2, 64
     *   64         4.6         6.9         6.1
     *   341       11.3         9.7        10.5
     *   932       25.1        17.5        20.5   (before, with its merge: 22.9)
     *   3000      71.3        49.0        53.6
     *   4001      94.8        82.0        72.3   (before: 185.7)
     * Few queries need few wavefronts; up to about 3,300 the key groups shorten
     * the last query tiles' walk; beyond it the larger query tile's half as
     * many passes over K and V tell. */
    if (P <= 256u) return launch<4, 1, 64, 2>(st, q, kcache, vcache, cap, P, ctx);
    if (P <= 3300u) return launch<2, 4, 32, 2>(st, q, kcache, vcache, cap, P, ctx);
    return launch<4, 2, 64, 2>(st, q, kcache, vcache, cap, P, ctx);
}
