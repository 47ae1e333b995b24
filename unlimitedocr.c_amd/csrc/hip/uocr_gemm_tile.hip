/*
 * uocr_gemm_tile.hip - the large-tile MFMA GEMM of the prompt prefill, the
 * operator API and the vision linears on gfx950 (replaces the reference's
 * tiled GEMMs gemm_q4.metal / gemm_q8.metal where a grid of large tiles fills
 * the chip).
 */
#include "uocr_async.h"
#include "uocr_gemm.h"

#define NA 3u  /* activation tiles in LDS: two steps of loads in flight */

namespace {

/* The block's tile.  Blocks go to the 8 XCDs in turn; each XCD takes a
 * contiguous run of row tiles (by_row; else of column tiles), so that its L2
 * fetches only its share of the activations (of the weights). */
__device__ __forceinline__ bool tile_of(u32 id, bool by_row, u32 nx, u32 ny, u32 &bx, u32 &by) {
    const u32 total = nx * ny, q = total / 8u, rem = total % 8u, x = id % 8u, slot = id / 8u;
    if (slot >= q + (x < rem ? 1u : 0u)) return false;
    const u32 l = x * q + min(x, rem) + slot;
    if (by_row) {
        bx = l / ny;
        by = l % ny;
    } else {
        bx = l % nx;
        by = l / nx;
    }
    return true;
}

/* Groups of 64 columns in the 128 bytes of a weight row. */
template <int QT>
constexpr int groups_per_line() {
    return QT == 4 ? 4 : (QT == 3 ? 2 : 1);
}

template <u32 ACT>
__device__ __forceinline__ float vision_act(float v) {
    return ACT == UOCR_VISION_ACT_QUICKGELU ? quick_gelu(v) : (ACT == UOCR_VISION_ACT_GELU_ERF ? gelu_erf_as(v) : v);
}

/* f(integral_constant<u32, act>): the activation is chosen once, around an
 * epilogue.  Chosen per value, the branches and the code they step over took
 * 2.3 us of a 64 x 128 tile (1600 x 768 x 768 Q8 11.1 -> 8.9) and 3.6 of a
 * large one (4096 x 768 x 768 19.4 -> 15.7). */
template <typename F>
__device__ __forceinline__ void with_act(u32 act, F &&f) {
    if (act == UOCR_VISION_ACT_QUICKGELU) f(std::integral_constant<u32, UOCR_VISION_ACT_QUICKGELU>{});
    else if (act == UOCR_VISION_ACT_GELU_ERF) f(std::integral_constant<u32, UOCR_VISION_ACT_GELU_ERF>{});
    else f(std::integral_constant<u32, UOCR_VISION_ACT_NONE>{});
}

/* LDS of one K group: the activation tiles and its wavefronts' weight lines. */
template <int RT, int WN>
constexpr u32 group_lds_bytes() {
    return NA * 32u * RT * 128u + WN * 8192u;
}

template <int RT, int WN, int WK>
constexpr u32 tile_lds_bytes(bool rope) {
    constexpr u32 main = WK * group_lds_bytes<RT, WN>(), stage = 32u * RT * (64u * WN + 8u) * 2u;
    return rope && stage > main ? stage : main;
}

template <int QT, int EPI, bool GROUPED, bool PACKED, int RT, int WN, int WK>
__device__ __forceinline__ void tile_body(const GemmArgs &p, u32 bx, u32 by, uint8_t *sm, const RopeDst &rd) {
    constexpr int NG = groups_per_line<QT>();
    constexpr bool SW = EPI == GE_SWIGLU;
    constexpr u32 CW = SW ? 32u : 64u; /* output columns of a wavefront */
    constexpr u32 ROWS = 32u * RT, ABUF = ROWS * 128u, TT = 64u * WN * WK;
    constexpr int AL = RT * 4 / WN; /* activation loads of a wavefront per step */
    static_assert(AL * WN == RT * 4, "activation rows");
    constexpr u32 RB = QT == 4 ? 32u : 64u; /* packed: bytes of a row's group */
    const u32 t = threadIdx.x, lane = t & 63u, r = lane & 31u, h = lane >> 5;
    const u32 wave = uni(t >> 6) % WN, kg = uni(t >> 6) / WN; /* column group, K group */
    u32 e = 0, s0 = bx * ROWS, rows;
    if (GROUPED) {
        e = uni((u32)p.tile_e[bx]);
        s0 = uni((u32)p.tile_s0[bx]);
        rows = uni((u32)p.tile_s1[bx]) - s0;
    } else {
        rows = min(ROWS, p.M - s0);
    }
    const u32 K = p.K;
    /* K group kg takes steps [ks, ks + NT) of its matrix; all groups run the
     * same number of steps (NS) for the block's barriers */
    const u32 NTA = K / 64u, NS = (NTA + WK - 1u) / WK, ks = min(kg * NS, NTA - 1u), NT = kg * NS < NTA ? min(NS, NTA - ks) : 0u;
    const u32 NCH = (NS + NG - 1u) / NG;
    const u32 rowb = QT == 4 ? K / 2u : (QT == 3 ? K : 2u * K);
    const u32 n0 = by * WN * CW;
    const uocr_qmat *W0 = &p.W[0];
    u32 nbase = 0, nmax = p.N;
    if (p.nseg != 0u) {
        const u32 sg = n0 / p.nseg;
        W0 = &p.W[sg];
        nbase = sg * p.nseg;
        nmax = p.nseg;
    }
    const uint8_t *w[2];
    const unsigned short *sc[2];
    u32 cb[2]; /* first weight row of the wavefront's two column groups */
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const uocr_qmat &m = SW ? p.W[j] : *W0;
        w[j] = (const uint8_t *)m.w + (GROUPED ? e * p.w_stride : 0);
        sc[j] = (const unsigned short *)m.s + (GROUPED ? e * p.s_stride : 0);
        cb[j] = n0 - nbase + CW * wave + (SW ? 0u : 32u * j);
    }

    /* activation staging: this lane's rows, 16-byte piece (lane % 8) ^ (row /
     * 2 % 8) of the row's 128 bytes; two rows span the 64 banks, so this
     * swizzle keeps the reads free of bank conflicts (16 reads by 4 wavefronts
     * 118 ns; by row % 8, two rows to a bank, 230 ns).  The wavefront loads RT
     * groups of 8 rows; pc(i): the piece's offset in group i */
    auto pc = [&](u32 i) { return 16u * ((lane & 7u) ^ (lane >> 4)) ^ (64u * (i & 1u)); };
    u32 va[AL];
#pragma unroll
    for (int q = 0; q < AL; ++q) {
        const u32 rr = min(8u * (AL * wave + q) + (lane >> 3), rows - 1u);
        const u32 ar = GROUPED ? (u32)p.a_idx[s0 + rr] : s0 + rr;
        va[q] = ar * p.lda * 2u + pc(AL * wave + q);
    }
    const u32 lds0 = uni((u32)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)sm);
    uint8_t *gsm = sm + kg * group_lds_bytes<RT, WN>();
    const u32 ldsg = lds0 + kg * group_lds_bytes<RT, WN>(), lds_a = ldsg + wave * AL * 1024u, lds_b = ldsg + NA * ABUF + wave * 8192u;
    const uint8_t *Ab = (const uint8_t *)p.A + (size_t)ks * 128u;
    auto issue_a = [&](u32 s, u32 buf, int q) { lds_load16(Ab + (size_t)s * 128u, va[q], lds_a + buf + 1024u * q); };
    /* weight staging: the wavefront's own 64 rows, a line of 128 bytes (NG
     * groups) of each; pieces past the row's end re-read its last 16 bytes */
    u32 vb[PACKED ? 1 : 8];
    const uint8_t *pb[2];
    const u32 room = rowb - ks * (rowb / NTA) - 16u; /* a row's last 16 bytes, from the group's first */
    if constexpr (PACKED) {
        vb[0] = 16u * lane;
#pragma unroll
        for (int j = 0; j < 2; ++j) pb[j] = w[j] + (size_t)min(cb[j] / 32u, nmax / 32u - 1u) * NTA * (32u * RB) + (size_t)ks * (32u * RB);
    } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) vb[i] = min(cb[i >> 2] + 8u * (i & 3) + (lane >> 3), nmax - 1u) * rowb;
        pb[0] = w[0] + ks * (rowb / NTA);
        pb[1] = w[1] + ks * (rowb / NTA);
    }
    auto issue_b = [&](u32 c, int i) {
        if constexpr (PACKED) {
            const u32 cc = min(c, (NTA - ks - 1u) / NG), left = (NTA - ks - cc * NG) * 32u * RB, o = 1024u * (i & 3); /* left: bytes to the run's end */
            lds_load16(pb[i >> 2] + (size_t)cc * 4096u + (o < left ? o : 0u), vb[0], lds_b + 1024u * i);
        } else {
            lds_load16(pb[i >> 2], vb[i] + min(c * 128u + pc(i & 1), room), lds_b + 1024u * i);
        }
    };
    u32 sn[2][NG];
    const unsigned short *srow[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        srow[j] = sc[j] + (size_t)min(cb[j] + r, nmax - 1u) * NTA + ks;
#pragma unroll
        for (int g = 0; g < NG; ++g) sn[j][g] = 0u;
    }
    auto load_s = [&](u32 c) {
        if constexpr (QT != 1) {
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int g = 0; g < NG; ++g) sn[j][g] = srow[j][min(c * NG + g, NTA - ks - 1u)];
        }
    };

    f32x16 acc[RT][2];
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int k = 0; k < 16; ++k) acc[i][j][k] = 0.0f;

    /* LDS offsets of this lane's activation operand of substep i (row r of a
     * 32-row tile) */
    u32 ao[4];
#pragma unroll
    for (u32 i = 0; i < 4; ++i) ao[i] = r * 128u + 16u * ((b_koff<QT>(i, h) / 8u) ^ ((r >> 1) & 7u));
    const uint8_t *bsm = gsm + NA * ABUF + wave * 8192u;

    load_s(0);
#pragma unroll
    for (int i = 0; i < 8; ++i) issue_b(0, i);
#pragma unroll
    for (int q = 0; q < AL; ++q) issue_a(0, 0u, q);
    const u32 sl = max(NT, 1u) - 1u; /* the group's last step */
#pragma unroll
    for (int q = 0; q < AL; ++q) issue_a(min(1u, sl), ABUF, q);
    u32 cur = 0, nxt = 2u * ABUF; /* LDS offsets of step s's activations and of step s + 2's */
    u32 br[2][16], sv[2][NG];
    for (u32 c = 0; c < NCH; ++c) {
#pragma unroll
        for (int g = 0; g < NG; ++g) {
            const u32 s = c * NG + g;
            if (g > 0 && s >= NS) break;
            /* A step issues the activations of step s + 2, then its share of
             * line c + 1 (f16, whose line lasts one step: the line first).
             * Loads complete in order, so what must have landed here is the
             * activations of step s, issued in step s - 2, and at g = 0 line c;
             * in flight may stay what was issued after them.  The weights,
             * which come from HBM, so have three steps to arrive (Q8: two). */
            constexpr int NB = NG == 4 ? 4 : 8, BS = 8 / NB; /* loads of a line per step, in the line's first BS steps */
            const int after = NG == 1 ? 0 : (g >= 1 && g <= BS ? NB : 0) + (g >= 2 && g <= BS + 1 ? NB : 0);
            if (after == 2 * NB && c + 1u < NCH) wait_barrier<AL + 2 * NB>();
            else if (after == NB && c + 1u < NCH) wait_barrier<AL + NB>();
            else wait_barrier<AL>();
            if (g == 0) {
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int q = 0; q < NG; ++q) {
                        asm volatile("" : "+v"(sn[j][q])); /* the scales' wait belongs here, before later loads */
                        sv[j][q] = sn[j][q];
                    }
                load_s(min(c + 1u, NCH - 1u));
            }
            if (g == 0) {
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        u32 o;
                        if constexpr (PACKED) {
                            o = QT == 4 ? 1024u * q + 16u * lane : 2048u * (q >> 1) + 32u * lane + 16u * (q & 1);
                        } else {
                            const u32 ch = QT == 4 ? 2u * q + h : (QT == 3 ? 4u * (q >> 1) + 2u * h + (q & 1) : 4u * h + q);
                            o = r * 128u + 16u * (ch ^ ((r >> 1) & 7u));
                        }
                        const uint4 x = *(const uint4 *)(bsm + 4096u * j + o);
                        br[j][4 * q] = x.x;
                        br[j][4 * q + 1] = x.y;
                        br[j][4 * q + 2] = x.z;
                        br[j][4 * q + 3] = x.w;
                    }
            }
            if (WK == 1 || s < NT) {
            const uint8_t *abuf = gsm + cur;
            /* computing goes before the CU's other block's loads and waits */
            __builtin_amdgcn_s_setprio(1);
            U4H8 a[2][RT]; /* substep i's operands and the next one's */
#pragma unroll
            for (int k = 0; k < RT; ++k) a[0][k].u = *(const uint4 *)(abuf + ao[0] + 4096u * k);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (i < 3) {
#pragma unroll
                    for (int k = 0; k < RT; ++k) a[(i + 1) & 1][k].u = *(const uint4 *)(abuf + ao[i < 3 ? i + 1 : 3] + 4096u * k);
                }
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    h16x8 wv;
                    if (QT == 4) wv = dequant_q4(br[j][4 * g + 2 * (i & 1)], br[j][4 * g + 2 * (i & 1) + 1], (i & 2) != 0, sv[j][g]);
                    else if (QT == 3) wv = dequant_q8(br[j][(8 * g + 2 * i) & 15], br[j][(8 * g + 2 * i + 1) & 15], sv[j][g]);
                    else wv = operand_f16(br[j][4 * i], br[j][4 * i + 1], br[j][4 * i + 2], br[j][4 * i + 3]);
#pragma unroll
                    for (int k = 0; k < RT; ++k) acc[k][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(wv, a[i & 1][k].v, acc[k][j], 0, 0, 0);
                    /* the loads spread over the step, between its MFMAs: issued
                     * together they fill the memory pipe's queue and the
                     * wavefront's MFMAs wait behind them */
                    const int slot = 2 * i + j, bslot = NG > 1 ? 4 : 1, aslot = NG > 1 ? 0 : 4;
                    /* (past the end the last step again, which nothing reads:
                     * the count of loads in flight stays the same) */
                    auto slot_a = [&]() {
#pragma unroll
                        for (int q = 0; q < AL; ++q)
                            if (aslot + q * 4 / AL == slot) issue_a(min(s + 2u, sl), nxt, q);
                    };
                    if (NG > 1) slot_a();
                    if (g < BS && slot >= bslot && slot < bslot + 4 && c + 1u < NCH) {
                        /* the line is in registers: its LDS takes the next one */
                        if (slot == bslot) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
                        for (int x = 0; x < NB / 4; ++x) issue_b(c + 1u, NB * g + NB / 4 * (slot - bslot) + x);
                    }
                    if (NG == 1) slot_a();
                }
            }
            __builtin_amdgcn_s_setprio(0);
            }
            nxt = cur;
            cur = cur + ABUF == NA * ABUF ? 0u : cur + ABUF;
        }
    }

    if constexpr (WK > 1) {
        /* the K groups' sums, added in order by group 0 */
        wait_barrier<0>();
        if (kg > 0) {
            uint8_t *dst = sm + ((kg - 1u) * WN + wave) * (RT * 8192u) + 16u * lane;
#pragma unroll
            for (int k = 0; k < RT; ++k)
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        *(float4 *)(dst + ((k * 2 + j) * 4 + q) * 1024u) =
                            make_float4(acc[k][j][4 * q], acc[k][j][4 * q + 1], acc[k][j][4 * q + 2], acc[k][j][4 * q + 3]);
        }
        __syncthreads();
        if (kg == 0) {
            for (u32 g = 1; g < WK; ++g) {
                const uint8_t *src = sm + ((g - 1u) * WN + wave) * (RT * 8192u) + 16u * lane;
#pragma unroll
                for (int k = 0; k < RT; ++k)
#pragma unroll
                    for (int j = 0; j < 2; ++j)
#pragma unroll
                        for (int q = 0; q < 4; ++q) {
                            const float4 v = *(const float4 *)(src + ((k * 2 + j) * 4 + q) * 1024u);
                            acc[k][j][4 * q] += v.x;
                            acc[k][j][4 * q + 1] += v.y;
                            acc[k][j][4 * q + 2] += v.z;
                            acc[k][j][4 * q + 3] += v.w;
                        }
            }
        }
    }
    /* Lane l holds row l % 32 of each 32-row tile and, of column group j,
     * columns 8q + 4 (l / 32) + 0..3 in elements 4q..4q+3. */
    if constexpr (EPI == GE_ROPE) {
        constexpr u32 LD = 64u * WN + 8u; /* padded row (halves) */
        h16 *tile = (h16 *)sm;
        wait_barrier<0>();
        if (WK == 1 || kg == 0) {
#pragma unroll
        for (int k = 0; k < RT; ++k)
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    union {
                        h16 x[4];
                        uint2 u;
                    } o;
#pragma unroll
                    for (int x = 0; x < 4; ++x) o.x[x] = (h16)acc[k][j][4 * q + x];
                    *(uint2 *)(tile + (32u * k + r) * LD + 64u * wave + 32u * j + 8u * q + 4u * h) = o.u;
                }
        }
        __syncthreads();
        const u32 seg = n0 / p.nseg, h0 = (n0 - seg * p.nseg) / 128u;
        /* 8 pairs (d, d + 64) of one head and row per thread and turn */
        for (u32 it = t; it < rows * 4u * WN; it += TT) {
            const u32 row = it / (4u * WN), hd = (it / 8u) % (WN / 2u), d = 8u * (it % 8u), tok = s0 + row;
            U4H8 a, b;
            a.u = *(const uint4 *)(tile + row * LD + 128u * hd + d);
            b.u = *(const uint4 *)(tile + row * LD + 128u * hd + d + 64u);
            h16 *dst = seg == 0u ? rd.q + (size_t)tok * UOCR_K_HIDDEN + (h0 + hd) * 128u + d
                                 : (seg == 1u ? rd.k : rd.v) + ((size_t)(h0 + hd) * rd.cap + tok) * 128u + d;
            if (seg != 2u) {
                const float4 *cs = (const float4 *)(rd.cs + (size_t)tok * 64u + d);
                U4H8 x, y;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const float4 f = cs[q];
                    const float a0 = (float)a.h[2 * q], b0 = (float)b.h[2 * q], a1 = (float)a.h[2 * q + 1], b1 = (float)b.h[2 * q + 1];
                    x.h[2 * q] = (h16)(a0 * f.x - b0 * f.y);
                    y.h[2 * q] = (h16)(a0 * f.y + b0 * f.x);
                    x.h[2 * q + 1] = (h16)(a1 * f.z - b1 * f.w);
                    y.h[2 * q + 1] = (h16)(a1 * f.w + b1 * f.z);
                }
                a = x;
                b = y;
            }
            *(uint4 *)dst = a.u;
            *(uint4 *)(dst + 64) = b.u;
        }
        return;
    }
    /* Through LDS, so that the stores (and the residual's loads) cover whole
     * rows of the tile: 16-byte pieces, swizzled by row.  Stored from the
     * registers, 8 bytes of 32 rows at a time, every piece was a write request
     * of its own. */
    constexpr bool F32O = EPI == GE_F32;
    constexpr u32 CPP = F32O ? 4u : 8u;        /* columns per piece */
    constexpr u32 CH = WN * CW / CPP;          /* pieces per row */
    constexpr int PASS_RT = F32O ? (RT == 4 ? 2 : 1) : RT; /* 32-row tiles per pass */
    static_assert(PASS_RT * 32u * CH * 16u <= tile_lds_bytes<RT, WN, WK>(false), "staging fits");
    const u32 ch = t % CH, col = n0 + CPP * ch; /* the piece this thread moves, in rows t / CH, + TT / CH, .. */
#pragma unroll
    for (int k0 = 0; k0 < RT; k0 += PASS_RT) {
        wait_barrier<0>();
        if (EPI == GE_F16 && p.res != nullptr) {
            /* the residual's tile into the pieces' places; columns past N and
             * rows past the tile re-read valid ones */
            constexpr u32 RPL = 64u / CH; /* rows per load */
#pragma unroll 4
            for (u32 q = uni(t >> 6); q < ROWS / RPL; q += WN * WK) {
                const u32 row = q * RPL + lane / CH;
                const u32 c = min(n0 + CPP * ((lane % CH) ^ (row % CH)), p.N - CPP);
                const u32 rr = min(row, rows - 1u);
                const size_t orow = GROUPED ? (size_t)p.o_idx[s0 + rr] : (size_t)(s0 + rr);
                lds_load16(p.res, (u32)((orow * p.ldr + c) * 2u), lds0 + q * 1024u);
            }
            wait_barrier<0>();
        }
        auto put = [&](auto ACT) {
#pragma unroll
        for (int j = 0; j < (SW ? 1 : 2); ++j) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                float bias[4] = {0.0f, 0.0f, 0.0f, 0.0f};
                if constexpr (EPI == GE_VISION) {
                    union {
                        h16 x[4];
                        uint2 u;
                    } b;
                    b.u = *(const uint2 *)(p.bias + min(n0 + CW * wave + 32u * j + 8u * q + 4u * h, p.N - 4u));
#pragma unroll
                    for (int x = 0; x < 4; ++x) bias[x] = (float)b.x[x];
                }
                const u32 pcs = F32O ? 16u * wave + 8u * j + 2u * q + h : (SW ? 4u * wave + q : 8u * wave + 4u * j + q);
#pragma unroll
                for (int k = 0; k < PASS_RT; ++k) {
                    uint8_t *at = sm + ((32u * k + r) * CH + (pcs ^ (r % CH))) * 16u + (F32O ? 0u : 8u * h);
                    float v[4];
#pragma unroll
                    for (int x = 0; x < 4; ++x) {
                        v[x] = acc[k0 + k][j][4 * q + x];
                        if (SW) v[x] = silu_p(v[x]) * acc[k0 + k][1][4 * q + x];
                        if constexpr (EPI == GE_VISION) v[x] = vision_act<decltype(ACT)::value>(v[x] + bias[x]);
                    }
                    if constexpr (F32O) {
                        *(float4 *)at = make_float4(v[0], v[1], v[2], v[3]);
                    } else {
                        union {
                            h16 x[4];
                            uint2 u;
                        } o;
                        if (EPI == GE_F16 && p.res != nullptr) {
                            o.u = *(const uint2 *)at;
#pragma unroll
                            for (int x = 0; x < 4; ++x) v[x] += (float)o.x[x];
                        }
#pragma unroll
                        for (int x = 0; x < 4; ++x) o.x[x] = (h16)v[x];
                        *(uint2 *)at = o.u;
                    }
                }
            }
        }
        };
        if (WK == 1 || kg == 0) {
            if constexpr (EPI == GE_VISION) with_act(p.act, put);
            else put(std::integral_constant<u32, UOCR_VISION_ACT_NONE>{});
        }
        __syncthreads();
        if (col < p.N) {
            uint8_t *out = (uint8_t *)p.out;
            u32 c = col, ld = p.ldo;
            if (EPI == GE_VISION && p.split != 0u) {
                const u32 pj = col / p.split;
                out = (uint8_t *)(pj == 0u ? p.out : (pj == 1u ? p.out1 : p.out2));
                c = col - pj * p.split;
                ld = p.split;
            }
#pragma unroll 4
            for (u32 row = t / CH; row < PASS_RT * 32u; row += TT / CH) {
                const u32 rr = 32u * k0 + row;
                if (rr >= rows) break;
                const size_t orow = GROUPED ? (size_t)p.o_idx[s0 + rr] : (size_t)(s0 + rr);
                const uint4 v = *(const uint4 *)(sm + (row * CH + (ch ^ (row % CH % 32u))) * 16u);
                *(uint4 *)(out + (orow * ld + c) * (F32O ? 4u : 2u)) = v;
            }
        }
    }
}

/* One block of a tile grid.  A bucket's last tile of 128 rows takes the body
 * of 32, 64 or 96 rows when that is all it holds (an expert's bucket of a
 * 932-token prompt is about 87 rows). */
template <int QT, int EPI, bool GROUPED, bool PACKED, int RT, int WN, int WK>
__device__ __forceinline__ void tile_block(const GemmArgs &p, u32 id, uint8_t *sm, const RopeDst &rd) {
    u32 bx, by;
    if (!tile_of(id, p.by_row != 0u, GROUPED ? (u32)*p.ntiles : p.nx, p.ny, bx, by)) return;
    if constexpr (GROUPED && RT == 4) {
        const u32 rows = uni((u32)p.tile_s1[bx]) - uni((u32)p.tile_s0[bx]);
        if (rows <= 32u) return tile_body<QT, EPI, GROUPED, PACKED, 1, WN, WK>(p, bx, by, sm, rd);
        if (rows <= 64u) return tile_body<QT, EPI, GROUPED, PACKED, 2, WN, WK>(p, bx, by, sm, rd);
        if (rows <= 96u) return tile_body<QT, EPI, GROUPED, PACKED, 3, WN, WK>(p, bx, by, sm, rd);
    }
    tile_body<QT, EPI, GROUPED, PACKED, RT, WN, WK>(p, bx, by, sm, rd);
}

template <int QT, int EPI, bool GROUPED, bool PACKED, int RT, int WN, int WK>
__global__ __launch_bounds__(64 * WN * WK, 2) void k_gemm_tile(GemmArgs p) {
    __shared__ __attribute__((aligned(1024))) uint8_t sm[tile_lds_bytes<RT, WN, WK>(false)];
    tile_block<QT, EPI, GROUPED, PACKED, RT, WN, WK>(p, blockIdx.x, sm, RopeDst{});
}

/* The Q | K | V projection with RoPE and the cache scatter as its epilogue. */
template <int QT, bool PACKED, int RT, int WN, int WK>
__global__ __launch_bounds__(64 * WN * WK, 2) void k_gemm_tile_rope(GemmArgs p, RopeDst rd) {
    __shared__ __attribute__((aligned(1024))) uint8_t sm[tile_lds_bytes<RT, WN, WK>(true)];
    tile_block<QT, GE_ROPE, false, PACKED, RT, WN, WK>(p, blockIdx.x, sm, rd);
}

/* One of the two GEMMs of a launch: weight type, epilogue, layout and tile. */
template <int QT_, int EPI_, bool GROUPED_, bool PACKED_, int RT_, int WN_, int WK_>
struct Half {
    static constexpr int QT = QT_, EPI = EPI_, RT = RT_, WN = WN_, WK = WK_;
    static constexpr bool GROUPED = GROUPED_, PACKED = PACKED_;
    static constexpr u32 LDS = tile_lds_bytes<RT_, WN_, WK_>(false), CW = (EPI_ == GE_SWIGLU ? 32u : 64u) * WN_;
    static_assert(WN_ * WK_ == 4, "both halves run 256 threads");
    static __device__ __forceinline__ void block(const GemmArgs &p, u32 id, uint8_t *sm) {
        tile_block<QT, EPI, GROUPED, PACKED, RT, WN, WK>(p, id, sm, RopeDst{});
    }
};

/* The router's fp32 logits [M][64] of fp16 rows and weights.  Each logit is one
 * sum over K in steps of 16 in ascending order, as the general kernel forms it:
 * the six experts are chosen from the logits, and another order of the sum picks
 * another expert where the 6th and 7th logit are a rounding apart (K in four
 * partial sums: one row of 1.9 million).  So K cannot be split, and what bounds a
 * block is the latency of its 20 steps: 4 of them are in flight, in lines of 128
 * bytes (64 lanes on 64 rows, straight to registers, took 8.5 us more at 64 rows
 * and above).  A block takes 64 rows, a wavefront 32 rows and 32 experts. */
struct RouterHalf {
    static constexpr u32 ROWS = 64u, CW = UOCR_K_EXPERTS, STAGE = (ROWS + CW) * 128u, RD = 5u, LDS = RD * STAGE;
    static constexpr bool GROUPED = false;
    static __device__ __forceinline__ void block(const GemmArgs &p, u32 id, uint8_t *sm) {
        constexpr int NT = UOCR_K_HIDDEN / 64, NL = (int)(STAGE / 4096u); /* K steps, loads of a wavefront per step */
        static_assert(UOCR_K_EXPERTS == 64, "two wavefronts along the experts");
        const u32 lane = threadIdx.x & 63u, r = lane & 31u, h = lane >> 5, wave = uni(threadIdx.x >> 6);
        const u32 row0 = id * ROWS;
        if (row0 >= p.M) return;
        const u32 lds0 = uni((u32)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)sm) + 2048u * wave;
        /* the wavefront's 16 activation rows and 16 weight rows, swizzled as in tile_body */
        u32 vx[2], vw[2];
#pragma unroll
        for (u32 i = 0; i < 2; ++i) {
            const u32 row = 16u * wave + 8u * i + (lane >> 3), pc = 16u * ((lane & 7u) ^ (row >> 1 & 7u));
            vx[i] = min(row0 + row, p.M - 1u) * p.lda * 2u + pc;
            vw[i] = row * (UOCR_K_HIDDEN * 2u) + pc;
        }
        auto issue = [&](u32 s) {
#pragma unroll
            for (u32 i = 0; i < 2; ++i) {
                lds_load16((const uint8_t *)p.A + 128u * s, vx[i], lds0 + s % RD * STAGE + 1024u * i);
                lds_load16((const uint8_t *)p.W[0].w + 128u * s, vw[i], lds0 + s % RD * STAGE + ROWS * 128u + 1024u * i);
            }
        };
        f32x16 acc;
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[i] = 0.0f;
#pragma unroll
        for (u32 s = 0; s + 1u < RD; ++s) issue(s);
        const uint8_t *xs = sm + 4096u * (wave >> 1) + 128u * r, *ws = sm + ROWS * 128u + 4096u * (wave & 1u) + 128u * r;
        static_for<NT>([&](auto S) {
            constexpr int s = decltype(S)::value, after = NT - 1 - s < (int)RD - 2 ? NT - 1 - s : (int)RD - 2;
            /* step s has landed for all wavefronts; step s - 1's place is free */
            wait_barrier<NL * after>();
            if constexpr (s + (int)RD - 1 < NT) issue(s + RD - 1u);
#pragma unroll
            for (u32 i = 0; i < 4; ++i) {
                const u32 at = s % RD * STAGE + 16u * ((b_koff<1>(i, h) / 8u) ^ (r >> 1 & 7u));
                U4H8 x, w;
                x.u = *(const uint4 *)(xs + at);
                w.u = *(const uint4 *)(ws + at);
                acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(w.v, x.v, acc, 0, 0, 0);
            }
        });
        const u32 row = row0 + 32u * (wave >> 1) + r;
        if (row < p.M) {
            float *o = (float *)p.out + (size_t)row * p.ldo + 32u * (wave & 1u) + 4u * h;
#pragma unroll
            for (int q = 0; q < 4; ++q) *(float4 *)(o + 8 * q) = make_float4(acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]);
        }
    }
};

/* Two GEMMs that do not read each other's output in one launch: blocks [0, na)
 * take A's tiles, the others B's. */
template <typename A, typename B>
__global__ __launch_bounds__(256, 2) void k_gemm_tile_pair(GemmArgs a, u32 na, GemmArgs b) {
    __shared__ __attribute__((aligned(1024))) uint8_t sm[A::LDS > B::LDS ? A::LDS : B::LDS];
    if (blockIdx.x < na) A::block(a, blockIdx.x, sm);
    else B::block(b, blockIdx.x - na, sm);
}

/* ---- narrow tiles, K split over the block's wavefronts ---------------------- */

#define KS_WAVES 8u                     /* wavefronts of a block at most */
#define KS_PLANE (8u * 1040u)           /* bytes of a wavefront's 32 x 64 partials: 8 pieces of 64 float4, padded */

template <int QT, int EPI, bool GROUPED, bool PACKED>
__device__ __forceinline__ void lines_block(const GemmArgs &p, u32 id, uint8_t *ksm) {
    constexpr int NG = groups_per_line<QT>();
    constexpr bool SW = EPI == GE_SWIGLU;
    /* 32 rows (64 measured slower at 32 to 4096 rows) */
    constexpr u32 CW = SW ? 32u : 64u, ROWS = 32u, RB = QT == 4 ? 32u : 64u;
    const u32 t = threadIdx.x, lane = t & 63u, wave = uni(t >> 6), r = lane & 31u, h = lane >> 5, nw = blockDim.x / 64u;
    u32 bx, by;
    if (!tile_of(id, p.by_row != 0u, GROUPED ? (u32)*p.ntiles : p.nx, p.ny, bx, by)) return;
    const u32 n0 = by * CW;
    u32 e = 0, s0 = bx * ROWS, rows;
    if (GROUPED) {
        e = uni((u32)p.tile_e[bx]);
        s0 = uni((u32)p.tile_s0[bx]);
        rows = uni((u32)p.tile_s1[bx]) - s0;
    } else {
        rows = min(ROWS, p.M - s0);
    }
    const u32 K = p.K, NT = K / 64u, NCH = (NT + NG - 1u) / NG;
    const u32 rowb = QT == 4 ? K / 2u : (QT == 3 ? K : 2u * K);
    const uint8_t *pb[2];
    const unsigned short *srow[2];
    u32 vb[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const uocr_qmat &m = SW ? p.W[j] : p.W[0];
        const u32 cb = n0 + (SW ? 0u : 32u * j), row = min(cb + r, p.N - 1u);
        pb[j] = (const uint8_t *)m.w + (GROUPED ? e * p.w_stride : 0);
        if (PACKED) pb[j] += (size_t)min(cb / 32u, p.N / 32u - 1u) * NT * (32u * RB);
        vb[j] = PACKED ? 0u : row * rowb;
        srow[j] = (const unsigned short *)m.s + (GROUPED ? e * p.s_stride : 0) + (size_t)row * NT;
    }
    const u32 ar = GROUPED ? (u32)p.a_idx[s0 + min(r, rows - 1u)] : s0 + min(r, rows - 1u);
    const u32 va = ar * p.lda * 2u + 2u * b_koff<QT>(0u, h);
    u32 bn[2][16], sn[2][NG], bc[2][16], sc[2][NG];
    U4H8 an[4], ac[4];
    /* line c of the lane's two weight rows: its half of every group (past the
     * row's end the last piece again) */
    auto load_b = [&](u32 c) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
#pragma unroll
            for (u32 q = 0; q < 4; ++q) {
                uint4 x;
                if constexpr (PACKED) {
                    const u32 left = (NT - c * NG) * 32u * RB, o = QT == 4 ? 1024u * q : 2048u * (q >> 1);
                    x = *(const uint4 *)(pb[j] + (size_t)c * 4096u + (o < left ? o : 0u) + (QT == 4 ? 16u * lane : 32u * lane + 16u * (q & 1u)));
                } else {
                    const u32 ch = QT == 4 ? 2u * q + h : (QT == 3 ? 4u * (q >> 1) + 2u * h + (q & 1) : 4u * h + q);
                    x = *(const uint4 *)(pb[j] + (vb[j] + min(c * 128u + 16u * ch, rowb - 16u)));
                }
                bn[j][4 * q] = x.x;
                bn[j][4 * q + 1] = x.y;
                bn[j][4 * q + 2] = x.z;
                bn[j][4 * q + 3] = x.w;
            }
            if constexpr (QT != 1) {
#pragma unroll
                for (int g = 0; g < NG; ++g) sn[j][g] = srow[j][min(c * NG + g, NT - 1u)];
            }
        }
    };
    auto load_a = [&](u32 s) {
        const uint8_t *base = (const uint8_t *)p.A + (size_t)s * 128u;
#pragma unroll
        for (u32 i = 0; i < 4; ++i) an[i].u = *(const uint4 *)(base + (va + 2u * b_koff<QT>(i, 0u)));
    };
    f32x16 acc[2];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int x = 0; x < 16; ++x) acc[j][x] = 0.0f;

    if (wave < NCH) {
        load_b(wave);
        load_a(wave * NG);
    }
    for (u32 c = wave; c < NCH; c += nw) {
        const bool more = c + nw < NCH;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
#pragma unroll
            for (int x = 0; x < 16; ++x) bc[j][x] = bn[j][x];
#pragma unroll
            for (int g = 0; g < NG; ++g) sc[j][g] = sn[j][g];
        }
#pragma unroll
        for (int g = 0; g < NG; ++g) {
            const u32 s = c * NG + g;
            if (g > 0 && s >= NT) break;
#pragma unroll
            for (int i = 0; i < 4; ++i) ac[i] = an[i];
            if (g + 1 < NG) load_a(min(s + 1u, NT - 1u));
            if (g == 0 && more) load_b(c + nw);
            if (g + 1 == NG && more) load_a((c + nw) * NG);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    h16x8 wv;
                    if (QT == 4) wv = dequant_q4(bc[j][4 * g + 2 * (i & 1)], bc[j][4 * g + 2 * (i & 1) + 1], (i & 2) != 0, sc[j][g]);
                    else if (QT == 3) wv = dequant_q8(bc[j][(8 * g + 2 * i) & 15], bc[j][(8 * g + 2 * i + 1) & 15], sc[j][g]);
                    else wv = operand_f16(bc[j][4 * i], bc[j][4 * i + 1], bc[j][4 * i + 2], bc[j][4 * i + 3]);
                    acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(wv, ac[i].v, acc[j], 0, 0, 0);
                }
            }
        }
    }

    /* The wavefronts' partials are added in order, 8 columns of a row per
     * thread and turn.  Piece (j, q) of a plane: the four values of row r and
     * half h at 16 (32 h + r). */
    constexpr u32 CH = CW / 8u;
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q)
            *(float4 *)(ksm + wave * KS_PLANE + (4u * j + q) * 1040u + 16u * lane) =
                make_float4(acc[j][4 * q], acc[j][4 * q + 1], acc[j][4 * q + 2], acc[j][4 * q + 3]);
    __syncthreads();
    for (u32 it = t; it < 32u * CH; it += blockDim.x) {
        const u32 row = it / CH, pc = it % CH, col = n0 + 8u * pc;
        if (row >= rows || col >= p.N) continue;
        const size_t orow = GROUPED ? (size_t)p.o_idx[s0 + row] : (size_t)(s0 + row);
        U4H8 rs;
        if (EPI == GE_F16 && p.res != nullptr) rs.u = *(const uint4 *)(p.res + orow * p.ldr + col);
        if (EPI == GE_VISION) rs.u = *(const uint4 *)(p.bias + col);
        float v[8], u[8];
        auto sum = [&](u32 piece, float (&o)[8]) {
            const uint8_t *src = ksm + piece * 1040u + 16u * row;
#pragma unroll
            for (int x = 0; x < 8; ++x) o[x] = 0.0f;
            for (u32 w = 0; w < nw; ++w) {
                const float4 a = *(const float4 *)(src + w * KS_PLANE), b = *(const float4 *)(src + w * KS_PLANE + 512u);
                o[0] += a.x;
                o[1] += a.y;
                o[2] += a.z;
                o[3] += a.w;
                o[4] += b.x;
                o[5] += b.y;
                o[6] += b.z;
                o[7] += b.w;
            }
        };
        sum(pc, v);
        if constexpr (SW) {
            sum(pc + 4u, u);
#pragma unroll
            for (int x = 0; x < 8; ++x) v[x] = silu_p(v[x]) * u[x];
        }
        if constexpr (EPI == GE_F32) {
            float4 *o = (float4 *)((float *)p.out + orow * p.ldo + col);
            o[0] = make_float4(v[0], v[1], v[2], v[3]);
            o[1] = make_float4(v[4], v[5], v[6], v[7]);
            continue;
        }
        h16 *dst = (h16 *)p.out + orow * p.ldo + col;
        if (EPI == GE_VISION && p.split != 0u) {
            const u32 pj = col / p.split;
            dst = (h16 *)(pj == 0u ? p.out : (pj == 1u ? p.out1 : p.out2)) + orow * p.split + (col - pj * p.split);
        }
        U4H8 o;
        if constexpr (EPI == GE_VISION) {
            with_act(p.act, [&](auto ACT) {
#pragma unroll
                for (int x = 0; x < 8; ++x) v[x] = vision_act<decltype(ACT)::value>(v[x] + (float)rs.h[x]);
            });
        }
#pragma unroll
        for (int x = 0; x < 8; ++x) {
            if (EPI == GE_F16 && p.res != nullptr) v[x] += (float)rs.h[x];
            o.h[x] = (h16)v[x];
        }
        *(uint4 *)dst = o.u;
    }
}

template <int QT, int EPI, bool GROUPED, bool PACKED>
__global__ __launch_bounds__(64u * KS_WAVES) void k_gemm_lines(GemmArgs p) {
    extern __shared__ __attribute__((aligned(16))) uint8_t ksm[];
    lines_block<QT, EPI, GROUPED, PACKED>(p, blockIdx.x, ksm);
}

template <int QT, int EA, int EB, bool PACKED>
__global__ __launch_bounds__(64u * KS_WAVES) void k_gemm_lines_pair(GemmArgs a, u32 na, GemmArgs b) {
    extern __shared__ __attribute__((aligned(16))) uint8_t ksm[];
    if (blockIdx.x < na) lines_block<QT, EA, false, PACKED>(a, blockIdx.x, ksm);
    else lines_block<QT, EB, true, PACKED>(b, blockIdx.x - na, ksm);
}

/* The launch's blocks and the order of its tiles. */
dim3 tile_grid(GemmArgs &a, u32 row_tiles, u32 col_tiles, u32 qt, bool grouped) {
    a.nx = row_tiles;
    a.ny = col_tiles;
    const uint64_t wb = (uint64_t)a.N * a.K * (qt == UOCR_QT_F16 ? 4u : (qt == UOCR_QT_Q8 ? 2u : 1u)), ab = (uint64_t)a.M * a.K * 4u;
    a.by_row = grouped || ab > wb ? 1u : 0u;
    return dim3((row_tiles * col_tiles + 7u) / 8u * 8u);
}

/* Wavefronts per block: as many lines of 128 bytes each, at most KS_WAVES. */
u32 lines_waves(u32 qt, u32 K) {
    const u32 ng = qt == UOCR_QT_Q4 ? 4u : (qt == UOCR_QT_Q8 ? 2u : 1u), nch = (K / 64u + ng - 1u) / ng;
    const u32 per = (nch + KS_WAVES - 1u) / KS_WAVES;
    return (nch + per - 1u) / per;
}

template <int EPI, bool GROUPED>
hipError_t launch_lines(hipStream_t st, u32 qt, GemmArgs a, u32 row_tiles) {
    const u32 nw = lines_waves(qt, a.K), cw = EPI == GE_SWIGLU ? 32u : 64u;
    const dim3 grid = tile_grid(a, row_tiles, (a.N + cw - 1u) / cw, qt, GROUPED);
#define GO(Q, PK) hipLaunchKernelGGL((k_gemm_lines<Q, EPI, GROUPED, PK>), grid, dim3(64u * nw), nw * KS_PLANE, st, a)
    if (qt == UOCR_QT_F16) GO(1, false);
    else if (qt == UOCR_QT_Q8 && a.packed) GO(3, true);
    else if (qt == UOCR_QT_Q8) GO(3, false);
    else if (a.packed) GO(4, true);
    else GO(4, false);
#undef GO
    return hipGetLastError();
}

template <int EPI, bool GROUPED, int RT, int WN, int WK>
hipError_t launch(hipStream_t st, u32 qt, GemmArgs a, u32 row_tiles) {
    const u32 cw = (EPI == GE_SWIGLU ? 32u : 64u) * WN;
    const dim3 grid = tile_grid(a, row_tiles, (a.N + cw - 1u) / cw, qt, GROUPED);
#define GO(Q, PK) hipLaunchKernelGGL((k_gemm_tile<Q, EPI, GROUPED, PK, RT, WN, WK>), grid, dim3(64 * WN * WK), 0, st, a)
    if (qt == UOCR_QT_F16) GO(1, false);
    else if (qt == UOCR_QT_Q8 && a.packed) GO(3, true);
    else if (qt == UOCR_QT_Q8) GO(3, false);
    else if (a.packed) GO(4, true);
    else GO(4, false);
#undef GO
    return hipGetLastError();
}

template <int RT, int WN, int WK>
hipError_t plain(hipStream_t st, int epi, u32 qt, const GemmArgs &a) {
    const u32 tiles = (a.M + 32u * RT - 1u) / (32u * RT);
    switch (epi) {
        case GE_F16: return launch<GE_F16, false, RT, WN, WK>(st, qt, a, tiles);
        case GE_VISION: return launch<GE_VISION, false, RT, WN, WK>(st, qt, a, tiles);
        case GE_SWIGLU: return launch<GE_SWIGLU, false, RT, WN, WK>(st, qt, a, tiles);
        default: return hipErrorInvalidValue;
    }
}

hipError_t plain_lines(hipStream_t st, int epi, u32 qt, const GemmArgs &a) {
    const u32 tiles = (a.M + 31u) / 32u;
    switch (epi) {
        case GE_F16: return launch_lines<GE_F16, false>(st, qt, a, tiles);
        case GE_VISION: return launch_lines<GE_VISION, false>(st, qt, a, tiles);
        case GE_SWIGLU: return launch_lines<GE_SWIGLU, false>(st, qt, a, tiles);
        default: return hipErrorInvalidValue;
    }
}

/* Which kernel a plain GEMM of M x N (SwiGLU: N pairs) x K takes, by the blocks
 * of its grids (large, mid, narrow: tiles of 128 x 256, 64 x 128, 32 x 64).  A K
 * step of a block takes 0.6-0.9 us whatever it computes (its loads' latency):
 *  - the large tile, the cheapest per output, once the mid grid is over its two
 *    blocks per CU;
 *  - up to a narrow block per CU, K split over the block's wavefronts: by lines
 *    while a line holds several K steps, in 8 groups for long sums;
 *  - else the mid tile, K in 2 groups, or in 4 where the sums are long and each
 *    block has a CU of its own (at 1280 the groups' merge costs more: 932 x 1280
 *    x 1280 13.9 -> 14.5).  Q4 lines hold 4 K steps, so K by lines stays the
 *    better one there for another half a round.
 * The general kernel (64 x 128, K split over blocks for long vision sums) is
 * the better one for vision linears
 *  - with long sums on so few rows that its K splits are what fills the CUs, and,
 *    for quantised weights, between a narrow block per CU and 100 mid tiles;
 *  - with Q4 weights and an activation at up to one and a half rounds: its
 *    weights skip LDS and all its wavefronts share the epilogue;
 * and for plain Q4 GEMMs from 513 to 768 mid tiles, where three of its blocks fit
 * a CU and large tiles leave a quarter of the CUs and more idle: 1-6% over K from
 * 64 to 6848; above, in its second round, it is 10-25% slower from K = 256 on.
 * Measured (us): general / large / mid, K in 2 / in 4 / narrow, K in 8 / lines
 *   Q8   3500 x 1280 x 6848   123  /  97  / 118  / 128  / 200  / 229    550 mid
 *   Q8   2000 x 1280 x 6848   78.7 / 93.9 / 65.8 / 85.2 / 113  / 130    320
 *   Q4   3584 x 1280 x 1280   23.7 / 24.4                               560
 *   Q4   3600 x 1280 x 6848   114  / 118     (in a prompt)              570
 *   Q4   4928 x 1280 x 1280   33.9 / 27.3                               770
 *   Q8    932 x 1280 x 6848   68.9 / 94.5 / 46.9 / 41.5                 150
 *   F16   500 x 1280 x 6848   52.3 / 92.4 / 45.6 / 39.9 / 43.1 / 74.5   320 narrow
 *   Q8    257 x 1280 x 6848   67.5 / 94.7 / 46.3 / 41.5 / 23.4 / 28.3   180
 *   Q4    500 x 1280 x 1280   16.2 / 25.1 / 12.8 / 12.8 / 16.7 / 12.2   320
 *   Q8    500 x 1280 x 1280   16.9 / 23.6 / 11.9 / 11.7 / 15.8 / 15.0   320
 *   Q4    257 x 1280 x 1280   16.2 / 25.0 / 12.7 / 12.6 /  9.1 /  7.3   180
 *   F16   257 x 1280 x 1792   23.0 / 26.3 / 11.7 / 12.0 /  8.3 / 12.6   180
 *  vision:
 *   Q8   1960 x 2304 x 768    20.0 / 16.7 / 18.7 / 25.8                 558 mid
 *   Q8   1600 x 768 x 768     10.9 / 15.1 /  8.9 /  9.5 / 18.5 / 13.6   150
 *   Q4   1600 x 3072 x 768    19.8 / 21.1 / 23.6   (GELU)               600
 *   Q4   1176 x 3072 x 768    15.3 / 20.5 / 15.9   (GELU)               456
 *   Q4    514 x 1024 x 4096   21.8 / 60.6 / 28.6 / 26.3 / 29.8 / 32.4   272 narrow
 *   F16   514 x 1024 x 4096   25.4 / 55.6 / 26.6 / 23.9 / 24.9 / 41.6   272
 *   Q8    257 x 1024 x 4096   17.5 / 57.1 / 26.3 / 24.4 / 14.8 / 21.1   144
 *   Q4    300 x 768 x 3072    13.1 /                      14.2          120
 *   Q4    101 x 1024 x 4096   12.1 / 60.0 / 28.6 / 26.4 / 15.7 / 17.2    64 */
int choose(int epi, u32 qt, u32 M, u32 N, u32 K, u32 act) {
    const u32 n2 = epi == GE_SWIGLU ? 2u * N : N;
    const u32 mid = ((M + 63u) / 64u) * ((n2 + 127u) / 128u), narrow = ((M + 31u) / 32u) * ((n2 + 63u) / 64u);
    if (epi == GE_VISION) {
        if (K >= 2048u && (narrow < (qt == UOCR_QT_Q4 ? 128u : 100u) || (qt != UOCR_QT_F16 && narrow > 256u && mid < 100u))) return UOCR_GEMM_KERNEL_GENERAL;
        if (qt == UOCR_QT_Q4 && act != UOCR_VISION_ACT_NONE && K <= 1024u && mid > 256u && mid <= 768u) return UOCR_GEMM_KERNEL_GENERAL;
    }
    if (epi == GE_F16 && qt == UOCR_QT_Q4 && mid > 512u && mid <= 768u) return UOCR_GEMM_KERNEL_GENERAL;
    if (mid > 512u) return UOCR_GEMM_KERNEL_LARGE;
    if (narrow <= 256u) return K >= (qt == UOCR_QT_F16 ? 1280u : 3072u) ? UOCR_GEMM_KERNEL_NARROW : UOCR_GEMM_KERNEL_LINES;
    if (qt == UOCR_QT_Q4 && K < 3072u && narrow <= 384u) return UOCR_GEMM_KERNEL_LINES;
    return K >= 3072u && mid <= 256u ? UOCR_GEMM_KERNEL_MID_K4 : UOCR_GEMM_KERNEL_MID;
}

}  // namespace

bool uocr_gemm_tile_fits(int epi, u32 qt, const GemmArgs &a) {
    const uint64_t rowb = qt == UOCR_QT_Q4 ? a.K / 2u : (qt == UOCR_QT_Q8 ? a.K : 2ull * a.K), lim = 1ull << 32;
    uintptr_t al = (uintptr_t)a.A | (uintptr_t)a.W[0].w | (epi == GE_SWIGLU ? (uintptr_t)a.W[1].w : 0u);
    /* a plain fp32 GEMM is the router's: its sums keep their order (RouterHalf, or the general kernel) */
    const bool known = epi == GE_F16 || (epi == GE_F32 && a.tile_e != nullptr) || epi == GE_SWIGLU || epi == GE_VISION;
    return a.vec != 0u && known && a.nseg == 0u && al % 16u == 0u &&
           (uint64_t)a.M * a.lda * 2u < lim && (uint64_t)a.M * a.ldr * 2u < lim && a.N * rowb < lim && (!a.packed || a.N % 32u == 0u);
}

bool uocr_gemm_tile_takes(int epi, u32 qt, const GemmArgs &a) {
    return uocr_gemm_tile_fits(epi, qt, a) && choose(epi, qt, a.M, a.N, a.K, a.act) != UOCR_GEMM_KERNEL_GENERAL;
}

bool uocr_gemm_router_fits(const GemmArgs &a) {
    const uintptr_t al = (uintptr_t)a.A | (uintptr_t)a.W[0].w;
    return a.vec != 0u && a.tile_e == nullptr && a.nseg == 0u && a.res == nullptr && a.N == UOCR_K_EXPERTS && a.K == UOCR_K_HIDDEN && al % 16u == 0u &&
           (uint64_t)a.M * a.lda * 2u < 1ull << 32;
}

hipError_t uocr_gemm_tile_rope(hipStream_t st, u32 qt, GemmArgs a, const RopeDst &rd) {
    /* 932 rows: 64 x 128 tiles, K in 2 (450 blocks); over two of them per CU
     * large tiles (a head pair per tile) */
    const bool large = choose(GE_ROPE, qt, a.M, a.N, a.K, 0u) == UOCR_GEMM_KERNEL_LARGE;
    const dim3 grid = tile_grid(a, (a.M + (large ? 127u : 63u)) / (large ? 128u : 64u), a.N / (large ? 256u : 128u), qt, false);
#define GO(Q, PK)                                                                                                      \
    do {                                                                                                               \
        if (large) hipLaunchKernelGGL((k_gemm_tile_rope<Q, PK, 4, 4, 1>), grid, dim3(256), 0, st, a, rd);              \
        else hipLaunchKernelGGL((k_gemm_tile_rope<Q, PK, 2, 2, 2>), grid, dim3(256), 0, st, a, rd);                    \
    } while (0)
    if (qt == UOCR_QT_F16) GO(1, false);
    else if (qt == UOCR_QT_Q8 && a.packed) GO(3, true);
    else if (qt == UOCR_QT_Q8) GO(3, false);
    else if (a.packed) GO(4, true);
    else GO(4, false);
#undef GO
    return hipGetLastError();
}

/* Row tiles of a grouped launch at most: a bucket's last tile may be partial. */
static u32 grouped_tiles(u32 pairs, u32 tile_rows) {
    const u32 t = pairs / tile_rows + UOCR_K_EXPERTS;
    return t < pairs ? t : pairs;
}

u32 uocr_gemm_grouped_rows(u32 pairs, u32 table) {
    /* whole MoE of P rows (us, 128-row tiles / weight lines): Q4 P = 2: 56 / 43,
     * 9: 67 / 66, 23: 77 / 86; Q8 2: 55 / 47, 9: 75 / 84 */
    return pairs <= 36u && grouped_tiles(pairs, 32u) <= table ? 32u : 128u;
}

hipError_t uocr_gemm_tile_grouped(hipStream_t st, int epi, u32 qt, const GemmArgs &a, u32 pairs, u32 rows) {
    const u32 tiles = grouped_tiles(pairs, rows);
#define GO(E) return rows == 32u ? launch_lines<E, true>(st, qt, a, tiles) : launch<E, true, 4, 4, 1>(st, qt, a, tiles)
    switch (epi) {
        case GE_F16: GO(GE_F16);
        case GE_F32: GO(GE_F32);
        case GE_SWIGLU: GO(GE_SWIGLU);
        default: return hipErrorInvalidValue;
    }
#undef GO
}

namespace {

template <typename A, typename B>
void launch_halves(hipStream_t st, u32 qa, GemmArgs a, u32 ta, u32 qb, GemmArgs b, u32 tb) {
    const dim3 ga = tile_grid(a, ta, (a.N + A::CW - 1u) / A::CW, qa, A::GROUPED);
    const dim3 gb = tile_grid(b, tb, (b.N + B::CW - 1u) / B::CW, qb, B::GROUPED);
    hipLaunchKernelGGL((k_gemm_tile_pair<A, B>), dim3(ga.x + gb.x), dim3(256), 0, st, a, ga.x, b);
}

/* The plain GEMM a, EPI GE_F16, beside the grouped b. */
template <int EB>
hipError_t launch_pair(hipStream_t st, u32 qt, GemmArgs a, GemmArgs b, u32 pairs, u32 rows) {
    const u32 tiles = grouped_tiles(pairs, rows), ta = (a.M + 63u) / 64u;
    if (rows == 32u) {
        const u32 wa = lines_waves(qt, a.K), wb = lines_waves(qt, b.K), nw = wa > wb ? wa : wb;
        const dim3 ga = tile_grid(a, (a.M + 31u) / 32u, (a.N + 63u) / 64u, qt, false), gb = tile_grid(b, tiles, (b.N + 63u) / 64u, qt, true);
#define GO(Q, PK) hipLaunchKernelGGL((k_gemm_lines_pair<Q, GE_F16, EB, PK>), dim3(ga.x + gb.x), dim3(64u * nw), nw * KS_PLANE, st, a, ga.x, b)
        if (qt == UOCR_QT_F16) GO(1, false);
        else if (qt == UOCR_QT_Q8 && a.packed) GO(3, true);
        else if (qt == UOCR_QT_Q8) GO(3, false);
        else if (a.packed) GO(4, true);
        else GO(4, false);
#undef GO
        return hipGetLastError();
    }
#define GO(Q, PK) launch_halves<Half<Q, GE_F16, false, PK, 2, 2, 2>, Half<Q, EB, true, PK, 4, 4, 1>>(st, qt, a, ta, qt, b, tiles)
    if (qt == UOCR_QT_F16) GO(1, false);
    else if (qt == UOCR_QT_Q8 && a.packed) GO(3, true);
    else if (qt == UOCR_QT_Q8) GO(3, false);
    else if (a.packed) GO(4, true);
    else GO(4, false);
#undef GO
    return hipGetLastError();
}

}  // namespace

hipError_t uocr_gemm_tile_pair(hipStream_t st, int eb, u32 qt, const GemmArgs &a, const GemmArgs &b, u32 pairs, u32 rows) {
    return eb == GE_F16 ? launch_pair<GE_F16>(st, qt, a, b, pairs, rows) : launch_pair<GE_F32>(st, qt, a, b, pairs, rows);
}

hipError_t uocr_gemm_tile_router(hipStream_t st, u32 qt, const GemmArgs &a, const GemmArgs &b) {
    const u32 ta = (a.M + 63u) / 64u, tb = (b.M + RouterHalf::ROWS - 1u) / RouterHalf::ROWS;
    /* the router first: its blocks are the longest chains of the launch */
#define GO(Q, PK) launch_halves<RouterHalf, Half<Q, GE_SWIGLU, false, PK, 2, 2, 2>>(st, UOCR_QT_F16, b, tb, qt, a, ta)
    if (qt == UOCR_QT_F16) GO(1, false);
    else if (qt == UOCR_QT_Q8 && a.packed) GO(3, true);
    else if (qt == UOCR_QT_Q8) GO(3, false);
    else if (a.packed) GO(4, true);
    else GO(4, false);
#undef GO
    return hipGetLastError();
}

hipError_t uocr_gemm_tile_plain(hipStream_t st, int epi, u32 qt, const GemmArgs &a) {
    switch (choose(epi, qt, a.M, a.N, a.K, a.act)) {
        case UOCR_GEMM_KERNEL_LARGE: return plain<4, 4, 1>(st, epi, qt, a);
        case UOCR_GEMM_KERNEL_MID: return plain<2, 2, 2>(st, epi, qt, a);
        case UOCR_GEMM_KERNEL_MID_K4: return plain<2, 2, 4>(st, epi, qt, a);
        case UOCR_GEMM_KERNEL_NARROW: return plain<1, 1, 8>(st, epi, qt, a);
        default: return plain_lines(st, epi, qt, a);
    }
}

extern "C" int uocr_gemm_kernel_choice(uint32_t qtype, uint32_t M, uint32_t N, uint32_t K, int vision, uint32_t act) {
    return choose(vision ? GE_VISION : GE_F16, qtype, M, N, K, act);
}
