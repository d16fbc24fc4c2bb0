/*
 * Batched products in the exact w64 order, on the fp32 matrix units.
 *
 * The order (k3_rocm_mxfp4_gemv_bf16, k3_rocm_q8_128_gemv_bf16): a row's
 * 32-column groups g belong to partial l = g % 64; a group sum gs is an fmaf
 * chain over its columns from +0, partial_l = fmaf(gs, scale_g, partial_l)
 * with a partial's groups in ascending order, and the 64 partials meet in the
 * butterfly 32, 16, .. 1. V_MFMA_F32_4X4X1_16B_F32 is one rounded fmaf per
 * output (K = 1), so chaining it through C over a group's columns is that
 * chain, bit for bit, for 64 weight rows x 4 tokens per instruction: 32
 * multiply-adds per cycle and SIMD where the vector unit has 16, and one
 * conversion of a weight serves every token.
 *
 * A block computes 64 weight rows (B: lane = row) x up to 16 tokens (A: lane
 * = 4 column + token, broadcast to all 16 blocks of the instruction). The
 * rows' bytes pass through a ring of LDS stages (256 or 512 bytes of each
 * row, whole lines, direct-to-LDS) shared by the eight waves: wave w takes
 * the groups with l % 8 == w, so butterfly levels 32 .. 8 stay in the wave's
 * registers (8 partials per output) and only levels 4 .. 1 cross the waves,
 * through LDS at the end. Token columns come straight from memory (L1/L2)
 * into the A registers, one stage ahead; the rows' scales are staged in LDS.
 *
 * What bounds it: matrix and vector instructions of a SIMD take turns (they
 * do not overlap, measured at two and four waves per SIMD), so a group of 64
 * rows costs 8.1 cycles per MFMA plus its conversions and sums. Per group and
 * SIMD, operands in registers: one quad of tokens 195 ns, two 300, four 545
 * (124 TFLOP/s; Q8-128 614). Measured on the vector units before and here:
 * K3 layer of 333 tokens 19.6 -> 8.0 ms, of 5 tokens 732 -> 403 us (both with
 * the router's logits, 28 -> 10 us at 5); one expert's 77 rows 326 -> 93 us;
 * Q8-128 6144 x 7168 at 300 tokens 1.50 -> 0.39 ms.
 */
#include "k3_device.h"
#include "k3_exact.h"
#include "k3_exact_rule.h"
#include "k3_lds.h"

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

namespace k3 {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr uint32_t kRows = 64;         /* weight rows of a block */
constexpr uint32_t W = 8;              /* waves of a block */
constexpr uint32_t kRing = 3;          /* LDS stages */
constexpr uint32_t kScaleGroups = 256; /* groups whose scales are staged together */

typedef const __attribute__((address_space(4))) uint32_t *ScalarWords;

struct Mx4 { /* e2m1 codes, E8M0 scale per group */
    static constexpr int kGroupBytes = 16;
};
struct Q8 { /* int8 codes, f32 scale per four groups: as many scale bytes as groups */
    static constexpr int kGroupBytes = 32;
};

/* Weight rows of a block, 0 .. 31 from w[0] and 32 .. 63 from w[1] (two
 * matrices for gate/up), scales likewise. Rows past the matrix (whole ==
 * false) repeat the half's last one and are not stored. */
struct BlockRows {
    const uint8_t *w[2], *s[2];
    uint32_t last[2];
    bool whole;
    __device__ __forceinline__ uint32_t row(uint32_t r) const { /* of its half */
        const uint32_t q = r & 31u, end = r < 32u ? last[0] : last[1];
        return whole || q < end ? q : end;
    }
};

/* 16 bytes a lane into consecutive LDS from a wave-uniform LDS address (a
 * number: from a pointer the compiler tests it for null at every use). */
__device__ __forceinline__ void dma16(const uint8_t *src, uint32_t lds) {
    __builtin_amdgcn_global_load_lds((const void *)src, (lds_void *)(uintptr_t)lds, 16, 0, 0);
}

/* What a block carries from one tile to the next. */
struct Pipe {
    uint32_t lds;  /* LDS address of the ring, then two scale buffers */
    uint32_t slot; /* ring slot of the tile's stage 0 */
    uint32_t buf;  /* its scale buffer */
    bool primed;   /* stages 0 and 1 and the scales are on their way */
};

/* RB weight rows (64 or 16; the lanes hold them 64 / RB times, each for token
 * quads of its own) against NT x 64 / RB quads of tokens on the matrix units
 * and NV more tokens on the vector unit (RB = 64); SB bytes of each weight
 * row per stage. */
template <class Fmt, int NT, int NV, int SB, int RB>
struct Core {
    static constexpr int kQuads = 64 / RB;             /* token quads of an instruction */
    static constexpr int kTokens = 4 * kQuads * NT + NV;
    static constexpr int kSG = SB / Fmt::kGroupBytes;  /* groups of a stage */
    static constexpr int kGW = kSG / (int)W;           /* of them, a wave's */
    static constexpr int kSP = 64 / kSG;               /* stages until l repeats */
    static constexpr int kC = 128 * kGW / RB;          /* columns a lane holds of a stage */
    static constexpr int kLG = RB / 4 / kGW;           /* lanes (per token) of a group */
    static constexpr int kCbsz = RB == 64 ? 4 : 2;     /* RB / 4 blocks share an A block */
    static constexpr int kNA = 64 / (int)W;            /* partials of a wave per output */
    static constexpr int kDma = RB * SB / 8192;        /* DMA instructions of a wave per stage */
    static constexpr uint32_t kDmaRows = 1024 / SB;    /* rows of one of them */
    static constexpr int kPieces = Fmt::kGroupBytes / 16;
    static constexpr uint32_t kStage = RB * SB;
    static constexpr uint32_t kScaleBytes = RB * kScaleGroups;
    static constexpr int MT = NT ? NT : 1, MV = NV ? NV : 1;

    struct Rows { /* token rows: the lane's of each quad, and the wave-uniform ones */
        const uint16_t *quad[MT];
        const uint16_t *one[MV];
    };
    struct Result {
        f32x4 quad[MT];
        float one[MV];
    };
    struct Columns { /* one lane's token columns of a stage */
        uint32_t d[MT][kC / 2];
    };
    struct Acc {
        f32x4 quad[MT][kNA];
        float one[MV][kNA];
    };

    static __device__ __forceinline__ void load_x(Columns &v, const Rows &X, uint32_t off) {
#pragma unroll
        for (int t = 0; t < NT; t++) {
            if constexpr (kC >= 8) {
#pragma unroll
                for (int i = 0; i < kC / 8; i++) {
                    const uint4 q = ((const uint4 *)(X.quad[t] + off))[i];
                    v.d[t][4 * i] = q.x; v.d[t][4 * i + 1] = q.y;
                    v.d[t][4 * i + 2] = q.z; v.d[t][4 * i + 3] = q.w;
                }
            } else if constexpr (kC == 4) {
                const uint2 q = *(const uint2 *)(X.quad[t] + off);
                v.d[t][0] = q.x; v.d[t][1] = q.y;
            } else {
                v.d[t][0] = *(const uint32_t *)(X.quad[t] + off);
            }
        }
    }
    /* Pinned between the step's wait and the next loads, which take x's
     * registers: a use elsewhere would drain the DMA or cost copies. */
    static __device__ __forceinline__ void unpack_x(float (&a)[MT][kC], Columns &x) {
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int i = 0; i < kC / 2; i++) asm volatile("" : "+v"(x.d[t][i]));
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int i = 0; i < kC / 2; i++) {
                a[t][2 * i] = bf16_lo(x.d[t][i]);
                a[t][2 * i + 1] = bf16_hi(x.d[t][i]);
                asm volatile("" : "+v"(a[t][2 * i]), "+v"(a[t][2 * i + 1]) : : "memory");
            }
    }

    /* columns 8 D .. 8 D + 7 of the group as fp32 */
    template <int D>
    static __device__ __forceinline__ void weights8(float (&b)[8], const u32x4_t (&p)[kPieces]) {
        if constexpr (std::is_same<Fmt, Mx4>::value) {
            const float2 v0 = fp4x2<0>(p[0][D]), v1 = fp4x2<1>(p[0][D]);
            const float2 v2 = fp4x2<2>(p[0][D]), v3 = fp4x2<3>(p[0][D]);
            b[0] = v0.x; b[1] = v0.y; b[2] = v1.x; b[3] = v1.y;
            b[4] = v2.x; b[5] = v2.y; b[6] = v3.x; b[7] = v3.y;
        } else {
#pragma unroll
            for (int i = 0; i < 8; i++)
                b[i] = (float)(int8_t)(p[D >> 1][2 * (D & 1) + i / 4] >> (8 * (i & 3)));
        }
    }
    static __device__ __forceinline__ float scale(uint32_t raw) {
        /* e8m0_to_f32 in one instruction: 2^-127 2^raw, +inf at 255 */
        if constexpr (std::is_same<Fmt, Mx4>::value)
            return __builtin_amdgcn_ldexpf(__uint_as_float(0x00400000u), (int)raw);
        else return __uint_as_float(raw);
    }

    template <class Fn, int... Is>
    static __device__ __forceinline__ bool period(Fn &&f, uint32_t s,
                                                  std::integer_sequence<int, Is...>) {
        return (f(s + (uint32_t)Is, std::integral_constant<int, Is>{}) && ...);
    }

    /* Whole rows' scales, contiguous bytes per half. */
    static __device__ __forceinline__ void fetch_scales(uint32_t sc, const BlockRows &R,
                                                        uint32_t G, uint32_t w, uint32_t L) {
        constexpr uint32_t kHalf = RB < 32 ? RB : 32; /* rows from s[0] */
        const uint32_t half = kHalf * G / 16u, all = RB * G / 16u;
        for (uint32_t i = 64u * w; i < all; i += 64u * W) {
            uint32_t p = i + L;
            p = p < all ? p : all - 1u;
            dma16(p < half ? R.s[0] + 16u * p : R.s[1] + 16u * (p - half), sc + 16u * i);
        }
    }

    /* The wave's levels 32 .. W of the lane's weight row, per token; the last
     * steps fetch the first stages of the block's next tile (more). */
    static __device__ __forceinline__ void run(Result &out, Pipe &pipe, const BlockRows &R,
                                               const Rows &X, uint32_t G, bool more,
                                               const BlockRows &N) {
        const uint32_t tid = threadIdx.x, L = tid & 63u;
        const uint32_t w = __builtin_amdgcn_readfirstlane(tid >> 6);
        const uint32_t rbytes = G * Fmt::kGroupBytes;
        /* DMA: instruction m of a wave fills kDmaRows rows of the stage from
         * row kDmaRows (w + W m) on, a row's pieces in consecutive lanes;
         * slot p of row r holds the row's piece p ^ (r % 16), so 16 lanes
         * reading one piece of 16 rows touch every bank once */
        constexpr uint32_t kRowPieces = SB / 16;
        const uint32_t dr = kDmaRows * w + L / kRowPieces;
        const uint32_t dp = (L % kRowPieces) ^ (dr & 15u);
        /* the lane's offset from its half's first row; in a partial last stage
         * the pieces past the row's end repeat its last one */
        uint32_t voff[kDma], vend[kDma];
        const uint32_t pieces = rbytes / 16u, rest = pieces % kRowPieces;
        const uint32_t whole = pieces / kRowPieces;
#pragma unroll
        for (int m = 0; m < kDma; m++) {
            voff[m] = R.row(dr + kDmaRows * W * (uint32_t)m) * rbytes + 16u * dp;
            vend[m] = dp < rest ? voff[m] : voff[m] - 16u * (dp + 1u - rest);
        }
        const uint32_t ring = __builtin_amdgcn_readfirstlane(pipe.lds);
        /* no branches: the waits on the token columns count these loads */
        auto fetch = [&](const uint8_t *w0, const uint8_t *w1, uint32_t s, uint32_t slot) {
            const uint32_t dst = ring + kStage * slot + 1024u * w;
            const bool last = s == whole;
#pragma unroll
            for (int m = 0; m < kDma; m++)
                dma16((m * kDmaRows * W >= 32u ? w1 : w0) + (uint64_t)s * SB +
                          (last ? vend[m] : voff[m]),
                      dst + 1024u * W * m);
        };
        /* A: lane 4 c + i (of RB lanes) holds kC columns of token i: of the
         * wave's group c / kLG, columns kC (c % kLG) .. */
        const uint32_t c = (L % RB) >> 2;
        const uint32_t xgroup = w + W * (c / (uint32_t)kLG);
        const uint32_t xoff = 32u * xgroup + kC * (c % (uint32_t)kLG);
        auto xat = [&](uint32_t s) { /* groups past the row are not used */
            return (uint32_t)kSG * s + xgroup < G ? 32u * (uint32_t)kSG * s + xoff : 0u;
        };
        Acc acc;
#pragma unroll
        for (int a = 0; a < kNA; a++) {
#pragma unroll
            for (int t = 0; t < NT; t++) acc.quad[t][a] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int t = 0; t < NV; t++) acc.one[t][a] = 0.0f;
        }
        /* LDS offsets of the wave's groups in the lane's row of a stage */
        uint32_t at[kGW][kPieces];
#pragma unroll
        for (int q = 0; q < kGW; q++)
#pragma unroll
            for (int i = 0; i < kPieces; i++)
                at[q][i] = ring + SB * (L % RB) +
                           (((kPieces * (w + W * (uint32_t)q) + (uint32_t)i) ^ (L & 15u)) << 4);
        for (uint32_t g0 = 0; g0 < G; g0 += kScaleGroups) {
            const uint32_t gn = G - g0 < kScaleGroups ? G - g0 : kScaleGroups;
            const uint32_t s_end = (g0 + gn + kSG - 1u) / kSG, s_begin = g0 / kSG;
            const uint32_t sc = ring + kRing * kStage + kScaleBytes * pipe.buf;
            if (!pipe.primed) {
                wait_vm<0>();
                __syncthreads(); /* the last reads of what is filled now are done */
                if (G <= kScaleGroups && R.whole) {
                    fetch_scales(sc, R, G, w, L);
                } else {
                    const uint32_t r = L % RB;
                    const uint8_t *row = (r < 32u ? R.s[0] : R.s[1]) + (uint64_t)R.row(r) * G + g0;
#pragma unroll 1
                    for (uint32_t i = w; i < gn; i += W)
                        *(__attribute__((address_space(3))) uint8_t *)(uintptr_t)(sc + gn * r + i) =
                            row[i];
                    __syncthreads();
                }
                fetch(R.w[0], R.w[1], s_begin, pipe.slot);
                const uint32_t s1 = pipe.slot == kRing - 1u ? 0u : pipe.slot + 1u;
                fetch(R.w[0], R.w[1], s_begin + 1u < s_end ? s_begin + 1u : s_begin, s1);
            }
            pipe.primed = false;
            const uint32_t sc_lds = sc + gn * (L % RB) + w;
            Columns xs;
            load_x(xs, X, xat(s_begin));
            wait_vm<0>(); /* here, so that the loop's own waits need not drain */
            uint32_t slot = __builtin_amdgcn_readfirstlane(pipe.slot);
            auto step = [&](uint32_t s, auto SM) { /* false after the last stage */
                /* only the next stage's DMA stays in flight */
                wait_vm<kDma>();
                asm volatile("" ::: "memory");
                __builtin_amdgcn_s_barrier();
                asm volatile("" ::: "memory");
                float a[MT][kC]; /* the stage's token columns as fp32 */
                unpack_x(a, xs);
                load_x(xs, X, xat(s + 1u));
                asm volatile("" ::: "memory");
                const uint32_t f = s + 2u, fslot = slot >= 1u ? slot - 1u : kRing - 1u;
                /* after the last stage: the next tile's scales and stages 0
                 * and 1, or (none) any stage into the free slot */
                if (f == s_end && more)
                    fetch_scales(ring + kRing * kStage + kScaleBytes * (pipe.buf ^ 1u), N, G, w, L);
                const bool cur = f < s_end, nxt = !cur && more;
                fetch(nxt ? N.w[0] : R.w[0], nxt ? N.w[1] : R.w[1],
                      cur ? f : nxt ? f - s_end : s_begin, fslot);
                asm volatile("" ::: "memory");
                stage<(int)SM>(acc, a, X, at, kStage * slot, sc_lds, w, (uint32_t)kSG * s, g0, G);
                slot = slot == kRing - 1u ? 0u : slot + 1u;
                return s + 1u < s_end;
            };
            uint32_t s = s_begin;
            while (period(step, s, std::make_integer_sequence<int, kSP>{})) s += kSP;
            pipe.slot = slot;
        }
        pipe.primed = more;
        pipe.buf ^= 1u;
        /* butterfly levels 32 .. W: partial a of the wave is l = W a + w */
#pragma unroll
        for (int h = kNA / 2; h >= 1; h /= 2)
#pragma unroll
            for (int a = 0; a < h; a++) {
#pragma unroll
                for (int t = 0; t < NT; t++)
#pragma unroll
                    for (int i = 0; i < 4; i++)
                        acc.quad[t][a][i] = __fadd_rn(acc.quad[t][a][i], acc.quad[t][a + h][i]);
#pragma unroll
                for (int t = 0; t < NV; t++)
                    acc.one[t][a] = __fadd_rn(acc.one[t][a], acc.one[t][a + h]);
            }
#pragma unroll
        for (int t = 0; t < NT; t++) out.quad[t] = acc.quad[t][0];
#pragma unroll
        for (int t = 0; t < NV; t++) out.one[t] = acc.one[t][0];
    }

    template <int SM>
    static __device__ __forceinline__ void stage(Acc &acc, const float (&a)[MT][kC], const Rows &X,
                                                 const uint32_t (&at)[kGW][kPieces], uint32_t ring,
                                                 uint32_t sc, uint32_t w, uint32_t gs0,
                                                 uint32_t g0, uint32_t G) {
        static_for<kGW>([&](auto Q) {
            const uint32_t g = gs0 + w + W * (uint32_t)Q;
            if (g >= G) return;
            uint32_t xv[MV][16]; /* the uniform tokens' columns, in scalar registers */
#pragma unroll
            for (int t = 0; t < NV; t++)
#pragma unroll
                for (int i = 0; i < 16; i++)
                    xv[t][i] = ((ScalarWords)(uintptr_t)X.one[t])[16u * g + (uint32_t)i];
            u32x4_t p[kPieces];
            uint32_t raw;
            if constexpr (std::is_same<Fmt, Mx4>::value) {
                asm volatile("ds_read_b128 %0, %2\n\tds_read_u8 %1, %3\n\ts_waitcnt lgkmcnt(0)"
                             : "=&v"(p[0]), "=&v"(raw)
                             : "v"(at[(int)Q][0] + ring), "v"(sc + (g - w - g0)));
            } else { /* one scale word per four groups */
                asm volatile("ds_read_b128 %0, %3\n\tds_read_b128 %1, %4\n\tds_read_b32 %2, %5\n\t"
                             "s_waitcnt lgkmcnt(0)"
                             : "=&v"(p[0]), "=&v"(p[1]), "=&v"(raw)
                             : "v"(at[(int)Q][0] + ring), "v"(at[(int)Q][1] + ring),
                               "v"(sc - w + ((g - g0) & ~3u)));
            }
            f32x4 gs[MT];
            float gv[MV];
#pragma unroll
            for (int t = 0; t < NT; t++) gs[t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int t = 0; t < NV; t++) gv[t] = 0.0f;
            static_for<4>([&](auto D) {
                float b[8];
                weights8<(int)D>(b, p);
                static_for<8>([&](auto I) {
                    constexpr int k = 8 * (int)D + (int)I, ab = (int)Q * kLG + k / kC;
#pragma unroll
                    for (int t = 0; t < NT; t++)
                        gs[t] = __builtin_amdgcn_mfma_f32_4x4x1f32(a[t][k % kC], b[(int)I], gs[t],
                                                                   kCbsz, ab, 0);
#pragma unroll
                    for (int t = 0; t < NV; t++) {
                        const uint32_t v = xv[t][k / 2];
                        gv[t] = fmaf(b[(int)I], k & 1 ? bf16_hi(v) : bf16_lo(v), gv[t]);
                    }
                });
            });
            const float s = scale(raw);
            constexpr int A = SM * kGW + (int)Q;
#pragma unroll
            for (int t = 0; t < NT; t++)
#pragma unroll
                for (int i = 0; i < 4; i++)
                    acc.quad[t][A][i] = fmaf(gs[t][i], s, acc.quad[t][A][i]);
#pragma unroll
            for (int t = 0; t < NV; t++) acc.one[t][A] = fmaf(gv[t], s, acc.one[t][A]);
        });
    }

    /* Butterfly levels W / 2 .. 1 across the waves: partials [wave][token]
     * [row] (token 4 t + i of quad t, then the uniform ones) in the ring slot
     * of the tile's last stage, which no load in flight fills. The LDS
     * accesses are asm: the compiler would drain the DMA before its own. */
    static __device__ __forceinline__ uint32_t meet(const Pipe &pipe, const Result &v) {
        const uint32_t w = threadIdx.x >> 6, L = threadIdx.x & 63u;
        const uint32_t last = pipe.slot >= 1u ? pipe.slot - 1u : kRing - 1u;
        const uint32_t red = pipe.lds + kStage * last;
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier(); /* the stage's last reads are done */
        asm volatile("" ::: "memory");
        const uint32_t o = red + 4u * ((w * (uint32_t)kTokens + 4u * (L / RB)) * RB + L % RB);
#pragma unroll
        for (int t = 0; t < 4 * NT + NV; t++) {
            const float f = t < 4 * NT ? v.quad[t / 4 % MT][t & 3] : v.one[(t - 4 * NT + MV) % MV];
            const uint32_t token = (uint32_t)(t < 4 * NT ? t / 4 * 4 * kQuads + (t & 3) : t);
            asm volatile("ds_write_b32 %0, %1" ::"v"(o + 4u * RB * token), "v"(f) : "memory");
        }
        wait_lgkm<0>();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        return red;
    }
    static __device__ __forceinline__ float value(uint32_t red, uint32_t token, uint32_t row) {
        static_assert(W == 8u, "eight partials");
        constexpr int S = 4 * RB * kTokens; /* bytes of a wave's partials */
        float v[W];
        asm volatile("ds_read_b32 %0, %8\n\tds_read_b32 %1, %8 offset:%9\n\t"
                     "ds_read_b32 %2, %8 offset:%10\n\tds_read_b32 %3, %8 offset:%11\n\t"
                     "ds_read_b32 %4, %8 offset:%12\n\tds_read_b32 %5, %8 offset:%13\n\t"
                     "ds_read_b32 %6, %8 offset:%14\n\tds_read_b32 %7, %8 offset:%15\n\t"
                     "s_waitcnt lgkmcnt(0)"
                     : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]), "=&v"(v[4]),
                       "=&v"(v[5]), "=&v"(v[6]), "=&v"(v[7])
                     : "v"(red + 4u * (token * RB + row)), "i"(S), "i"(2 * S), "i"(3 * S),
                       "i"(4 * S), "i"(5 * S), "i"(6 * S), "i"(7 * S));
#pragma unroll
        for (int h = (int)W / 2; h >= 1; h /= 2)
#pragma unroll
            for (int i = 0; i < h; i++) v[i] = __fadd_rn(v[i], v[i + h]);
        return v[0];
    }
    /* Token rows of a tile of n <= kTokens tokens (the missing ones of the
     * last quad repeat the last token). */
    template <class RowFn>
    static __device__ __forceinline__ void rows(Rows &X, uint32_t n, RowFn &&row) {
        const uint32_t L = threadIdx.x & 63u;
#pragma unroll
        for (int t = 0; t < NT; t++) {
            const uint32_t i = 4u * (kQuads * t + L / RB) + (L & 3u);
            X.quad[t] = row(i < n ? i : n - 1u);
        }
#pragma unroll
        for (int t = 0; t < NV; t++) X.one[t] = row(4u * NT + t);
    }
};

/* ---- users of the core --------------------------------------------------- */

/* An expert's descriptor through scalar loads (uniform pointers). */
struct ScalarExpert {
    const uint8_t *gate_packed, *gate_scales, *down_packed, *down_scales, *up_packed, *up_scales;
};
__device__ __forceinline__ ScalarExpert scalar_expert(const k3_moe_expert *e) {
    const auto p = (const __attribute__((address_space(4))) uint64_t *)(uintptr_t)e;
    return ScalarExpert{(const uint8_t *)p[0], (const uint8_t *)p[1], (const uint8_t *)p[2],
                        (const uint8_t *)p[3], (const uint8_t *)p[4], (const uint8_t *)p[5]};
}

struct GateUpArgs {
    ExactGroup g;
    uint16_t *act;
    const uint16_t *x;
    uint32_t kind;
    float beta, lb;

    __device__ __forceinline__ uint32_t cols() const { return g.F / 32u; }
    __device__ __forceinline__ uint32_t groups() const { return g.H / 32u; }
    /* 32 gate and 32 up rows of expert e */
    __device__ __forceinline__ BlockRows weights(const ScalarExpert &e, uint32_t col) const {
        const uint64_t f0 = 32ull * col;
        BlockRows R;
        R.w[0] = e.gate_packed + f0 * (g.H / 2u);
        R.w[1] = e.up_packed + f0 * (g.H / 2u);
        R.s[0] = e.gate_scales + f0 * (g.H / 32u);
        R.s[1] = e.up_scales + f0 * (g.H / 32u);
        R.last[0] = R.last[1] = 31u;
        R.whole = true;
        return R;
    }
    __device__ __forceinline__ const uint16_t *token(uint32_t row) const {
        return x + (uint64_t)g.token_index[row] * g.H;
    }
    template <class C>
    __device__ __forceinline__ void store(uint32_t red, uint32_t row0, uint32_t n,
                                          uint32_t col) const {
        for (uint32_t o = threadIdx.x; o < 32u * n; o += 64u * W) {
            const uint32_t t = o >> 5, f = o & 31u;
            const float gv = bf16_to_f32(f32_to_bf16(C::value(red, t, f)));
            const float uv = bf16_to_f32(f32_to_bf16(C::value(red, t, 32u + f)));
            act[(uint64_t)(row0 + t) * g.F + 32u * col + f] =
                f32_to_bf16(gated_act(gv, uv, kind, beta, lb));
        }
    }
};

struct DownArgs {
    ExactGroup g;
    uint16_t *y;
    const uint16_t *act;

    __device__ __forceinline__ uint32_t cols() const { return (g.H + kRows - 1u) / kRows; }
    __device__ __forceinline__ uint32_t groups() const { return g.F / 32u; }
    /* 64 rows, or (H % 64 == 32) the last 32 twice */
    __device__ __forceinline__ BlockRows weights(const ScalarExpert &e, uint32_t col) const {
        const uint64_t h0 = (uint64_t)kRows * col, h1 = g.H - h0 > 32u ? h0 + 32u : h0;
        BlockRows R;
        R.w[0] = e.down_packed + h0 * (g.F / 2u);
        R.w[1] = e.down_packed + h1 * (g.F / 2u);
        R.s[0] = e.down_scales + h0 * (g.F / 32u);
        R.s[1] = e.down_scales + h1 * (g.F / 32u);
        R.last[0] = R.last[1] = 31u;
        R.whole = true;
        return R;
    }
    __device__ __forceinline__ const uint16_t *token(uint32_t row) const {
        return act + (uint64_t)row * g.F;
    }
    template <class C>
    __device__ __forceinline__ void store(uint32_t red, uint32_t row0, uint32_t n,
                                          uint32_t col) const {
        const uint32_t h0 = kRows * col;
        for (uint32_t o = threadIdx.x; o < kRows * n; o += 64u * W) {
            const uint32_t t = o >> 6, r = o & 63u;
            if (h0 + r < g.H)
                y[(uint64_t)g.route_index[row0 + t] * g.H + h0 + r] =
                    f32_to_bf16(C::value(red, t, r));
        }
    }
};

/* One tile: plan rows [row0, row0 + n), the weight rows R of column block col. */
struct Tile {
    BlockRows R;
    uint32_t row0, n, col;
};

template <class Args, int NT, int NV, int SB>
__device__ __forceinline__ void run_tile(const Args &A, Pipe &pipe, const Tile &T, bool more,
                                         const BlockRows &next) {
    using C = Core<Mx4, NT, NV, SB, 64>;
    typename C::Rows X;
    C::rows(X, T.n, [&](uint32_t i) { return A.token(T.row0 + i); });
    typename C::Result v;
    C::run(v, pipe, T.R, X, A.groups(), more, next);
    A.template store<C>(C::meet(pipe, v), T.row0, T.n, T.col);
}

/* n <= 16 rows: whole quads on the matrix units and of a short tile one or
 * two rows on the vector unit. Per 64 rows x 32 columns (two waves per SIMD,
 * operands in registers) the conversions take 34 ns, a vector row 61, a quad
 * 150: one vector row costs less than a second quad, two do not. */
template <bool Heavy, int SB, class Args>
__device__ __forceinline__ void any_tile(const Args &A, Pipe &pipe, const Tile &T, bool more,
                                         const BlockRows &next) {
    switch (T.n) {
        case 1u: run_tile<Args, 0, 1, SB>(A, pipe, T, more, next); break;
        case 2u: run_tile<Args, 0, 2, SB>(A, pipe, T, more, next); break;
        case 3u:
        case 4u: run_tile<Args, 1, 0, SB>(A, pipe, T, more, next); break;
        case 5u: run_tile<Args, 1, 1, SB>(A, pipe, T, more, next); break;
        case 6u:
        case 7u:
        case 8u: run_tile<Args, 2, 0, SB>(A, pipe, T, more, next); break;
        default:
            if constexpr (Heavy) {
                if (T.n <= 12u) run_tile<Args, 3, 0, SB>(A, pipe, T, more, next);
                else run_tile<Args, 4, 0, SB>(A, pipe, T, more, next);
            }
    }
}

/* Tile of work wk: experts in address order over the whole chip. Blocks are
 * dealt to the XCDs round robin: within an expert, eight columns at a time
 * with the expert's tiles in between, so the tiles that read the same weight
 * rows run together on one XCD. False past the last. */
struct Walk {
    uint32_t wk, q; /* next work; list mode: of list entry q */
};
template <bool Heavy, class Args>
__device__ __forceinline__ bool next_tile(const Args &A, Walk &p, Tile &T) {
    const ExactGroup &g = A.g;
    const uint32_t ncol = A.cols();
    const ScalarWords counts = (ScalarWords)(uintptr_t)g.lists;
    const ScalarWords light = counts + 4;
    if constexpr (!Heavy) {
        if (p.wk >= counts[0] * ncol) return false;
        const ScalarWords rec = light + 4u * (p.wk / ncol);
        T.col = p.wk % ncol;
        T.row0 = rec[1];
        T.n = rec[2];
        T.R = A.weights(scalar_expert(g.experts + rec[0]), T.col);
    } else {
        uint32_t e, base, rows, local;
        if (g.list) { /* listed experts, their works one after the other */
            const ScalarWords list = (ScalarWords)(uintptr_t)g.list;
            for (;; p.q++) {
                if (p.q >= list[0]) return false;
                e = list[1u + p.q];
                rows = ((ScalarWords)(uintptr_t)g.counts)[e];
                const uint32_t works = (rows + kHeavyTile - 1u) / kHeavyTile * ncol;
                if (p.wk < works) break;
                p.wk -= works;
            }
            base = ((ScalarWords)(uintptr_t)g.offsets)[e];
            local = p.wk;
        } else {
            if (p.wk >= counts[1] * ncol) return false;
            const ScalarWords rec = light + 4u * ((g.routes < g.E ? g.routes : g.E) + p.wk / ncol);
            e = rec[0];
            base = rec[1];
            rows = rec[2];
            local = p.wk - rec[3] * ncol;
        }
        const uint32_t nsub = (rows + kHeavyTile - 1u) / kHeavyTile;
        const uint32_t cg = local / (8u * nsub), r = local - cg * 8u * nsub;
        const uint32_t width = ncol - 8u * cg < 8u ? ncol - 8u * cg : 8u;
        const uint32_t p0 = (r / width) * kHeavyTile;
        T.col = 8u * cg + r % width;
        T.row0 = base + p0;
        T.n = rows - p0 < kHeavyTile ? rows - p0 : kHeavyTile;
        T.R = A.weights(scalar_expert(g.experts + e), T.col);
    }
    p.wk += gridDim.x;
    return true;
}

/* Persistent blocks: two a CU with 16 KB stages for the light tiles, which
 * stream; one with 32 KB stages (half the barriers) for the heavy ones, whose
 * partials take 128 registers. A block's next tile is known one tile ahead,
 * and its first loads run under the current one's last steps. */
template <bool Heavy, class Args>
__global__ __launch_bounds__(512, Heavy ? 2 : 4) void exact_tiles_run_kernel(Args A) {
    constexpr int SB = Heavy ? 512 : 256;
    __shared__ __attribute__((aligned(16))) uint8_t smem[kRows * (kRing * SB + 2 * kScaleGroups)];
    const uint32_t G = A.groups();
    /* short rows (a stage or less) and many scales: no look-ahead */
    const bool ahead = G <= kScaleGroups && G > SB / 16;
    Walk p{blockIdx.x, 0u};
    Pipe pipe{lds_addr(smem), 0u, 0u, false};
    Tile T, N;
    bool have = next_tile<Heavy>(A, p, T);
    while (have) {
        have = next_tile<Heavy>(A, p, N);
        any_tile<Heavy, SB>(A, pipe, T, have && ahead, N.R);
        T = N;
    }
}

/* One block of 1024 threads: the tile lists, experts ascending. */
__global__ __launch_bounds__(1024) void exact_tiles_kernel(ExactGroup g) {
    __shared__ uint32_t first[1025]; /* each expert's first heavy tile */
    __shared__ uint32_t wave_tot[2][16];
    const uint32_t e = threadIdx.x, lane = e & 63u, wave = e >> 6;
    const uint32_t n = e < g.E ? g.counts[e] : 0u;
    const uint32_t light = n != 0u && n <= kLightRows ? 1u : 0u;
    const uint32_t nt = n > kLightRows ? (n + kHeavyTile - 1u) / kHeavyTile : 0u;
    uint32_t inc = nt, linc = light;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t a = __shfl_up(inc, o, 64), b = __shfl_up(linc, o, 64);
        if ((int)lane >= o) { inc += a; linc += b; }
    }
    if (lane == 63u) { wave_tot[0][wave] = inc; wave_tot[1][wave] = linc; }
    __syncthreads();
    uint32_t before = 0u, lbefore = 0u;
    for (uint32_t w = 0; w < wave; w++) { before += wave_tot[0][w]; lbefore += wave_tot[1][w]; }
    first[e] = before + inc - nt;
    ExactTile *lights = (ExactTile *)(g.lists + 16);
    if (light) {
        const uint32_t at = lbefore + linc - 1u;
        lights[at] = ExactTile{e, g.offsets[e], n, at};
    }
    if (e == 1023u) {
        first[1024] = before + inc;
        ((uint32_t *)g.lists)[0] = lbefore + linc;
        ((uint32_t *)g.lists)[1] = before + inc;
    }
    __syncthreads();
    const uint32_t total = first[1024];
    ExactTile *heavy = lights + (g.routes < g.E ? g.routes : g.E);
    for (uint32_t t = e; t < total; t += 1024u) {
        uint32_t lo = 0u, hi = 1024u; /* first[lo] <= t < first[hi] */
        while (hi - lo > 1u) {
            const uint32_t m = (lo + hi) / 2u;
            if (first[m] <= t) lo = m;
            else hi = m;
        }
        heavy[t] = ExactTile{lo, g.offsets[lo], g.counts[lo], first[lo]};
    }
}

struct DenseArgs {
    uint16_t *out;
    const uint8_t *w, *s;
    const uint16_t *x;
    uint32_t tokens, rows, cols, token_tiles, works;
};

/* Work -> (row block, token tile): eight row blocks at a time, one per XCD
 * (blocks are dealt to the XCDs round robin), the token tiles in between, so
 * the tiles that read the same rows run together on one XCD. */
template <class Fmt, uint32_t RB, uint32_t TT>
__device__ __forceinline__ bool dense_tile(const DenseArgs &A, uint32_t wk, uint32_t &r0,
                                           uint32_t &t0, BlockRows &R) {
    if (wk >= A.works) return false;
    const uint32_t nrb = (A.rows + RB - 1u) / RB, tt = A.token_tiles;
    const uint32_t cg = wk / (8u * tt), r = wk - cg * 8u * tt;
    const uint32_t width = nrb - 8u * cg < 8u ? nrb - 8u * cg : 8u;
    r0 = (8u * cg + r % width) * RB;
    t0 = (r / width) * TT;
    const uint32_t G = A.cols / 32u, live = A.rows - r0 < RB ? A.rows - r0 : RB;
    const uint64_t rbytes = (uint64_t)G * Fmt::kGroupBytes;
    const uint32_t h1 = live > 32u ? 32u : live - 1u; /* no second half: the last row */
    R.w[0] = A.w + r0 * rbytes;
    R.w[1] = A.w + (r0 + h1) * rbytes;
    R.s[0] = A.s + (uint64_t)r0 * G;
    R.s[1] = A.s + (uint64_t)(r0 + h1) * G;
    R.last[0] = live < 32u ? live - 1u : 31u;
    R.last[1] = live > 32u ? live - 33u : 0u;
    R.whole = live == RB;
    return true;
}

template <class Fmt, int NT, int RB>
__global__ __launch_bounds__(512, RB == 64 && NT > 2 ? 2 : 4) void exact_dense_kernel(DenseArgs A) {
    constexpr int SB = RB == 64 && NT <= 2 ? 256 : 512;
    __shared__ __attribute__((aligned(16))) uint8_t smem[RB * (kRing * SB + 2 * kScaleGroups)];
    using C = Core<Fmt, NT, 0, SB, RB>;
    constexpr uint32_t TT = C::kTokens;
    const uint32_t G = A.cols / 32u;
    const bool ahead = G <= kScaleGroups && G > (uint32_t)C::kSG;
    Pipe pipe{lds_addr(smem), 0u, 0u, false};
    BlockRows R, N;
    uint32_t r0, t0, nr0, nt0, wk = blockIdx.x;
    bool have = dense_tile<Fmt, RB, TT>(A, wk, r0, t0, R);
    while (have) {
        wk += gridDim.x;
        have = dense_tile<Fmt, RB, TT>(A, wk, nr0, nt0, N);
        const uint32_t n = A.tokens - t0 < TT ? A.tokens - t0 : TT;
        typename C::Rows X;
        C::rows(X, n, [&](uint32_t i) { return A.x + (uint64_t)(t0 + i) * A.cols; });
        typename C::Result v;
        C::run(v, pipe, R, X, G, have && ahead && R.whole && N.whole, N);
        const uint32_t red = C::meet(pipe, v);
        for (uint32_t o = threadIdx.x; o < RB * n; o += 64u * W) {
            const uint32_t t = o / RB, r = o % RB;
            if (r0 + r < A.rows)
                A.out[(uint64_t)(t0 + t) * A.rows + r0 + r] = f32_to_bf16(C::value(red, t, r));
        }
        R = N;
        r0 = nr0;
        t0 = nt0;
    }
}

/* persistent grids: blocks of a CU times the CUs */
uint32_t grid_of(uint64_t works, uint32_t per_cu) {
    return (uint32_t)(works < per_cu * kCus ? works : per_cu * kCus);
}

template <class Fmt, int NT, int RB>
bool launch_dense_tiles(DenseArgs A, const DenseForm &f, hipStream_t st) {
    A.token_tiles = (A.tokens + f.tokens() - 1u) / f.tokens();
    const uint64_t works = (uint64_t)((A.rows + RB - 1u) / RB) * A.token_tiles;
    if (works > 0xffff0000ull) return false;
    A.works = (uint32_t)works;
    hipLaunchKernelGGL(HIP_KERNEL_NAME(exact_dense_kernel<Fmt, NT, RB>),
                       dim3(grid_of(works, f.per_cu)), dim3(64 * W), 0, st, A);
    return hipGetLastError() == hipSuccess;
}

template <class Fmt>
bool launch_dense(uint16_t *out, const void *w, const void *s, const void *x, uint32_t tokens,
                  uint32_t rows, uint32_t cols, hipStream_t st) {
    const DenseArgs A{out, (const uint8_t *)w, (const uint8_t *)s, (const uint16_t *)x, tokens,
                      rows, cols, 0u, 0u};
    const DenseForm f = dense_form(tokens, rows);
    if (f.rows == 16u) return launch_dense_tiles<Fmt, 1, 16>(A, f, st);
    if (f.quads == 1u) return launch_dense_tiles<Fmt, 1, 64>(A, f, st);
    if (f.quads == 2u) return launch_dense_tiles<Fmt, 2, 64>(A, f, st);
    return launch_dense_tiles<Fmt, 4, 64>(A, f, st);
}

/* The light and the heavy tiles' launches (a token has an expert at most
 * once, so few tokens make no heavy tiles). A list of experts (tensors that the
 * scaled-MFMA tiles cannot take; none as a rule) runs on the heavy kernel, one
 * block a CU: an empty list costs no more than on 64 blocks, on which a layer
 * of 128 such experts (3584 / 2048) took 762 us for 9 tokens and 2240 for 64
 * against 273 and 663 here. */
template <class Args>
bool launch_grouped(const Args &A, uint32_t ncol, hipStream_t st) {
    const ExactGroup &g = A.g;
    const dim3 block(64 * W);
    if (g.list) {
        hipLaunchKernelGGL(HIP_KERNEL_NAME(exact_tiles_run_kernel<true, Args>), dim3(kCus),
                           block, 0, st, A);
        return hipGetLastError() == hipSuccess;
    }
    const uint64_t lights = exact_light_cap(g.routes, g.E), tiles = exact_heavy_cap(g.routes, g.E);
    hipLaunchKernelGGL(HIP_KERNEL_NAME(exact_tiles_run_kernel<false, Args>),
                       dim3(grid_of(lights * ncol, 2u)), block, 0, st, A);
    if (g.tokens > kLightRows)
        hipLaunchKernelGGL(HIP_KERNEL_NAME(exact_tiles_run_kernel<true, Args>),
                           dim3(grid_of(tiles * ncol, 1u)), block, 0, st, A);
    return hipGetLastError() == hipSuccess;
}

}  // namespace

bool launch_exact_tiles(const ExactGroup &g, hipStream_t st) {
    if (g.E > 1024u) return false;
    hipLaunchKernelGGL(exact_tiles_kernel, dim3(1), dim3(1024), 0, st, g);
    return hipGetLastError() == hipSuccess;
}

bool launch_exact_gateup(const ExactGroup &g, uint16_t *act, const uint16_t *x, uint32_t kind,
                         float beta, float lb, hipStream_t st) {
    return launch_grouped(GateUpArgs{g, act, x, kind, beta, lb}, g.F / 32u, st);
}

bool launch_exact_down(const ExactGroup &g, uint16_t *y, const uint16_t *act, hipStream_t st) {
    return launch_grouped(DownArgs{g, y, act}, (g.H + kRows - 1u) / kRows, st);
}

bool launch_exact_mxfp4(uint16_t *out, const void *packed, const void *scales, const void *x,
                        uint32_t tokens, uint32_t rows, uint32_t cols, hipStream_t st) {
    return launch_dense<Mx4>(out, packed, scales, x, tokens, rows, cols, st);
}

bool launch_exact_q8(uint16_t *out, const void *codes, const void *scales, const void *x,
                     uint32_t tokens, uint32_t rows, uint32_t cols, hipStream_t st) {
    return launch_dense<Q8>(out, codes, scales, x, tokens, rows, cols, st);
}

}  // namespace k3
