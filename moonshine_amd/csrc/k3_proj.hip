/*
 * Static projections of a token batch on bf16 MFMA, for the MXFP8
 * precisions of the K3-native block (the exact precision keeps the VALU
 * rows kernels of k3_rocm_q8_128_gemm_bf16 / k3_rocm_bf16_gemm_bf16,
 * k3_rocm_ops.cu:663-835, 1694-2038, and their bits).
 *
 *   out[t, r] = bf16(sum_b s[r, b] * sum_{k in block b} q[r, k] x[t, k])   Q8-128
 *   out[t, r] = bf16(sum_k w[r, k] x[t, k])                                bf16
 *
 * Int8 codes are exact in bf16 (|q| <= 127 has at most 7 significant
 * bits), so every product is the exact product and only the fp32
 * summation order differs from the exact kernels (which sum 32-column
 * groups and scale each): a tolerance of fp32 reassociation, far inside
 * one bf16 rounding of the output.
 *
 * Block tile 128 tokens x 128 rows, 8 waves of 32 x 64 (2 x 4
 * V_MFMA_F32_16X16X32_BF16 tiles), K steps of 64 through two LDS buffers
 * (rows padded to 144 bytes), global loads two steps ahead. Codes are
 * converted to bf16 on their way into LDS. A Q8-128 block is two K steps:
 * its four MFMAs per tile chain in a block sum that is then scaled into
 * the accumulator with one fma per output; the next block's scales are
 * loaded a block ahead. Tiles are dealt to the XCDs in contiguous ranges,
 * a token tile's row tiles together.
 */
#include "k3_device.h"
#include "k3_internal.h"
#include "k3_lds.h"

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

namespace k3 {
namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

constexpr uint32_t kPT = 128, kPK = 64, kPPad = 144;

typedef uint8_t ProjStage[2][kPT * kPPad]; /* [A tokens | B weight rows] */

struct ProjArgs {
    uint16_t *out;        /* [T, N] bf16 */
    const uint16_t *x;    /* [T, K] bf16 */
    const void *w;        /* [N, K] int8 codes or bf16 */
    const float *scales;  /* [N, K / 128] (Q8-128) */
    uint32_t T, N, K;
};

/* Eight int8 codes as eight bf16 (exact). */
__device__ __forceinline__ uint4 codes_to_bf16(uint2 v) {
    uint32_t o[4];
    const uint32_t u[2] = {v.x, v.y};
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
        for (int p = 0; p < 2; p++) {
            const float lo = (float)(int8_t)(u[h] >> (16 * p));
            const float hi = (float)(int8_t)(u[h] >> (16 * p + 8));
            /* the two upper halves */
            o[2 * h + p] = __builtin_amdgcn_perm(__float_as_uint(hi), __float_as_uint(lo), 0x07060302u);
        }
    return make_uint4(o[0], o[1], o[2], o[3]);
}

/* The thread's two rows of one K step: x as 16 bytes, weights as 16
 * (bf16) or 8 (codes) bytes, converted to bf16 on the store. */
template <bool Q8>
using WeightPiece = typename std::conditional<Q8, uint2, uint4>::type;

template <bool Q8>
__device__ __forceinline__ void proj_load(uint4 &a0, uint4 &a1, WeightPiece<Q8> &b0,
                                          WeightPiece<Q8> &b1, const uint8_t *xb,
                                          const uint8_t *wb, uint32_t ao0, uint32_t ao1,
                                          uint32_t bo0, uint32_t bo1, uint32_t s) {
    const uint32_t ka = 2u * kPK * s, kw = (Q8 ? 1u : 2u) * kPK * s;
    a0 = *(const uint4 *)(xb + ao0 + ka);
    a1 = *(const uint4 *)(xb + ao1 + ka);
    b0 = *(const WeightPiece<Q8> *)(wb + bo0 + kw);
    b1 = *(const WeightPiece<Q8> *)(wb + bo1 + kw);
}

__device__ __forceinline__ uint4 as_bf16x8(uint2 codes) { return codes_to_bf16(codes); }
__device__ __forceinline__ uint4 as_bf16x8(uint4 bf16) { return bf16; }

template <bool Q8>
__device__ __forceinline__ void proj_store(ProjStage &buf, uint32_t off, const uint4 &a0,
                                           const uint4 &a1, const WeightPiece<Q8> &b0,
                                           const WeightPiece<Q8> &b1) {
    constexpr uint32_t R64 = 64u * kPPad;
    *(uint4 *)(buf[0] + off) = a0;
    *(uint4 *)(buf[0] + off + R64) = a1;
    *(uint4 *)(buf[1] + off) = as_bf16x8(b0);
    *(uint4 *)(buf[1] + off + R64) = as_bf16x8(b1);
}

/* acc[i][j] += A(wave rows i) . B(wave rows j) over one K step. */
__device__ __forceinline__ void proj_compute(f32x4_t (&acc)[2][4], const ProjStage &buf,
                                             uint32_t a_off, uint32_t b_off) {
#pragma unroll
    for (int ks = 0; ks < 2; ks++) {
        bf16x8_t af[2], bf[4];
#pragma unroll
        for (int i = 0; i < 2; i++)
            af[i] = __builtin_bit_cast(bf16x8_t, *(const uint4 *)(buf[0] + a_off + 16u * kPPad * i +
                                                                  64u * ks));
#pragma unroll
        for (int j = 0; j < 4; j++)
            bf[j] = __builtin_bit_cast(bf16x8_t, *(const uint4 *)(buf[1] + b_off + 16u * kPPad * j +
                                                                  64u * ks));
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int j = 0; j < 4; j++)
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[i], bf[j], acc[i][j], 0, 0, 0);
    }
}

template <bool Q8>
__global__ __launch_bounds__(512) void proj_mfma_kernel(ProjArgs P) {
    __shared__ __attribute__((aligned(16))) ProjStage lds[2];
    const uint32_t T = P.T, N = P.N, K = P.K;
    const uint32_t ntt = (T + kPT - 1u) / kPT, nnt = (N + kPT - 1u) / kPT;
    const uint32_t works = ntt * nnt, per = (works + 7u) / 8u;
    const uint32_t L = blockIdx.x, j8 = L >> 3, wk = (L & 7u) * per + j8;
    if (j8 >= per || wk >= works) return;
    const uint32_t t0 = (wk / nnt) * kPT, n0 = (wk % nnt) * kPT;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    const uint32_t wm = wave >> 1, wn = wave & 1u, g = lane >> 4, c = lane & 15u;
    /* thread tid loads piece tid % 8 (8 columns) of rows tid / 8 and tid /
     * 8 + 64; rows past T or N clamp to the last one (not stored) */
    const uint32_t r0 = tid >> 3, pc = tid & 7u;
    constexpr uint32_t wbytes = Q8 ? 1u : 2u;
    uint32_t ao[2], bo[2];
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const uint32_t ta = t0 + r0 + 64u * i, nb = n0 + r0 + 64u * i;
        ao[i] = ((ta < T ? ta : T - 1u) * K + 8u * pc) * 2u;
        bo[i] = ((nb < N ? nb : N - 1u) * K + 8u * pc) * wbytes;
    }
    const uint8_t *xb = (const uint8_t *)P.x, *wb = (const uint8_t *)P.w;
    const uint32_t soff = r0 * kPPad + 16u * pc;
    const uint32_t a_off = (32u * wm + c) * kPPad + 16u * g;
    const uint32_t b_off = (64u * wn + c) * kPPad + 16u * g;
    /* Q8: the scales of this lane's four weight rows (one per n-tile) */
    const uint32_t nblk = K / 128u;
    const float *srow[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const uint32_t r = n0 + 64u * wn + 16u * (uint32_t)j + c;
        srow[j] = P.scales + (uint64_t)(r < N ? r : N - 1u) * nblk;
    }
    f32x4_t acc[2][4], blk[2][4];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) {
            acc[i][j] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
            blk[i][j] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
        }
    float sc[4] = {1.0f, 1.0f, 1.0f, 1.0f};
    if constexpr (Q8) {
#pragma unroll
        for (int j = 0; j < 4; j++) sc[j] = srow[j][0];
    }
    const uint32_t nsteps = K / kPK, last = nsteps - 1u;
    /* two register sets: step s + 2's loads are issued at the start of
     * step s; loads and stores are unconditional (steps past the end
     * reload the last one into a buffer nobody reads) */
    uint4 a0, a1, p0, p1;
    WeightPiece<Q8> b0, b1, q0, q1;
    proj_load<Q8>(a0, a1, b0, b1, xb, wb, ao[0], ao[1], bo[0], bo[1], 0u);
    proj_load<Q8>(p0, p1, q0, q1, xb, wb, ao[0], ao[1], bo[0], bo[1], 1u < last ? 1u : last);
    proj_store<Q8>(lds[0], soff, a0, a1, b0, b1);
    __syncthreads();
    for (uint32_t s = 0; s < nsteps; s += 2u) {
        /* Q8: steps s, s + 1 are 128-column block s / 2 (K % 128 == 0);
         * the next block's scales load during this block's two steps */
        float nx[4] = {1.0f, 1.0f, 1.0f, 1.0f};
        if constexpr (Q8) {
            const uint32_t b1 = s / 2u + 1u < nblk ? s / 2u + 1u : s / 2u;
#pragma unroll
            for (int j = 0; j < 4; j++) nx[j] = srow[j][b1];
        }
        proj_load<Q8>(a0, a1, b0, b1, xb, wb, ao[0], ao[1], bo[0], bo[1],
                      s + 2u < last ? s + 2u : last);
        if constexpr (Q8) proj_compute(blk, lds[0], a_off, b_off);
        else proj_compute(acc, lds[0], a_off, b_off);
        proj_store<Q8>(lds[1], soff, p0, p1, q0, q1);
        __syncthreads();
        if (s + 1u < nsteps) {
            proj_load<Q8>(p0, p1, q0, q1, xb, wb, ao[0], ao[1], bo[0], bo[1],
                          s + 3u < last ? s + 3u : last);
            if constexpr (Q8) proj_compute(blk, lds[1], a_off, b_off);
            else proj_compute(acc, lds[1], a_off, b_off);
            proj_store<Q8>(lds[0], soff, a0, a1, b0, b1);
            __syncthreads();
        }
        if constexpr (Q8) {
            /* acc += scale * block sum */
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
                for (int j = 0; j < 4; j++) {
#pragma unroll
                    for (int r = 0; r < 4; r++) acc[i][j][r] = fmaf(blk[i][j][r], sc[j], acc[i][j][r]);
                    blk[i][j] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
                }
#pragma unroll
            for (int j = 0; j < 4; j++) sc[j] = nx[j];
        }
    }
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const uint32_t n = n0 + 64u * wn + 16u * (uint32_t)j + c;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const uint32_t t = t0 + 32u * wm + 16u * (uint32_t)i + 4u * g + (uint32_t)r;
                if (t < T && n < N) P.out[(uint64_t)t * N + n] = f32_to_bf16(acc[i][j][r]);
            }
        }
}

/*
 * The Q8-128 form for many tokens: block tile 256 tokens x 128 rows, eight
 * waves of 64 x 64, so a stage of 64 columns (32 KB of tokens, 16 KB of codes
 * as bf16) feeds 32 MFMAs a wave from 16 LDS reads (the 32 x 64 wave tile
 * above reads 12 for 16, and its LDS reads outlast its MFMAs). Three stages:
 * tokens by direct-to-LDS loads two stages ahead (whole 128-byte lines,
 * swizzled as the expert kernels' A tiles), codes into registers two stages
 * ahead, converted and written one ahead, after the stage's MFMAs. LDS
 * accesses and their waits are explicit: the compiler would drain the loads
 * in flight before each. 2048 tokens, before -> after, us: 6144 x 7168
 * 308 -> 251, 7168 x 3584 201 -> 127; 8192 tokens 1231 -> 805, 724 -> 468.
 */
constexpr uint32_t kWT = 256, kWN = 128;              /* block tile */
constexpr uint32_t kWA = kWT * 128u, kWB = kWN * 128u; /* bytes of a stage */

/* Both kernels hold one block a CU, and a round of tiles over the 256 CUs
 * takes the wide one 6/5 as long for twice the work (7168 columns: 123 and
 * 103 us, 1024 columns: 21 and 17 us): wide where that pays for its rounds. */
static bool wide_pays(uint32_t T, uint32_t N) {
    auto rounds = [&](uint32_t tt) {
        return ((T + tt - 1u) / tt * (uint64_t)((N + 127u) / 128u) + 255u) / 256u;
    };
    return 6u * rounds(kWT) < 5u * rounds(kPT);
}

__global__ __launch_bounds__(512, 2) void proj_wide_kernel(ProjArgs P) {
    __shared__ __attribute__((aligned(16))) uint8_t smem[3u * (kWA + kWB)];
    const uint32_t T = P.T, N = P.N, K = P.K;
    const uint32_t ntt = (T + kWT - 1u) / kWT, nnt = (N + kWN - 1u) / kWN;
    const uint32_t works = ntt * nnt, per = (works + 7u) / 8u;
    const uint32_t j8 = blockIdx.x >> 3, wk = (blockIdx.x & 7u) * per + j8;
    if (j8 >= per || wk >= works) return;
    const uint32_t t0 = (wk / nnt) * kWT, n0 = (wk % nnt) * kWN;
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t wm = wave >> 1, wn = wave & 1u, g = lane >> 4, c = lane & 15u;
    const uint32_t lds = lds_addr(smem);
    /* tokens: wave w fills rows 32 w .. + 32 (four 8-row chunks); rows past
     * T repeat the last one (not stored) */
    const uint8_t *xs[4];
#pragma unroll
    for (int m = 0; m < 4; m++) {
        const uint32_t h = (uint32_t)m & 1u;
        const uint32_t r = t0 + 32u * wave + 16u * ((uint32_t)m >> 1) + a_dma_row(lane, h);
        xs[m] = (const uint8_t *)P.x + 2ull * (r < T ? r : T - 1u) * K + 16u * a_dma_piece(lane, h);
    }
    /* codes: thread t loads 16 of row t / 4 per stage */
    const uint32_t br = tid >> 2, bq = tid & 3u;
    const uint8_t *ws = (const uint8_t *)P.w + (uint64_t)(n0 + br < N ? n0 + br : N - 1u) * K + 16u * bq;
    const uint32_t b_dst = kWA + 2048u * (br >> 4) + a_slot(br & 15u, 2u * bq);
    const uint32_t b_dst2 = kWA + 2048u * (br >> 4) + a_slot(br & 15u, 2u * bq + 1u);
    const uint32_t nblk = K / 128u, nsteps = K / kPK, last = nsteps - 1u;
    const float *srow[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const uint32_t r = n0 + 64u * wn + 16u * (uint32_t)j + c;
        srow[j] = P.scales + (uint64_t)(r < N ? r : N - 1u) * nblk;
    }
    auto fetch = [&](uint32_t s, uint32_t slot) { /* past the end: the last stage again */
        const uint32_t off = 128u * (s < last ? s : last);
#pragma unroll
        for (int m = 0; m < 4; m++)
            __builtin_amdgcn_global_load_lds(
                (const void *)(xs[m] + off),
                (lds_void *)(uintptr_t)(lds + (kWA + kWB) * slot + 4096u * wave + 1024u * m), 16, 0,
                0);
    };
    auto codes = [&](uint32_t s) { return *(const u32x4_t *)(ws + kPK * (s < last ? s : last)); };
    auto write = [&](const u32x4_t &q, uint32_t slot) {
        const uint32_t base = lds + (kWA + kWB) * slot;
        const uint4 lo = codes_to_bf16(make_uint2(q[0], q[1])), hi = codes_to_bf16(make_uint2(q[2], q[3]));
        const u32x4_t l = {lo.x, lo.y, lo.z, lo.w}, h = {hi.x, hi.y, hi.z, hi.w};
        asm volatile("ds_write_b128 %0, %1\n\tds_write_b128 %2, %3" ::"v"(base + b_dst), "v"(l),
                     "v"(base + b_dst2), "v"(h)
                     : "memory");
    };
    f32x4_t acc[4][4], blk[4][4];
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) acc[i][j] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    /* the fragments of 32 columns: rows 64 wm + 16 i + c and 64 wn + 16 j + c */
    const uint32_t a_base = lds + 2048u * 4u * wm, b_base = lds + kWA + 2048u * 4u * wn;
    const uint32_t slot0 = a_slot(c, g), slot1 = a_slot(c, 4u + g);
    float sc[4];
    u32x4_t q0 = codes(0u), q1 = codes(1u);
    write(q0, 0u);
    asm volatile("" : "+v"(q1) : : "memory");
    fetch(0u, 0u);
    asm volatile("" ::: "memory");
    q0 = codes(2u); /* the order the stages' waits count */
#pragma unroll
    for (int j = 0; j < 4; j++) sc[j] = srow[j][0];
    asm volatile("" ::: "memory");
    fetch(1u, 1u);
    uint32_t slot = 0u;
    /* stage s from `slot`; next: the codes of s + 1, refilled with s + 3 */
    auto stage = [&](uint32_t s, u32x4_t &next, auto Odd) {
        constexpr bool odd = decltype(Odd)::value;
        /* younger than stage s's tokens: those of s + 1, a code load and four
         * scales at least */
        wait_vm<9>();
        wait_lgkm<0>(); /* this wave's code writes */
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        const uint32_t s1 = slot == 2u ? 0u : slot + 1u, s2 = slot == 0u ? 2u : slot - 1u;
        fetch(s + 2u, s2);
        if constexpr (odd) wait_vm<9>(); /* this block's scales: nine loads ago */
        asm volatile("" ::: "memory");
        const uint32_t st = (kWA + kWB) * slot;
#pragma unroll
        for (int ks = 0; ks < 2; ks++) {
            u32x4_t af[4], bf[4];
            const uint32_t o = st + (ks ? slot1 : slot0);
            asm volatile(
                "ds_read_b128 %0, %8\n\tds_read_b128 %1, %8 offset:2048\n\t"
                "ds_read_b128 %2, %8 offset:4096\n\tds_read_b128 %3, %8 offset:6144\n\t"
                "ds_read_b128 %4, %9\n\tds_read_b128 %5, %9 offset:2048\n\t"
                "ds_read_b128 %6, %9 offset:4096\n\tds_read_b128 %7, %9 offset:6144\n\t"
                "s_waitcnt lgkmcnt(0)"
                : "=&v"(af[0]), "=&v"(af[1]), "=&v"(af[2]), "=&v"(af[3]), "=&v"(bf[0]),
                  "=&v"(bf[1]), "=&v"(bf[2]), "=&v"(bf[3])
                : "v"(a_base + o), "v"(b_base + o));
#pragma unroll
            for (int i = 0; i < 4; i++)
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const f32x4_t in = !odd && ks == 0 ? f32x4_t{0.0f, 0.0f, 0.0f, 0.0f} : blk[i][j];
                    blk[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                        __builtin_bit_cast(bf16x8_t, af[i]), __builtin_bit_cast(bf16x8_t, bf[j]), in,
                        0, 0, 0);
                }
        }
        /* used here and not before the products: the loads are still out */
        asm volatile("" : "+v"(next) : : "memory");
        write(next, s1);
        next = codes(s + 3u);
        slot = s1;
        if constexpr (odd) { /* acc += scale x block sum; the next block's scales */
            const uint32_t b = s / 2u + 1u < nblk ? s / 2u + 1u : s / 2u;
#pragma unroll
            for (int i = 0; i < 4; i++)
#pragma unroll
                for (int j = 0; j < 4; j++)
#pragma unroll
                    for (int r = 0; r < 4; r++) acc[i][j][r] = fmaf(blk[i][j][r], sc[j], acc[i][j][r]);
#pragma unroll
            for (int j = 0; j < 4; j++) sc[j] = srow[j][b];
        }
    };
    for (uint32_t s = 0u; s < nsteps; s += 2u) { /* K % 128 == 0: an even count */
        stage(s, q1, std::false_type{});
        stage(s + 1u, q0, std::true_type{});
    }
    wait_vm<0>(); /* the loads past the end land before the LDS is given back */
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const uint32_t n = n0 + 64u * wn + 16u * (uint32_t)j + c;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const uint32_t t = t0 + 64u * wm + 16u * (uint32_t)i + 4u * g + (uint32_t)r;
                if (t < T && n < N) P.out[(uint64_t)t * N + n] = f32_to_bf16(acc[i][j][r]);
            }
        }
}

}  // namespace

bool proj_mfma_supported(uint32_t tokens, uint32_t rows, uint32_t cols, bool q8,
                         const void *weights, const void *x) {
    const uint64_t xbytes = 2ull * tokens * cols, wbytes = (q8 ? 1ull : 2ull) * rows * cols;
    return tokens > 0u && rows > 0u && cols > 0u && cols % (q8 ? 128u : kPK) == 0u &&
           xbytes < (1ull << 31) && wbytes < (1ull << 31) &&
           ((uintptr_t)x % 16u) == 0u && ((uintptr_t)weights % (q8 ? 8u : 16u)) == 0u;
}

bool launch_proj_mfma(uint16_t *out, const void *x, const void *weights, const float *scales,
                      uint32_t T, uint32_t N, uint32_t K, bool q8, hipStream_t st) {
    if (!proj_mfma_supported(T, N, K, q8, weights, x) || (q8 && !scales)) return false;
    const ProjArgs A{out, (const uint16_t *)x, weights, scales, T, N, K};
    if (q8 && wide_pays(T, N) && ((uintptr_t)weights % 16u) == 0u) {
        const uint32_t wide = ((T + kWT - 1u) / kWT) * ((N + kWN - 1u) / kWN);
        hipLaunchKernelGGL(proj_wide_kernel, dim3(8u * ((wide + 7u) / 8u)), dim3(512), 0, st, A);
        return hipGetLastError() == hipSuccess;
    }
    const uint32_t works = ((T + kPT - 1u) / kPT) * ((N + kPT - 1u) / kPT);
    const dim3 grid(8u * ((works + 7u) / 8u));
    if (q8)
        hipLaunchKernelGGL(HIP_KERNEL_NAME(proj_mfma_kernel<true>), grid, dim3(512), 0, st, A);
    else
        hipLaunchKernelGGL(HIP_KERNEL_NAME(proj_mfma_kernel<false>), grid, dim3(512), 0, st, A);
    return hipGetLastError() == hipSuccess;
}

}  // namespace k3

extern "C" bool k3_moe_proj_mfma_bf16(void *output, const void *weights, const float *scales,
                                      const void *input, uint32_t vector_count, uint32_t rows,
                                      uint32_t columns, bool q8, void *stream) {
    if (!output || !weights || !input) return false;
    return k3::launch_proj_mfma((uint16_t *)output, input, weights, scales, vector_count, rows,
                                columns, q8, (hipStream_t)stream);
}
