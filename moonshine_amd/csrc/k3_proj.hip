/*
 * Static projections of a token batch on bf16 MFMA, for the MXFP8
 * precisions of the K3-native block (the exact precision runs
 * k3_rocm_q8_128_gemm_bf16 / k3_rocm_bf16_gemm_bf16, k3_rocm_ops.cu:663-835,
 * 1694-2038, in their w64 order).
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
 * bf16 weights: block tile 128 tokens x 128 rows, 8 waves of 32 x 64 (2 x 4
 * V_MFMA_F32_16X16X32_BF16 tiles), K steps of 64 through two LDS buffers
 * (rows padded to 144 bytes), global loads two steps ahead. Codes: tiles of
 * 64 x 64 to 256 x 128 fed by direct-to-LDS loads, chosen by the rounds they
 * take (q8_tile); the four MFMAs of a 128-column block chain in a block sum
 * that is then scaled into the accumulator with one fma per output, in every
 * tile alike: the same bits. Tiles are dealt to the XCDs in contiguous ranges,
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
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4_a8_t __attribute__((ext_vector_type(4), aligned(8)));

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

/* The thread's two rows of one K step of x and of the weights. */
__device__ __forceinline__ void proj_load(uint4 &a0, uint4 &a1, uint4 &b0, uint4 &b1,
                                          const uint8_t *xb, const uint8_t *wb, uint32_t ao0,
                                          uint32_t ao1, uint32_t bo0, uint32_t bo1, uint32_t s) {
    const uint32_t k = 2u * kPK * s;
    a0 = *(const uint4 *)(xb + ao0 + k);
    a1 = *(const uint4 *)(xb + ao1 + k);
    b0 = *(const uint4 *)(wb + bo0 + k);
    b1 = *(const uint4 *)(wb + bo1 + k);
}

__device__ __forceinline__ void proj_store(ProjStage &buf, uint32_t off, const uint4 &a0,
                                           const uint4 &a1, const uint4 &b0, const uint4 &b1) {
    constexpr uint32_t R64 = 64u * kPPad;
    *(uint4 *)(buf[0] + off) = a0;
    *(uint4 *)(buf[0] + off + R64) = a1;
    *(uint4 *)(buf[1] + off) = b0;
    *(uint4 *)(buf[1] + off + R64) = b1;
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
    uint32_t ao[2], bo[2];
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const uint32_t ta = t0 + r0 + 64u * i, nb = n0 + r0 + 64u * i;
        ao[i] = ((ta < T ? ta : T - 1u) * K + 8u * pc) * 2u;
        bo[i] = ((nb < N ? nb : N - 1u) * K + 8u * pc) * 2u;
    }
    const uint8_t *xb = (const uint8_t *)P.x, *wb = (const uint8_t *)P.w;
    const uint32_t soff = r0 * kPPad + 16u * pc;
    const uint32_t a_off = (32u * wm + c) * kPPad + 16u * g;
    const uint32_t b_off = (64u * wn + c) * kPPad + 16u * g;
    f32x4_t acc[2][4];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) acc[i][j] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    const uint32_t nsteps = K / kPK, last = nsteps - 1u;
    /* two register sets: step s + 2's loads are issued at the start of
     * step s; loads and stores are unconditional (steps past the end
     * reload the last one into a buffer nobody reads) */
    uint4 a0, a1, b0, b1, p0, p1, q0, q1;
    proj_load(a0, a1, b0, b1, xb, wb, ao[0], ao[1], bo[0], bo[1], 0u);
    proj_load(p0, p1, q0, q1, xb, wb, ao[0], ao[1], bo[0], bo[1], 1u < last ? 1u : last);
    proj_store(lds[0], soff, a0, a1, b0, b1);
    __syncthreads();
    for (uint32_t s = 0; s < nsteps; s += 2u) {
        proj_load(a0, a1, b0, b1, xb, wb, ao[0], ao[1], bo[0], bo[1],
                      s + 2u < last ? s + 2u : last);
        proj_compute(acc, lds[0], a_off, b_off);
        proj_store(lds[1], soff, p0, p1, q0, q1);
        __syncthreads();
        if (s + 1u < nsteps) {
            proj_load(p0, p1, q0, q1, xb, wb, ao[0], ao[1], bo[0], bo[1],
                      s + 3u < last ? s + 3u : last);
            proj_compute(acc, lds[1], a_off, b_off);
            proj_store(lds[0], soff, a0, a1, b0, b1);
            __syncthreads();
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
 * 308 -> 251 (226 on the 128 x 128 tiles below, which q8_tile gives that size),
 * 7168 x 3584 201 -> 127; 8192 tokens 1231 -> 805, 724 -> 468.
 */
constexpr uint32_t kWT = 256, kWN = 128;              /* block tile */
constexpr uint32_t kWA = kWT * 128u, kWB = kWN * 128u; /* bytes of a stage */

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
    auto codes = [&](uint32_t s) { return (u32x4_t) * (const u32x4_a8_t *)(ws + kPK * (s < last ? s : last)); };
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
    fetch(1u, 1u);
    asm volatile("" ::: "memory");
    q0 = codes(2u); /* the order the stages' waits count */
#pragma unroll
    for (int j = 0; j < 4; j++) sc[j] = srow[j][0];
    asm volatile("" ::: "memory");
    uint32_t slot = 0u;
    /* stage s from `slot`; next: the codes of s + 1, refilled with s + 3 */
    auto stage = [&](uint32_t s, u32x4_t &next, auto Odd) {
        constexpr bool odd = decltype(Odd)::value;
        /* This wave's loads of stage s are done before the barrier, behind
         * which its neighbours read them. Issued after those four: for stage
         * 0 fetch(1), the codes of 2 and four scales (9); for stage 1 these
         * five, fetch(2) and the codes of 3 (10); from stage 2 on fetch(s + 1),
         * the codes of s + 1 and s + 2 and, at the odd stage of the two, four
         * scales (10). */
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

/*
 * The Q8-128 form for fewer tokens: 16 WT WM tokens x 16 NR WN rows of eight
 * waves, everything by direct-to-LDS loads into a ring of RING stages of one
 * scale block (128 columns: tokens as bf16, codes as bytes, each wave's
 * scales), explicit LDS accesses and waits as above. Codes become bf16 after
 * their LDS read. A stage is LDS reads (12 to 20 KB a wave), then conversions
 * and MFMAs. With two row subtiles a wave the two waves of a SIMD take turns:
 * waves 4..7 run one barrier behind, so one half reads while the other
 * multiplies (64 x 128 tiles, 7168 columns: 53 -> 43 us a round, 128 x 128 72
 * -> 70; with conversions and scaling in the reading phase 59 and 83; 64 x 64
 * tiles 36 either way, 1024 columns 7.8 and 8.2; the 256 x 128 tiles above 124
 * either way, 3584 columns 62 and 65). Conversions (1.5 instructions a code,
 * once per token half) and MFMAs share the SIMD's issue: without any load in
 * the loop a round still takes 29, 38 and 55 us. A 128 x 128 tile staged
 * through registers two steps ahead took 103 us for 7168 columns at any token
 * count up to a round. Before -> after, us: 6144 x 7168, 96 tokens 102 -> 36,
 * 300 tokens 103 -> 45, 512 tokens 104 -> 72, 1536 tokens 305 (248 on the tile
 * above) -> 211; 7168 x 3584, 96 tokens 51 -> 19; 1024 x 1024, 96 tokens 17 ->
 * 7.8.
 */
/* The fragments of two 32-column steps, and of a stage where they fit, each
 * read by one statement that waits for them. */
template <int WT, int NR>
struct RingFrags {
    u32x4_t a[2][WT];
    u32x2_t b[2][NR];
};
__device__ __forceinline__ void ring_read(RingFrags<4, 2> &f, uint32_t a0, uint32_t a1, uint32_t b0,
                                          uint32_t b1) {
    asm volatile(
        "ds_read_b128 %0, %12\n\tds_read_b128 %1, %12 offset:2048\n\t"
        "ds_read_b128 %2, %12 offset:4096\n\tds_read_b128 %3, %12 offset:6144\n\t"
        "ds_read_b64 %8, %14\n\tds_read_b64 %9, %14 offset:2048\n\t"
        "ds_read_b128 %4, %13\n\tds_read_b128 %5, %13 offset:2048\n\t"
        "ds_read_b128 %6, %13 offset:4096\n\tds_read_b128 %7, %13 offset:6144\n\t"
        "ds_read_b64 %10, %15\n\tds_read_b64 %11, %15 offset:2048\n\ts_waitcnt lgkmcnt(0)"
        : "=&v"(f.a[0][0]), "=&v"(f.a[0][1]), "=&v"(f.a[0][2]), "=&v"(f.a[0][3]), "=&v"(f.a[1][0]),
          "=&v"(f.a[1][1]), "=&v"(f.a[1][2]), "=&v"(f.a[1][3]), "=&v"(f.b[0][0]), "=&v"(f.b[0][1]),
          "=&v"(f.b[1][0]), "=&v"(f.b[1][1])
        : "v"(a0), "v"(a1), "v"(b0), "v"(b1)
        : "memory");
}


template <uint32_t H> /* bytes between the two halves of the tokens */
__device__ __forceinline__ void ring_read(RingFrags<2, 1> (&f)[2], const uint32_t (&a)[2],
                                          const uint32_t (&b)[4]) {
    asm volatile(
        "ds_read_b128 %0, %12\n\tds_read_b128 %1, %12 offset:2048\n\tds_read_b64 %8, %14\n\t"
        "ds_read_b128 %2, %13\n\tds_read_b128 %3, %13 offset:2048\n\tds_read_b64 %9, %15\n\t"
        "ds_read_b128 %4, %12 offset:%18\n\tds_read_b128 %5, %12 offset:%19\n\tds_read_b64 %10, %16\n\t"
        "ds_read_b128 %6, %13 offset:%18\n\tds_read_b128 %7, %13 offset:%19\n\tds_read_b64 %11, %17\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(f[0].a[0][0]), "=&v"(f[0].a[0][1]), "=&v"(f[0].a[1][0]), "=&v"(f[0].a[1][1]),
          "=&v"(f[1].a[0][0]), "=&v"(f[1].a[0][1]), "=&v"(f[1].a[1][0]), "=&v"(f[1].a[1][1]),
          "=&v"(f[0].b[0][0]), "=&v"(f[0].b[1][0]), "=&v"(f[1].b[0][0]), "=&v"(f[1].b[1][0])
        : "v"(a[0]), "v"(a[1]), "v"(b[0]), "v"(b[1]), "v"(b[2]), "v"(b[3]), "i"(H), "i"(H + 2048u)
        : "memory");
}
template <uint32_t H>
__device__ __forceinline__ void ring_read(RingFrags<2, 2> (&f)[2], const uint32_t (&a)[2],
                                          const uint32_t (&b)[4]) {
    asm volatile(
        "ds_read_b128 %0, %16\n\tds_read_b128 %1, %16 offset:2048\n\t"
        "ds_read_b64 %8, %18\n\tds_read_b64 %9, %18 offset:2048\n\t"
        "ds_read_b128 %2, %17\n\tds_read_b128 %3, %17 offset:2048\n\t"
        "ds_read_b64 %10, %19\n\tds_read_b64 %11, %19 offset:2048\n\t"
        "ds_read_b128 %4, %16 offset:%22\n\tds_read_b128 %5, %16 offset:%23\n\t"
        "ds_read_b64 %12, %20\n\tds_read_b64 %13, %20 offset:2048\n\t"
        "ds_read_b128 %6, %17 offset:%22\n\tds_read_b128 %7, %17 offset:%23\n\t"
        "ds_read_b64 %14, %21\n\tds_read_b64 %15, %21 offset:2048\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(f[0].a[0][0]), "=&v"(f[0].a[0][1]), "=&v"(f[0].a[1][0]), "=&v"(f[0].a[1][1]),
          "=&v"(f[1].a[0][0]), "=&v"(f[1].a[0][1]), "=&v"(f[1].a[1][0]), "=&v"(f[1].a[1][1]),
          "=&v"(f[0].b[0][0]), "=&v"(f[0].b[0][1]), "=&v"(f[0].b[1][0]), "=&v"(f[0].b[1][1]),
          "=&v"(f[1].b[0][0]), "=&v"(f[1].b[0][1]), "=&v"(f[1].b[1][0]), "=&v"(f[1].b[1][1])
        : "v"(a[0]), "v"(a[1]), "v"(b[0]), "v"(b[1]), "v"(b[2]), "v"(b[3]), "i"(H), "i"(H + 2048u)
        : "memory");
}

/* Between two phases of the alternating form. */
__device__ __forceinline__ void phase_barrier() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}

template <int WT, int NR, int WM, int RING>
struct Ring {
    static constexpr uint32_t WN = 8 / WM, TT = 16 * WT * WM, TN = 16 * NR * WN;
    static constexpr uint32_t A = 256u * TT, B = 128u * TN, S = 2048u; /* bytes of a stage */
    static constexpr uint32_t STAGE = A + B + S;
    static constexpr int DA = TT / 32, DB = TN / 64, D = DA + DB + 1; /* loads a wave and stage */
    static constexpr bool ALT = NR == 2; /* the halves of the block alternate */
    static_assert(WT == 2 || ALT, "four token subtiles read by halves of a stage");
    static_assert(RING * STAGE <= 160u * 1024u, "LDS");
};

template <int WT, int NR, int WM, int RING>
__global__ __launch_bounds__(512) void proj_ring_kernel(ProjArgs P) {
    using C = Ring<WT, NR, WM, RING>;
    __shared__ __attribute__((aligned(16))) uint8_t smem[RING * C::STAGE];
    const uint32_t T = P.T, N = P.N, K = P.K;
    const uint32_t ntt = (T + C::TT - 1u) / C::TT, nnt = (N + C::TN - 1u) / C::TN;
    const uint32_t works = ntt * nnt, per = (works + 7u) / 8u;
    const uint32_t j8 = blockIdx.x >> 3, wk = (blockIdx.x & 7u) * per + j8;
    if (j8 >= per || wk >= works) return;
    const uint32_t t0 = (wk / nnt) * C::TT, n0 = (wk % nnt) * C::TN;
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t wm = wave / C::WN, wn = wave % C::WN, g = lane >> 4, c = lane & 15u;
    const uint32_t lds = lds_addr(smem);
    /* 1 KB chunks (8 rows x 128 bytes) of each wave: tokens [64 columns][16
     * rows][8 rows], codes [16 rows][8 rows]; rows past T or N repeat the
     * last one (not stored) */
    const uint8_t *xs[C::DA], *ws[C::DB];
#pragma unroll
    for (int m = 0; m < C::DA; m++) {
        const uint32_t q = C::DA * wave + (uint32_t)m, h = q & 1u, col = q / (C::TT / 8u);
        const uint32_t r = t0 + 16u * (q % (C::TT / 8u) >> 1) + a_dma_row(lane, h);
        xs[m] = (const uint8_t *)P.x + 2ull * (r < T ? r : T - 1u) * K + 128u * col + 16u * a_dma_piece(lane, h);
    }
#pragma unroll
    for (int m = 0; m < C::DB; m++) {
        const uint32_t q = C::DB * wave + (uint32_t)m, h = q & 1u;
        const uint32_t r = n0 + 16u * (q >> 1) + a_dma_row(lane, h);
        ws[m] = (const uint8_t *)P.w + (uint64_t)(r < N ? r : N - 1u) * K + 16u * a_dma_piece(lane, h);
    }
    const uint32_t nblk = K / 128u, last = nblk - 1u;
    const uint32_t sr = n0 + 16u * NR * wn + (lane & (16u * NR - 1u));
    const float *sp = P.scales + (uint64_t)(sr < N ? sr : N - 1u) * nblk;
    auto fetch = [&](uint32_t s, uint32_t base) { /* past the end: the last stage again */
        const uint32_t b = s < last ? s : last;
#pragma unroll
        for (int m = 0; m < C::DB; m++)
            __builtin_amdgcn_global_load_lds((const void *)(ws[m] + 128u * b),
                                             (lds_void *)(uintptr_t)(base + C::A + 1024u * (C::DB * wave + m)),
                                             16, 0, 0);
        __builtin_amdgcn_global_load_lds((const void *)(sp + b),
                                         (lds_void *)(uintptr_t)(base + C::A + C::B + 256u * wave), 4, 0, 0);
#pragma unroll
        for (int m = 0; m < C::DA; m++)
            __builtin_amdgcn_global_load_lds((const void *)(xs[m] + 256u * b),
                                             (lds_void *)(uintptr_t)(base + 1024u * (C::DA * wave + m)), 16,
                                             0, 0);
    };
    f32x4_t acc[WT][NR];
#pragma unroll
    for (int i = 0; i < WT; i++)
#pragma unroll
        for (int j = 0; j < NR; j++) acc[i][j] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    const uint32_t a_base = 2048u * WT * wm, b_base = C::A + 2048u * NR * wn;
    const uint32_t aslot[2] = {a_base + a_slot(c, g), a_base + a_slot(c, 4u + g)};
    uint32_t bslot[4];
#pragma unroll
    for (uint32_t k = 0; k < 4u; k++) bslot[k] = b_base + a_slot(c, 2u * k + (g >> 1)) + 8u * (g & 1u);
    const uint32_t s_slot = C::A + C::B + 256u * wave + 4u * c;
#pragma unroll
    for (uint32_t s = 0; s < RING - 1u; s++) fetch(s, lds + C::STAGE * s);
    uint32_t cur = lds, free_ = lds + C::STAGE * (RING - 1u);
    const uint32_t end = lds + C::STAGE * RING;
    if constexpr (C::ALT) {
        wait_vm<C::D *(RING - 2)>(); /* stage 0 */
        phase_barrier();
        if (wave >= 4u) phase_barrier();
    }
    for (uint32_t s = 0; s < nblk; s++) {
        if constexpr (!C::ALT) {
            wait_vm<C::D *(RING - 2)>(); /* this wave's loads of stage s */
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
        }
        fetch(s + RING - 1u, free_); /* stage s - 1's slot: every wave has read it */
        f32x4_t blk[WT][NR];
        float sc[NR];
        if constexpr (NR == 1)
            asm volatile("ds_read_b32 %0, %1\n\ts_waitcnt lgkmcnt(0)" : "=&v"(sc[0]) : "v"(cur + s_slot) : "memory");
        else
            asm volatile("ds_read_b32 %0, %2\n\tds_read_b32 %1, %2 offset:64\n\ts_waitcnt lgkmcnt(0)"
                         : "=&v"(sc[0]), "=&v"(sc[1])
                         : "v"(cur + s_slot)
                         : "memory");
        const uint32_t as[2] = {cur + aslot[0], cur + aslot[1]};
        const uint32_t bs[4] = {cur + bslot[0], cur + bslot[1], cur + bslot[2], cur + bslot[3]};
        RingFrags<WT, NR> fr[2];
        if constexpr (WT == 2) {
            ring_read<128u * C::TT>(fr, as, bs);
            if constexpr (C::ALT) {
                wait_vm<C::D *(RING - 2)>(); /* this wave's loads of stage s + 1 */
                phase_barrier();
            }
        }
#pragma unroll
        for (int h = 0; h < 2; h++) {
            RingFrags<WT, NR> &f = fr[h];
            if constexpr (WT == 4) {
                ring_read(f, as[0] + 128u * C::TT * h, as[1] + 128u * C::TT * h, bs[2 * h], bs[2 * h + 1]);
                if (h == 1) wait_vm<C::D *(RING - 2)>();
                phase_barrier();
            }
#pragma unroll
            for (int ks = 0; ks < 2; ks++)
#pragma unroll
                for (int j = 0; j < NR; j++) {
                    const bf16x8_t b = __builtin_bit_cast(
                        bf16x8_t, codes_to_bf16(make_uint2(f.b[ks][j][0], f.b[ks][j][1])));
#pragma unroll
                    for (int i = 0; i < WT; i++)
                        blk[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                            __builtin_bit_cast(bf16x8_t, f.a[ks][i]), b,
                            h == 0 && ks == 0 ? f32x4_t{0.0f, 0.0f, 0.0f, 0.0f} : blk[i][j], 0, 0, 0);
                }
            if (WT == 4 && h == 0) phase_barrier();
        }
#pragma unroll
        for (int i = 0; i < WT; i++)
#pragma unroll
            for (int j = 0; j < NR; j++)
#pragma unroll
                for (int r = 0; r < 4; r++) acc[i][j][r] = fmaf(blk[i][j][r], sc[j], acc[i][j][r]);
        if constexpr (C::ALT) phase_barrier();
        free_ = cur;
        cur += C::STAGE;
        if (cur == end) cur = lds;
    }
    if constexpr (C::ALT) {
        if (wave < 4u) phase_barrier();
    }
    wait_vm<0>(); /* the loads past the end land before the LDS is given back */
#pragma unroll
    for (int i = 0; i < WT; i++)
#pragma unroll
        for (int j = 0; j < NR; j++) {
            const uint32_t n = n0 + 16u * (NR * wn + (uint32_t)j) + c;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const uint32_t t = t0 + 16u * (WT * wm + (uint32_t)i) + 4u * g + (uint32_t)r;
                if (t < T && n < N) P.out[(uint64_t)t * N + n] = f32_to_bf16(acc[i][j][r]);
            }
        }
}

template <int WT, int NR, int WM, int RING>
bool launch_ring(const ProjArgs &A, hipStream_t st) {
    using C = Ring<WT, NR, WM, RING>;
    const uint32_t works = ((A.T + C::TT - 1u) / C::TT) * ((A.N + C::TN - 1u) / C::TN);
    hipLaunchKernelGGL(HIP_KERNEL_NAME(proj_ring_kernel<WT, NR, WM, RING>),
                       dim3(8u * ((works + 7u) / 8u)), dim3(512), 0, st, A);
    return hipGetLastError() == hipSuccess;
}

/* Every Q8 tile holds one block a CU, so a call takes its rounds of tiles over
 * the 256 CUs times a round: 64 x 64 tokens x rows 36 us of 7168 columns, 64 x
 * 128 43, 128 x 128 71 and 256 x 128 124. The cheapest, the larger tile of
 * equals. (6144 x 7168, us: 300 tokens 45 on 64 x 128, 68 on 64 x 64; 512
 * tokens 72 on 128 x 128, 101 on 64 x 64; 1280 tokens 129 on 256 x 128, 151 on
 * 128 x 128; 1536 tokens 211 on 128 x 128, 248 on 256 x 128.)
 */
int q8_tile(uint32_t T, uint32_t N) {
    static constexpr uint32_t tt[4] = {64u, 64u, 128u, 256u}, tn[4] = {64u, 128u, 128u, 128u};
    static constexpr uint32_t cost[4] = {10u, 12u, 20u, 35u};
    int best = 0;
    uint64_t least = ~0ull;
    for (int i = 0; i < 4; i++) {
        const uint64_t works = (uint64_t)((T + tt[i] - 1u) / tt[i]) * ((N + tn[i] - 1u) / tn[i]);
        const uint64_t t = (works + 255u) / 256u * cost[i];
        if (t <= least) least = t, best = i;
    }
    return best;
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
    if (q8) {
        const int tile = q8_tile(T, N);
        /* One scale block: nothing to prefetch and the output's stores bound
         * it, so 64 x 64 tiles of two stages, three a CU, in place of all but
         * the largest. 128 columns, us, the tiles of longer rows -> here: 20000
         * rows, 300 tokens 11.9 -> 9.1, 1024 28.3 -> 22.1; 14879 rows, 2167
         * tokens 42.5 -> 32.9 (20000 rows, 5000 tokens: 89 on the largest, 99). */
        if (K == 128u && tile != 3) return launch_ring<2, 1, 2, 2>(A, st);
        switch (tile) {
        case 0: return launch_ring<2, 1, 2, 6>(A, st);
        case 1: return launch_ring<2, 2, 2, 4>(A, st);
        case 2: return launch_ring<4, 2, 2, 3>(A, st);
        }
        const uint32_t works = ((T + kWT - 1u) / kWT) * ((N + kWN - 1u) / kWN);
        hipLaunchKernelGGL(proj_wide_kernel, dim3(8u * ((works + 7u) / 8u)), dim3(512), 0, st, A);
        return hipGetLastError() == hipSuccess;
    }
    const uint32_t works = ((T + kPT - 1u) / kPT) * ((N + kPT - 1u) / kPT);
    hipLaunchKernelGGL(proj_mfma_kernel, dim3(8u * ((works + 7u) / 8u)), dim3(512), 0, st, A);
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
