/*
 * Which kernel an exact per-matrix product takes (k3_rocm_mxfp4_gemm_bf16,
 * k3_rocm_q8_128_gemm_bf16): the one-wave-per-row kernels of k3_ops.hip or the
 * tiles of k3_exact.hip, and which tile. Plain C++, so that it can be checked
 * without a GPU.
 */
#pragma once

#include <stdint.h>

namespace k3 {

/* 64 or 16 weight rows of a tile, its quads of tokens per instruction group,
 * and the tiles (persistent blocks) a CU holds: 16 tokens of 64 rows take all
 * its registers. */
struct DenseForm {
    uint32_t rows, quads, per_cu;
    constexpr uint32_t tokens() const { return quads * 256u / rows; }
};

/* 16-row tiles where 64-row ones would leave CUs idle: a tile's time is the
 * floor then, and the smaller tile's is a third. Measured, 64-row against
 * 16-row: MXFP4 3072 x 3584 at 32 tokens (96 works of 64 rows x 16 tokens)
 * 23.9 against 19.2 us, at 48 (144) 24.0 against 25.2; 2048 x 7168 at 64
 * (128) 41.8 against 33.0, at 96 (192) 42.4 against 44.1. Up to 8 tokens the
 * 64-row tile is itself shorter: Q8-128 6144 x 7168 at 8 tokens (96) 32.6
 * against 35.3, 3584 x 7168 (56) 32.0 against 23.7. */
inline DenseForm dense_form(uint32_t tokens, uint32_t rows) {
    const uint64_t works = (rows / 64u + (rows % 64u != 0u)) * (uint64_t)((tokens + 15u) / 16u);
    if (works <= (tokens <= 8u ? 64u : 128u)) return {16u, 1u, 2u};
    if (tokens <= 4u) return {64u, 1u, 2u};
    if (tokens <= 8u) return {64u, 2u, 2u};
    return {64u, 4u, 1u};
}

constexpr uint32_t kCus = 256;

/* The tiles' row offsets within 32 rows are 32-bit byte counts. */
constexpr uint32_t kTileMaxColumns = 1u << 27;

/*
 * Whether the product stays on the row kernels. Their vector arithmetic takes
 * 0.0040 ns per output and 32-column group up to 16 tokens and 0.0046 above, in
 * passes of 64 groups (a wave's lanes). The tiles take their rounds over the
 * CUs times a tile's time per group (ns below; a sixth or a third more where
 * the scales no longer fit their buffer whole, over 256 groups). Up to 16384
 * outputs the row kernels, which fill the chip with less. Measured, rows against
 * tiles, us: Q8-128 6144 x 7168 at 3 tokens 21 against 25, at 4 26.2 against
 * 25.5, 7168 x 6144 at 4 28.5 against 22.9, 3000 x 16512 at 6 39 against 60,
 * 2566 x 12544 at 7 34 against 45, 252 x 9600 at 66 24 against 35, 1183 x 6528
 * at 18 30 against 24; MXFP4 3000 x 16512 at 6 38 against 50, 1596 x 9920 at 11
 * 26 against 31, 3072 x 3584 at 8 13.8 against 12.0. Of 1497 products of 16385
 * to 8 * 10^7 outputs the choice is more than 5% off the better kernel for 30
 * (the worst 6.6 against 8.1 us, MXFP4 512 x 2048 at 33 tokens).
 */
inline bool dense_rows_form(uint32_t tokens, uint32_t rows, uint32_t columns, bool q8) {
    const uint64_t outputs = (uint64_t)tokens * rows, groups = columns / 32u;
    if (tokens == 1u || outputs <= 16384u || columns > kTileMaxColumns) return true;
    const DenseForm f = dense_form(tokens, rows);
    const uint64_t works = (uint64_t)((rows + f.rows - 1u) / f.rows) *
                           ((tokens + f.tokens() - 1u) / f.tokens());
    const uint64_t rounds = (works + f.per_cu * kCus - 1u) / (f.per_cu * kCus);
    uint64_t tile = f.rows == 16u ? (q8 ? 102u : 76u)
                                  : f.quads == 1u ? (q8 ? 112u : 74u)
                                                  : f.quads == 2u ? (q8 ? 135u : 108u)
                                                                  : (q8 ? 200u : 163u);
    if (groups > 256u) tile = tile * (f.rows == 16u ? 115u : 130u) / 100u;
    const uint64_t passes = (groups + 63u) / 64u, rate = tokens <= 16u ? 40u : 46u;
    return outputs * 64u * passes * rate < rounds * groups * tile * 10000u;
}

}  // namespace k3
