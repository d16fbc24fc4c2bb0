/*
 * Token batches in the exact w64 order on the fp32 matrix units
 * (k3_exact.hip): the routed experts of a batch, and the per-matrix MXFP4 and
 * Q8-128 entry points. Same bits as the one-wave-per-row kernels.
 */
#pragma once

#include "k3_moe.h"

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace k3 {

/* Tile lists of the selected experts: an expert of at most kLightRows plan
 * rows is one record of the light list; the others have one record of the
 * heavy list per kHeavyTile rows, an expert's tiles together. */
constexpr uint32_t kLightRows = 8, kHeavyTile = 16;
struct ExactTile {
    uint32_t expert, base, rows, first; /* expert, its plan rows [base, base + rows), its first
                                           record's index */
};
inline uint32_t exact_light_cap(uint32_t routes, uint32_t E) { return routes < E ? routes : E; }
inline uint32_t exact_heavy_cap(uint32_t routes, uint32_t E) {
    const uint32_t experts = routes / (kLightRows + 1u);
    return routes / kHeavyTile + (experts < E ? experts : E);
}
inline size_t exact_list_bytes(uint32_t routes, uint32_t E) { /* counts, light, heavy */
    return 16u + sizeof(ExactTile) * ((size_t)exact_light_cap(routes, E) +
                                      exact_heavy_cap(routes, E));
}

struct ExactGroup {
    uint8_t *lists;              /* exact_list_bytes, 16-byte aligned */
    const uint32_t *list;        /* instead of the tile lists: a count, then expert ids */
    const uint32_t *counts, *offsets; /* of the plan */
    const uint32_t *token_index, *route_index;
    const k3_moe_expert *experts;
    uint32_t tokens, routes, E, H, F;
};

/* The plan is on the stream already; E <= 1024. */
bool launch_exact_tiles(const ExactGroup &g, hipStream_t st);
/* act[plan row, F] = bf16(act(bf16(gate . x), bf16(up . x))), x [tokens, H] */
bool launch_exact_gateup(const ExactGroup &g, uint16_t *act, const uint16_t *x, uint32_t kind,
                         float beta, float lb, hipStream_t st);
/* y[route, H] = bf16(down . act[plan row]) */
bool launch_exact_down(const ExactGroup &g, uint16_t *y, const uint16_t *act, hipStream_t st);

/* out [tokens, rows] = w [rows, cols] . x [tokens, cols]; x 16-byte aligned.
 * MXFP4: cols % 32 == 0; Q8-128 (int8 codes, f32 scales): cols % 128 == 0;
 * which products come here: dense_rows_form (k3_exact_rule.h). */
bool launch_exact_mxfp4(uint16_t *out, const void *packed, const void *scales, const void *x,
                        uint32_t tokens, uint32_t rows, uint32_t cols, hipStream_t st);
bool launch_exact_q8(uint16_t *out, const void *codes, const void *scales, const void *x,
                     uint32_t tokens, uint32_t rows, uint32_t cols, hipStream_t st);

}  // namespace k3
