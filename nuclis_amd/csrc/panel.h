// The panel tile's shapes, plan and launchers (panel.hip, panel_plan.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace nuq {

// Shape index, TG (32-token groups), RG (32-row groups per wave), WR (waves
// over the rows), WK (wave sets over K), DEPTH (activation slabs in LDS).
#define NUQ_PANEL_SHAPES(X)                                                                                         \
    X(0, 1, 1, 4, 1, 4)                                                                                            \
    X(1, 1, 1, 2, 4, 2)                                                                                            \
    X(2, 2, 1, 2, 2, 2)                                                                                            \
    X(3, 3, 1, 4, 2, 2)                                                                                            \
    X(4, 4, 1, 4, 2, 2)                                                                                            \
    X(5, 4, 1, 2, 2, 2)                                                                                            \
    X(6, 4, 1, 4, 1, 2)                                                                                            \
    X(7, 4, 2, 4, 1, 2)                                                                                            \
    X(8, 6, 2, 4, 1, 2)                                                                                            \
    X(9, 8, 2, 4, 1, 2)
constexpr int PANEL_SHAPE_COUNT = 10;
constexpr uint32_t PANEL_GROUP = 4;  // token tiles per group of the tile order (2 to 8 measured alike)

// Workgroups [0, full) each own a whole tile; the `tail` tiles after them are
// split along K into `splits` ranges of whole 256-column blocks each.
struct PanelPlan {
    int shape;
    uint32_t full, tail, splits;
    uint64_t work_floats;  // partial tiles of the split
    float cost;            // predicted time, us
};

struct PanelArgs {
    const uint8_t *w;
    uint64_t stride;
    uint32_t rows, columns;
    const _Float16 *x;
    uint64_t in_stride;
    float *y;
    uint64_t out_stride;
    uint32_t tokens;
};

// The fastest plan by the cost model on `cus` compute units with at most
// max_floats of workspace; false when the tile does not take the product.
bool panel_plan(uint32_t encoding, uint32_t rows, uint32_t columns, uint32_t tokens, uint64_t stride,
                uint64_t in_stride, uint64_t max_floats, uint32_t cus, PanelPlan *plan);
hipError_t launch_panel(hipStream_t s, uint32_t encoding, const PanelArgs &a, const PanelPlan &p, float *work);
// f32 rows of `columns` values, `in_stride` apart, to packed f16 rows.
hipError_t launch_to_f16(hipStream_t s, const float *x, uint64_t in_stride, uint32_t columns, uint32_t tokens,
                         _Float16 *out);

// One encoding's kernels, compiled on their own.
template <uint32_t ENC>
hipError_t launch_panel_enc(hipStream_t s, const PanelArgs &a, const PanelPlan &p, float *work);

// Tile id -> (token tile, row tile), XCD-contiguous and `group` token tiles deep
__device__ __forceinline__ void panel_coords(uint32_t id, uint32_t tm, uint32_t tn, uint32_t group, uint32_t *pm,
                                             uint32_t *pn) {
    const uint32_t total = tm * tn;
    if (total % 8 == 0) id = (id % 8) * (total / 8) + id / 8;
    const uint32_t per = group * tn, g = id / per, first = g * group, gm = min(tm - first, group), in = id % per;
    *pm = first + in % gm;
    *pn = in / gm;
}

}  // namespace nuq
