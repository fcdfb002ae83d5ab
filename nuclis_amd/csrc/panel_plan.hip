// Host side of the panel tile: the choice of shape and K split, the reduction
// of split tiles and the f32 -> f16 pass over the activations.
#include <algorithm>

#include "kernels.h"
#include "panel.h"

namespace nuq {

// Predicted time of one launch. A CU holds `occ` workgroups of a shape at once
// (its LDS and registers); a round of the grid with q workgroups on the busiest
// CU takes a + n (b + c (q - 1)) us, n the 256-column blocks of a wave set. A
// split adds r0 us and r1 us per MB of partial sums. Fitted per encoding and
// shape to 11,421 timings on MI355X (six matrices from 1024 x 5120 to 17408 x
// 5120, 4 to 4096 tokens; profiles/fit_costs.py prints this table from them):
// relative error 5-10 % rms, and the plan chosen takes 1.02 of the best measured
// plan's time on average (at most 1.32). Encodings 8, 12, 13, 14, 23.
struct PanelCost {
    uint8_t occ;
    float a, b, c, r0, r1;
};
static const PanelCost PANEL_COST[5][PANEL_SHAPE_COUNT] = {
    {  // q8_0
        {3, 0.67f, 2.250f, 1.871f, 8.9f, 0.215f},
        {1, 3.22f, 4.659f, 0.000f, 6.2f, 0.000f},
        {2, 1.93f, 2.998f, 2.094f, 6.8f, 0.227f},
        {1, 1.91f, 5.594f, 0.000f, 9.3f, 0.281f},
        {1, 2.97f, 6.253f, 0.000f, 8.3f, 0.255f},
        {1, 3.79f, 3.794f, 0.000f, 6.2f, 0.164f},
        {2, 1.88f, 3.235f, 2.191f, 9.5f, 0.206f},
        {1, 2.97f, 5.908f, 0.000f, 7.9f, 0.337f},
        {1, 4.17f, 6.897f, 0.000f, 7.6f, 0.337f},
        {1, 6.09f, 7.944f, 0.000f, 7.0f, 0.348f},
    },
    {  // q4_k
        {4, 1.50f, 1.299f, 0.694f, 7.5f, 0.319f},
        {2, 2.38f, 2.236f, 1.591f, 6.0f, 0.000f},
        {3, 2.30f, 1.980f, 0.940f, 6.8f, 0.193f},
        {1, 3.34f, 3.107f, 0.000f, 9.3f, 0.150f},
        {1, 3.44f, 4.004f, 0.000f, 7.7f, 0.249f},
        {1, 4.56f, 3.001f, 0.000f, 6.7f, 0.005f},
        {2, 0.69f, 2.415f, 1.487f, 11.1f, 0.145f},
        {2, 1.50f, 3.912f, 3.380f, 10.3f, 0.222f},
        {1, 5.52f, 5.013f, 0.000f, 7.6f, 0.280f},
        {1, 6.53f, 6.067f, 0.000f, 7.6f, 0.312f},
    },
    {  // q5_k
        {4, 0.83f, 1.510f, 0.821f, 8.5f, 0.266f},
        {2, 2.43f, 2.545f, 1.838f, 6.1f, 0.000f},
        {2, 2.67f, 2.063f, 0.917f, 6.9f, 0.093f},
        {1, 2.93f, 3.361f, 0.000f, 8.9f, 0.200f},
        {1, 3.02f, 4.285f, 0.000f, 7.6f, 0.273f},
        {1, 4.21f, 3.099f, 0.000f, 6.6f, 0.038f},
        {2, 2.60f, 2.407f, 1.691f, 9.0f, 0.167f},
        {2, 0.00f, 5.073f, 3.105f, 10.2f, 0.274f},
        {1, 4.88f, 5.206f, 0.000f, 7.8f, 0.297f},
        {1, 5.97f, 6.167f, 0.000f, 7.9f, 0.322f},
    },
    {  // q6_k
        {3, 0.41f, 1.741f, 0.880f, 9.5f, 0.251f},
        {1, 2.96f, 3.188f, 0.000f, 5.7f, 0.000f},
        {2, 2.71f, 2.454f, 1.180f, 7.3f, 0.131f},
        {1, 2.91f, 4.180f, 0.000f, 9.3f, 0.218f},
        {1, 3.04f, 5.144f, 0.000f, 8.1f, 0.268f},
        {1, 4.59f, 3.674f, 0.000f, 6.7f, 0.070f},
        {2, 2.89f, 2.739f, 1.953f, 9.1f, 0.180f},
        {1, 2.84f, 4.866f, 0.000f, 8.8f, 0.309f},
        {1, 4.64f, 6.014f, 0.000f, 8.0f, 0.316f},
        {1, 4.99f, 7.191f, 0.000f, 7.1f, 0.360f},
    },
    {  // iq4_xs
        {4, 0.42f, 1.779f, 0.939f, 8.7f, 0.300f},
        {2, 2.15f, 3.031f, 2.017f, 6.3f, 0.021f},
        {3, 1.76f, 2.506f, 1.178f, 7.4f, 0.171f},
        {1, 2.30f, 4.096f, 0.000f, 11.0f, 0.089f},
        {1, 2.59f, 5.228f, 0.000f, 9.2f, 0.215f},
        {1, 4.34f, 3.379f, 0.000f, 7.2f, 0.014f},
        {2, 1.77f, 3.763f, 1.335f, 10.5f, 0.178f},
        {2, 0.36f, 4.202f, 3.839f, 11.3f, 0.224f},
        {1, 5.03f, 5.159f, 0.000f, 8.0f, 0.291f},
        {1, 6.02f, 6.189f, 0.000f, 8.6f, 0.316f},
    },
};

struct PanelShape {
    uint8_t tg, rg, wr, wk, depth;
};
#define NUQ_PANEL_ROW(I, T, R, W, K, D) {T, R, W, K, D},
static const PanelShape PANEL_SHAPES[PANEL_SHAPE_COUNT] = {NUQ_PANEL_SHAPES(NUQ_PANEL_ROW)};
#undef NUQ_PANEL_ROW

static int encoding_index(uint32_t encoding) {
    return encoding == 8 ? 0 : encoding == 12 ? 1 : encoding == 13 ? 2 : encoding == 14 ? 3 : encoding == 23 ? 4 : -1;
}

// `count` workgroups of `blocks` 256-column blocks each
static float rounds_cost(const PanelCost &k, uint32_t cus, uint32_t wk, uint32_t count, uint32_t blocks) {
    if (count == 0) return 0.f;
    const uint32_t cap = cus * k.occ, whole = count / cap, rest = count % cap;
    const float n = (float)((blocks + wk - 1) / wk);
    float t = (float)whole * (k.a + n * (k.b + k.c * (float)(k.occ - 1)));
    if (rest) t += k.a + n * (k.b + k.c * (float)((rest + cus - 1) / cus - 1));
    return t;
}

bool panel_plan(uint32_t encoding, uint32_t rows, uint32_t columns, uint32_t tokens, uint64_t stride,
                uint64_t in_stride, uint64_t max_floats, uint32_t cus, PanelPlan *plan) {
    const int e = encoding_index(encoding);
    if (e < 0 || columns % 256 != 0 || tokens == 0) return false;
    // copies use 32-bit offsets within a tile (at most 256 rows or tokens)
    if (256 * stride > 0xffffffffull || 256 * in_stride * 2 + 2ull * columns > 0xffffffffull) return false;
    const uint32_t nb = columns / 256;
    const uint32_t groups = (tokens + 31) / 32;
    // Shapes of more token groups than the tokens fill only add padding, and
    // small ones decode the weights once more per token tile: not considered
    // beyond two tiles, except for rows of one block, where only the one-group
    // shape and those of four groups and more have no second K set, and a tile
    // is bound by its start-up (4096 x 256 at 96 tokens on one / four groups:
    // IQ4_XS 5.5 / 12.7 us, Q4_K 5.0 / 8.1; at 200 tokens 6.0 / 14.1, 5.6 / 8.9).
    bool found = false;
    for (int i = 0; i < PANEL_SHAPE_COUNT; ++i) {
        const PanelShape &s = PANEL_SHAPES[i];
        const PanelCost &k = PANEL_COST[e][i];
        if (s.tg > groups || (s.tg < 4 && groups > 2u * s.tg && nb > 1) || nb < s.wk) continue;
        const uint32_t bm = 32 * s.tg, bn = 32 * s.rg * s.wr, cap = cus * k.occ;
        const uint64_t tiles64 = (uint64_t)((tokens + bm - 1) / bm) * ((rows + bn - 1) / bn);
        if (tiles64 > 0x7fffffffu / 32) continue;
        const uint32_t tiles = (uint32_t)tiles64;
        const auto consider = [&](uint32_t tail, uint32_t splits, float margin = 1.f) {
            const uint64_t floats = splits > 1 ? (uint64_t)tail * splits * bm * bn : 0;
            if (floats > max_floats) return;
            float t;
            if (splits == 1) {
                t = rounds_cost(k, cus, s.wk, tiles, nb);
            } else {
                // the reduction moves the partial sums of real tokens and rows once in, and the results out
                const float sums = tail == tiles ? std::min((float)tail * bm * bn, (float)tokens * rows) : (float)tail * bm * bn;
                t = rounds_cost(k, cus, s.wk, tiles - tail, nb) + rounds_cost(k, cus, s.wk, tail * splits, (nb + splits - 1) / splits) +
                    k.r0 + k.r1 * 4e-6f * sums * ((float)splits + 0.5f);
            }
            t *= margin;
            if (found && t >= plan->cost) return;
            found = true;
            *plan = {i, splits > 1 ? tiles - tail : tiles, splits > 1 ? tail : 0, splits, floats, t};
        };
        consider(0, 1);
        // all tiles split, to one to four workgroups per CU, or as far as the
        // blocks go where the tiles are too few for one: 64 x 17408 at 200 tokens
        // 14.7 (Q4_K) to 15.8 us (IQ4_XS) split 24 ways, 104 and 119 in whole
        // tiles. The model is a little low with idle CUs (Q6_K 1024 x 5120 at 128
        // tokens 15.4 us against 13.4 on the next plan), so there a split has to
        // win by 15 %.
        if (tiles < 2 * cap) {
            const uint32_t most = std::min(24u, nb / s.wk);
            if (cus / tiles > most && most > 1) consider(tiles, most, 1.15f);
            for (uint32_t u = cus; u <= 4 * cus; u += cus)
                for (uint32_t r = 0; r < 2; ++r) {
                    const uint32_t sp = r ? (u + tiles - 1) / tiles : u / tiles;
                    if (sp > 1 && sp <= most) consider(tiles, sp);
                }
        }
        // only the tiles of a partial last round split
        if (tiles > cap && tiles % cap != 0)
            for (uint32_t sp = 2; sp <= 4 && sp * s.wk <= nb; ++sp) consider(tiles % cap, sp);
    }
    return found;
}

// The plan as plain numbers (shape, full, tail, splits, partial floats, then the
// shape's tokens and rows of a tile, its K sets and the predicted ns), for
// checks on the host; 0 when the tile does not take the product.
extern "C" int nuq_panel_plan(uint32_t encoding, uint32_t rows, uint32_t columns, uint32_t tokens, uint64_t stride,
                              uint64_t in_stride, uint64_t max_floats, uint32_t cus, uint64_t out[9]) {
    PanelPlan p;
    if (!panel_plan(encoding, rows, columns, tokens, stride, in_stride, max_floats, cus, &p)) return 0;
    const PanelShape &s = PANEL_SHAPES[p.shape];
    const uint64_t v[9] = {(uint64_t)p.shape, p.full, p.tail, p.splits, p.work_floats,
                           32ull * s.tg, 32ull * s.rg * s.wr, s.wk, (uint64_t)(p.cost * 1e3f)};
    std::copy(v, v + 9, out);
    return 1;
}

// Adds a split tile's partial sums in split order (results do not depend on
// which split ran first) and stores them, four rows of one token a thread.
// Bound by the latency of the loads, whose lines other XCDs wrote: four splits'
// go out together (the last one's again past the end, not added). One load per
// turn of the loop waited for each in turn: with the product, Q6_K 5120 x 17408
// at 8 tokens 32.1 us against 28.8, Q5_K 5120 x 6144 at 77 tokens 22.3 against 21.6.
__global__ void __launch_bounds__(256) panel_reduce_kernel(const float *__restrict__ work, float *__restrict__ y,
                                                           uint64_t out_stride, uint32_t rows, uint32_t tokens,
                                                           uint32_t bm, uint32_t bn, uint32_t full, uint32_t splits,
                                                           uint32_t group) {
    const uint32_t tile_f = bm * bn, per = tile_f / 1024;
    const uint32_t t = blockIdx.x / per, e = ((blockIdx.x % per) * 256 + threadIdx.x) * 4;
    uint32_t pm, pn;
    panel_coords(full + t, (tokens + bm - 1) / bm, (rows + bn - 1) / bn, group, &pm, &pn);
    const uint32_t m = pm * bm + e / bn, n = pn * bn + e % bn;
    if (m >= tokens || n >= rows) return;
    const float *p = work + (uint64_t)t * splits * tile_f + e;
    float4 v = *(const float4 *)p;
    for (uint32_t q0 = 1; q0 < splits; q0 += 4) {
        float4 o[4];
#pragma unroll
        for (uint32_t j = 0; j < 4; ++j) o[j] = *(const float4 *)(p + (uint64_t)min(q0 + j, splits - 1) * tile_f);
#pragma unroll
        for (uint32_t j = 0; j < 4; ++j) {
            const bool live = q0 + j < splits;
            v.x = live ? v.x + o[j].x : v.x;
            v.y = live ? v.y + o[j].y : v.y;
            v.z = live ? v.z + o[j].z : v.z;
            v.w = live ? v.w + o[j].w : v.w;
        }
    }
    float *out = y + (uint64_t)m * out_stride + n;  // rows is a multiple of 8: all four are inside
    out[0] = v.x;
    out[1] = v.y;
    out[2] = v.z;
    out[3] = v.w;
}

#define NUQ_PANEL_DECLARE(E) \
    template <> hipError_t launch_panel_enc<E>(hipStream_t, const PanelArgs &, const PanelPlan &, float *);
NUQ_PANEL_DECLARE(8)
NUQ_PANEL_DECLARE(12)
NUQ_PANEL_DECLARE(13)
NUQ_PANEL_DECLARE(14)
NUQ_PANEL_DECLARE(23)
#undef NUQ_PANEL_DECLARE

hipError_t launch_panel(hipStream_t s, uint32_t encoding, const PanelArgs &a, const PanelPlan &p, float *work) {
    hipError_t e = hipErrorInvalidValue;
    switch (encoding) {
    case 8: e = launch_panel_enc<8>(s, a, p, work); break;
    case 12: e = launch_panel_enc<12>(s, a, p, work); break;
    case 13: e = launch_panel_enc<13>(s, a, p, work); break;
    case 14: e = launch_panel_enc<14>(s, a, p, work); break;
    case 23: e = launch_panel_enc<23>(s, a, p, work); break;
    }
    if (e != hipSuccess || p.tail == 0) return e;
    const PanelShape &sh = PANEL_SHAPES[p.shape];
    const uint32_t bm = 32 * sh.tg, bn = 32 * sh.rg * sh.wr;
    hipLaunchKernelGGL(panel_reduce_kernel, dim3(p.tail * (bm * bn / 1024)), dim3(256), 0, s, work, a.y, a.out_stride,
                       a.rows, a.tokens, bm, bn, p.full, p.splits, PANEL_GROUP);
    return hipGetLastError();
}

// For checks: the fields of shape i (TG, RG, WR, WK, DEPTH), 0 past the last
// shape, and one product on a given plan.
extern "C" int nuq_panel_shape(uint32_t i, uint32_t out[5]) {
    if (i >= (uint32_t)PANEL_SHAPE_COUNT) return 0;
    const PanelShape &s = PANEL_SHAPES[i];
    const uint32_t v[5] = {s.tg, s.rg, s.wr, s.wk, s.depth};
    std::copy(v, v + 5, out);
    return 1;
}

extern "C" int nuq_panel_run(void *stream, uint32_t encoding, const void *w, uint64_t stride, uint32_t rows,
                             uint32_t columns, const void *x, uint64_t in_stride, void *y, uint64_t out_stride,
                             uint32_t tokens, uint32_t shape, uint32_t full, uint32_t tail, uint32_t splits,
                             void *work) {
    if (shape >= (uint32_t)PANEL_SHAPE_COUNT || splits == 0 || tokens == 0 || columns % 256 != 0)
        return (int)hipErrorInvalidValue;
    const PanelShape &sh = PANEL_SHAPES[shape];
    const uint32_t bm = 32 * sh.tg, bn = 32 * sh.rg * sh.wr;
    if (full + tail != (tokens + bm - 1) / bm * ((rows + bn - 1) / bn) || splits * sh.wk > columns / 256)
        return (int)hipErrorInvalidValue;
    const PanelPlan p{(int)shape, full, tail, splits, (uint64_t)tail * splits * bm * bn, 0.f};
    const PanelArgs a{(const uint8_t *)w, stride, rows, columns, (const _Float16 *)x, in_stride, (float *)y, out_stride,
                      tokens};
    return (int)launch_panel((hipStream_t)stream, encoding, a, p, (float *)work);
}

// Eight values a thread, rounded to nearest even as the tiles' own conversion.
__global__ void __launch_bounds__(256) to_f16_kernel(const float *__restrict__ x, uint64_t in_stride,
                                                     uint32_t columns, _Float16 *__restrict__ out) {
    typedef _Float16 half8 __attribute__((ext_vector_type(8)));
    const uint32_t c = (blockIdx.x * 256 + threadIdx.x) * 8, t = blockIdx.y;
    if (c >= columns) return;
    const float4 *p = (const float4 *)(x + (uint64_t)t * in_stride + c);
    const float4 a = p[0], b = p[1];
    *(half8 *)(out + (uint64_t)t * columns + c) =
        half8{(_Float16)a.x, (_Float16)a.y, (_Float16)a.z, (_Float16)a.w,
              (_Float16)b.x, (_Float16)b.y, (_Float16)b.z, (_Float16)b.w};
}

hipError_t launch_to_f16(hipStream_t s, const float *x, uint64_t in_stride, uint32_t columns, uint32_t tokens,
                         _Float16 *out) {
    // a grid's y dimension holds 65535 blocks
    for (uint32_t t0 = 0; t0 < tokens; t0 += 65535) {
        const uint32_t n = std::min(tokens - t0, 65535u);
        hipLaunchKernelGGL(to_f16_kernel, dim3((columns / 8 + 255) / 256, n), dim3(256), 0, s,
                           x + (uint64_t)t0 * in_stride, in_stride, columns, out + (uint64_t)t0 * columns);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace nuq
