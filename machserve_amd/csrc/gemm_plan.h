// What a product costs in each of the tiles of whole K steps (two-byte elements): host code, shared by the plain products (gemm.hip) and
// those over the rows of routed experts (routed.hip).
#pragma once
#include "common.cuh"

namespace ms {

// The choice of a tile (and of the K slices, where the reader adds them up) for more than 64 rows and whole K steps: the
// one whose predicted time is least.  A block of a tile takes `step[n]` us a K step of 64 where n + 1 such blocks share a CU, `slope` more of it in
// proportion as the chip is full, and `store32` or `store16` for each block a CU to store its sums; `start` is paid once a product.  The
// numbers are a fit (non-negative least squares, 8 to 15 % off) to the times of 168 products: 96 to 3,001 rows of the projections
// of the 0.5B, 1.5B and 7B layer sizes and of widths of 1,024 and 2,048, cold operands, one to six slices.  The choice is 2 % slower
// than the best tile measured, on average; against the rules it replaces (rounds of 128x128 blocks, with borders
// for wider tiles, in a loop of one burst of loads a step) the products are 1.26 times as fast (geometric mean).
struct TileCost {
    int bm, bn, per_cu;
    float step[4], store32, store16, start, slope;
};
enum Tile { TILE_256x256, TILE_256x192, TILE_256x128, TILE_128x128, TILE_64x64, TILE_64x64_DEEP, TILE_COUNT };
static constexpr TileCost kTiles[TILE_COUNT] = {
    {256, 256, 1, {1.12f}, 8.64f, 0.85f, 8.26f, 0.22f},
    {256, 192, 1, {0.96f}, 7.82f, 0.00f, 7.22f, 0.14f},
    {256, 128, 1, {0.65f}, 5.95f, 1.97f, 4.09f, 0.17f},
    {128, 128, 2, {0.42f, 0.67f}, 1.99f, 0.12f, 3.70f, 0.31f},
    {64, 64, 4, {0.27f, 0.29f, 0.40f, 0.51f}, 0.31f, 0.00f, 2.87f, 0.37f},
    {64, 64, 2, {0.25f, 0.45f}, 0.79f, 0.09f, 2.79f, 0.04f},
};

static inline float tile_time(const TileCost& t, long blocks, int k_per_split, bool store32) {
    const long cus = compute_units(), round = cus * t.per_cu;
    const float steps = (float)ceil_div(k_per_split, 64), store = store32 ? t.store32 : t.store16;
    const long full = blocks / round, rest = blocks % round;
    float us = t.start + (float)full * (steps * (t.step[t.per_cu - 1] + t.slope) + store * t.per_cu);
    if (rest) {
        const float fill = (float)rest / (float)round;
        us += steps * (t.step[ceil_div(rest, cus) - 1] + t.slope * fill) + store * t.per_cu * fill;
    }
    return us;
}

}  // namespace ms
