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
enum Tile { TILE_256x256, TILE_256x192, TILE_256x128, TILE_128x128, TILE_64x64, TILE_64x64_DEEP, TILE_COUNT, TILE_256x320 = TILE_COUNT, TILE_COUNT_GATED };
static constexpr TileCost kTiles[TILE_COUNT_GATED] = {
    {256, 256, 1, {1.12f}, 8.64f, 0.85f, 8.26f, 0.22f},
    {256, 192, 1, {0.96f}, 7.82f, 0.00f, 7.22f, 0.14f},
    {256, 128, 1, {0.65f}, 5.95f, 1.97f, 4.09f, 0.17f},
    {128, 128, 2, {0.42f, 0.67f}, 1.99f, 0.12f, 3.70f, 0.31f},
    {64, 64, 4, {0.27f, 0.29f, 0.40f, 0.51f}, 0.31f, 0.00f, 2.87f, 0.37f},
    {64, 64, 2, {0.25f, 0.45f}, 0.79f, 0.09f, 2.79f, 0.04f},
    // Gated products only, where 256x192 tiles are a round and a half: 130 to 4,160 rows of five gate/up sizes (70 products), 4 to 14 % faster than the best
    // of the other tiles in twelve of them, and the choice is within 0.1 % of the best tile on average.  Its prediction is 3 % off; the others' are 4 % (256x192 where these win: up to 12 %) short
    // of these products' times, and this is 7 % short.  2,048 x 9,728 x 896: 42.3 us in 256x192, 38.9 in these; 1,536 x 11,264 x 2,048 76.0 (128x128) and 67.2.
    {256, 320, 1, {1.57f}, 5.69f, 5.69f, 5.52f, 0.21f},
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

// Products of few rows (few_rows.cuh: four waves that share out K).  A block of `nt` tiles of 16 columns takes `step[n]` us for each of a wave's K steps
// where n + 1 such blocks share a CU, `slope` more of it in proportion as the chip is full; the product takes `start` and `per_mb` for each MB of the weight.
// A fit (non-negative least squares, 6 to 10 % off) to 1,416 products of 1 to 16 rows, their weights read as a model has them (past the last-level cache or through it), and 224 each of
// 32 and 64: 37 and 40 weights of 64 to 151,936 columns and K of 320 to 18,944, cold, in one to eight slices.  Up to 16 rows the choice of tiles and slices takes 1.006 times the
// best measured, where that of a fit to weights through the cache took 1.034: 37,888 x 3,584 gated 48.1 us in 64 columns a block, 43.1 in 32; 17,920 x 1,536 gated 14.4 and
// 12.2; 2,048 x 2,048 4.35 in eight slices, 3.94 in two.
struct FewCost {
    int nt, stages, per_cu;
    float step[3], slope, start, per_mb;
};
constexpr int FEW_WAVES = 4, FEW_TILES = 3;
static constexpr FewCost kFew[3][FEW_TILES] = {  // up to 16, 32 and 64 rows
    {{1, 3, 3, {0.143f, 0.265f, 0.419f}, 0.194f, 2.49f, 0.085f}, {2, 3, 2, {0.203f, 0.404f}, 0.349f, 2.44f, 0.081f}, {4, 2, 2, {0.387f, 0.733f}, 0.000f, 2.45f, 0.120f}},
    {{1, 3, 2, {0.261f, 0.436f}, 0.557f, 2.21f, 0.149f}, {2, 2, 2, {0.358f, 0.620f}, 0.483f, 2.34f, 0.143f}, {4, 2, 1, {0.646f}, 1.792f, 2.50f, 0.118f}},
    {{1, 2, 2, {0.406f, 0.717f}, 0.604f, 2.26f, 0.167f}, {2, 2, 1, {0.595f}, 1.792f, 2.52f, 0.114f}, {4, 2, 1, {0.935f}, 3.220f, 3.42f, 0.101f}},
};
static inline int few_row_tiles(int M) { return M <= 16 ? 0 : M <= 32 ? 1 : 2; }
static inline float few_time(const FewCost& t, long blocks, int k_per_split, long N, long K) {
    const long cus = compute_units(), round = cus * t.per_cu, full = blocks / round, rest = blocks % round;
    const float steps = (float)ceil_div(k_per_split, 64 * FEW_WAVES);
    float us = t.start + (float)(N * K) * 2e-6f * t.per_mb + (float)full * steps * (t.step[t.per_cu - 1] + t.slope);
    if (rest) us += steps * (t.step[ceil_div(rest, cus) - 1] + t.slope * (float)rest / (float)round);
    return us;
}
struct FewPlan {
    int tile, splits;
    float us;
};
// The best tile for `splits` slices, or, with splits == 0, the best tile and number of slices (a plane of sums more is written and read again, and
// no slice is shorter than a step for every wave).  `pairs`: gate and up columns lie side by side.  Up to 32 rows the slices are those of 16, so that a row's
// sums do not depend on how many rows come with it.
// K in numbers of two bytes: one of four counts twice (a slice is a multiple of 64 numbers of either).
constexpr int FEW_BYTES = (int)sizeof(elem_t) / 2, FEW_SLICE = 64 * FEW_BYTES;
static inline FewPlan plan_few(int M, int N, int K, int splits, bool pairs) {
    if (splits == 0 && M <= 32 && M != 16) return plan_few(M, N, K, plan_few(16, N, K, 0, pairs).splits, pairs);
    FewPlan best{0, 1, INFINITY};
    // (up to sixteen slices only in 32-bit and of very few columns, 128 x 16,384 6.4 us in eight, 4.8 in sixteen: the norm that adds them up takes longer by more than the
    // prediction knows, a pass of three requests of the 0.5B sizes 20.4 ms and 20.5 with ten of the down projection)
    for (int s = splits ? splits : 1; s <= (splits ? splits : kHalf || N > 256 ? 8 : 16); ++s) {
        const int per = ceil_div(ceil_div(K, s), FEW_SLICE) * FEW_SLICE;
        if (splits == 0 && s > 1 && (ceil_div(K, per) != s || per < 64 * FEW_WAVES)) continue;
        for (int i = pairs ? 1 : 0; i < FEW_TILES; ++i) {
            const FewCost& t = kFew[few_row_tiles(M)][i];
            // (a plane of sums more: its bytes, and up to 16 rows 0.05 us of the reader's time)
            const float us = few_time(t, (long)ceil_div(N, 16 * t.nt) * s, per, N, K) + (float)(s - 1) * ((float)M * (float)N * (8.0f / 4.5e6f) + (M <= 16 ? 0.05f : 0.0f));
            if (us < best.us) best = {i, s, us};
        }
    }
    return best;
}

}  // namespace ms
