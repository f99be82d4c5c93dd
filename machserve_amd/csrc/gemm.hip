// out[M, N] = A[M, K] * W[N, K]^T on the matrix cores, with the epilogue fused:
// bias add, residual accumulation into the 32-bit stream, or SiLU(gate) * up.
//
// Role in the reference: hipBLAS Sgemm / GemmEx plus separate add_bias, add and silu_mul
// kernels (crates/mach-model/src/kernels.rs:5772-5798, 6416-6455, 131-160).
//
// A block's loop over K and its epilogues are in gemm_tile.cuh; here are the choice of the tile and the entry points.
#include "few_rows.cuh"
#include "gemm_plan.h"
#include "gemm_tile.cuh"

namespace ms {

// The order of the tiles.  Blocks go to the eight dies in turn, each die with an L2 of its own, and what a die's blocks read beside one another goes over the
// fabric once: so a die takes a run of the order in which `group` row tiles stand under every column in turn, K slice by K slice, and what it has in
// work is nearly a square.  What bounds the tiles' loops is this traffic: W comes from memory, at 23 bytes a clock into a CU whatever is asked for ahead, from
// the last-level cache at 40, and what the die has already read at 53.  us before (by turns or a run of whole columns, every slice in every die)
// and so, cold W: 2,048 x 3,584 x 18,944 in two slices 195 -> 182, 3,001 x 11,264 x 2,048 108 -> 101, 2,048 x 2,048 x 5,632 in two 41.6 -> 40.1, 512 x 9,728 x 896
// (64x64) 23.4 -> 20.9; W in the last-level cache: 181 -> 173, 99 -> 98, 37.8 -> 36.0, 22.6 -> 14.6.
struct TilePlace {
    int m, n, split;
};
// x / d by a reciprocal: a whole division is twenty instructions one behind the other, four of them 1 us ahead of a block's first load.  With x + 1/2 the quotient is
// no nearer to a whole number than 1 / 2d, and wrong by 2^-22 of itself.
__device__ __forceinline__ int quotient(int x, int d) {
    if (x >= 1 << 20) return x / d;
    return __builtin_amdgcn_readfirstlane((int)(((float)x + 0.5f) * __builtin_amdgcn_rcpf((float)d)));
}
__device__ __forceinline__ TilePlace tile_of_block(int tiles_m, int group) {
    const int tiles = gridDim.x, all = tiles * gridDim.y, id = blockIdx.x + tiles * blockIdx.y;
    const int per = all / 8, rest = all % 8, die = id % 8;
    int at = die * per + min(die, rest) + id / 8, split = 0;
    if (gridDim.y > 1) {
        split = quotient(at, tiles);
        at -= split * tiles;
    }
    const int band = group * quotient(tiles, tiles_m), g = quotient(at, band), in = at - g * band, rows = min(group, tiles_m - g * group), n = quotient(in, rows);
    return {g * group + in - n * rows, n, split};
}

template <int BM, int BN, int WM, int WN, int BK, int EPI, int STAGES = 2, bool SCALED = false>
__global__ __launch_bounds__(64 * WM * WN) void gemm_kernel(const elem_t* __restrict__ A, const elem_t* __restrict__ W,
                                                   int M, int N, int K, EpiArgs ep) {
    arguments_now(A, W, M, N, K, ep.out, ep.bias, ep.ldo, ep.n_out, ep.k_per_split, ep.split_stride, ep.group);
    if constexpr (SCALED) arguments_now(ep.row_ss, ep.ss_parts, ep.ss_eps);
    if constexpr (STAGES == 4 && BM == 64) arguments_now(ep.past);
    const int tiles_m = ceil_div(M, BM);
    // (Tiles with four buffers are few, and gain nothing by it: 2,048 x 64 x 2,048 12.0 us by turns, 13.1 so; 32-bit, 32x32 tiles, prompts of 100 and 250 rows of the
    // further designs' small sizes 0.6 % by turns, and 1 % the other way round where K is 2,048 and more.)
    constexpr bool BY_TURNS = STAGES == 4 && EPI != EPI_QKV_ROPE;
    const TilePlace at = BY_TURNS || tiles_m == 1 ? TilePlace{(int)blockIdx.x % tiles_m, (int)blockIdx.x / tiles_m, (int)blockIdx.y} : tile_of_block(tiles_m, ep.group);
    gemm_tile<BM, BN, WM, WN, BK, EPI, STAGES, SCALED>(A, W, M, N, K, ep, at.m * BM, at.n * BN, at.split, NoExperts{});
}

// Row tiles side by side (see tile_of_block): the power of two nearest to what makes the rows and the columns that a die has in work, of which it holds `per_cu`
// tiles a CU, equally many.
static int row_group(int bm, int bn, int per_cu, long blocks) {
    const double run = (double)min(ceil_div(blocks, 8L), (long)max(1, compute_units() / 8) * per_cu);
    return 1 << max(0, (int)lround(0.5 * log2(run * bn / bm)));
}

#ifdef MS_MEASURE  // switches for measurements, in no library that serves
static int g_gemm_config = 0;  // 0: chosen by shape; else a fixed tile
#else
static constexpr int g_gemm_config = 0;
#endif

static int tiled_slices(int M, int N, int K);

#ifdef MS_ELEM_HALF
struct GemmPlan {
    int tile, splits;
};
// The best tile for `splits` slices, or, with splits == 0, the best tile and number of slices: a slice more is a plane of sums more to
// write and to read again (4.5 TB/s), and never less than three K steps.
static GemmPlan plan_gemm(int M, int N, int K, int splits, bool store32, bool gated = false) {
    GemmPlan best{0, max(1, splits)};
    float best_us = INFINITY;
    for (int s = splits ? splits : 1; s <= (splits ? splits : 6); ++s) {
        const int per = ceil_div(ceil_div(K, s), 64) * 64;
        if (splits == 0 && s > 1 && (ceil_div(K, per) != s || per < 192)) continue;
        for (int i = 0; i < (gated ? TILE_COUNT_GATED : TILE_COUNT); ++i) {
            const long blocks = (long)ceil_div(M, kTiles[i].bm) * ceil_div(N, kTiles[i].bn) * s;
            const float us = tile_time(kTiles[i], blocks, per, store32) + (float)(s - 1) * (float)M * (float)N * (8.0f / 4.5e6f);
            if (us < best_us) {
                best_us = us;
                best = {i, s};
            }
        }
    }
    return best;
}
#endif
template <int MT, int NT, int STAGES, int EPI, bool SCALED>
__global__ __launch_bounds__(64 * FEW_WAVES) void gemm_few_kernel(const elem_t* __restrict__ A, const elem_t* __restrict__ W, int M, int N, int K, EpiArgs ep) {
    arguments_now(A, W, M, N, K, ep.out, ep.bias, ep.ldo, ep.n_out, ep.k_per_split, ep.split_stride, ep.past);
    if constexpr (SCALED) arguments_now(ep.row_ss, ep.ss_parts, ep.ss_eps);
    if constexpr (EPI == EPI_PRENORM) arguments_now(ep.norm_w, ep.hn, ep.ss_part);
    few_rows_tile<MT, NT, FEW_WAVES, STAGES, EPI, SCALED>(A, W, M, N, K, ep, 0, blockIdx.x * 16 * NT, blockIdx.y, NoExperts{});
}

template <int NT, int STAGES>
__global__ __launch_bounds__(64 * FEW_WAVES) void gemm_few_normed_kernel(const elem_t* __restrict__ W, int M, int N, int K, EpiArgs ep) {
    arguments_now(W, M, N, K, ep.out, ep.ldo, ep.k_per_split, ep.split_stride, ep.past, ep.stream, ep.pending, ep.n_pending, ep.norm_w, ep.stream_out, ep.ss_eps);
    few_rows_tile<1, NT, FEW_WAVES, STAGES, EPI_STORE_F32, false, NoExperts, true>(W, W, M, N, K, ep, 0, blockIdx.x * 16 * NT, blockIdx.y, NoExperts{});
}

template <int EPI, bool SCALED = false>
static int launch_few(const elem_t* A, const elem_t* W, int M, int N, int K, const EpiArgs& ep, hipStream_t stream, int ns) {
    constexpr bool PAIRS = EPI == EPI_SWIGLU;
    const int rows = few_row_tiles(M), tile = plan_few(M, N, K * FEW_BYTES, ns, PAIRS).tile;
#define MS_FEW(ROWS_, TILE_)                                                                                                                          \
    do {                                                                                                                                              \
        constexpr FewCost t = kFew[ROWS_][TILE_];                                                                                                     \
        if constexpr (!(PAIRS && t.nt == 1) && !(EPI == EPI_PRENORM && ROWS_ > 0) && !(!kHalf && ROWS_ > 1)) {                                                                   \
            hipLaunchKernelGGL((gemm_few_kernel<1 << ROWS_, t.nt, t.stages, EPI, SCALED>), dim3((unsigned)ceil_div(N, 16 * t.nt), (unsigned)ns),      \
                               dim3(64 * FEW_WAVES), 0, stream, A, W, M, N, K, ep);                                                                   \
            return check_launch("gemm, few rows");                                                                                                    \
        }                                                                                                                                             \
    } while (0)
    if (rows == 0) {
        if (tile == 0) MS_FEW(0, 0);
        if (tile == 1) MS_FEW(0, 1);
        MS_FEW(0, 2);
    }
    if (rows == 1) {
        if (tile == 0) MS_FEW(1, 0);
        if (tile == 1) MS_FEW(1, 1);
        MS_FEW(1, 2);
    }
    if (tile == 0) MS_FEW(2, 0);
    if (tile == 1) MS_FEW(2, 1);
    MS_FEW(2, 2);
#undef MS_FEW
    MS_REQUIRE(false, "few-rows product: M=%d N=%d K=%d is not taken", M, N, K);
}

// Whether a product runs in few_rows.cuh, with K cut over several blocks (`slices`) or not: whole K steps, at least one for every wave, up to 16 rows, in 32-bit up to 32; in the two-byte builds up to
// 64 where it is predicted not to be slower than 64x64 tiles.  Their prediction (made for more rows) is an eighth short there: over 240
// products of 32, 48 and 64 rows, cut and uncut, the choice takes 1.00 to 1.02 times the better of the two, which is 1.08 to 1.6 times as fast as the tiles.
static bool few_rows(int M, int N, int K, bool slices, bool pairs) {
    // (32-bit: a wave of two steps is no better than one of skinny.hip, 40,000 x 256 10.9 us and 10.2)
    if (M > 64 || K % FEW_STEP != 0 || K < FEW_STEP * FEW_WAVES * (kHalf ? 1 : 3) || g_gemm_config != 0) return false;
    if (M <= (kHalf ? 16 : 32)) return true;  // (in 32-bit all rows whose sums are those of a row by itself)
#ifdef MS_ELEM_HALF
    const int ns = slices ? tiled_slices(M, N, K) : 1, per = ceil_div(ceil_div(K, ns), 64) * 64;
    const float tiled = fmaxf(tile_time(kTiles[TILE_64x64_DEEP], (long)ceil_div(N, 64) * ns, per, true), 2.5f + (float)N * (float)K * 4e-7f) +
                        (float)(ns - 1) * (float)M * (float)N * (8.0f / 4.5e6f);
    return plan_few(M, N, K, slices ? 0 : 1, pairs).us < 1.12f * tiled;
#else
    (void)N; (void)slices; (void)pairs;
    return false;
#endif
}
#ifdef MS_ELEM_HALF
// products of more than 64 rows over whole K steps: what is planned as above
static bool planned(int M, int K) { return M > 64 && K % 64 == 0 && g_gemm_config == 0; }
#endif

#ifndef MS_ELEM_HALF
// Whether a 32-bit product runs in parts of 16 bits (GEMM_SPLIT): whole K steps, K in slices or an output of at least 4,096 columns in which the 32-bit instructions would fill
// rounds badly.  Those have 32x32 tiles below two of 64x64 a CU, and parts are faster from six and a half of them on; else three of 64x64 a CU at a time, which take as long with
// two and a bit as with three, and parts, 0.6 us a step for each that a CU has, are faster behind two up to 2.6 of them, and beyond a round.  us, 32-bit instructions and parts: 192 x
// 9,728 x 896 (7.1 tiles of 32x32 a CU) 38 and 34, 160 rows (5.9) 32 and 35, 128 x 12,288 x 896 (6) 30 and 34, 65 rows (4.5) 28 and 35; 512 x 4,096 x 1,024 (2 of 64x64) 37.7 and 39.6,
// 256 x 8,192 x 2,048 (2) 70 and 77, 400 x 4,864 x 896 (2.1) 46 and 42.6, 300 x 8,192 x 2,048 (2.5) 99 and 95, 700 x 4,096 x 1,024 (2.75) 53 and 54, 300 x 9,728 x 896 (2.97) 48.6 and
// 50.8, 400 rows (4.2) 85 and 73, 1,024 x 4,096 x 1,024 (4) 95 and 57.  The rows' number is part of the rule, as it is of the number of slices: a row's sums are those of other
// batches to rounding only.
static bool parted(int M, int N, int K, int slices) {
    const long cus = compute_units(), tiles = (long)ceil_div(M, 64) * ceil_div(N, 64), small = (long)ceil_div(M, 32) * ceil_div(N, 32);
    const bool faster = tiles < 2 * cus ? 2 * small >= 13 * cus : tiles > 3 * cus || (tiles > 2 * cus && 5 * tiles <= 13 * cus);
    return K % 32 == 0 && M > 64 && (slices > 1 || (N >= 4096 && faster));
}
// ... in tiles of 128x128, a block a CU, which take 1.7 us a K step and round, or of 64x64, 0.55 us for each that a CU has: 768 x 9,728 x 896 (two rounds, 7.1 a CU) 100 and
// 114 us, 512 rows (two rounds, 4.8) 97 and 79, 1,024 rows (three, 9.5) 137 and 142; 512 x 896 x 4,864 in eight slices (one round, 3.5) 38 and 46, 192 x 2,048 x 5,632 (one, 3)
// 44 and 42, 512 x 2,048 x 5,632 in four (one, 4) 83 and 102.
static bool parted_wide(int M, int N, int slices) {
    const long cus = compute_units(), wide = (long)ceil_div(M, 128) * ceil_div(N, 128) * slices, narrow = (long)ceil_div(M, 64) * ceil_div(N, 64) * slices;
    return 1.7 * (double)ceil_div(wide, cus) < 0.55 * (double)narrow / (double)cus;
}
#endif

template <int EPI>
static int launch_gemm(const elem_t* A, const elem_t* W, int M, int N, int K, EpiArgs ep, hipStream_t stream,
                       int nsplit = 1) {
    MS_REQUIRE(M > 0 && N > 0 && K > 0, "gemm: empty problem M=%d N=%d K=%d", M, N, K);
    MS_REQUIRE(K % 8 == 0, "gemm: the reduction size K=%d must be a multiple of 8", K);
    MS_REQUIRE((reinterpret_cast<uintptr_t>(A) & 15) == 0 && (reinterpret_cast<uintptr_t>(W) & 15) == 0,
               "gemm: operands must be 16-byte aligned");
    MS_REQUIRE(nsplit >= 1 && (nsplit == 1 || EPI == EPI_STORE_F32), "gemm: %d K slices need the float store", nsplit);
    // slices of a multiple of 64; rounding up may leave fewer slices than asked for
    ep.k_per_split = ceil_div(ceil_div(K, nsplit), 64) * 64;
    ep.split_stride = (size_t)M * N;
    const unsigned ns = (unsigned)ceil_div(K, ep.k_per_split);
    MS_REQUIRE(nsplit == 1 || (int)ns == nsplit, "gemm: %d K slices asked for, %u fit", nsplit, ns);
#define MS_GEMM_DEEP(BM_, BN_, WM_, WN_, BK_, ST_)                                                                         \
    do {                                                                                                                  \
        const long nb = (long)ceil_div(M, BM_) * ceil_div(N, BN_);                                                        \
        ep.group = row_group(BM_, BN_, BM_ >= 256 ? 1 : BM_ == 128 ? 2 : 4, nb * ns);                                     \
        hipLaunchKernelGGL((gemm_kernel<BM_, BN_, WM_, WN_, BK_, EPI, ST_>), dim3((unsigned)nb, ns), dim3(64 * WM_ * WN_), 0, stream, \
                           A, W, M, N, K, ep);                                                                            \
        return check_launch("gemm " #BM_ "x" #BN_ "x" #BK_ " deep");                                                      \
    } while (0)
#define MS_GEMM(BM_, BN_, WM_, WN_, BK_)                                                                              \
    do {                                                                                                              \
        const long nb = (long)ceil_div(M, BM_) * ceil_div(N, BN_);                                                    \
        ep.group = row_group(BM_, BN_, BM_ >= 256 ? 1 : BM_ == 128 ? 2 : 4, nb * ns);                                 \
        hipLaunchKernelGGL((gemm_kernel<BM_, BN_, WM_, WN_, BK_, EPI>), dim3((unsigned)nb, ns), dim3(64 * WM_ * WN_), 0, stream, \
                           A, W, M, N, K, ep);                                                                        \
        return check_launch("gemm " #BM_ "x" #BN_ "x" #BK_);                                                          \
    } while (0)
    if (few_rows(M, N, K, ns > 1, EPI == EPI_SWIGLU)) return launch_few<EPI>(A, W, M, N, K, ep, stream, (int)ns);
#ifdef MS_ELEM_HALF
    const int forced = g_gemm_config;
    if (forced == 1) MS_GEMM(128, 128, 2, 2, 32);
    if (forced == 2) MS_GEMM(128, 128, 2, 2, 64);
    if (forced == 5) MS_GEMM(128, 64, 2, 2, 64);
    if (forced == 6) MS_GEMM(64, 64, 2, 2, 64);
    const bool whole_steps = ep.k_per_split % 64 == 0 && K % 64 == 0;
    if (planned(M, K)) {
        switch (plan_gemm(M, N, K, (int)ns, EPI == EPI_STORE_F32 || EPI == EPI_RESIDUAL, EPI == EPI_SWIGLU).tile) {
            case TILE_256x320:
                if constexpr (EPI == EPI_SWIGLU) MS_GEMM_DEEP(256, 320, 2, 4, 64, GEMM_PIPED);
            case TILE_256x256: MS_GEMM_DEEP(256, 256, 2, 4, 64, GEMM_PIPED);
            case TILE_256x192: MS_GEMM_DEEP(256, 192, 4, 2, 64, GEMM_PIPED);
            case TILE_256x128: MS_GEMM_DEEP(256, 128, 4, 2, 64, GEMM_PIPED);
            case TILE_128x128: MS_GEMM_DEEP(128, 128, 2, 4, 64, GEMM_PIPED);
            case TILE_64x64: MS_GEMM_DEEP(64, 64, 2, 2, 64, GEMM_PIPED);
            default: MS_GEMM_DEEP(64, 64, 2, 2, 64, 4);
        }
    }
    if (forced == 8 && whole_steps) MS_GEMM_DEEP(64, 64, 2, 2, 64, 4);
    if (forced == 9) MS_GEMM(256, 256, 2, 4, 64);
    // What is left are products of at most 64 rows, and those whose last K step is not a whole one, which run in the loop of one
    // burst of loads a step: the largest tile that still gives every CU of the chip a block or two, with K steps of 64 (half
    // the barriers of steps of 32).  The borders were found with whole steps in this loop, which are planned above now, and hold for
    // partial ones: over 92 products (130 to 4,096 rows, 1,160 to 18,952 columns, K of 904, 1,544, 3,592, 4,872 and 9,000) the choice takes 1.03 times
    // the best of 256x256, 128x128, 128x64 and 64x64 (1.26 at most: 130 rows of 9,736 columns, 17.6 us against 14.0 in 64x64), and each of these
    // and 128x160 is the best somewhere.
    // two 128x128 blocks a CU are a round of the chip (512 on 256 CUs); a tile is taken when its blocks fill
    // six tenths of a round
    const long round_blocks = 2L * compute_units(), enough = round_blocks * 300 / 512;
    if (M > 64 && (ns == 1 || K >= 16384) && ep.k_per_split >= 128 && forced == 0) {
        // Tiles of 256x256 under eight waves (each 128 rows by 64 columns: 128 accumulator registers, 220 in all, two
        // waves a SIMD; 128 KB of LDS: one block a CU) bring half the bytes of two 128x128 tiles from the L2 into the CUs,
        // which is what bounds the large products.  They pay where the last of their rounds of one block a CU is well filled; a short K
        // (few steps between a tile's start and its 256x256 stores) wants the rounds fuller.  us, 256x256 against 128x128: 4,096 x 18,952 x 1,544
        // (1,200 tiles, 0.94 of five rounds) 275 and 354; 4,096 x 9,736 x 4,872 (0.81 of three) 418 and 488; 2,048 x 9,736 x 4,872
        // (0.61 of two) 294 and 288; 1,024 x 4,616 x 4,872 (0.30 of one) 140 and 122.
        // (with K cut over `ns` blocks - a very long K under few tiles, see plan_tiled_splits - the slices fill the round)
        const long t256 = (long)ceil_div(M, 256) * ceil_div(N, 256) * ns, cus = compute_units();
        const long rounds = ceil_div(t256, cus);
        if (t256 * 100 >= rounds * cus * (K >= 1536 ? 72 : 85)) MS_GEMM(256, 256, 2, 4, 64);
    }
    if (M > 64) {
        const long b128 = (long)ceil_div(M, 128) * ceil_div(N, 128), b12864 = (long)ceil_div(M, 128) * ceil_div(N, 64);
        // The chip holds a round of such blocks at a time and a round that is nearly empty takes as long as a full one:
        // the time is rounds times the tile's width.  Where tiles a quarter wider save more in rounds than they
        // cost, they are taken (2,048 x 9,736 x 4,872: 1,232 tiles of 128x128 are two rounds and four tenths, 976 of 128x160 two rounds less
        // a twentieth: 288 -> 245 us; 2,048 x 4,616 x 4,872, one round and an eighth: 189 -> 128).
        if (ns == 1 && ep.k_per_split >= 128 && b128 >= enough) {
            const long rounds128 = ceil_div(b128, round_blocks), rounds160 = ceil_div((long)ceil_div(M, 128) * ceil_div(N, 160), round_blocks);
            if (rounds160 * 160 < rounds128 * 128) MS_GEMM(128, 160, 4, 1, 64);
        }
        if (b128 * ns >= enough) {
            if (ep.k_per_split >= 128) MS_GEMM(128, 128, 2, 2, 64);
            MS_GEMM(128, 128, 2, 2, 32);
        }
        if (b12864 * ns >= enough) {
            if (ep.k_per_split >= 128) MS_GEMM(128, 64, 2, 2, 64);
            MS_GEMM(128, 64, 2, 2, 32);
        }
    }
    // At most two blocks a CU, each a chain of K steps: four LDS buffers keep three steps in flight (0.5B
    // gate/up product at 64 rows, 152 blocks of 14 steps: 10.5 -> 7.8 us; 1.5B: 23.7 -> 21.1; with more
    // blocks than that the blocks hide each other's loads and the two-buffer kernel is as fast).
    if ((long)ceil_div(M, 64) * ceil_div(N, 64) * ns <= round_blocks && whole_steps && ep.k_per_split >= 256) MS_GEMM_DEEP(64, 64, 2, 2, 64, 4);
    MS_GEMM(64, 64, 2, 2, 64);
#else
    // Whole K steps straight to LDS, three or two of them in flight (the loop through registers waits for a trip to memory every step:
    // 1,024 x 2,048 x 2,048 in 512 tiles of 64x64 90 -> 69 us); where the 64x64 tiles are less than two a CU, four times as many of
    // 32x32 (512 x 896 x 4,864 118 -> 50 us, 512 x 896 x 896 25 -> 12; at two a CU 69 against 75).  The sums keep their order.
    if (parted(M, N, K, (int)ns)) {
        if (parted_wide(M, N, (int)ns)) MS_GEMM_DEEP(128, 128, 2, 4, 32, GEMM_SPLIT);
        MS_GEMM_DEEP(64, 64, 2, 2, 32, GEMM_SPLIT);
    }
    if (K % 32 == 0) {
        const bool few = (long)ceil_div(M, 64) * ceil_div(N, 64) < 2L * compute_units();
        if constexpr (EPI == EPI_SWIGLU) {  // gate and up columns lie side by side: 32 columns a wave
            if (few) MS_GEMM_DEEP(32, 64, 2, 2, 32, 4);
        } else {
            if (few) MS_GEMM_DEEP(32, 32, 2, 2, 32, 4);
        }
        MS_GEMM_DEEP(64, 64, 2, 2, 32, 3);
    }
    MS_GEMM(64, 64, 2, 2, 32);
#endif
#undef MS_GEMM
#undef MS_GEMM_DEEP
}

#ifdef MS_ELEM_HALF
// The columns of a wave in the tile that a product into the residual stream is planned in: those of a part of the rows' sums of squares (EPI_PRENORM).
static int wave_columns(int tile) {
    constexpr int cols[TILE_COUNT] = {256 / 4, 192 / 2, 128 / 2, 128 / 4, 64 / 2, 64 / 2};
    return cols[tile];
}
// Steps of more than 64 rows: the product before a norm, which prepares it (EPI_PRENORM), and the gated product behind it, which applies the rows' factors (SCALED), in the
// tiles that they are planned in without the norm.
template <int EPI, bool SCALED>
static int launch_around_norm(const elem_t* A, const elem_t* W, int M, int N, int K, EpiArgs ep, hipStream_t stream) {
    ep.k_per_split = K;
#define MS_AROUND(BM_, BN_, WM_, WN_, ST_)                                                                                                                 \
    do {                                                                                                                                                   \
        ep.group = row_group(BM_, BN_, BM_ >= 256 ? 1 : BM_ == 128 ? 2 : 4, (long)ceil_div(M, BM_) * ceil_div(N, BN_));                                    \
        hipLaunchKernelGGL((gemm_kernel<BM_, BN_, WM_, WN_, 64, EPI, ST_, SCALED>), dim3((unsigned)((long)ceil_div(M, BM_) * ceil_div(N, BN_)), 1),       \
                           dim3(64 * WM_ * WN_), 0, stream, A, W, M, N, K, ep);                                                                            \
        return check_launch("gemm around a norm, " #BM_ "x" #BN_);                                                                                         \
    } while (0)
    switch (plan_gemm(M, N, K, 1, EPI == EPI_PRENORM, SCALED).tile) {
        case TILE_256x320:
            if constexpr (SCALED) MS_AROUND(256, 320, 2, 4, GEMM_PIPED);
        case TILE_256x256: MS_AROUND(256, 256, 2, 4, GEMM_PIPED);
        case TILE_256x192: MS_AROUND(256, 192, 4, 2, GEMM_PIPED);
        case TILE_256x128: MS_AROUND(256, 128, 4, 2, GEMM_PIPED);
        case TILE_128x128: MS_AROUND(128, 128, 2, 4, GEMM_PIPED);
        case TILE_64x64: MS_AROUND(64, 64, 2, 2, GEMM_PIPED);
        default: MS_AROUND(64, 64, 2, 2, 4);
    }
#undef MS_AROUND
}
#endif

// K slices for a product whose consumer adds partial sums: enough 128x128 blocks to fill the chip,
// at least 512 of K each.  The 32-bit build does not slice here: its sums keep one order.
#ifdef MS_MEASURE
static int g_force_splits = 0;
#else
static constexpr int g_force_splits = 0;
#endif

// K slices of a product in tiles.
static int tiled_slices(int M, int N, int K) {
#ifdef MS_ELEM_HALF
    const long b128 = (long)ceil_div(M, 128) * ceil_div(N, 128);
    const long round_blocks = 2L * compute_units();  // two 128x128 blocks a CU
    // A very long K under few output tiles (the 7B down projection: K = 18,944, 14 column tiles of 256): tiles of 256x256
    // bring half the bytes of 128x128 tiles from the L2, but one or two thousand rows of them do not fill the chip's round of
    // one block a CU; with K cut in two to four they do, and the norm that follows adds the slices (2,048 rows: 221 us in two slices and
    // 13 for the second plane, 238 uncut in tiles of 256x128).  Other K, and rows that leave the round less full, as planned
    // above.
    if (M > 64 && K >= 16384 && g_force_splits == 0) {
        const long t256 = (long)ceil_div(M, 256) * ceil_div(N, 256), cus = compute_units();
        if (t256 * 100 < 72 * cus)
            for (int sl = 2; sl <= 4; ++sl)
                if (t256 * sl * 100 >= 85 * cus && t256 * sl <= cus) return ceil_div(K, ceil_div(ceil_div(K, sl), 64) * 64);
    }
    if (planned(M, K) && g_force_splits == 0) return plan_gemm(M, N, K, 0, true).splits;
    if (b128 >= round_blocks * 300 / 512 && g_force_splits == 0) return 1;
    // More than six slices cost more in the consumer's sums than they gain here (with very few tiles - a
    // portion of a few hundred rows - slices of 256 still pay).  With few rows the partial sums are small
    // and the weight is all the traffic: a long K is then cut up to 16 times (7B down projection at 64
    // rows: 49 us with 6 slices, 33 with 12 to 16).
    // (measured again at 33 and 64 rows of the three layer sizes: 1.5B down projection, K = 8,960, 9.0 us in 10
    // slices, 10.0 in 16, and its consumer sums fewer planes)
    // (and again once few blocks ran with four LDS buffers in turn: with its 56 column tiles in four slices the 7B down
    // projection stays within a round of blocks and takes that kernel, 30 to 34 us at 16 to 64 rows with the sum of its
    // planes, against 31 to 36 in thirteen; the 7B decode step at 16 to 64 requests 0.5 to 1 % shorter)
    const int most = M <= 128 ? (K >= 16384 ? (M <= 64 ? 4 : 16) : (K >= 8192 ? 10 : 8)) : 6;
    // (a handful of tiles under few rows - a small projection in a decode step of 33 to 64 requests:
    // slices of 128, or the step's few blocks leave the chip idle)
    // (from K = 1,536 on slices of 256, which run with four LDS buffers in turn: 1.5B output projection at 64
    // rows 5.1 us in 6 slices, 5.5 in 8)
    const int shortest = b128 <= 16 && M <= 128 ? (K >= 1536 ? 256 : 128) : (b128 <= 32 ? 256 : 512);
    const int limit = max(1, min(K / shortest, most));
    // The chip holds two of the 128x128 blocks a CU at a time (512 on 256 CUs), and a last round that is nearly
    // empty takes as long as a full one: the fewest slices that fill their rounds to 70 %, else the
    // count that fills them best (1.5B down projection at 2,048 rows, 192 tiles: 3 slices make a
    // full round and an eighth, 118 us; 2 slices one round three quarters full, 97 us).
    int want = 1;
    double best = 0.0;
    for (int sl = 1; sl <= limit; ++sl) {
        const long blocks = b128 * sl, rounds = ceil_div(blocks, round_blocks);
        const double filled = (double)blocks / (double)(rounds * round_blocks);
        if (filled > best + 1e-9) {
            best = filled;
            want = sl;
        }
        if (filled >= 0.7) break;
    }
    if (g_force_splits > 0) want = g_force_splits;
    // what the launcher's rounding of a slice to a multiple of 64 really yields
    const int k_per_split = ceil_div(ceil_div(K, want), 64) * 64;
    return ceil_div(K, k_per_split);
#else
    (void)M; (void)N; (void)K;
    return 1;
#endif
}

static int plan_tiled_splits(int M, int N, int K) {
    if (g_force_splits == 0 && few_rows(M, N, K, true, false)) return plan_few(M, N, K * FEW_BYTES, 0, false).splits;
    return tiled_slices(M, N, K);
}

}  // namespace ms

using namespace ms;

// Each product has two entry points: `..._past` reads the weight of up to 64 rows past the last-level cache where few_rows.cuh or 64x64 tiles with four
// buffers serve it (see few_rows.cuh); the sums are the same.

// out[M, N] = a[M, K] w[N, K]^T (+ bias[N]); out is float when out_f32 != 0, else the element type.
static int linear(const void* a, const void* w, const float* bias, void* out, int out_f32, int M, int N, int K,
                         hipStream_t stream, bool past) {
    EpiArgs ep{out, bias, N, N, 0, 0};
    ep.past = past && M <= 64;
    if (out_f32) return launch_gemm<EPI_STORE_F32>((const elem_t*)a, (const elem_t*)w, M, N, K, ep, stream);
    return launch_gemm<EPI_STORE_ELEM>((const elem_t*)a, (const elem_t*)w, M, N, K, ep, stream);
}
extern "C" int ms_linear(const void* a, const void* w, const float* bias, void* out, int out_f32, int M, int N, int K,
                         hipStream_t stream) {
    return linear(a, w, bias, out, out_f32, M, N, K, stream, false);
}
extern "C" int ms_linear_past(const void* a, const void* w, const float* bias, void* out, int out_f32, int M, int N, int K,
                         hipStream_t stream) {
    return linear(a, w, bias, out, out_f32, M, N, K, stream, true);
}

// x[M, N] += a[M, K] w[N, K]^T, x being the 32-bit residual stream.
static int linear_residual(const void* a, const void* w, float* x, int M, int N, int K, hipStream_t stream, bool past) {
    EpiArgs ep{x, nullptr, N, N, 0, 0};
    ep.past = past && M <= 64;
    return launch_gemm<EPI_RESIDUAL>((const elem_t*)a, (const elem_t*)w, M, N, K, ep, stream);
}
extern "C" int ms_linear_residual(const void* a, const void* w, float* x, int M, int N, int K, hipStream_t stream) {
    return linear_residual(a, w, x, M, N, K, stream, false);
}
extern "C" int ms_linear_residual_past(const void* a, const void* w, float* x, int M, int N, int K, hipStream_t stream) {
    return linear_residual(a, w, x, M, N, K, stream, true);
}

// out[M, I] = act(a g^T) * (a u^T) where w holds gate and up rows interleaved in blocks of 16:
// rows [32 t, 32 t + 16) are gate rows [16 t, 16 t + 16), rows [32 t + 16, 32 t + 32) the same
// up rows; w has 2 * ceil16(I) rows, the padding rows being zero.
static int linear_swiglu(const void* a, const void* w, void* out, int M, int I, int K, int act, hipStream_t stream, bool past) {
    MS_REQUIRE(act >= 0 && act < ACT_COUNT, "gated product: no activation %d", act);
    const int n = 2 * ceil_div(I, 16) * 16;
    EpiArgs ep{out, nullptr, I, I, 0, 0, nullptr, 0, 0.f, act};
    ep.past = past && M <= 64;
    return launch_gemm<EPI_SWIGLU>((const elem_t*)a, (const elem_t*)w, M, n, K, ep, stream);
}
extern "C" int ms_linear_swiglu(const void* a, const void* w, void* out, int M, int I, int K, int act, hipStream_t stream) {
    return linear_swiglu(a, w, out, M, I, K, act, stream, false);
}
extern "C" int ms_linear_swiglu_past(const void* a, const void* w, void* out, int M, int I, int K, int act, hipStream_t stream) {
    return linear_swiglu(a, w, out, M, I, K, act, stream, true);
}

// out[M, N] = act(a[M, K] w[N, K]^T) in the element type, the activation (UnaryActivation) in the product's epilogue.
static int linear_act(const void* a, const void* w, void* out, int M, int N, int K, int act, hipStream_t stream, bool past) {
    MS_REQUIRE(act >= 0 && act < UNARY_COUNT, "product with an activation: no activation %d", act);
    EpiArgs ep{out, nullptr, N, N, 0, 0, nullptr, 0, 0.f, act};
    ep.past = past && M <= 64;
    return launch_gemm<EPI_ACT>((const elem_t*)a, (const elem_t*)w, M, N, K, ep, stream);
}
extern "C" int ms_linear_act(const void* a, const void* w, void* out, int M, int N, int K, int act, hipStream_t stream) {
    return linear_act(a, w, out, M, N, K, act, stream, false);
}
extern "C" int ms_linear_act_past(const void* a, const void* w, void* out, int M, int N, int K, int act, hipStream_t stream) {
    return linear_act(a, w, out, M, N, K, act, stream, true);
}

// Whether ms_linear_swiglu_scaled takes this shape: bfloat16, whole K steps of 64.
extern "C" int ms_swiglu_scaled_takes(int M, int I, int K) {
#ifdef MS_ELEM_HALF
    (void)I;
    return kRoundsBeforeTheNormIsSafe && M >= 1 && K % 64 == 0 && K >= 256;
#else
    (void)M; (void)I; (void)K;
    return 0;
#endif
}

// ... and whether it pays to hand it rows that lack their norm's division: few rows, or tiles that are at most a round of the chip.  Every tile reads its rows' factors at its start and
// applies them at its end, which in the first round is less than the norm's kernel, and is paid again in each further one.  us a layer, output projection to gated product, with
// the norm between them and without: 0.5B sizes 2,048 rows (248 tiles) 48.7 and 48.2, 3,001 (372) 68.6 and 70.2; 1.5B 1,024 (224) 77.6 and 76.6, 1,500 (336) 105.8 and 107.9,
// 4,096 (896) 232 and 242; 7B 1,024 (476) 287 and 290; width 1,024 and 2,816 in the middle, 3,001 rows (216) 57.0 and 55.8.
extern "C" int ms_swiglu_scaled_pays(int M, int I, int K) {
#ifdef MS_ELEM_HALF
    if (!ms_swiglu_scaled_takes(M, I, K)) return 0;
    if (!planned(M, K)) return 1;
    const int n = 2 * ceil_div(I, 16) * 16;
    const auto& t = kTiles[plan_gemm(M, n, K, 1, false, true).tile];
    return (long)ceil_div(M, t.bm) * ceil_div(n, t.bn) <= (long)compute_units() * t.per_cu;
#else
    (void)M; (void)I; (void)K;
    return 0;
#endif
}

// ms_linear_swiglu for rows that came in multiplied by a norm's weight only: both products of a row are
// divided by the row's root mean square, 1 / sqrt(sum_p row_ss[p, row] / K + eps), before the activation.
static int linear_swiglu_scaled(const void* a, const float* row_ss, int ss_parts, float eps, const void* w, void* out, int M, int I,
                                       int K, int act, hipStream_t stream, bool past) {
#ifdef MS_ELEM_HALF
    MS_REQUIRE(act >= 0 && act < ACT_COUNT, "gated product: no activation %d", act);
    MS_REQUIRE(ms_swiglu_scaled_takes(M, I, K), "gated product with row factors: M=%d K=%d is not taken", M, K);
    MS_REQUIRE(row_ss && ss_parts >= 1, "gated product with row factors: the rows' sums of squares are missing");
    MS_REQUIRE((reinterpret_cast<uintptr_t>(a) & 15) == 0 && (reinterpret_cast<uintptr_t>(w) & 15) == 0, "gemm: operands must be 16-byte aligned");
    const int n = 2 * ceil_div(I, 16) * 16;
    EpiArgs ep{out, nullptr, I, I, K, 0, row_ss, ss_parts, eps, act};
    ep.past = past && M <= 64;
    if (planned(M, K)) {
        if constexpr (kRoundsBeforeTheNormIsSafe) return launch_around_norm<EPI_SWIGLU, true>((const elem_t*)a, (const elem_t*)w, M, n, K, ep, stream);
    }
    if (few_rows(M, n, K, false, true)) return launch_few<EPI_SWIGLU, true>((const elem_t*)a, (const elem_t*)w, M, n, K, ep, stream, 1);
    hipLaunchKernelGGL((gemm_kernel<64, 64, 2, 2, 64, EPI_SWIGLU, 4, true>), dim3((unsigned)ceil_div(n, 64), 1), dim3(256), 0, stream,
                       (const elem_t*)a, (const elem_t*)w, M, n, K, ep);
    return check_launch("gemm 64x64x64 deep, row factors");
#else
    (void)a; (void)row_ss; (void)ss_parts; (void)eps; (void)w; (void)out; (void)M; (void)I; (void)K; (void)act; (void)stream;
    MS_REQUIRE(false, "gated product with row factors: built for bfloat16 only");
#endif
}
extern "C" int ms_linear_swiglu_scaled(const void* a, const float* row_ss, int ss_parts, float eps, const void* w, void* out, int M, int I,
                                       int K, int act, hipStream_t stream) {
    return linear_swiglu_scaled(a, row_ss, ss_parts, eps, w, out, M, I, K, act, stream, false);
}
extern "C" int ms_linear_swiglu_scaled_past(const void* a, const float* row_ss, int ss_parts, float eps, const void* w, void* out, int M, int I,
                                       int K, int act, hipStream_t stream) {
    return linear_swiglu_scaled(a, row_ss, ss_parts, eps, w, out, M, I, K, act, stream, true);
}

// Column tiles of ms_linear_residual_prenorm for this shape (the first size of its ss_part), or 0 if it is not taken: up to 16 rows over whole K steps,
// uncut, where that is predicted to take no longer than the slices and the norm that would add them up (2.5 us: a launch and a trip to memory); more than 64
// rows where the product is not cut: of the norm's 5.1 us a layer of 2,048 rows of the 0.5B sizes 1 goes to this product's epilogue and 2.4 to the gated product's
// start and end, and a prompt takes 3.14 ms for 3.17.
extern "C" int ms_prenorm_parts(int M, int N, int K) {
#ifdef MS_ELEM_HALF
    if (kRoundsBeforeTheNormIsSafe && planned(M, K) && plan_tiled_splits(M, N, K) == 1) return ceil_div(N, wave_columns(plan_gemm(M, N, K, 1, true).tile));
    if (!kRoundsBeforeTheNormIsSafe || M < 1 || M > 16 || !few_rows(M, N, K, false, false)) return 0;
    return plan_few(16, N, K, 1, false).us < plan_few(16, N, K, 0, false).us + 2.5f ? ceil_div(N, 16) : 0;
#else
    (void)M; (void)N; (void)K;
    return 0;
#endif
}

// x[M, N] += a w^T, and beside it hn[M, N] = x * norm_w in the element type and ss_part[parts, M], whose sum over parts is the rows' sums of
// squares of x (parts = ms_prenorm_parts).
static int linear_residual_prenorm(const void* a, const void* w, float* x, const float* norm_w, void* hn, float* ss_part, int M, int N, int K,
                                          hipStream_t stream, bool past) {
#ifdef MS_ELEM_HALF
    MS_REQUIRE(ms_prenorm_parts(M, N, K) > 0, "product that prepares the norm: M=%d N=%d K=%d is not taken", M, N, K);
    MS_REQUIRE(norm_w && hn && ss_part, "product that prepares the norm: its outputs are missing");
    MS_REQUIRE((reinterpret_cast<uintptr_t>(a) & 15) == 0 && (reinterpret_cast<uintptr_t>(w) & 15) == 0, "gemm: operands must be 16-byte aligned");
    EpiArgs ep{x, nullptr, N, N, K, 0};
    ep.past = past && M <= 64;
    ep.norm_w = norm_w;
    ep.hn = (elem_t*)hn;
    ep.ss_part = ss_part;
    if (planned(M, K)) {
        if constexpr (kRoundsBeforeTheNormIsSafe) return launch_around_norm<EPI_PRENORM, false>((const elem_t*)a, (const elem_t*)w, M, N, K, ep, stream);
    }
    return launch_few<EPI_PRENORM>((const elem_t*)a, (const elem_t*)w, M, N, K, ep, stream, 1);
#else
    (void)a; (void)w; (void)x; (void)norm_w; (void)hn; (void)ss_part; (void)M; (void)N; (void)K; (void)stream;
    MS_REQUIRE(false, "product that prepares the norm: built for bfloat16 only");
#endif
}
extern "C" int ms_linear_residual_prenorm(const void* a, const void* w, float* x, const float* norm_w, void* hn, float* ss_part, int M, int N, int K,
                                          hipStream_t stream) {
    return linear_residual_prenorm(a, w, x, norm_w, hn, ss_part, M, N, K, stream, false);
}
extern "C" int ms_linear_residual_prenorm_past(const void* a, const void* w, float* x, const float* norm_w, void* hn, float* ss_part, int M, int N, int K,
                                          hipStream_t stream) {
    return linear_residual_prenorm(a, w, x, norm_w, hn, ss_part, M, N, K, stream, true);
}

// Whether ms_linear_qkv_rope takes this shape: two-byte elements, more rows than the few-rows kernels take, heads of
// 64 (a tile's columns are one head, so that both elements of a rotated pair lie in one lane), K in whole chunks.
// Heads of 128 are left to the plain product and the rotation kernel: tiles of one head's width, four waves above one
// another, give those shapes a worse count of blocks and less reuse in a wave than the plain product's wider tiles
// (7B layer sizes, 2,048 rows: 133 us in one launch against 81 + 17 in two; 1.5B, 512 rows: the step 6 % longer).
// So are steps of up to 256 rows: their few tiles are each a chain of all K steps, which takes 10 us whatever the
// number of LDS buffers, while the plain product cuts K over several blocks (0.5B sizes, 128 rows: 8.9 us in two
// kernels, 9.7 to 11.8 in one; from 384 rows on the one kernel is ahead: 10.0 against 10.9).
extern "C" int ms_qkv_rope_takes(int M, int H, int KV, int hd, int K) {
#ifdef MS_ELEM_HALF
    return M > 256 && H > 0 && KV > 0 && hd == 64 && K % 8 == 0 && K >= 128;
#else
    (void)M; (void)H; (void)KV; (void)hd; (void)K;
    return 0;
#endif
}

// The q/k/v projection of a step of many rows with what follows it in its epilogue: w [(H + 2 KV) * hd, K] holds the
// query heads, the key heads and the value heads; bias [(H + 2 KV) * hd] or null is added, queries and keys are rotated
// by the rows' angles (rope_cs [M, hd / 2, 2], cosine and sine, as ms_rope_table makes them), queries go to q_out
// [M, H * hd], keys and values into their pages at slot_map[row] (a negative slot is not written).  The same values as
// ms_linear (32-bit output) followed by ms_rope_kv_write, without the 32-bit sums' trip through memory and without
// the second launch.
extern "C" int ms_linear_qkv_rope(const void* a, const void* w, const float* bias, const float* rope_cs, const int* slot_map,
                                  void* q_out, void* kpool, void* vpool, int M, int H, int KV, int hd, int ps, int K,
                                  hipStream_t stream) {
#ifdef MS_ELEM_HALF
    MS_REQUIRE(ms_qkv_rope_takes(M, H, KV, hd, K), "q/k/v product with rotation: M=%d, %d + 2 x %d heads of %d, K=%d is not taken", M, H, KV, hd, K);
    MS_REQUIRE(rope_cs && slot_map && q_out && kpool && vpool && ps > 0, "q/k/v product with rotation: a buffer is missing");
    MS_REQUIRE((reinterpret_cast<uintptr_t>(a) & 15) == 0 && (reinterpret_cast<uintptr_t>(w) & 15) == 0, "gemm: operands must be 16-byte aligned");
    const int N = (H + 2 * KV) * hd;
    EpiArgs ep{q_out, bias, H * hd, N, K, 0, nullptr, 0, 0.f, 0, rope_cs, slot_map, (elem_t*)kpool, (elem_t*)vpool, H, KV, ps};
    const long round_blocks = 2L * compute_units();
#define MS_QKV(BM_, BN_)                                                                                                 \
    do {                                                                                                                 \
        const long nb = (long)ceil_div(M, BM_) * (N / BN_);                                                              \
        ep.group = row_group(BM_, BN_, BM_ == 128 ? 2 : 4, nb);                                                          \
        hipLaunchKernelGGL((gemm_kernel<BM_, BN_, 4, 1, 64, EPI_QKV_ROPE>), dim3((unsigned)nb, 1), dim3(256), 0, stream, \
                           (const elem_t*)a, (const elem_t*)w, M, N, K, ep);                                             \
        return check_launch("gemm q/k/v with rotation " #BM_ "x" #BN_);                                                  \
    } while (0)
    // rows in tiles of 128 where that still gives the chip a round of blocks, else of 64
    const bool tall = (long)ceil_div(M, 128) * (N / hd) >= round_blocks * 300 / 512;
    if (tall) MS_QKV(128, 64);
    if (K % 64 == 0 && K >= 256) {
        // three LDS buffers in turn (two K steps in flight, three blocks a CU): 0.5B, 2,048 rows, 17.0 -> 16.4 us; tiles of
        // 128x64 take 20.3 (288 blocks, barely one a CU, each step a trip to the L2); four buffers where the blocks are
        // at most two a CU (512 to 1,536 rows: 10.6 -> 10.0, 11.8 -> 11.4 us; at 2,048 rows 13.4 -> 17.9)
        const long nb = (long)ceil_div(M, 64) * (N / 64);
        ep.group = row_group(64, 64, 4, nb);
        if (nb <= round_blocks) {
            hipLaunchKernelGGL((gemm_kernel<64, 64, 4, 1, 64, EPI_QKV_ROPE, 4>), dim3((unsigned)nb, 1), dim3(256), 0, stream,
                               (const elem_t*)a, (const elem_t*)w, M, N, K, ep);
            return check_launch("gemm q/k/v with rotation 64x64 deeper");
        }
        hipLaunchKernelGGL((gemm_kernel<64, 64, 4, 1, 64, EPI_QKV_ROPE, 3>), dim3((unsigned)nb, 1), dim3(256), 0, stream,
                           (const elem_t*)a, (const elem_t*)w, M, N, K, ep);
        return check_launch("gemm q/k/v with rotation 64x64 deep");
    }
    MS_QKV(64, 64);
#undef MS_QKV
#else
    (void)a; (void)w; (void)bias; (void)rope_cs; (void)slot_map; (void)q_out; (void)kpool; (void)vpool; (void)M; (void)H; (void)KV;
    (void)hd; (void)ps; (void)K; (void)stream;
    MS_REQUIRE(false, "q/k/v product with rotation: built for two-byte elements only");
#endif
}

// Number of partial sums ms_linear_split_tiled writes for this problem (1 = the complete product).
extern "C" int ms_tiled_partials(int M, int N, int K) { return plan_tiled_splits(M, N, K); }

// The tile that a product over whole K steps runs in with that many K slices (an index into kTiles), or -1 where it is not planned (up to
// 64 rows, a partial K step, the 32-bit build).
extern "C" int ms_tiled_tile(int M, int N, int K, int splits, int store32) {
#ifdef MS_ELEM_HALF
    return planned(M, K) ? plan_gemm(M, N, K, max(1, splits), store32 != 0).tile : -1;
#else
    (void)M; (void)N; (void)K; (void)splits; (void)store32;
    return -1;
#endif
}

// Whether a 32-bit product with that many K slices runs in parts of 16 bits: 1 in tiles of 64x64, 2 of 128x128, else 0 (the two-byte builds: 0).
extern "C" int ms_parted(int M, int N, int K, int slices) {
#ifdef MS_ELEM_HALF
    (void)M; (void)N; (void)K; (void)slices;
    return 0;
#else
    return parted(M, N, K, slices) ? 1 + parted_wide(M, N, slices) : 0;
#endif
}

// The same of a gated product of `N` columns, gate and up.
extern "C" int ms_gated_tile(int M, int N, int K) {
#ifdef MS_ELEM_HALF
    return planned(M, K) ? plan_gemm(M, N, K, 1, false, true).tile : -1;
#else
    (void)M; (void)N; (void)K;
    return -1;
#endif
}

// Whether the entry points of the tiled products run this product in few_rows.cuh (then they are the ones to call): `slices` if its reader adds up
// K slices, `pairs` for the gated product.
extern "C" int ms_few_rows_takes(int M, int N, int K, int slices, int pairs) {
    return M >= 1 && N >= 1 && few_rows(M, N, K, slices != 0, pairs != 0);
}

// Whether a product of one row norms it itself, each of its blocks for itself, and how many slices it then leaves: with sums pending, where what a block keeps is within 64 KB
// and what all blocks read of it within 24 MB.  A kernel of the chain goes, its launch and its trips to memory; the product waits for the row instead.  Passes of one request, us,
// without and with: 0.5B sizes 8,340 and 8,090 (thirteen steps), 1.5B (23 MB) 16,240 and 16,010, 32-bit 0.5B (13 MB) 8,700 and 8,650; of two to four requests the same.
extern "C" int ms_few_normed_takes(int M, int N, int K, int n_pending) {
    if (M != 1 || n_pending < 1 || n_pending > 16 || !few_rows(M, N, K, true, false)) return 0;
    const FewPlan p = plan_few(M, N, K * FEW_BYTES, 0, false);
    const size_t lds = few_normed_lds(K, n_pending);
    return lds <= 64 * 1024 && lds * ceil_div(N, 16 * kFew[0][p.tile].nt) * p.splits <= 24u << 20 ? p.splits : 0;
}

// out[slices, 1, N] (float) = partial sums of rmsnorm(x + sum pending; norm_w, eps) w^T over ms_few_normed_takes slices of K, x_out = x + sum pending (another buffer than x).
static int linear_few_normed(const float* x, const float* pending, int n_pending, const float* norm_w, float eps, float* x_out, const void* w, float* out, int M, int N,
                             int K, hipStream_t stream, bool past) {
    const int ns = ms_few_normed_takes(M, N, K, n_pending);
    MS_REQUIRE(ns > 0, "product that norms its row: M=%d N=%d K=%d with %d pending sums is not taken", M, N, K, n_pending);
    MS_REQUIRE(x && pending && norm_w && x_out && x_out != x, "product that norms its row: a buffer is missing, or the stream would be written where it is read");
    MS_REQUIRE(((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(pending) | reinterpret_cast<uintptr_t>(norm_w) | reinterpret_cast<uintptr_t>(x_out) |
                 reinterpret_cast<uintptr_t>(w)) & 15) == 0, "product that norms its row: operands must be 16-byte aligned");
    EpiArgs ep{out, nullptr, N, N, ceil_div(ceil_div(K, ns), 64) * 64, (size_t)M * N};
    ep.past = past;
    ep.norm_w = norm_w, ep.ss_eps = eps;
    ep.stream = x, ep.pending = pending, ep.n_pending = n_pending, ep.stream_out = x_out;
    const unsigned lds = (unsigned)few_normed_lds(K, n_pending);
    const int tile = plan_few(M, N, K * FEW_BYTES, ns, false).tile;
#define MS_NORMED(TILE_)                                                                                                                                       \
    do {                                                                                                                                                       \
        constexpr FewCost t = kFew[0][TILE_];                                                                                                                  \
        hipLaunchKernelGGL((gemm_few_normed_kernel<t.nt, t.stages>), dim3((unsigned)ceil_div(N, 16 * t.nt), (unsigned)ns), dim3(64 * FEW_WAVES), lds, stream,  \
                           (const elem_t*)w, M, N, K, ep);                                                                                                     \
        return check_launch("gemm, few rows, normed");                                                                                                         \
    } while (0)
    if (tile == 0) MS_NORMED(0);
    if (tile == 1) MS_NORMED(1);
    MS_NORMED(2);
#undef MS_NORMED
}
extern "C" int ms_linear_few_normed(const float* x, const float* pending, int n_pending, const float* norm_w, float eps, float* x_out, const void* w, float* out, int M,
                                    int N, int K, hipStream_t stream) {
    return linear_few_normed(x, pending, n_pending, norm_w, eps, x_out, w, out, M, N, K, stream, false);
}
extern "C" int ms_linear_few_normed_past(const float* x, const float* pending, int n_pending, const float* norm_w, float eps, float* x_out, const void* w, float* out, int M,
                                         int N, int K, hipStream_t stream) {
    return linear_few_normed(x, pending, n_pending, norm_w, eps, x_out, w, out, M, N, K, stream, true);
}

// Of the products that few_rows.cuh does not take (a K that is no whole number of steps, 17 to 64 rows of some shapes, 32-bit), and of norms that could be
// folded in: whether a product of M rows is better served by the tiled kernel than by the one of skinny.hip (which
// takes at most 64 rows).  The few-rows kernel reads its rows again for every 32 or 64 columns; with
// many rows and a large weight that traffic outweighs the weight itself, and the tiled kernel, which
// shares the rows of a block through LDS, streams the weight faster (measured at the 0.5B, 1.5B and 7B
// layer sizes, 8 to 64 rows).  The choice changes the order of the sums, so results differ in rounding.
extern "C" int ms_prefers_tiled(int M, int N, int K) {
    if (M > 64) return 1;
#ifdef MS_ELEM_HALF
    // Above 32 rows the tiled kernel, with K cut over enough blocks, beats the few-rows kernel for every
    // weight (0.5B q/k/v projection at 64 rows: 9.7 us few-rows, 4.9 us tiled in seven slices).
    if (M > 32) return 1;
    const double nk = (double)N * (double)K;
    if (N >= 2048) {
        // A large weight under a wide output: the tiled kernel's blocks each stream their columns' rows of the
        // weight step after step, several steps in flight, while every wave of the few-rows kernel asks for its
        // whole share at once and then waits.  From one row on (decode steps of the 1.5B and 7B layer sizes at
        // batch 1, 2, 4, 8: 7 to 12 % shorter; the vocabulary-sized head of every shape); a smaller weight
        // (0.5B gate/up) from 17 rows on, where the few-rows kernel can no longer apply the norm itself and
        // re-reads its rows for every 32 columns (batch 32: 1.53 -> 1.40 ms a step); from 9 rows on where the output
        // is wide (0.5B gate/up, 9,728 columns), together with the narrow projections below: the norm between them
        // then runs by itself and adds the K slices (0.5B decode step at batch 12 and 16: 1.085 -> 1.056 ms; a
        // 2,048-wide output, the 1.5B q/k/v projection, loses 1 % by it and keeps the few-rows kernel up to 16 rows).
        return nk >= 10e6 || M >= 17 || (M >= 9 && N >= 4096);
    }
    if (N >= 1024) {
        // a projection of the width (q/k/v, output): from 16 rows, or 8 if it is not small (batch 32: 1.40 ->
        // 1.36 ms a step; 0.5B q/k/v at 8 rows is faster in the few-rows kernel); a large weight (the 1.5B down
        // projection: 27 MB) from one row on (1.5B decode step at batch 1 and 4: 1.5 % shorter)
        return M >= 16 || (M >= 8 && nk >= 2e6) || nk >= 10e6;
    }
    // a narrow output (the 0.5B output and down projections, 896 columns): from 9 rows on the tiled kernel with K cut
    // over many blocks (0.5B decode step at batch 24 and 32: 1.195 -> 1.129 and 1.200 -> 1.138 ms, all of it from the
    // output projection; at 9 to 16 rows only together with the gate/up product above)
    return M >= 9;
#else
    return 0;
#endif
}

// K slices of a product that is added to the residual stream, whose next norm adds them up: those of ms_tiled_partials, and in the 32-bit build those of a long K
// under a narrow output, whose uncut 32x32 tiles are each a chain of all K steps: slices that fill the chip with 128x128 tiles, eight at most.  us, uncut and in slices:
// 512 x 896 x 4,864 53 and 38 (eight), 192 rows 43 and 25, 1,024 rows 92 and 66 (four).
extern "C" int ms_residual_partials(int M, int N, int K) {
#ifndef MS_ELEM_HALF
    if (M > 64 && N < 4096 && K >= 4096 && K % 32 == 0) {
        const int want = max(1, min(8, (int)(compute_units() / ((long)ceil_div(M, 128) * ceil_div(N, 128)))));
        return ceil_div(K, ceil_div(ceil_div(K, want), 64) * 64);
    }
#endif
    return plan_tiled_splits(M, N, K);
}

// out[slices, M, N] (float) = partial sums of a w^T over that many slices of K.
static int linear_slices(const void* a, const void* w, float* out, int M, int N, int K, int slices, hipStream_t stream, bool past) {
    EpiArgs ep{out, nullptr, N, N, 0, 0};
    ep.past = past && M <= 64;
    return launch_gemm<EPI_STORE_F32>((const elem_t*)a, (const elem_t*)w, M, N, K, ep, stream, slices);
}
extern "C" int ms_linear_slices(const void* a, const void* w, float* out, int M, int N, int K, int slices, hipStream_t stream) {
    return linear_slices(a, w, out, M, N, K, slices, stream, false);
}
extern "C" int ms_linear_slices_past(const void* a, const void* w, float* out, int M, int N, int K, int slices, hipStream_t stream) {
    return linear_slices(a, w, out, M, N, K, slices, stream, true);
}

// out[ks, M, N] (float) = partial sums of a w^T over ms_tiled_partials(M, N, K) slices of K.
static int linear_split_tiled(const void* a, const void* w, float* out, int M, int N, int K, hipStream_t stream, bool past) {
    EpiArgs ep{out, nullptr, N, N, 0, 0};
    ep.past = past && M <= 64;
    return launch_gemm<EPI_STORE_F32>((const elem_t*)a, (const elem_t*)w, M, N, K, ep, stream, plan_tiled_splits(M, N, K));
}
extern "C" int ms_linear_split_tiled(const void* a, const void* w, float* out, int M, int N, int K, hipStream_t stream) {
    return linear_split_tiled(a, w, out, M, N, K, stream, false);
}
extern "C" int ms_linear_split_tiled_past(const void* a, const void* w, float* out, int M, int N, int K, hipStream_t stream) {
    return linear_split_tiled(a, w, out, M, N, K, stream, true);
}

// Measurements only: force one tile configuration (0 = choose by shape).
#ifdef MS_MEASURE
extern "C" void ms_gemm_force_config(int c) { g_gemm_config = c; }
extern "C" void ms_gemm_force_splits(int n) { g_force_splits = n; }
#endif
