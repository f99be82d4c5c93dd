// One block of out[M, N] = A[M, K] * W[N, K]^T on the matrix cores: the K loop and the fused epilogues that the plain products
// (gemm.hip) and the products over the rows of routed experts (routed.hip) share.
//
// Both operands are contiguous along K, so a 16x32 MFMA fragment of either is "row
// l % 16, elements (l / 16) * 8 .. + 8".  Two LDS buffers and one barrier a K step, three or four buffers with as many steps less one in
// flight, or two buffers and two barriers in phases (GEMM_PIPED).  LDS has 64 banks
// of 4 bytes; the 16-byte fragment reads of a wave are free of bank conflicts when the row pitch is
// 32 modulo 64 bytes (measured: pitches of 80 or 144 bytes take twice as long), or, with unpadded
// rows of 128 bytes, when chunk c of row r lies at position c ^ (r & 7).
// bfloat16 with K steps of 64: tiles go global -> LDS directly (global_load_lds_dwordx4, a wave's
// 64 lanes fill 1 KB = 8 unpadded rows in lane order, so the swizzle is applied to the global
// address), and the next step's tile is in flight while this one is multiplied (how far ahead, and with how many buffers, see the
// loops below); only a partial last step goes through registers, where what lies beyond K is masked.  K steps of 32 of
// two-byte elements, and in 32-bit whatever has a partial last step, go global -> registers -> LDS (padded rows); the other
// products of the 32-bit build go straight to LDS as well (its K steps of 32 are rows of 128 bytes too).
// Every output element is the sum over K in steps of 32 in ascending order whatever the
// tile shape, so a row's result does not depend on the tile that its batch runs in.  What does go by the number of rows is whether K is cut into slices whose sums the
// reader adds (the 32-bit build: under a narrow output alone), and which 32-bit products are worked out in parts, with sums of their own (GEMM_SPLIT).
#pragma once
#include <type_traits>

#include "common.cuh"

namespace ms {

#ifdef MS_ELEM_HALF
constexpr int EPC = 8;   // elements per 16-byte chunk
constexpr int KPAD = 16;  // row padding in elements: rows of 96 (BK 32) or 160 (BK 64) bytes
#else
constexpr int EPC = 4;
constexpr int KPAD = 8;  // rows of 160 bytes (BK 32)
#endif

constexpr int GEMM_PIPED = 1;  // in the place of a number of LDS buffers: two of them, in phases (see gemm_tile)
constexpr int GEMM_SPLIT = 8;  // 32-bit: two buffers, and every number in three parts of 16 bits (see gemm_tile)

enum EpiKind {
    EPI_STORE_F32 = 0, EPI_STORE_ELEM = 1, EPI_RESIDUAL = 2, EPI_SWIGLU = 3, EPI_QKV_ROPE = 4, EPI_ACT = 5,
    EPI_EXPERT_GATED = 6, EPI_EXPERT_PLAIN = 7, EPI_EXPERT_DOWN = 8,  // over the rows that chose an expert (routed.hip)
    EPI_PRENORM = 9,  // into the residual stream, and what the norm that follows needs
};

struct NoExperts {
    static constexpr bool GATHERS = false;  // A's rows lie one behind the other
    __device__ __forceinline__ int source(int m) const { return m; }
    __device__ __forceinline__ int pitch(int K) const { return K; }    // elements from a row of A to the next
    __device__ __forceinline__ int w_pitch(int K) const { return K; }  // ... of W
};

struct EpiArgs {
    void* out;          // [M, ldo]
    const float* bias;  // [N] or null
    int ldo;
    int n_out;          // SWIGLU: number of output columns (intermediate size)
    int k_per_split;    // K range of one blockIdx.y slice (multiple of 32); K itself without split
    size_t split_stride;  // STORE_F32 with gridDim.y > 1: elements between the slices' outputs
    // a factor a row for the finished sums (the RMS norm of rows that came in multiplied by the norm's weight only):
    // 1 / sqrt(sum over parts of row_ss[part, row] / K + ss_eps)
    const float* row_ss;  // [ss_parts, M] or null
    int ss_parts;
    float ss_eps;
    int act;            // SWIGLU: the activation on the gate (GateActivation); ACT: the activation (UnaryActivation)
    // QKV_ROPE: the columns are H query heads, KV key heads and KV value heads of the tile's width; bias added, queries
    // and keys rotated by the rows' angles (pairs (j, j + half a head)), queries to `out` [M, H * hd], keys and values
    // into their pages
    const float* rope_cs;  // [M, hd / 2, 2]: cosine and sine of each row's angles
    const int* slot_map;   // [M]: page * ps + offset of each row's key and value, or negative: not written
    elem_t* kpool;         // [pages, KV, ps, hd]
    elem_t* vpool;         // [pages, KV, hd, ps]
    int H, KV, ps;
    // PRENORM: the new values of the stream times the norm's weight, not yet divided by the rows' root mean square, and each tile's (of 16 columns; in
    // tiles of more than 64 rows each column of waves') share of the rows' sums of squares
    const float* norm_w;  // [N]
    elem_t* hn;           // [M, N]
    float* ss_part;       // [N / 16, or the columns of a wave, rounded up, M]
    // a row that its product norms: the stream [K], its pending sums [n_pending, K], and where the stream with them goes (norm_w and ss_eps as above)
    const float* stream = nullptr;
    const float* pending = nullptr;
    int n_pending = 0;
    float* stream_out = nullptr;
    int group = 1;        // row tiles that a run of the tiles' order has side by side (see tile_of_block)
    int past = 0;         // W is read past the last-level cache (see few_rows.cuh): up to 64 rows, where every block reads its own columns of it
};

// The block of rows m0 .. m0 + BM and columns n0 .. n0 + BN.  `rows` says which row of A the block's row i is and, for the
// experts' epilogues, what becomes of it (NoExperts: the rows as they come).
template <int BM, int BN, int WM, int WN, int BK, int EPI, int STAGES, bool SCALED, class Rows>
__device__ __forceinline__ void gemm_tile(const elem_t* __restrict__ A, const elem_t* __restrict__ W, int M, int N, int K, const EpiArgs& ep,
                                          int m0, int n0, int split, const Rows& rows) {
    static_assert(WM * WN == 4 || WM * WN == 8, "four waves, or eight for the widest tiles");
    constexpr int NT = 64 * WM * WN;  // threads of the block
    static_assert(BK % 32 == 0, "K step in MFMA steps of 32");
#ifdef MS_ELEM_HALF
    constexpr bool DIRECT = BK == 64;
#else
    constexpr bool DIRECT = STAGES > 2 && STAGES != GEMM_SPLIT;
#endif
    constexpr bool PIPED = STAGES == GEMM_PIPED, SPLIT = STAGES == GEMM_SPLIT;
    constexpr int BUFS = PIPED || SPLIT ? 2 : STAGES;
    // Tiles of more than 256 columns (256x320 under eight waves of 128x80: 160 registers of sums and 72 of fragments) have no register to spare for a lane's
    // offsets into the operands: rows of W go in eights with a scalar base (N is a multiple of 8), those of A are worked out at each load.
    constexpr bool WIDE = BN > 256;
    static_assert(!WIDE || (PIPED && !Rows::GATHERS), "wide tiles: in phases, rows as they come");
    constexpr int LDS_LD = SPLIT ? BK * 3 / 2 : DIRECT ? BK : BK + KPAD;
    constexpr int CPR = BK / EPC;  // chunks per tile row
    // where chunk `chunk` of tile row `row` lies in a buffer
    auto at = [](int row, int chunk) { return row * LDS_LD + (DIRECT ? (chunk ^ (row & 7)) : chunk) * EPC; };
    constexpr int TM = BM / WM / 16, TN = BN / WN / 16;
    constexpr int A_CHUNKS = BM * CPR / NT, W_CHUNKS = BN * CPR / NT;
    static_assert(BM * CPR % NT == 0 && BN * CPR % NT == 0, "tile loads divide over the block");
    static_assert(NT == 256 || !SCALED || PIPED, "the row factors' shares are dealt to four waves");
    static_assert(STAGES == 2 || DIRECT || SPLIT, "more than two LDS buffers, and phases, only with direct loads");
    static_assert(!SCALED || ((STAGES > 2 || PIPED) && EPI == EPI_SWIGLU), "row factors: built for the gated product with several steps in flight");
    static_assert(256 % BM == 0 || !SCALED, "threads are dealt to the rows");
    // the rows' sums of squares, in 256 / BM interleaved shares; in phases the rows' factors
    __shared__ float ss_q[SCALED && !PIPED ? 256 / BM : 1][SCALED ? BM : 1];
    float ss_v[SCALED ? 8 : 1];
    int ss_r = 0;
    __shared__ __attribute__((aligned(16))) elem_t As[BUFS][BM * LDS_LD];
    __shared__ __attribute__((aligned(16))) elem_t Ws[BUFS][BN * LDS_LD];

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave / WN, wn = wave % WN;
    const int r16 = lane & 15, grp = lane >> 4;

    const int k_end = min(K, (split + 1) * ep.k_per_split);
    // Loads are unconditional, on one straight path: a row beyond the operand reads the last row
    // (its results are never stored), and only the last K step of a slice, if it is a partial one,
    // masks what lies beyond the slice.
    u32x4 ra[A_CHUNKS], rw[W_CHUNKS];
    const elem_t* pa[A_CHUNKS];
    const elem_t* pw[W_CHUNKS];
    // Thread t owns position (t + i * NT) % CPR of tile row (t + i * NT) / CPR; with swizzled rows that
    // position holds another chunk of K, the same one for every i (NT / CPR rows on is a multiple of 8).
    const int my_chunk = DIRECT ? (tid % CPR) ^ ((tid / CPR) & 7) : tid % CPR;
#pragma unroll
    for (int i = 0; i < A_CHUNKS; ++i) {
        const int c = tid + i * NT;
        pa[i] = A + (size_t)rows.source(min(m0 + c / CPR, M - 1)) * rows.pitch(K) + my_chunk * EPC;
    }
#pragma unroll
    for (int i = 0; i < W_CHUNKS; ++i) {
        const int c = tid + i * NT;
        pw[i] = W + (size_t)min(n0 + c / CPR, N - 1) * rows.w_pitch(K) + my_chunk * EPC;
    }
    auto load_global = [&](int k0) {
#pragma unroll
        for (int i = 0; i < A_CHUNKS; ++i) ra[i] = *reinterpret_cast<const u32x4*>(pa[i] + k0);
#pragma unroll
        for (int i = 0; i < W_CHUNKS; ++i) rw[i] = *reinterpret_cast<const u32x4*>(pw[i] + k0);
    };
    auto load_global_tail = [&](int k0) {
        const int kk = k0 + my_chunk * EPC;  // the same K chunk for all of a thread's loads
        const bool in = kk < k_end;
        const uint32_t keep = opaque(in ? 0xffffffffu : 0u);
#pragma unroll
        for (int i = 0; i < A_CHUNKS; ++i) {
            u32x4 v = *reinterpret_cast<const u32x4*>(in ? pa[i] + k0 : A);  // the operand's start when beyond the slice
            ra[i] = (u32x4){v[0] & keep, v[1] & keep, v[2] & keep, v[3] & keep};
        }
#pragma unroll
        for (int i = 0; i < W_CHUNKS; ++i) {
            u32x4 v = *reinterpret_cast<const u32x4*>(in ? pw[i] + k0 : W);
            rw[i] = (u32x4){v[0] & keep, v[1] & keep, v[2] & keep, v[3] & keep};
        }
    };
    auto store_lds = [&](int buf) {
#pragma unroll
        for (int i = 0; i < A_CHUNKS; ++i) {
            const int c = tid + i * NT, row = c / CPR;
            *reinterpret_cast<u32x4*>(&As[buf][at(row, my_chunk)]) = ra[i];
        }
#pragma unroll
        for (int i = 0; i < W_CHUNKS; ++i) {
            const int c = tid + i * NT, row = c / CPR;
            *reinterpret_cast<u32x4*>(&Ws[buf][at(row, my_chunk)]) = rw[i];
        }
    };
    // One K step of both tiles straight into LDS buffer `buf`: lane l of a wave's load lands at the wave's
    // base + 16 l.  Written in assembly: of a load that it knows to write LDS the compiler makes every later
    // LDS read wait (vmcnt(0)), and nothing would be in flight during the multiplications; the waits are
    // explicit instead (`step_barrier`).  The bases are scalars, and so are the operands' with a lane's offset of 32 bits
    // (a tile's rows lie within 4 GiB): kept a lane, the places in LDS alone took 32 registers, and the 256-row tiles spilled.
    const int swave = __builtin_amdgcn_readfirstlane(wave);
    // The first of the eight tile rows that this wave loads in round i.  In phases, the rounds' first half brings the rows that the waves' first
    // halves of row tiles read.
    auto a_row = [&](int i) {
        if constexpr (PIPED) {
            constexpr int HR = BM / WM / 2;
            const int at8 = (i % (A_CHUNKS / 2)) * (NT / 64) + swave;
            return at8 / (HR / 8) * (BM / WM) + (i / (A_CHUNKS / 2)) * HR + at8 % (HR / 8) * 8;
        } else {
            return i * (NT / 8) + swave * 8;
        }
    };
    const uint32_t lds_a = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)&As[0][0];
    const uint32_t lds_w = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)&Ws[0][0];
    const elem_t* base_a = A + (size_t)rows.source(m0) * rows.pitch(K);
    const elem_t* base_w = W + (size_t)n0 * rows.w_pitch(K);
    uint32_t oa[A_CHUNKS], ow[W_CHUNKS];
    // (a product of 32 bits is made in 64, and its upper half would keep a register)
    auto alone = [](uint32_t x) {
        uint32_t y;
        asm("v_mov_b32 %0, %1" : "=v"(y) : "v"(x));
        return y;
    };
    auto a_offset = [&](int row) {  // of row m0 + `row`, or the last one
        return ((uint32_t)min(row, M - 1 - m0) * (uint32_t)rows.pitch(K) + my_chunk * EPC) * (uint32_t)sizeof(elem_t);
    };
    const elem_t* ga[Rows::GATHERS ? A_CHUNKS : 1];
    if constexpr (DIRECT) {
#pragma unroll
        for (int i = 0; i < A_CHUNKS; ++i) {
            if constexpr (Rows::GATHERS) ga[i] = A + (size_t)rows.source(min(m0 + a_row(i) + lane / 8, M - 1)) * rows.pitch(K) + my_chunk * EPC;
            else oa[i] = alone(a_offset(a_row(i) + lane / 8));
        }
#pragma unroll
        for (int i = 0; i < W_CHUNKS; ++i)
            ow[i] = alone(((uint32_t)(WIDE ? lane / 8 : min(n0 + (tid + i * NT) / CPR, N - 1) - n0) * (uint32_t)rows.w_pitch(K) + my_chunk * EPC) *
                          (uint32_t)sizeof(elem_t));
    }
    // load l of a step: A's rounds, then W's
    auto load_one = [&](int k0, int buf, int l) {
        if (l < A_CHUNKS) {
            const uint32_t to = lds_a + buf * (BM * LDS_LD * (int)sizeof(elem_t)) + a_row(l) * (LDS_LD * (int)sizeof(elem_t));
            if constexpr (Rows::GATHERS)
                asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(ga[l] + k0), "s"(to) : "memory", "m0");
            else
                asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(WIDE ? a_offset(a_row(l) + opaque(lane) / 8) : oa[l]), "s"(base_a + k0), "s"(to) : "memory", "m0");
        } else {
            const int i = l - A_CHUNKS;
            const uint32_t to = lds_w + buf * (BN * LDS_LD * (int)sizeof(elem_t)) + (i * (NT / 8) + swave * 8) * (LDS_LD * (int)sizeof(elem_t));
            const elem_t* from = WIDE ? W + (size_t)min(n0 + i * (NT / 8) + swave * 8, N - 8) * rows.w_pitch(K) : base_w;
            if (STAGES == 4 && BM == 64 && ep.past)
                asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1 nt" ::"v"(ow[WIDE ? 0 : i]), "s"(from + k0), "s"(to) : "memory", "m0");
            else asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(ow[WIDE ? 0 : i]), "s"(from + k0), "s"(to) : "memory", "m0");
        }
    };
    auto load_direct = [&](int k0, int buf) {
#pragma unroll
        for (int l = 0; l < A_CHUNKS + W_CHUNKS; ++l) load_one(k0, buf, l);
    };
    // End of a K step: this wave's loads and LDS accesses have completed, then everybody's.
    auto step_barrier = [&]() {
        if constexpr (DIRECT) {
            __builtin_amdgcn_sched_barrier(0);
            asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_s_barrier();
            __builtin_amdgcn_sched_barrier(0);
        } else {
            __syncthreads();
        }
    };

    // The first column of a wave's tile j.  Gate and up tiles alternate; where a wave has an odd number of them, the last is an even wave's
    // gate tile and the next wave's up tile to it.
    constexpr bool SPLIT_PAIR = EPI == EPI_SWIGLU && TN % 2 != 0;
    static_assert(!SPLIT_PAIR || (PIPED && WN % 2 == 0), "a pair between two waves: in phases");
    const bool second = SPLIT_PAIR && (swave & 1);
    const int col_first = wn * (BN / WN) + (second ? 16 : 0), col_last = wn * (BN / WN) + (second ? 0 : (TN - 1) * 16);
    auto tile_col = [&](int j) { return SPLIT_PAIR && j == TN - 1 ? col_last : col_first + j * 16; };

    f32x4 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};

    // a slice of K per blockIdx.y: partial sums that the consumer adds in slice order
    const int k_begin = split * ep.k_per_split;
    const int nk = ceil_div(k_end - k_begin, BK);
    const bool partial = (k_end - k_begin) % BK != 0;  // the last step is a partial one
    // 8 elements of a tile's row, of the K chunk of 32 at kk, in swizzled rows: one 16-byte chunk, or in 32-bit two
    auto tile_frag = [&](const elem_t* t, int row, int kk) {
#ifdef MS_ELEM_HALF
        return frag_load(&t[at(row, kk / EPC + grp)]);
#else
        Frag f;
        const f32x4 x = *reinterpret_cast<const f32x4*>(&t[at(row, kk / EPC + 2 * grp)]), y = *reinterpret_cast<const f32x4*>(&t[at(row, kk / EPC + 2 * grp + 1)]);
#pragma unroll
        for (int e = 0; e < 4; ++e) { f.v[e] = x[e]; f.v[4 + e] = y[e]; }
        return f;
#endif
    };
    auto multiply = [&](int buf) {
#pragma unroll
        for (int kk = 0; kk < BK; kk += 32) {
            Frag fa[TM], fb[TN];
            if constexpr (DIRECT) {
#pragma unroll
                for (int i = 0; i < TM; ++i) fa[i] = tile_frag(As[buf], wm * (BM / WM) + i * 16 + r16, kk);
#pragma unroll
                for (int j = 0; j < TN; ++j) fb[j] = tile_frag(Ws[buf], wn * (BN / WN) + j * 16 + r16, kk);
            } else {
#pragma unroll
                for (int i = 0; i < TM; ++i) fa[i] = frag_load(&As[buf][(wm * (BM / WM) + i * 16 + r16) * LDS_LD + kk + grp * 8]);
#pragma unroll
                for (int j = 0; j < TN; ++j) fb[j] = frag_load(&Ws[buf][(wn * (BN / WN) + j * 16 + r16) * LDS_LD + kk + grp * 8]);
            }
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) mma_16x16x32(acc[i][j], fa[i], fb[j]);
        }
    };
    if constexpr (SPLIT) {
#ifndef MS_ELEM_HALF
        // Numbers of 32 bits in three parts of 16 (bfloat16, which has their exponents): x = x1 + x2 + x3, each the rounding of what the ones before it
        // leave, so that nothing is lost, and eight of a product's nine terms on the 16-bit matrix instructions, where each is exact.  |x2| is at most 2^-8 |x| and |x3|
        // 2^-17 |x|: x3 y3, which is left out, is a thousandth of a product's rounding in 32 bits (x2 y3 and x3 y2 together are as much as that rounding).  x1 y1 has
        // sums of its own, which a step rounds once; the others, below 2^-6 of them, would round them seven times more.  The eight take 128 cycles where the 32-bit
        // instructions take 256.  Relative error against 64 bits, in those and here: normal inputs of K = 896 5.4e-7 and 1.7e-7, 2,048 8.1e-7 and 2.7e-7, 4,864 in
        // eight slices 4.5e-7 and 1.5e-7; positive inputs of K = 896 4.6e-7 and 1.7e-7; a single product at most 5.93e-8 and 5.96e-8 (with the six largest terms in
        // one set of sums 4.5e-7 and, of a single product, 1.28e-7).
        // The threads hold a step's numbers for two steps, part them two at a time between the matrix instructions, and store each part's rows of 64 bytes for
        // the next step; two buffers, one barrier a step.  What bounds it: a matrix instruction leaves the issue of two others free, and LDS takes stores at a third of
        // the rate of reads (with six terms in one set of sums, 128x128 of K = 4,864, one block a CU, 166 us: parting and storing alone 115, the matrix instructions
        // and LDS reads 110).  us, 32-bit instructions and here: 512 x 9,728 x 896 93 and 79 (64x64), 1,024 x 17,920 x 1,536 461 and 396 (128x128); with K in
        // slices 512 x 896 x 4,864 53 (uncut) and 38.  (Six terms: 67, 332 and 31.)
        static_assert(BK == 32 && BM * 4 % NT == 0 && BN * 4 % NT == 0, "four threads a row");
        constexpr int A_ROUNDS = BM * 4 / NT, W_ROUNDS = BN * 4 / NT, ROUNDS = A_ROUNDS + W_ROUNDS;
        // thread t has the eight numbers t % 4 of row t / 4 of every round
        const int t_row = tid / 4, t_chunk = tid % 4;
        const float* from[ROUNDS];
#pragma unroll
        for (int i = 0; i < ROUNDS; ++i) {
            const int row = (i < A_ROUNDS ? i : i - A_ROUNDS) * (NT / 4) + t_row;
            from[i] = (i < A_ROUNDS ? A + (size_t)rows.source(min(m0 + row, M - 1)) * rows.pitch(K) : W + (size_t)min(n0 + row, N - 1) * rows.w_pitch(K)) + k_begin + t_chunk * 8;
        }
        f32x4 held[2][ROUNDS][2];  // of two steps
        auto ask = [&](int kt, int set) {
#pragma unroll
            for (int i = 0; i < ROUNDS; ++i)
#pragma unroll
                for (int h = 0; h < 2; ++h) held[set][i][h] = *reinterpret_cast<const f32x4*>(from[i] + kt * 32 + h * 4);
        };
        auto place = [](int row, int chunk) { return row * LDS_LD + (chunk ^ ((row >> 1) & 2)) * 4; };  // in floats; a part's rows are 64 bytes, 192 apart
        u32x4 part[3];
        float most[ROUNDS];  // the largest size of the thread's numbers of each round
#pragma unroll
        for (int i = 0; i < ROUNDS; ++i) most[i] = 0.f;
        auto put = [&](int set, int buf, int unit) {  // two numbers of round unit / 4, and the round's stores behind its last
            const int i = unit / 4, e = unit % 4;
            float x = held[set][i][e / 2][e % 2 * 2], y = held[set][i][e / 2][e % 2 * 2 + 1];
            asm("v_max3_f32 %0, %0, |%1|, |%2|" : "+v"(most[i]) : "v"(x), "v"(y));
#pragma unroll
            for (int q = 0; q < 3; ++q) {
                const uint32_t xy = round_pair(x, y);
                part[q][e] = xy;
                if (q < 2) {
                    x -= __uint_as_float(xy << 16);
                    y -= __uint_as_float(xy & 0xffff0000u);
                }
            }
            if (e == 3) {
                float* to = (i < A_ROUNDS ? &As[buf][0] : &Ws[buf][0]) + place((i < A_ROUNDS ? i : i - A_ROUNDS) * (NT / 4) + t_row, t_chunk);
#pragma unroll
                for (int q = 0; q < 3; ++q) *reinterpret_cast<u32x4*>(to + q * 16) = part[q];
            }
        };
        constexpr int UNITS = ROUNDS * 4, FIRST = UNITS / 4;
        ask(0, 0);
        ask(min(1, nk - 1), 1);
#pragma unroll
        for (int u = 0; u < UNITS; ++u) put(0, 0, u);
        __syncthreads();
        f32x4 low[TM][TN];
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) low[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
        auto step = [&](int kt, int buf) {
            ask(min(kt + 2, nk - 1), buf);
            bf16x8 fa[TM][3], fb[TN][3];
#pragma unroll
            for (int q = 2; q >= 0; --q) {
#pragma unroll
                for (int i = 0; i < TM; ++i) fa[i][2 - q] = *reinterpret_cast<const bf16x8*>(&As[buf][place(wm * (BM / WM) + i * 16 + r16, grp) + (2 - q) * 16]);
#pragma unroll
                for (int j = 0; j < TN; ++j) fb[j][q] = *reinterpret_cast<const bf16x8*>(&Ws[buf][place(wn * (BN / WN) + j * 16 + r16, grp) + q * 16]);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < FIRST; ++u) put(buf ^ 1, buf ^ 1, u);  // (behind the last step: a place that nobody reads)
            __builtin_amdgcn_sched_barrier(0);
            constexpr int GR = TM * TN >= 4 ? 4 : TM * TN, GROUPS = 8 * TM * TN / GR;
#pragma unroll
            for (int g = 0; g < GROUPS; ++g) {  // the smallest products first
                constexpr int qa[8] = {2, 1, 2, 0, 1, 1, 0, 0}, qb[8] = {1, 2, 0, 2, 1, 0, 1, 0};
#pragma unroll
                for (int u = FIRST; u < UNITS; ++u)
                    if ((u - FIRST) * GROUPS / (UNITS - FIRST) == g) put(buf ^ 1, buf ^ 1, u);
#pragma unroll
                for (int m = g * GR; m < (g + 1) * GR; ++m) {
                    const int t = m / (TM * TN), i = m / TN % TM, j = m % TN;
                    f32x4& sum = t == 7 ? acc[i][j] : low[i][j];
                    sum = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[i][qa[t]], fb[j][qb[t]], sum, 0, 0, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            __syncthreads();
        };
        int kt = 0;
        for (; kt + 1 < nk; kt += 2) {
            step(kt, 0);
            step(kt + 1, 1);
        }
        if (kt < nk) step(kt, 0);
        // Parts lose what is below 2^-133, and 2^-126 if such numbers count as zeros: of a sum K 2^-126 (X + Y) at most, X and Y the largest sizes in its row and its
        // column of W.  A sum beneath 2^-80 of those is taken from the 32-bit matrix instructions, as is one beneath 2^-100, whose terms may round more often than once,
        // and one that is not finite (an infinity's second part is NaN, and so are those of a number whose first part rounds up to infinity).  Zeros of a
        // row or column of zeros are right as they are.  Only these sums are: no other row or column of the block shows what stands beside it.
        __shared__ float largest[BM + BN];
#pragma unroll
        for (int i = 0; i < ROUNDS; ++i) {
            float v = most[i];
            v = fmaxf(v, __shfl_xor(v, 1, WAVE));
            v = fmaxf(v, __shfl_xor(v, 2, WAVE));
            if (t_chunk == 0) largest[i * (NT / 4) + t_row] = v;
        }
        __syncthreads();
        auto sound = [](float v, float x, float y) {
            const float least = x == 0.f || y == 0.f ? 0.f : fmaxf(fmaxf(x, y) * 0x1p-80f, 0x1p-100f);
            return fabsf(v) >= least && fabsf(v) < INFINITY;
        };
        float row_max[TM][4], col_max[TN];
        bool again = false;
#pragma unroll
        for (int j = 0; j < TN; ++j) col_max[j] = largest[BM + wn * (BN / WN) + j * 16 + r16];
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) row_max[i][e] = largest[wm * (BM / WM) + i * 16 + grp * 4 + e];
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    acc[i][j][e] += low[i][j][e];
                    again |= !sound(acc[i][j][e], row_max[i][e], col_max[j]);
                }
        if (__syncthreads_or(again)) {
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) low[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
            for (int k = k_begin; k < k_end; k += 32) {
                Frag ra_[TM];
#pragma unroll
                for (int i = 0; i < TM; ++i)
                    ra_[i] = frag_load(A + (size_t)rows.source(min(m0 + wm * (BM / WM) + i * 16 + r16, M - 1)) * rows.pitch(K) + k + grp * 8);
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    const Frag rb = frag_load(W + (size_t)min(n0 + wn * (BN / WN) + j * 16 + r16, N - 1) * rows.w_pitch(K) + k + grp * 8);
#pragma unroll
                    for (int i = 0; i < TM; ++i) mma_16x16x32(low[i][j], ra_[i], rb);
                }
            }
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (!sound(acc[i][j][e], row_max[i][e], col_max[j])) acc[i][j][e] = low[i][j][e];
        }
#endif
    } else if constexpr (PIPED) {
#ifdef MS_ELEM_HALF
        // Two LDS buffers, whole K steps.  What bounds the loop with one burst of loads a step and all of a K chunk's fragments read before they are
        // multiplied (measured with parts of it left out, 256x256 tiles, 2,048 x 37,888 x 3,584: 493 us; without the loads
        // 351, without the matrix instructions 410, without both 124): a step waits for its burst, and LDS reads and
        // matrix instructions add up.  So:
        // * a step is four phases, (first half of the wave's rows, K chunk 0), (first, 1), (second, 0), (second, 1); in each the wave
        //   reads the fragments of the next one between groups of this one's matrix instructions;
        // * W and the first half's rows have been read when phase 0 ends, the second half's when phase 2 ends: the loads of the step
        //   after the next go out there, in two portions, into the places just read, and have a step and a half to
        //   come.  The wait at both places is for all but the last step's worth of loads; the two barriers a step say that
        //   everybody's have come and that everybody has read.
        // 256x256: 493 -> 429 us (with the order of the tiles); 256x192 of 2,048 x 11,264 x 2,048: 79 us (128x128 tiles in the old loop:
        // 103); 128x128 of 2,048 x 2,048 x 5,632, one block a CU: 80 -> 60.
        static_assert(TM % 2 == 0 && A_CHUNKS % 2 == 0, "a wave's rows in two halves");
        constexpr int TH = TM / 2;
        Frag fa[2][TH], fb[2][TN];
        // A lane's places in the tiles' first rows, for both K chunks: the others are constants further (rows 16 apart are swizzled alike).
        int lane_a[2], lane_b[2];
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
            lane_a[kk] = (int)opaque((uint32_t)at(wm * (BM / WM) + r16, kk * (32 / EPC) + grp));
            lane_b[kk] = (int)opaque((uint32_t)at(col_first + r16, kk * (32 / EPC) + grp));
        }
        const int last_b = col_last - col_first;
        auto fetch_a = [&](int buf, int half, int kk, int to, int i) {
            fa[to][i] = frag_load(&As[0][lane_a[kk] + (WIDE ? 0 : buf * BM * LDS_LD) + (half * TH + i) * 16 * LDS_LD]);
        };
        auto fetch_b = [&](int buf, int kk, int j) {
            const int at_j = SPLIT_PAIR && j == TN - 1 ? last_b * LDS_LD : j * 16 * LDS_LD;
            fb[kk][j] = frag_load(&Ws[0][lane_b[kk] + (WIDE ? 0 : buf * BN * LDS_LD) + at_j]);
        };
        constexpr int PER_STEP = A_CHUNKS + W_CHUNKS, EARLY = W_CHUNKS + A_CHUNKS / 2;
        static_assert(PER_STEP <= 63, "the wait count is a 6-bit field");
        auto load_nth = [&](int k0, int buf, int l) { load_one(k0, buf, l < W_CHUNKS ? A_CHUNKS + l : l - W_CHUNKS); };  // W, first half, second half
        auto arrive = [&](bool all_but_a_step) {
            __builtin_amdgcn_sched_barrier(0);
            if (all_but_a_step) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(PER_STEP) : "memory");
            else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_s_barrier();
            __builtin_amdgcn_sched_barrier(0);
        };
#pragma unroll
        for (int l = 0; l < PER_STEP; ++l) load_nth(k_begin, 0, l);
        if (nk > 1)
#pragma unroll
            for (int l = 0; l < PER_STEP; ++l) load_nth(k_begin + BK, 1, l);
        if constexpr (SCALED) {
            // A row's factor is its thread's: the parts of its sum of squares, written by the kernel before this one, are asked for behind the first steps,
            // thirty-two at a time, and come with them.
            if (tid < BM) {
                const int row = min(m0 + tid, M - 1);
                float sum = 0.f;
                for (int p0 = 0; p0 < ep.ss_parts; p0 += 32) {
                    float v[32];
#pragma unroll
                    for (int u = 0; u < 32; ++u) v[u] = ep.row_ss[(size_t)min(p0 + u, ep.ss_parts - 1) * M + row];
#pragma unroll
                    for (int u = 0; u < 32; ++u) sum += p0 + u < ep.ss_parts ? v[u] : 0.f;
                }
                ss_q[0][tid] = 1.0f / sqrtf(sum / (float)K + ep.ss_eps);
            }
        }
        arrive(nk > 1);
#pragma unroll
        for (int i = 0; i < TH; ++i) fetch_a(0, 0, 0, 0, i);
#pragma unroll
        for (int j = 0; j < TN; ++j) fetch_b(0, 0, j);
        constexpr int GR = TH * TN % 4 == 0 ? 4 : 2, GROUPS = TH * TN / GR;  // matrix instructions in groups, each with its share of reads and loads ahead
        static_assert(TH * TN % GR == 0, "groups of matrix instructions");
        auto step = [&](int kt, int buf) {
            const bool more = kt + 2 < nk;
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                const int np = (p + 1) & 3, nbuf = p == 3 ? buf ^ 1 : buf;  // (behind the last step: what is left there, and not used)
                const int reads = TH + (np < 2 ? TN : 0);
                if (WIDE && p == 3) {  // to the other buffer
                    const int turn = buf ? -1 : 1;
#pragma unroll
                    for (int kk = 0; kk < 2; ++kk) {
                        lane_a[kk] += turn * BM * LDS_LD;
                        lane_b[kk] += turn * BN * LDS_LD;
                    }
                }
                // phase 1: the second half's rows of this step have come; phase 3: W and the first half's rows of the next one
                if (p == 1) arrive(kt + 1 < nk);
                if (p == 3) arrive(more);
                const int first = p == 1 ? 0 : EARLY, loads = p == 1 ? EARLY : p == 3 ? PER_STEP - EARLY : 0;
#pragma unroll
                for (int g = 0; g < GROUPS; ++g) {
#pragma unroll
                    for (int r = 0; r < TH + TN; ++r) {
                        if (r >= reads || r * GROUPS / reads != g) continue;
                        if (r < TH) fetch_a(nbuf, np / 2, np & 1, np & 1, r);
                        else fetch_b(nbuf, np, r - TH);
                    }
#pragma unroll
                    for (int l = 0; l < PER_STEP; ++l)
                        if (l < loads && l * GROUPS / (loads > 0 ? loads : 1) == g && more) load_nth(k_begin + (kt + 2) * BK, buf, first + l);
#pragma unroll
                    for (int m = g * GR; m < (g + 1) * GR; ++m) mma_16x16x32(acc[p / 2 * TH + m / TN][m % TN], fa[p & 1][m / TN], fb[p & 1][m % TN]);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        };
        int kt = 0;
        if constexpr (WIDE) {  // one body for both buffers
#pragma unroll 1
            for (; kt < nk; ++kt) step(kt, kt & 1);
        } else {
            for (; kt + 1 < nk; kt += 2) {
                step(kt, 0);
                step(kt + 1, 1);
            }
            if (kt < nk) step(kt, 0);
        }
#endif
    } else if constexpr (DIRECT && STAGES > 2) {
        // A block that is alone on its CU (few tiles: one tile of rows under a weight of a few hundred column
        // tiles) has nobody to hide its loads behind, and with one step in flight every step costs a trip to
        // memory.  Here STAGES - 1 steps are in flight: the loads of step kt + STAGES - 1 go out before step
        // kt is multiplied, and the step's end waits only for the loads of step kt + 1 (a wave's loads
        // complete in order, so "all but the last (STAGES - 2) steps' loads" is a count).  The launcher
        // gives this variant whole K steps only.
        constexpr int PER_STEP = A_CHUNKS + W_CHUNKS;
        static_assert(PER_STEP * (STAGES - 2) <= 63, "the wait count is a 6-bit field");
        for (int s = 0; s < STAGES - 1; ++s)
            if (s < nk) load_direct(k_begin + s * BK, s);
        if constexpr (SCALED) {
            // The rows' sums of squares, asked for behind the first K steps and not used before the last one is
            // multiplied: what they are made of was written by the kernel before this one, a slow read that the
            // walk over K covers.  Thread (row, q) takes parts q, q + 256 / BM, ...
            ss_r = min(m0 + tid % BM, M - 1);
#pragma unroll
            for (int u = 0; u < 8; ++u) ss_v[u] = ep.row_ss[(size_t)min(tid / BM + u * (256 / BM), ep.ss_parts - 1) * M + ss_r];
        }
        // the first step's loads: the earliest of up to STAGES - 1 steps' loads
        __builtin_amdgcn_sched_barrier(0);
        if (nk >= STAGES - 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(PER_STEP * (STAGES - 2)) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        for (int kt = 0; kt < nk; ++kt) {
            const bool more = kt + STAGES - 1 < nk;
            if (more) load_direct(k_begin + (kt + STAGES - 1) * BK, (kt + STAGES - 1) % STAGES);
            multiply(kt % STAGES);
            __builtin_amdgcn_sched_barrier(0);
            // towards the end fewer steps are in flight behind step kt + 1: wait for everything
            if (more) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(PER_STEP * (STAGES - 2)) : "memory");
            else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_s_barrier();
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (SCALED) {
            constexpr int Q = 256 / BM;
            const int q = tid / BM;
            float ssum = 0.f;
#pragma unroll
            for (int u = 0; u < 8; ++u) ssum += q + u * Q < ep.ss_parts ? ss_v[u] : 0.f;
            for (int p = q + 8 * Q; p < ep.ss_parts; p += Q) ssum += ep.row_ss[(size_t)p * M + ss_r];  // more than 8 * Q parts: a very wide stream
            ss_q[q][tid % BM] = ssum;
            __syncthreads();
        }
    } else if constexpr (DIRECT) {
#ifdef MS_ELEM_HALF
        if (nk == 1 && partial) {
            load_global_tail(k_begin);
            store_lds(0);
        } else {
            load_direct(k_begin, 0);
        }
        step_barrier();
        for (int kt = 0; kt < nk; ++kt) {
            const int buf = kt & 1;
            // the next step: a whole one straight into the other buffer, a partial one into registers
            const bool tail_next = kt + 2 == nk && partial;
            if (kt + 1 < nk) {
                if (tail_next) load_global_tail(k_begin + (kt + 1) * BK);
                else load_direct(k_begin + (kt + 1) * BK, buf ^ 1);
            }
            multiply(buf);
            if (tail_next) store_lds(buf ^ 1);
            step_barrier();
        }
#endif
    } else {
        if (nk == 1 && partial) load_global_tail(k_begin);
        else load_global(k_begin);
        store_lds(0);
        __syncthreads();
        for (int kt = 0; kt < nk; ++kt) {
            const int buf = kt & 1;
            if (kt + 2 < nk || (kt + 2 == nk && !partial)) load_global(k_begin + (kt + 1) * BK);
            else if (kt + 1 < nk) load_global_tail(k_begin + (kt + 1) * BK);
            multiply(buf);
            if (kt + 1 < nk) store_lds(buf ^ 1);
            __syncthreads();
        }
    }

    // Epilogue.  Lane holds rows grp * 4 + e of column r16 in each 16x16 tile: sixteen lanes write
    // sixteen consecutive elements of a row.  (Four consecutive columns a lane - transposed tiles,
    // one 8-byte store - measured slower: neighbouring lanes then write to different rows, which
    // the memory pipeline does not merge.)  A tile wholly inside the output stores without checks:
    // sixty-four guarded stores cost a third of a whole 2,048 x 9,728 x 896 product.
    const int row_base = m0 + wm * (BM / WM) + grp * 4;
    const int col_base = n0 + wn * (BN / WN) + r16;
    const bool whole = m0 + BM <= M && n0 + BN <= N && (EPI != EPI_SWIGLU || (n0 + BN) / 2 <= ep.n_out);
    f32x4* over = nullptr;
    f32x4 last_up;
    if constexpr (SPLIT_PAIR) {  // the up tiles go over through LDS, when everybody's last fragments have been read
        static_assert(sizeof(As) >= (size_t)NT / 2 * TM * sizeof(f32x4), "room for the tiles that go over");
        over = reinterpret_cast<f32x4*>(&As[0][0]) + (size_t)(wave / 2) * TM * 64 + lane;
        __syncthreads();
        if (second)
#pragma unroll
            for (int i = 0; i < TM; ++i) over[i * 64] = acc[i][TN - 1];
        __syncthreads();
    }
    // The gate's activation in tile row i of a wave, in place; the up tiles are multiplied where the product is rounded (one instruction in half precision).
    auto activate = [&](auto act, int i) {
        float f[4] = {1.f, 1.f, 1.f, 1.f};  // SCALED: of the rows this lane holds
        if constexpr (SCALED) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int lr = wm * (BM / WM) + i * 16 + grp * 4 + e;
                if constexpr (PIPED) {
                    f[e] = ss_q[0][lr];
                    continue;
                }
                float ssum = 0.f;
#pragma unroll
                for (int qq = 0; qq < 256 / BM; ++qq) ssum += ss_q[PIPED ? 0 : qq][lr];
                f[e] = 1.0f / sqrtf(ssum / (float)K + ep.ss_eps);
            }
        }
        if constexpr (SPLIT_PAIR) {
            __builtin_amdgcn_sched_barrier(0);
            if (!second) last_up = over[i * 64];
        }
#pragma unroll
        for (int j = 0; j < TN; j += 2) {
            if (SPLIT_PAIR && j == TN - 1 && second) continue;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if constexpr (SCALED) {
                    acc[i][j][e] *= f[e];
                    if (SPLIT_PAIR && j == TN - 1) last_up[e] *= f[e];
                    else acc[i][min(j + 1, TN - 1)][e] *= f[e];
                }
                acc[i][j][e] = gate_activation(acc[i][j][e], act);
            }
        }
    };
    // Activations before the stores and for the one that the product has: their code is there once, not once a kind of store.  As a select an element, behind both
    // formulas, five of an element's twelve vector instructions were for the one that is not taken.  us from a tile's last step to its last store, before and now: 256x320
    // 6.3 and 5.4, 256x256 4.3 and 3.3, 256x192 3.2 and 2.6.  (The widest tiles have no registers for sums that come from either formula: there the stores are there twice.)
    if constexpr (EPI == EPI_SWIGLU && !WIDE) {
        with_gate_activation(ep.act, [&](auto act) {
#pragma unroll
            for (int i = 0; i < TM; ++i) activate(act, i);
        });
    } else if constexpr (EPI == EPI_ACT) {
        with_unary_activation(ep.act, [&](auto act) {
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    const float b = ep.bias ? ep.bias[min(col_base + j * 16, N - 1)] : 0.f;
#pragma unroll
                    for (int e = 0; e < 4; ++e) acc[i][j][e] = unary_activation(acc[i][j][e] + b, act);
                }
        });
    }
    // A tile at the lower edge of an output whose rows come in whole groups of sixteen (a decode step
    // of 48 requests in a 64-row tile) skips the groups beyond the last row and stores the others
    // without checks as well.
    auto emit = [&](auto checked, auto row_groups, auto act) {
        constexpr bool CHECKED = decltype(checked)::value, ROW_GROUPS = decltype(row_groups)::value;
        if constexpr (EPI == EPI_SWIGLU) {
            elem_t* out = reinterpret_cast<elem_t*>(ep.out);
#pragma unroll
            for (int i = 0; i < TM; ++i) {
                if (ROW_GROUPS && m0 + wm * (BM / WM) + i * 16 >= M) continue;
                if constexpr (WIDE) activate(act, i);
#pragma unroll
                for (int j = 0; j < TN; j += 2) {
                    if (SPLIT_PAIR && j == TN - 1 && second) continue;
                    const int col = (n0 + tile_col(j)) / 2 + r16;  // tiles 2t, 2t+1 -> output tile t
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const int row = row_base + i * 16 + e;
                        if (CHECKED && !(row < M && col < ep.n_out)) continue;
                        out[(size_t)row * ep.ldo + col] = from_f32<elem_t>(acc[i][j][e] * (SPLIT_PAIR && j == TN - 1 ? last_up[e] : acc[i][min(j + 1, TN - 1)][e]));
                    }
                }
            }
        } else if constexpr (EPI == EPI_QKV_ROPE) {
            // The tile's columns are one head (the launcher sees to it), and a wave holds all of them: lane (r16, grp)
            // has columns r16 + 16 j of rows grp * 4 + e, so both elements of a pair (j, j + TN / 2) are its own.
            static_assert(WN == 1 && TN % 2 == 0, "a wave holds whole heads");
            constexpr int HT = TN / 2, hd = BN, half = BN / 2;
            const int head = n0 / hd;
            const int kind = head < ep.H ? 0 : (head < ep.H + ep.KV ? 1 : 2);  // query, key or value head
            float bias_j[TN];
#pragma unroll
            for (int j = 0; j < TN; ++j) bias_j[j] = ep.bias ? ep.bias[n0 + j * 16 + r16] : 0.f;
#pragma unroll
            for (int i = 0; i < TM; ++i) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int row = row_base + i * 16 + e;
                    if (row >= M) continue;
                    float x[TN];
#pragma unroll
                    for (int j = 0; j < TN; ++j) x[j] = bias_j[j] + acc[i][j][e];
                    if (kind < 2) {
                        const float* cs = ep.rope_cs + (size_t)row * (2 * half);
#pragma unroll
                        for (int j = 0; j < HT; ++j) {
                            const float c = cs[2 * (j * 16 + r16)], sn = cs[2 * (j * 16 + r16) + 1];
                            const float x0 = x[j], x1 = x[j + HT];
                            x[j] = x0 * c - x1 * sn;
                            x[j + HT] = x0 * sn + x1 * c;
                        }
                    }
                    if (kind == 0) {
                        elem_t* o = reinterpret_cast<elem_t*>(ep.out) + ((size_t)row * ep.H + head) * hd + r16;
#pragma unroll
                        for (int j = 0; j < TN; ++j) o[j * 16] = from_f32<elem_t>(x[j]);
                    } else {
                        const int slot = ep.slot_map[row];
                        if (slot < 0) continue;
                        const int page = slot / ep.ps, off = slot - page * ep.ps;
                        if (kind == 1) {
                            elem_t* o = ep.kpool + (((size_t)page * ep.KV + (head - ep.H)) * ep.ps + off) * hd + r16;
#pragma unroll
                            for (int j = 0; j < TN; ++j) o[j * 16] = from_f32<elem_t>(x[j]);
                        } else {
                            elem_t* o = ep.vpool + (((size_t)page * ep.KV + (head - ep.H - ep.KV)) * hd + r16) * ep.ps + off;
#pragma unroll
                            for (int j = 0; j < TN; ++j) o[(size_t)(j * 16) * ep.ps] = cache_value(x[j]);
                        }
                    }
                }
            }
        } else {
            // RESIDUAL: what the stream holds is asked for a group of sixteen rows ahead of its stores.  Added to in place, every load stood behind the
            // stores before it, which may write the same address: 14.7 of 65 us in 256x128 tiles of 2,048 x 3,584 x 3,584.  Cold operands, before and
            // now: that product 69.6 -> 59.9 us, 2,048 x 1,536 x 1,536 (128x128) 24.2 -> 20.3, 2,048 x 896 x 896 (64x64) 10.0 -> 8.7.
            constexpr bool ADDS = EPI == EPI_RESIDUAL || EPI == EPI_PRENORM;
            constexpr int AHEAD = ADDS ? 2 : 1;
            float prior[AHEAD][ADDS ? TN : 1][4], nw[EPI == EPI_PRENORM ? TN : 1];
            if constexpr (EPI == EPI_PRENORM)
#pragma unroll
                for (int j = 0; j < TN; ++j) nw[j] = ep.norm_w[min(col_base + j * 16, N - 1)];
            auto ask = [&](int i) {
#pragma unroll
                for (int j = 0; j < TN; ++j)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const int row = row_base + i * 16 + e, col = col_base + j * 16;
                        prior[i % AHEAD][j][e] = reinterpret_cast<const float*>(ep.out)[(size_t)(CHECKED || ROW_GROUPS ? min(row, M - 1) : row) * ep.ldo + (CHECKED ? min(col, N - 1) : col)];
                    }
            };
            if constexpr (ADDS) ask(0);
#pragma unroll
            for (int i = 0; i < TM; ++i) {
                if constexpr (ADDS) {
                    if (i + 1 < TM) ask(i + 1);
                    __builtin_amdgcn_sched_barrier(0);
                }
                if (ROW_GROUPS && m0 + wm * (BM / WM) + i * 16 >= M) continue;
                float ss[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    const int col = col_base + j * 16;
                    const float b = EPI != EPI_ACT && ep.bias ? ep.bias[min(col, N - 1)] : 0.f;
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const int row = row_base + i * 16 + e;
                        if (CHECKED && !(row < M && col < N)) continue;
                        const size_t o = (size_t)row * ep.ldo + col;
                        const float v = acc[i][j][e] + b;
                        if constexpr (EPI == EPI_STORE_F32) reinterpret_cast<float*>(ep.out)[split * ep.split_stride + o] = v;
                        else if constexpr (EPI == EPI_STORE_ELEM) reinterpret_cast<elem_t*>(ep.out)[o] = from_f32<elem_t>(v);
                        else if constexpr (EPI == EPI_ACT) reinterpret_cast<elem_t*>(ep.out)[o] = from_f32<elem_t>(v);
                        else reinterpret_cast<float*>(ep.out)[o] = prior[i % AHEAD][j][e] + v;  // residual stream, 32-bit
                        if constexpr (EPI == EPI_PRENORM) {
                            const float x = prior[i % AHEAD][j][e] + v;
                            ep.hn[o] = from_f32<elem_t>(x * nw[j]);
                            ss[e] = fmaf(x, x, ss[e]);
                        }
                    }
                }
                if constexpr (EPI == EPI_PRENORM) {  // the sixteen lanes of a row, each of which then has the sum of one row of four to store
#pragma unroll
                    for (int e = 0; e < 4; ++e)
#pragma unroll
                        for (int o = 1; o < 16; o <<= 1) ss[e] += __shfl_xor(ss[e], o, WAVE);
                    const int row = row_base + i * 16 + r16;  // (of lanes 0 to 3 of the sixteen)
                    if (r16 < 4 && row < M && n0 + wn * (BN / WN) < N)  // (a wave behind the last column has no share)
                        ep.ss_part[(size_t)((n0 + wn * (BN / WN)) / (BN / WN)) * M + row] = r16 == 0 ? ss[0] : r16 == 1 ? ss[1] : r16 == 2 ? ss[2] : ss[3];
                }
            }
        }
    };
    if constexpr (EPI == EPI_EXPERT_GATED || EPI == EPI_EXPERT_PLAIN || EPI == EPI_EXPERT_DOWN) {
        // Half of the tiles are the last of an expert's rows: groups of sixteen that exist store without checks, those that do not are skipped.
        // up: the activations of the rows that chose the expert; down: their sums, each row's in its plane.
        constexpr int STEP = EPI == EPI_EXPERT_GATED ? 2 : 1;
        static_assert(TN % STEP == 0, "gate and up tiles come in pairs");
        using Out = std::conditional_t<EPI == EPI_EXPERT_DOWN, float, elem_t>;
        auto emit_group = [&](auto checked, int i) {
            constexpr bool CHECKED = decltype(checked)::value;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int row = row_base + i * 16 + e;
                if (CHECKED && row >= M) continue;
                Out* o = reinterpret_cast<Out*>(ep.out) + rows.out_row(row, m0) * ep.ldo;
#pragma unroll
                for (int j = 0; j < TN; j += STEP) {
                    const int col = STEP == 2 ? (col_base + j * 16 - r16) / 2 + r16 : col_base + j * 16;
                    if (CHECKED && col >= ep.n_out) continue;
                    o[col] = from_f32<Out>(acc[i][j][e]);
                }
            }
        };
        if constexpr (EPI != EPI_EXPERT_DOWN)  // in place, before the stores: the code of each activation is there once
            rows.with_activation([&](auto act) {
#pragma unroll
                for (int i = 0; i < TM; ++i) {
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float w = rows.weight(row_base + i * 16 + e, m0);
#pragma unroll
                        for (int j = 0; j < TN; j += STEP)
                            acc[i][j][e] = STEP == 2 ? rows.gated(act, acc[i][j][e], acc[i][j + STEP - 1][e], w) : rows.plain(act, acc[i][j][e], w);
                    }
                }
            });
        const int lower = m0 + wm * (BM / WM);
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            if (lower + i * 16 >= M) break;
            if (lower + i * 16 + 16 <= M && n0 + BN <= N) emit_group(std::false_type{}, i);
            else emit_group(std::true_type{}, i);
        }
        return;
    }
    const bool cols_whole = n0 + BN <= N && (EPI != EPI_SWIGLU || (n0 + BN) / 2 <= ep.n_out);
    auto finish = [&](auto act) {
        if (whole) emit(std::false_type{}, std::false_type{}, act);
        else if (cols_whole && M % 16 == 0) emit(std::false_type{}, std::true_type{}, act);
        else emit(std::true_type{}, std::false_type{}, act);
    };
    if constexpr (EPI == EPI_SWIGLU && WIDE) with_gate_activation(ep.act, finish);
    else finish(std::integral_constant<int, ACT_SILU>{});  // (not looked at)
}


}  // namespace ms
