// One block of out[M, N] = A[M, K] * W[N, K]^T for few rows (a decode step), two-byte elements, whole K steps of 64: the weight is read once
// and nothing of it is reused, so the block's waves share out K and not the columns.  Wave w of KW takes the steps w, w + KW, ... of 16 NT
// columns and 16 MT rows, through a ring of its own in LDS that loads straight from memory fill (global_load_lds_dwordx4: eight
// lanes bring 128 contiguous bytes of a row, swizzled as in gemm_tile.cuh): there is no barrier before the waves' sums are added, in
// wave order, and a wave waits for its own oldest step only.  How K falls to the waves depends on KW and the slice alone.  The slices are those of 16 rows
// up to 32 (plan_few), and up to 16 rows every product comes here, so that a row's sums do not depend on what else is in such a step; between 17 and 64
// rows it goes by their number whether a product comes here or goes in tiles, above 32 in how many slices.
//
// What bounds it: the weight's bytes (5 TB/s) behind 2.3 us of launch, first trip and end, and the rows, which every block reads again.  The kernel that
// this replaces for large weights shares 64 rows and 64 columns out over its waves, with a barrier a step of 0.36 us, so a wide output
// under a short K was few blocks of many steps; the one for small weights (skinny.hip) reads both operands as fragments, 16 rows by 64 bytes
// a load, which the CU's load path takes a quarter as fast as whole lines.  us at 8 rows, cold weights, few-rows / tiled / here: 5,632 x 2,048 with an
// activation 11.8 / 13.1 / 7.5; 11,264 x 2,048 gated 22.4 / 14.1 / 12.4; 9,728 x 896 gated 9.1 / 7.4 / 6.3; 37,888 x 3,584 gated 72 / 62 / 52;
// 2,048 x 5,632 in slices 11.3 / 8.4 / 6.9; 896 x 4,864 in slices 5.5 / 6.5 / 4.2; 151,936 x 896 69 / 60 / 54.
//
// `past`: the weight's loads are non-temporal ones, which leave nothing in the memory-side cache of 256 MB.  What comes from memory comes a tenth faster so, as the
// loads alone, cold, us without and with: 37,888 x 3,584 49.9 and 44.8 (6.1 TB/s), 3,584 x 18,944 in four slices 23.8 and 21.3, 152,064 x 896 44.6 and 40.4, 9,728 x 896
// 5.2 and 4.8; and weights that are read through the cache stay in it, if they fit.  A weight that would still be there from the step before is read slower so (11,264 x 2,048:
// 8.2 and 9.4), so the weights are marked by what all of a model's come to (engine/loading.py).  Sixteen requests of the 7B sizes, 16 steps and their prompts, 70.0 -> 65.7 ms;
// one of the 0.5B sizes 11.78 -> 10.98.
//
// In 32-bit a step is 32 numbers of K (rows of 128 bytes again), up to 32 rows; the fragments of skinny.hip, which it replaces
// there, are 64 bytes a row and load, and stream at half the rate.  us, skinny.hip and here, cold weights, 1 and 32 rows: 9,728 x 896 gated 13.0 and 9.1,
// 22.8 and 13.5; 896 x 4,864 in slices 7.3 and 5.9, 13.9 and 7.3; 11,264 x 2,048 gated 26.5 and 18.4, 47 and 27.6; 2,048 x 5,632 in slices 23.8 and 10.9, 24.9 and 13.5.
// Over 385 products of 1 to 32 rows, 96 to 40,000 columns and K of 256 to 16,384 1.45 times as fast (geometric mean); decode steps of the further designs' small sizes 1.13 to
// 1.35 times, of 24 requests of the 0.5B sizes 1.42.  Errors against 64 bits are the same (a pass of three requests 2.1e-6 and 2.0e-6).
#pragma once
#include "gemm_tile.cuh"

namespace ms {

constexpr int FEW_STEP = 128 / (int)sizeof(elem_t);  // numbers of K a step

// What a block that norms its one row itself (NORMED) keeps in dynamic LDS: the pending sums, the stream's row and the norm's weight as they come, whole kilobytes each, and the normed row.
static inline size_t few_normed_lds(int K, int n_pending) {
    auto whole = [](size_t floats) { return (floats * 4 + 1023) / 1024 * 1024; };
    return whole((size_t)n_pending * K) + 2 * whole(K) + (size_t)K * sizeof(elem_t);
}

template <int MT, int NT, int KW, int STAGES, int EPI, bool SCALED, class Rows, bool NORMED = false>
__device__ __forceinline__ void few_rows_tile(const elem_t* __restrict__ A, const elem_t* __restrict__ W, int M, int N, int K, const EpiArgs& ep, int m0,
                                              int n0, int split, const Rows& rows) {
    constexpr int RING = NT + (NORMED ? 0 : MT);  // tiles of sixteen rows in a ring
    constexpr int STEP = RING * 2048, PER_STEP = 2 * RING;  // bytes and loads of a step: rows of 128 bytes, eight a load
    constexpr int PAIR = EPI == EPI_SWIGLU || EPI == EPI_EXPERT_GATED ? 2 : 1;
    static_assert(NT % PAIR == 0, "gate and up tiles come in pairs");
    static_assert(PER_STEP * (STAGES - 1) <= 63, "the wait count is a 6-bit field");
    static_assert(STAGES >= 2 && STAGES <= 4, "one to three steps in flight behind the one that is waited for");
    static_assert(STAGES * STEP >= MT * NT * 1024, "the waves' sums lie where their rings were");
    __shared__ __attribute__((aligned(16))) char ring[KW][STAGES * STEP];
    __shared__ float ss_q[SCALED ? KW : 1][SCALED ? 16 * MT : 1];
    static_assert(!NORMED || (MT == 1 && EPI == EPI_STORE_F32 && !SCALED && !Rows::GATHERS), "a block that norms its row: one row, sums");
    extern __shared__ __attribute__((aligned(16))) char normed[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r16 = lane & 15, grp = lane >> 4;
    const int k_begin = split * ep.k_per_split, nk = (min(K, k_begin + ep.k_per_split) - k_begin) / FEW_STEP;
    const int mine = (nk - wave + KW - 1) / KW;  // steps of this wave

    // lane l of a load: row l / 8 of its eight, the chunk that the swizzle puts at place l % 8
    const int chunk = (lane & 7) ^ (lane >> 3);
    const elem_t* base_w = W + (size_t)n0 * rows.w_pitch(K) + k_begin + wave * FEW_STEP;
    const elem_t* base_a = A + (Rows::GATHERS ? (size_t)0 : (size_t)rows.source(m0) * rows.pitch(K)) + k_begin + wave * FEW_STEP;
    uint32_t ow[2 * NT], oa[2 * MT];
    const elem_t* ga[Rows::GATHERS ? 2 * MT : 1];
#pragma unroll
    for (int l = 0; l < 2 * NT; ++l)
        ow[l] = ((uint32_t)(min(n0 + l * 8 + (lane >> 3), N - 1) - n0) * (uint32_t)rows.w_pitch(K) + chunk * EPC) * (uint32_t)sizeof(elem_t);
#pragma unroll
    for (int l = 0; l < 2 * MT; ++l) {
        const int m = min(m0 + l * 8 + (lane >> 3), M - 1);
        if constexpr (Rows::GATHERS) ga[l] = base_a + (size_t)rows.source(m) * rows.pitch(K) + chunk * EPC;
        else oa[l] = ((uint32_t)(m - m0) * (uint32_t)rows.pitch(K) + chunk * EPC) * (uint32_t)sizeof(elem_t);
    }
    const uint32_t own = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)&ring[0][0] + wave * (STAGES * STEP);
    auto ask = [&](int i, int stage) {  // this wave's step i
        const size_t k = (size_t)i * (FEW_STEP * KW);
        const uint32_t to = own + stage * STEP;
        if (ep.past) {
#pragma unroll
            for (int l = 0; l < 2 * NT; ++l)
                asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1 nt" ::"v"(ow[l]), "s"(base_w + k), "s"(to + l * 1024) : "memory", "m0");
        } else {
#pragma unroll
            for (int l = 0; l < 2 * NT; ++l)
                asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(ow[l]), "s"(base_w + k), "s"(to + l * 1024) : "memory", "m0");
        }
#pragma unroll
        for (int l = 0; l < (NORMED ? 0 : 2 * MT); ++l) {
            if constexpr (Rows::GATHERS)
                asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(ga[l] + k), "s"(to + (2 * NT + l) * 1024) : "memory", "m0");
            else
                asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(oa[l]), "s"(base_a + k), "s"(to + (2 * NT + l) * 1024) : "memory", "m0");
        }
    };
    f32x4 acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};

    // NORMED: the row's sources are asked for ahead of the first steps, a kilobyte a load, shared out over the waves
    const int row4 = K / 4, row_kb = (K + 255) / 256 * 256;
    float* const src_p = reinterpret_cast<float*>(normed);
    float* const src_x = src_p + (ep.n_pending * K + 255) / 256 * 256;
    float* const src_w = src_x + row_kb;
    elem_t* const row_n = reinterpret_cast<elem_t*>(src_w + row_kb);
    if constexpr (NORMED) {
        auto bring = [&](const float* from, int quads, const float* to) {
            const uint32_t at = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const char*)to;
            for (int c = wave; c * 64 < quads; c += KW)
                asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"((uint32_t)min(c * 64 + lane, quads - 1) * 16u), "s"(from),
                             "s"(__builtin_amdgcn_readfirstlane(at + c * 1024)) : "memory", "m0");
        };
        bring(ep.pending, ep.n_pending * row4, src_p);
        bring(ep.stream, row4, src_x);
        bring(ep.norm_w, row4, src_w);
    }
#pragma unroll
    for (int s = 0; s < STAGES - 1; ++s)
        if (s < mine) ask(s, s);
    if constexpr (NORMED) {
        // As the norm's kernel does it, with its numbers: a thread's fours of the row, the sums added in order, squares over the waves in order.
        auto together = [&] {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
        };
        __shared__ float squares[KW];
        static_assert(KW == 4, "256 threads, as the norm's kernel has");
        __builtin_amdgcn_sched_barrier(0);
        if (mine >= STAGES - 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(PER_STEP * (STAGES - 1)) : "memory");  // all but the weight's
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        together();
        const bool writes = blockIdx.x == 0 && blockIdx.y == 0;
        float ss = 0.f;
        for (int c = threadIdx.x; c < row4; c += 256) {
            f32x4* x = reinterpret_cast<f32x4*>(src_x) + c;
            f32x4 v = *x;
            for (int p = 0; p < ep.n_pending; ++p) v += reinterpret_cast<const f32x4*>(src_p)[p * row4 + c];
            *x = v;
            if (writes) reinterpret_cast<f32x4*>(ep.stream_out)[c] = v;
            ss += v.x * v.x + v.y * v.y + v.z * v.z + v.w * v.w;
        }
        ss = wave_sum(ss);
        if (lane == 0) squares[wave] = ss;
        together();
        ss = 0.f;
#pragma unroll
        for (int w = 0; w < KW; ++w) ss += squares[w];
        const float inv = 1.0f / sqrtf(ss / (float)K + ep.ss_eps);
        for (int c = threadIdx.x; c < row4; c += 256) {
            // (with a zero added, as there: one rounding to half precision)
            const f32x4 o = reinterpret_cast<const f32x4*>(src_x)[c] * reinterpret_cast<const f32x4*>(src_w)[c] * inv + (f32x4){0.f, 0.f, 0.f, 0.f};
            typedef elem_t four_t __attribute__((ext_vector_type(4)));
            reinterpret_cast<four_t*>(row_n)[c] = (four_t){from_f32<elem_t>(o.x), from_f32<elem_t>(o.y), from_f32<elem_t>(o.z), from_f32<elem_t>(o.w)};
        }
        together();
    }
    // SCALED: the rows' sums of squares come in parts, shared out over the waves and their four groups of lanes; the first EARLY of each are asked
    // for here, behind the first steps
    constexpr int SHARES = 4 * KW, EARLY = 4;
    float ss_early[SCALED ? MT : 1][EARLY];
    if constexpr (SCALED) {
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int u = 0; u < EARLY; ++u)
                ss_early[i][u] = ep.row_ss[(size_t)min(wave * 4 + grp + u * SHARES, ep.ss_parts - 1) * M + min(m0 + i * 16 + r16, M - 1)];
    }
    // PRENORM: the stream's values and the norm's weights of the tile that this wave will finish, asked for with everything else
    static_assert(EPI != EPI_PRENORM || (MT == 1 && NT <= KW), "the form that prepares the norm: one tile a wave");
    float prior[4], nw = 0.f;
    if constexpr (EPI == EPI_PRENORM) {
        const int col = min(n0 + wave * 16 + r16, N - 1);
        nw = ep.norm_w[col];
#pragma unroll
        for (int e = 0; e < 4; ++e) prior[e] = reinterpret_cast<const float*>(ep.out)[(size_t)min(m0 + grp * 4 + e, M - 1) * ep.ldo + col];
    }
    auto wait_for = [&](int behind) {  // every step's loads but those of the last `behind`
        __builtin_amdgcn_sched_barrier(0);
        if (behind >= STAGES - 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(PER_STEP * (STAGES - 1)) : "memory");
        else if (STAGES > 3 && behind == 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(PER_STEP * 2) : "memory");
        else if (STAGES > 2 && behind == 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(PER_STEP) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    for (int i = 0, stage = 0; i < mine; ++i) {
        const int last = stage == 0 ? STAGES - 1 : stage - 1;  // where the step before this one was
        if (i + STAGES - 1 < mine) ask(i + STAGES - 1, last);
        wait_for(min(mine - 1 - i, STAGES - 1));
        const elem_t* t = reinterpret_cast<const elem_t*>(&ring[wave][stage * STEP]);
        constexpr int CHUNKS = FEW_STEP / 32;  // of 32 numbers
        auto fragment = [&](int row, int kk) {
#ifdef MS_ELEM_HALF
            return frag_load(t + row * FEW_STEP + ((kk * 4 + grp) ^ (r16 & 7)) * EPC);
#else
            Frag f;
            const f32x4 x = *reinterpret_cast<const f32x4*>(t + row * FEW_STEP + ((2 * grp) ^ (r16 & 7)) * EPC);
            const f32x4 y = *reinterpret_cast<const f32x4*>(t + row * FEW_STEP + ((2 * grp + 1) ^ (r16 & 7)) * EPC);
#pragma unroll
            for (int e = 0; e < 4; ++e) { f.v[e] = x[e]; f.v[4 + e] = y[e]; }
            return f;
#endif
        };
        Frag fa[CHUNKS][MT], fw[CHUNKS][NT];
#pragma unroll
        for (int kk = 0; kk < CHUNKS; ++kk) {
#pragma unroll
            for (int j = 0; j < NT; ++j) fw[kk][j] = fragment(j * 16 + r16, kk);
#pragma unroll
            for (int j = 0; j < MT; ++j)
                fa[kk][j] = NORMED ? frag_load(row_n + k_begin + (wave + i * KW) * FEW_STEP + kk * 32 + grp * 8) : fragment(NT * 16 + j * 16 + r16, kk);
        }
#pragma unroll
        for (int kk = 0; kk < CHUNKS; ++kk)
#pragma unroll
            for (int m = 0; m < MT; ++m)
#pragma unroll
                for (int j = 0; j < NT; ++j) mma_16x16x32(acc[m][j], fa[kk][m], fw[kk][j]);
        __builtin_amdgcn_sched_barrier(0);  // the fragments are in registers before their place is written again
        stage = stage == STAGES - 1 ? 0 : stage + 1;
    }
    if constexpr (SCALED) {
#pragma unroll
        for (int i = 0; i < MT; ++i) {
            const int share = wave * 4 + grp, row = min(m0 + i * 16 + r16, M - 1);
            float sq = 0.f;
#pragma unroll
            for (int u = 0; u < EARLY; ++u) sq += share + u * SHARES < ep.ss_parts ? ss_early[i][u] : 0.f;
            for (int p = share + EARLY * SHARES; p < ep.ss_parts; p += SHARES) sq += ep.row_ss[(size_t)p * M + row];  // a very wide stream
            sq += __shfl_xor(sq, 16, WAVE);
            sq += __shfl_xor(sq, 32, WAVE);
            if (grp == 0) ss_q[wave][i * 16 + r16] = sq;
        }
    }
    // The waves' sums go to LDS where the wave's own ring was (it has read all of it); then the tiles are dealt to the waves, which add them up in
    // wave order and store.
    {
        float* to = reinterpret_cast<float*>(&ring[wave][0]) + lane;
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e) to[((i * NT + j) * 4 + e) * 64] = acc[i][j][e];
    }
    __syncthreads();
    constexpr int ACROSS = NT / PAIR, UNITS = MT * ACROSS;
#pragma unroll
    for (int u0 = 0; u0 < UNITS; u0 += KW) {
        const int u = u0 + wave;
        if (UNITS % KW != 0 && u >= UNITS) break;
        const int i = u / ACROSS, j = u % ACROSS * PAIR;
        if (m0 + i * 16 >= M || n0 + j * 16 >= N) continue;  // the same for the whole wave; beyond the last column there is no share of ss_part either
        float v[PAIR][4];
#pragma unroll
        for (int p = 0; p < PAIR; ++p)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int at = ((i * NT + j + p) * 4 + e) * 64 + lane;
                float sum = reinterpret_cast<const float*>(&ring[0][0])[at];
#pragma unroll
                for (int w = 1; w < KW; ++w) sum += reinterpret_cast<const float*>(&ring[w][0])[at];
                v[p][e] = sum;
            }
        const int row0 = m0 + i * 16 + grp * 4, col = PAIR == 2 ? (n0 + j * 16) / 2 + r16 : n0 + j * 16 + r16;
        if constexpr (EPI == EPI_PRENORM) {
            float ss[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const bool on = col < N && row0 + e < M;
                const float x = prior[e] + v[0][e];
                if (on) {
                    reinterpret_cast<float*>(ep.out)[(size_t)(row0 + e) * ep.ldo + col] = x;
                    ep.hn[(size_t)(row0 + e) * ep.ldo + col] = from_f32<elem_t>(x * nw);
                }
                ss[e] = on ? x * x : 0.f;
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) {
#pragma unroll
                for (int o = 1; o < 16; o <<= 1) ss[e] += __shfl_xor(ss[e], o, WAVE);
                if (r16 == 0 && row0 + e < M) ep.ss_part[(size_t)(n0 / 16 + j) * M + row0 + e] = ss[e];
            }
            continue;
        }
        if (col >= (PAIR == 2 || EPI == EPI_EXPERT_DOWN || EPI == EPI_EXPERT_PLAIN ? ep.n_out : N)) continue;
        const float b = PAIR == 1 && EPI != EPI_EXPERT_DOWN && EPI != EPI_EXPERT_PLAIN && ep.bias ? ep.bias[col] : 0.f;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int row = row0 + e;
            if (row >= M) continue;
            if constexpr (EPI == EPI_SWIGLU) {
                float gv = v[0][e], uv = v[1][e];
                if constexpr (SCALED) {
                    float sq = 0.f;
#pragma unroll
                    for (int w = 0; w < KW; ++w) sq += ss_q[w][row - m0];
                    const float f = 1.0f / sqrtf(sq / (float)K + ep.ss_eps);
                    gv *= f;
                    uv *= f;
                }
                reinterpret_cast<elem_t*>(ep.out)[(size_t)row * ep.ldo + col] = from_f32<elem_t>(gate_activation(gv, ep.act) * uv);
            } else if constexpr (EPI == EPI_EXPERT_GATED || EPI == EPI_EXPERT_PLAIN || EPI == EPI_EXPERT_DOWN) {
                using Out = std::conditional_t<EPI == EPI_EXPERT_DOWN, float, elem_t>;
                float s = v[0][e];
                if constexpr (EPI != EPI_EXPERT_DOWN) {
                    const float w = rows.weight(row, m0);
                    rows.with_activation([&](auto act) { s = PAIR == 2 ? rows.gated(act, v[0][e], v[PAIR - 1][e], w) : rows.plain(act, v[0][e], w); });
                }
                reinterpret_cast<Out*>(ep.out)[rows.out_row(row, m0) * ep.ldo + col] = from_f32<Out>(s);
            } else {
                const size_t o = (size_t)row * ep.ldo + col;
                const float s = v[0][e] + b;
                if constexpr (EPI == EPI_STORE_F32) reinterpret_cast<float*>(ep.out)[split * ep.split_stride + o] = s;
                else if constexpr (EPI == EPI_STORE_ELEM) reinterpret_cast<elem_t*>(ep.out)[o] = from_f32<elem_t>(s);
                else if constexpr (EPI == EPI_ACT) reinterpret_cast<elem_t*>(ep.out)[o] = from_f32<elem_t>(unary_activation(s, ep.act));
                else reinterpret_cast<float*>(ep.out)[o] += s;  // residual stream, 32-bit
            }
        }
    }
}

}  // namespace ms
