// A feed-forward of many small experts of which a token uses a few: the router, and the experts' activation.
//
// The router's logits are 32-bit sums of 32-bit weights times the rows as the feed-forward's products read them (in the
// element type, which the 32-bit build does not round); a row's `top` largest logits choose its experts (the lower
// index wins a tie), and their weights are the softmax over the chosen logits alone.  The experts' up projections are one
// matrix [experts * ff (+ shared), width] and their down projections one matrix [width, experts * ff (+ shared)], so the
// weighted sum of the chosen experts' outputs is ONE product over activations in which an expert's columns are
// act(up) * (the row's weight for that expert), zero for an expert the row did not choose, and the columns of an
// expert that every row uses (beyond experts * ff) carry weight one.  Nothing here depends on what else is in the step.
//
// A second way to score (`softmax_all`): the scores are the softmax over every router output, the choice is by score plus
// a correction per output, and the weights are the chosen scores over their sum (+ 1e-20).  Gated experts
// act(gate) * up: the gates of all experts are the first half of the up product's columns.  Router outputs beyond the
// experts stand for experts that return their input: `add_scaled_rows` adds the input's rows with those weights.
//
// A third way (`sigmoid`): the weights are the sigmoids of the chosen logits as they are.  Rows of the router's matrix
// beyond the outputs to choose from (`extra`) are gates that every row has, the sigmoids of their own logits, left behind
// the experts' weights; the first of them can stand for the expert that every row uses.  A weight may also multiply a gated
// expert's input instead of its output: act(w gate) * (w up).
#include "few_rows.cuh"
#include "gemm_plan.h"

namespace ms {

constexpr int MAX_EXPERTS = 1024;
enum Scoring { SOFTMAX_CHOSEN = 0, SOFTMAX_ALL = 1, SIGMOID = 2 };

// What the router leaves for the products over the chosen rows alone: plane[t, e] numbers the experts that row t uses (chosen, with a
// weight that is not zero) in ascending order, -1 for the others; sums [top, T, width] will hold the k-th of them's output in plane k, and
// the rows of planes that row t does not use are zeroed here.
struct RouteSums {
    int* plane;   // [T, real], or null: not asked for
    float* sums;
    int real, width, T;
};

// gates[t, e] = the row's weight for expert e, 0 where it was not chosen.  A block takes R rows, a wave EW outputs at a time, whose weights it asks
// for together, V columns a lane; a logit is the sum of a lane's columns, then of the lanes, whatever R and EW.  The choice and all that follows are a wave's a row.
// An output at a time was a trip to memory for every fourth, and with one row a block every row brought the weights from the L2 again
// (us, warm: four rows of 2,048 over 9 outputs 7.1 -> 5.1, 2,048 rows 14.7 -> 8.5; 64 rows over 64 outputs 25.2 -> 17.6, 2,048 72.8 -> 33.2).
template <int R, int V, int EW, int AHEAD>
__global__ __launch_bounds__(256) void route_kernel(const elem_t* __restrict__ x, const float* __restrict__ w,
                                                    const float* __restrict__ bias, float* __restrict__ gates, int d, int E, int top,
                                                    int scoring, const float* __restrict__ correction, int extra, RouteSums rs) {
    static_assert(R == 1 || R == 4, "sums over the lanes of four rows at a time; a wave a row");
    const bool softmax_all = scoring == SOFTMAX_ALL;
    __shared__ float zs[R][MAX_EXPERTS];
    __shared__ float scores[R][MAX_EXPERTS];  // SOFTMAX_ALL: the outputs' scores; else `extra` logits
    __shared__ float chosen_zs[R][64];
    __shared__ int chosen_es[R][64];
    __shared__ int used_planes[R];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, t0 = blockIdx.x * R, outputs = E + extra;
    for (int e0 = wave; e0 < outputs; e0 += 4 * EW) {
        float v[EW][R];
#pragma unroll
        for (int k = 0; k < EW; ++k)
#pragma unroll
            for (int r = 0; r < R; ++r) v[k][r] = 0.f;
        if constexpr (AHEAD > 1) {
            // The loads of AHEAD steps on one straight path (beyond the row its end, not added).  Left to the compiler, the loop below asks for a step or two at a time: us,
            // warm, the same sums, that loop and here: four rows of 2,048 over 9 outputs 5.0 and 4.7, 64 rows over 64 outputs 15.9 and 13.3, 2,048 rows 8.0 and 7.7, 30.2 and
            // 25.6.  (With that loop behind this one, for the steps that fill no round, four rows of 2,048 over 4 outputs 4.4 for 3.7: the code is twice as long.
            // The loads are written out in both: through a function that both call they took 4 to 15 % longer.)
            for (int c0 = lane * V; c0 < d; c0 += 64 * V * AHEAD) {
                float we[AHEAD][EW][V], xr[AHEAD][R][V];
#pragma unroll
                for (int u = 0; u < AHEAD; ++u) {
                    const int c = min(c0 + u * 64 * V, d - V);
#pragma unroll
                    for (int k = 0; k < EW; ++k) {
                        const float* from = w + (size_t)min(e0 + 4 * k, outputs - 1) * d + c;
                        if constexpr (V == 4) {
                            const float4 four = *reinterpret_cast<const float4*>(from);
                            we[u][k][0] = four.x, we[u][k][1] = four.y, we[u][k][2] = four.z, we[u][k][3] = four.w;
                        } else {
                            we[u][k][0] = from[0];
                        }
                    }
#pragma unroll
                    for (int r = 0; r < R; ++r) {
                        const elem_t* row = x + (size_t)min(t0 + r, rs.T - 1) * d + c;
                        if constexpr (V == 4 && sizeof(elem_t) == 2) {
                            const u32x2 raw = *reinterpret_cast<const u32x2*>(row);
                            const elem_t* four = reinterpret_cast<const elem_t*>(&raw);
#pragma unroll
                            for (int i = 0; i < V; ++i) xr[u][r][i] = to_f32(four[i]);
                        } else if constexpr (V == 4) {
                            const float4 four = *reinterpret_cast<const float4*>(row);
                            xr[u][r][0] = four.x, xr[u][r][1] = four.y, xr[u][r][2] = four.z, xr[u][r][3] = four.w;
                        } else {
                            xr[u][r][0] = to_f32(row[0]);
                        }
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int u = 0; u < AHEAD; ++u) {
                    const bool in = c0 + u * 64 * V < d;
#pragma unroll
                    for (int k = 0; k < EW; ++k)
#pragma unroll
                        for (int r = 0; r < R; ++r)
#pragma unroll
                            for (int i = 0; i < V; ++i) {
                                const float sum = v[k][r] + xr[u][r][i] * we[u][k][i];
                                v[k][r] = in ? sum : v[k][r];
                            }
                }
            }
        } else {
#pragma unroll(R == 1 ? 8 : 4)
            for (int c = lane * V; c < d; c += 64 * V) {
                float we[EW][V], xr[R][V];
#pragma unroll
                for (int k = 0; k < EW; ++k) {
                    const float* from = w + (size_t)min(e0 + 4 * k, outputs - 1) * d + c;
                    if constexpr (V == 4) {
                        const float4 four = *reinterpret_cast<const float4*>(from);
                        we[k][0] = four.x, we[k][1] = four.y, we[k][2] = four.z, we[k][3] = four.w;
                    } else {
                        we[k][0] = from[0];
                    }
                }
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    const elem_t* row = x + (size_t)min(t0 + r, rs.T - 1) * d + c;
                    if constexpr (V == 4 && sizeof(elem_t) == 2) {
                        const u32x2 raw = *reinterpret_cast<const u32x2*>(row);
                        const elem_t* four = reinterpret_cast<const elem_t*>(&raw);
#pragma unroll
                        for (int i = 0; i < V; ++i) xr[r][i] = to_f32(four[i]);
                    } else if constexpr (V == 4) {
                        const float4 four = *reinterpret_cast<const float4*>(row);
                        xr[r][0] = four.x, xr[r][1] = four.y, xr[r][2] = four.z, xr[r][3] = four.w;
                    } else {
                        xr[r][0] = to_f32(row[0]);
                    }
                }
#pragma unroll
                for (int k = 0; k < EW; ++k)
#pragma unroll
                    for (int r = 0; r < R; ++r)
#pragma unroll
                        for (int i = 0; i < V; ++i) v[k][r] += xr[r][i] * we[k][i];
            }
        }
#pragma unroll
        for (int k = 0; k < EW; ++k) {
            // four rows: at the first two steps a lane hands half of its sums to its counterpart and adds what it gets to the other half
            int r = 0;
            if constexpr (R == 4) {
                const bool up = lane & 32, right = lane & 16;
                const float a = (up ? v[k][2] : v[k][0]) + __shfl_xor(up ? v[k][0] : v[k][2], 32, WAVE);
                const float b = (up ? v[k][3] : v[k][1]) + __shfl_xor(up ? v[k][1] : v[k][3], 32, WAVE);
                v[k][0] = (right ? b : a) + __shfl_xor(right ? a : b, 16, WAVE);
                r = (up ? 2 : 0) + (right ? 1 : 0);
            } else {
                v[k][0] += __shfl_xor(v[k][0], 32, WAVE);
                v[k][0] += __shfl_xor(v[k][0], 16, WAVE);
            }
#pragma unroll
            for (int o = 8; o > 0; o >>= 1) v[k][0] += __shfl_xor(v[k][0], o, WAVE);
            const int e = e0 + 4 * k;
            if ((lane & 15) == 0 && (R == 4 || lane == 0)) {
                if (e < E) zs[r][e] = v[k][0] + (bias ? bias[e] : 0.f);
                else if (e < outputs) scores[r][e - E] = v[k][0];
            }
        }
    }
    __syncthreads();
    auto settle = [] {  // what the wave's lanes have left in LDS is there for all of them
        __builtin_amdgcn_wave_barrier();
        __threadfence_block();
    };
    const int t = t0 + wave;
    if (wave < R && t < rs.T) {
        float *z = zs[wave], *score = scores[wave], *chosen_z = chosen_zs[wave];
        int* chosen_e = chosen_es[wave];
        if (softmax_all) {
            // scores over every output; what is compared below is the score plus the correction
            float m = -INFINITY;
            for (int e = lane; e < E; e += 64) m = fmaxf(m, z[e]);
            m = wave_max(m);
            float sum = 0.f;
            for (int e = lane; e < E; e += 64) sum += expf(z[e] - m);
            sum = wave_sum(sum);
            for (int e = lane; e < E; e += 64) {
                const float sc = expf(z[e] - m) / sum;
                score[e] = sc;
                z[e] = sc + (correction ? correction[e] : 0.f);
            }
            settle();
        }
        // `top` rounds of a maximum over the wave; the winner, of equals the first, leaves the list
        if (E <= 64) {
            float left = lane < E ? z[lane] : -INFINITY;
            for (int k = 0; k < top; ++k) {
                const float best = wave_max(left);
                const unsigned long long at = __ballot(left == best && best > -INFINITY);
                const int first = at ? __builtin_ctzll(at) : MAX_EXPERTS;
                if (lane == 0) {
                    chosen_z[k] = best;
                    chosen_e[k] = first;
                }
                if (lane == first) left = -INFINITY;
            }
            settle();
        } else {
            for (int k = 0; k < top; ++k) {
                float best = -INFINITY;
                int at = MAX_EXPERTS;
                for (int e = lane; e < E; e += 64)
                    if (z[e] > best) { best = z[e]; at = e; }
                for (int o = 32; o > 0; o >>= 1) {
                    const float ob = __shfl_xor(best, o, WAVE);
                    const int oa = __shfl_xor(at, o, WAVE);
                    if (ob > best || (ob == best && oa < at)) { best = ob; at = oa; }
                }
                if (lane == 0) {
                    chosen_z[k] = best;
                    chosen_e[k] = at;
                    if (at < E) z[at] = -INFINITY;
                }
                settle();
            }
        }
        // the weights of all outputs, in the place of the logits
        const int ek = lane < top ? chosen_e[lane] : MAX_EXPERTS;
        float weight = 0.f;
        if (scoring == SIGMOID) {
            if (lane < top) weight = 1.0f / (1.0f + expf(-chosen_z[lane]));
        } else if (softmax_all) {
            float sum = 0.f;
            for (int k = 0; k < top; ++k)
                if (chosen_e[k] < E) sum += score[chosen_e[k]];
            if (ek < E) weight = score[ek] / (sum + 1e-20f);
        } else {
            const float m = chosen_z[0];  // the first chosen is the largest
            float sum = 0.f;
            for (int k = 0; k < top; ++k) sum += expf(chosen_z[k] - m);
            if (lane < top) weight = expf(chosen_z[lane] - m) / sum;
        }
        for (int e = lane; e < E; e += 64) z[e] = 0.f;
        settle();
        if (ek < E) z[ek] = weight;
        settle();
        float* g = gates + (size_t)t * outputs;
        for (int e = lane; e < E; e += 64) g[e] = z[e];
        for (int i = lane; i < extra; i += 64) g[E + i] = 1.0f / (1.0f + expf(-score[i]));
        if (rs.plane) {
            const bool uses = ek < rs.real && weight != 0.f;
            int at = 0;
            for (int k = 0; k < top; ++k) {
                const int other = __shfl(uses ? ek : MAX_EXPERTS, k, WAVE);
                at += other < ek;
            }
            const unsigned long long all = __ballot(uses);
            settle();  // (the weights and the extra logits have been read)
            int* pl = reinterpret_cast<int*>(z);
            for (int e = lane; e < rs.real; e += 64) pl[e] = -1;
            settle();
            if (uses) pl[ek] = at;
            settle();
            for (int e = lane; e < rs.real; e += 64) rs.plane[(size_t)t * rs.real + e] = pl[e];
            const int used = __popcll(all);
            if (lane == 0) used_planes[wave] = used;
            if constexpr (R > 1)
                for (int p = used; p < top; ++p)
                    for (int c = lane; c < rs.width; c += 64) rs.sums[((size_t)p * rs.T + t) * rs.width + c] = 0.f;
        }
    }
    if constexpr (R == 1) {
        if (!rs.plane) return;
        __syncthreads();
        for (int p = used_planes[0]; p < top; ++p)
            for (int c = threadIdx.x; c < rs.width; c += 256) rs.sums[((size_t)p * rs.T + t0) * rs.width + c] = 0.f;
    }
}

// act: 0 the exact GELU (erf), 1 its tanh form, 2 SiLU
__device__ __forceinline__ float expert_activation(float z, int act) {
    if (act == 0) return 0.5f * z * (1.0f + erff(z * 0.7071067811865476f));
    if (act == 1) return 0.5f * z * (1.0f + tanhf(0.7978845608028654f * (z + 0.044715f * z * z * z)));
    return z / (1.0f + expf(-z));
}

// a[t, c] = act(up[t, c]) * gates[t, c / ff] for c < E * ff, act(up[t, c]) beyond (experts that every row uses, whose weight is
// one, or gates[t, E] with `shared_gate`).  `weigh_input` (gated experts): act(w gate) * (w up), for c < E * ff.
constexpr int ACT_COLS = 2048;  // columns of a row that a block takes
template <int V>  // columns a thread takes at once: 4 where an expert's columns and the row are multiples of four
__global__ __launch_bounds__(256) void expert_act_kernel(const float* __restrict__ up, const float* __restrict__ gates,
                                                         elem_t* __restrict__ out, int n, int E, int ff, int act, int ld_gates, int gated,
                                                         int weigh_input, int shared_gate, int interleaved) {
    const int t = blockIdx.x, c0 = blockIdx.y * ACT_COLS, c1 = min(n, c0 + ACT_COLS);
    const float* g = gates + (size_t)t * ld_gates;
    const float shared_w = shared_gate ? g[E] : 1.0f;
    if (gated) {  // up [T, 2 n]: the gates' columns, then the up projections', or both in blocks of 16 in turn
        const float* row = up + (size_t)t * 2 * n;
#pragma unroll 2
        for (int c = c0 + threadIdx.x * V; c < c1; c += 256 * V) {
            const int e = c / ff;  // V columns lie in one expert (ff is a multiple of V)
            const float w = e < E ? g[e] : shared_w;
            const bool inside = weigh_input && e < E;   // the weight stands inside the expert
            const float wi = inside ? w : 1.0f;         // what gate and up are multiplied by
            elem_t* o = out + (size_t)t * n + c;
            auto value = [&](float gv, float uv) {
                return w != 0.f ? expert_activation(wi * gv, act) * uv * w : 0.f;
            };
            if constexpr (V == 4) {
                float4 a = (float4){0.f, 0.f, 0.f, 0.f}, b = a;
                const int at = interleaved ? c / 16 * 32 + c % 16 : c;
                if (w != 0.f) {
                    a = *reinterpret_cast<const float4*>(row + at);
                    b = *reinterpret_cast<const float4*>(row + at + (interleaved ? 16 : n));
                }
                o[0] = from_f32<elem_t>(value(a.x, b.x));
                o[1] = from_f32<elem_t>(value(a.y, b.y));
                o[2] = from_f32<elem_t>(value(a.z, b.z));
                o[3] = from_f32<elem_t>(value(a.w, b.w));
            } else {
                o[0] = from_f32<elem_t>(value(row[c], row[n + c]));
            }
        }
        return;
    }
#pragma unroll 2
    for (int c = c0 + threadIdx.x * V; c < c1; c += 256 * V) {
        const int e = c / ff;
        const float w = e < E ? g[e] : shared_w;
        // an expert the row did not choose contributes an exact zero, whatever its product holds
        if constexpr (V == 4) {
            float4 v = (float4){0.f, 0.f, 0.f, 0.f};
            if (w != 0.f) v = *reinterpret_cast<const float4*>(up + (size_t)t * n + c);
            elem_t* o = out + (size_t)t * n + c;
            o[0] = from_f32<elem_t>(w != 0.f ? expert_activation(v.x, act) * w : 0.f);
            o[1] = from_f32<elem_t>(w != 0.f ? expert_activation(v.y, act) * w : 0.f);
            o[2] = from_f32<elem_t>(w != 0.f ? expert_activation(v.z, act) * w : 0.f);
            o[3] = from_f32<elem_t>(w != 0.f ? expert_activation(v.w, act) * w : 0.f);
        } else {
            out[(size_t)t * n + c] = from_f32<elem_t>(w != 0.f ? expert_activation(up[(size_t)t * n + c], act) * w : 0.f);
        }
    }
}

// x[t, c] += (sum of weights[t, first .. first + count]) * h[t, c]: rows of a part's input added with a weight a row
__global__ __launch_bounds__(256) void add_scaled_rows_kernel(float* __restrict__ x, const elem_t* __restrict__ h,
                                                              const float* __restrict__ weights, int ld_w, int first, int count, int d) {
    const int t = blockIdx.x;
    float w = 0.f;
    for (int i = 0; i < count; ++i) w += weights[(size_t)t * ld_w + first + i];
    if (w == 0.f) return;
    for (int c = blockIdx.y * 1024 + threadIdx.x; c < min(d, (int)(blockIdx.y + 1) * 1024); c += 256)
        x[(size_t)t * d + c] += w * to_f32(h[(size_t)t * d + c]);
}

// ---- products over the rows that chose an expert -------------------------------------------------------------------------
// Of E experts a row uses `top`, so a product over every expert's columns does E / top times the work (2,048 rows of 2,048, 8
// experts of 2,816 of which 2 are used, and one that every row uses: up, activation and down 366 + 73 + 366 us a layer where this
// does it all in 179 + 83).  Here a block's tile of rows belongs to one expert: the up product gathers the rows that chose it, applies
// the activation and the weight in its epilogue (the 32-bit sums of all experts never go through memory), and leaves the
// activations tile after tile; the down product multiplies them by the expert's own matrix and stores the sums in the planes that
// the reader adds up, one for each expert that a row uses, in ascending order.  Who reads what is found by the blocks themselves: a step of
// at most 64 rows has one tile an expert, whose rows a wave finds with one ballot; above, `expert_rows_kernel` lists them
// and a block finds its expert by a prefix sum over the lists' lengths.  Blocks of tiles that do not exist end at once.
struct ExpertArgs {
    const int* plane;     // [T, E]
    const float* gates;   // [T, ld_gates]
    const int* rows;      // [E, T] lists of the experts' rows, or null: T <= 64
    const int* counts;    // [E] their lengths
    int T, E, ld_gates, top;
    int routed_tiles, shared_tiles;  // row tiles of the grid: those of the experts (as many as there can be), those of the expert that every row uses
    int routed_slots;     // rows of the activations before those of the expert that every row uses
    int ff, shared;       // columns of an expert, and of the one that every row uses (0: there is none)
    int width;            // of the rows
    int shared_gate, weigh_input, act;
    int past;             // the weights are read past the last-level cache (few_rows.cuh); up to 32 rows
};

__global__ __launch_bounds__(1024) void expert_rows_kernel(const int* __restrict__ plane, int* __restrict__ rows, int* __restrict__ counts, int T, int E) {
    __shared__ int part[2][16];
    const int e = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int n = 0;
    for (int t0 = 0, turn = 0; t0 < T; t0 += 1024, turn ^= 1) {  // two sets of partial counts in turn: one barrier a round
        const int t = t0 + threadIdx.x;
        const bool mine = t < T && plane[(size_t)min(t, T - 1) * E + e] >= 0;
        const unsigned long long all = __ballot(mine);
        if (lane == 0) part[turn][wave] = __popcll(all);
        __syncthreads();
        int before = n;
        for (int w = 0; w < 16; ++w) {
            if (w < wave) before += part[turn][w];
            n += part[turn][w];
        }
        if (mine) rows[(size_t)e * T + before + __popcll(all & ((1ull << lane) - 1))] = t;
    }
    if (threadIdx.x == 0) counts[e] = n;
}

template <bool GATHERS_>  // A's rows are the step's rows (the up product), else the tiles' activations (the down product)
struct ExpertRows {
    static constexpr bool GATHERS = GATHERS_;
    const ExpertArgs& g;
    const int* list;  // of the expert's rows; null: every row
    int e, first;     // e == E: the expert that every row uses; where its activations begin
    const int* of_row;  // LDS: the weight of each of the tile's rows (up), the row of its sums (down)
    __device__ __forceinline__ int row_of(int m) const { return list ? list[m] : m; }
    __device__ __forceinline__ int slot(int m) const { return first + m; }
    __device__ __forceinline__ int source(int m) const { return GATHERS ? row_of(m) : slot(m); }
    __device__ __forceinline__ int pitch(int) const { return GATHERS ? g.width : max(g.ff, g.shared); }
    __device__ __forceinline__ int w_pitch(int) const { return GATHERS ? g.width : g.E * g.ff + g.shared; }
    __device__ __forceinline__ float weight(int m, int m0) const { return __int_as_float(of_row[m - m0]); }
    __device__ __forceinline__ size_t out_row(int m, int m0) const { return GATHERS ? slot(m) : of_row[m - m0]; }
    template <typename F>
    __device__ __forceinline__ void with_activation(F f) const {
        if (g.act == 0) f(std::integral_constant<int, 0>{});
        else if (g.act == 1) f(std::integral_constant<int, 1>{});
        else f(std::integral_constant<int, 2>{});
    }
    // as expert_act: the weight on the output, or inside the expert
    template <int ACT>
    __device__ __forceinline__ float gated(std::integral_constant<int, ACT>, float gv, float uv, float w) const {
        const float wi = g.weigh_input && e < g.E ? w : 1.0f;
        return w != 0.f ? expert_activation(wi * gv, ACT) * uv * w : 0.f;
    }
    template <int ACT>
    __device__ __forceinline__ float plain(std::integral_constant<int, ACT>, float z, float w) const {
        return w != 0.f ? expert_activation(z, ACT) * w : 0.f;
    }
};

template <int BM, int BN, int WM, int WN, int BK, int EPI, int STAGES>
__global__ __launch_bounds__(64 * WM * WN) void expert_gemm_kernel(const elem_t* __restrict__ A, const elem_t* __restrict__ W, void* out, ExpertArgs g) {
    __shared__ int few[64];
    constexpr int PER = EPI == EPI_EXPERT_GATED ? 2 : 1;  // columns of the up product for one of the activations
    constexpr int GROUP = BM >= 256 ? 4 : 1024 / BM;      // tiles of rows that go over the columns together
    const int lane = threadIdx.x & 63;
    int e = g.E, m0 = 0, count = g.T, first = g.routed_slots, col;
    const int* list = nullptr;
    if (!g.rows) {
        const int tiles = g.routed_tiles + g.shared_tiles, tile = blockIdx.x % tiles;
        col = blockIdx.x / tiles;
        if (tile < g.routed_tiles) {
            e = tile;
            first = tile * g.T;
            const bool mine = lane < g.T && g.plane[(size_t)min(lane, g.T - 1) * g.E + e] >= 0;
            const unsigned long long all = __ballot(mine);
            count = __popcll(all);
            if (mine) few[__popcll(all & ((1ull << lane) - 1))] = lane;
            list = few;
        }
    } else {
        // The blocks of one XCD (every 8th) take a run of the tiles that there are, first of the expert that every row uses, then of the others; in it
        // GROUP tiles, mostly of one or two experts, go over the columns together and share both operands in the XCD's L2.
        const int cols_all = EPI == EPI_EXPERT_DOWN ? ceil_div(g.width, BN) : ceil_div(PER * g.shared, BN);
        const int cols_one = EPI == EPI_EXPERT_DOWN ? ceil_div(g.width, BN) : ceil_div(PER * g.ff, BN);
        const int xcd = blockIdx.x & 7, run_all = ceil_div(g.shared_tiles * cols_all, 8);
        int nth = blockIdx.x >> 3, tiles = g.shared_tiles, cols = cols_all, run = run_all;
        const bool routed = nth >= run_all;
        if (routed) {
            nth -= run_all;
            tiles = 0;
            for (int e0 = 0; e0 < g.E; e0 += 64) {
                int mine = e0 + lane < g.E ? ceil_div(g.counts[e0 + lane], BM) : 0;
#pragma unroll
                for (int o = 1; o < 64; o <<= 1) mine += __shfl_xor(mine, o, WAVE);
                tiles += mine;
            }
            tiles = __builtin_amdgcn_readfirstlane(tiles);
            cols = cols_one;
            run = ceil_div(tiles * cols, 8);
        }
        const int at = xcd * run + nth;
        if (nth >= run || at >= tiles * cols) return;
        const int group = at / (GROUP * cols), in = at - group * (GROUP * cols), size = min(GROUP, tiles - group * GROUP);
        const int tile = group * GROUP + in % size;
        col = in / size;
        if (routed) {
            // the expert whose tiles hold this one, 64 experts' counts at a time
            int base = 0, slots = 0;
            count = 0;
            for (int e0 = 0; e0 < g.E; e0 += 64) {
                const int c = e0 + lane < g.E ? g.counts[e0 + lane] : 0;
                const int mine = ceil_div(c, BM), own = ceil_div(c, 64) * 64;
                int upto = mine, upto_slots = own;
#pragma unroll
                for (int o = 1; o < 64; o <<= 1) {
                    const int v = __shfl_up(upto, o, WAVE), u = __shfl_up(upto_slots, o, WAVE);
                    if (lane >= o) {
                        upto += v;
                        upto_slots += u;
                    }
                }
                const unsigned long long behind = __ballot(base + upto > tile);
                if (behind) {
                    const int l = __builtin_ctzll(behind);
                    e = e0 + l;
                    count = __shfl(c, l, WAVE);
                    m0 = (tile - (base + __shfl(upto - mine, l, WAVE))) * BM;
                    first = slots + __shfl(upto_slots - own, l, WAVE);
                    break;
                }
                base += __shfl(upto, 63, WAVE);
                slots += __shfl(upto_slots, 63, WAVE);
            }
            list = g.rows + (size_t)e * g.T;
        } else {
            m0 = tile * BM;
        }
    }
    // Into scalar registers for good (the tile's loads take their bases from there): seen through, the compiler may keep them in vector ones.
    auto scalar = [](int v) {
        asm volatile("" : "+v"(v));
        return __builtin_amdgcn_readfirstlane(v);
    };
    e = scalar(e), count = scalar(count), m0 = scalar(m0), first = scalar(first), col = scalar(col);
    const int cols = e == g.E ? g.shared : g.ff;
    const int N = EPI == EPI_EXPERT_DOWN ? g.width : PER * cols, K = EPI == EPI_EXPERT_DOWN ? cols : g.width;
    const int n0 = col * BN;
    if (m0 >= count || n0 >= N) return;  // the whole block: these are the block's own numbers
    __syncthreads();
    // What the epilogue needs of each row, read once by the whole block: read row by row between the stores the two dependent loads
    // were 9 to 12 us of a block's 35 to 72.
    __shared__ int of_row[BM];
    int own_e = e;
    asm volatile("" : "+v"(own_e));  // a copy for the branches: what they merge is kept in vector registers
    for (int i = threadIdx.x; i < BM; i += 64 * WM * WN) {
        const int m = min(m0 + i, count - 1), t = list ? list[m] : m;
        if (EPI == EPI_EXPERT_DOWN) of_row[i] = (own_e == g.E ? g.top : g.plane[(size_t)t * g.E + own_e]) * g.T + t;
        else of_row[i] = __float_as_int(own_e == g.E && !g.shared_gate ? 1.0f : g.gates[(size_t)t * g.ld_gates + own_e]);
    }
    EpiArgs ep{out, nullptr, EPI == EPI_EXPERT_DOWN ? g.width : max(g.ff, g.shared), EPI == EPI_EXPERT_DOWN ? g.width : cols, K, 0};
    const ExpertRows<EPI != EPI_EXPERT_DOWN> rows{g, list, e, first, of_row};
    const elem_t* own = W + (size_t)e * g.ff * (EPI == EPI_EXPERT_DOWN ? 1 : PER * g.width);  // its columns, or its rows
    gemm_tile<BM, BN, WM, WN, BK, EPI, STAGES, false>(A, own, count, N, K, ep, m0, n0, 0, rows);
}

#ifdef MS_ELEM_HALF
// A step of at most 32 rows, a step of K or more for every wave: four waves share out K (few_rows.cuh), a block an expert and 16 NT of its columns.  The rows
// that chose the expert, and what the epilogue needs of them, are one trip: every wave reads all rows' planes, lane t row t's.
// Bound by the chosen experts' weights.  32 columns a block (72 and 64 KB of LDS, two blocks a CU) are better than 64: four rows that use 5 of 8 experts of 2,816
// and one for every row, width 2,048 (us up + down): 64x64 tiles 44.5 + 21.6, 64 columns 38.3 + 21.8, 32 columns 34.4 + 17.1; sixteen rows 49.3 + 25.4,
// 47.2 + 25.5, 39.2 + 21.1; 24 rows 49.8 + 26, 50.4 + 27, 41.0 + 22.3; eight rows, 6 of 64 experts of 1,408, 94 + 49 and 79 + 42.  Above 32 rows the tiles are
// the better ones (48 rows 52.1 + 28.3; as two or three row tiles here 58.8 + 30.5 and 44 + 25, but 64 rows 44 + 18 against 54 + 26 and 84 + 40).
template <int MT, int NT, int STAGES, int EPI>
__global__ __launch_bounds__(64 * FEW_WAVES) void expert_few_kernel(const elem_t* __restrict__ A, const elem_t* __restrict__ W, void* out, ExpertArgs g) {
    constexpr bool DOWN = EPI == EPI_EXPERT_DOWN;
    constexpr int PER = EPI == EPI_EXPERT_GATED ? 2 : 1;
    __shared__ int few[16 * MT], of_row[16 * MT];
    const int lane = threadIdx.x & 63, tiles = g.routed_tiles + g.shared_tiles, tile = blockIdx.x % tiles, n0 = blockIdx.x / tiles * (16 * NT);
    const bool shared = tile >= g.routed_tiles;
    const int e = shared ? g.E : tile, cols = shared ? g.shared : g.ff;
    const int N = DOWN ? g.width : PER * cols, K = DOWN ? cols : g.width;
    if (n0 >= N) return;
    const int t = min(lane, g.T - 1);
    const int plane = shared ? g.top : g.plane[(size_t)t * g.E + e];
    const float gate = DOWN || (shared && !g.shared_gate) ? 1.0f : g.gates[(size_t)t * g.ld_gates + e];
    const bool mine = lane < g.T && plane >= 0;
    const unsigned long long all = __ballot(mine);
    const int count = __builtin_amdgcn_readfirstlane(__popcll(all));
    if (count == 0) return;  // the whole block
    if (threadIdx.x < 64 && mine) {
        const int at = __popcll(all & ((1ull << lane) - 1));
        few[at] = lane;
        of_row[at] = DOWN ? plane * g.T + lane : __float_as_int(gate);
    }
    __syncthreads();
    EpiArgs ep{out, nullptr, DOWN ? g.width : max(g.ff, g.shared), DOWN ? g.width : cols, K, 0};
    ep.k_per_split = K;
    ep.past = g.past;
    const ExpertRows<!DOWN> rows{g, shared ? nullptr : few, e, shared ? g.routed_slots : tile * g.T, of_row};
    const elem_t* own = W + (size_t)e * g.ff * (DOWN ? 1 : PER * g.width);  // its columns, or its rows
    few_rows_tile<MT, NT, FEW_WAVES, STAGES, EPI, false>(A, own, count, N, K, ep, 0, n0, 0, rows);
}
#endif

// The tile of a product.  A step of 33 to 64 rows (and of any number up to 64 in 32-bit) has one tile of 64 rows an expert, its weight's columns streamed by blocks with
// three steps in flight; above, the tile of the least predicted time, its tiles counted from how many rows
// an expert can be expected to have.
// With half of every expert's last tile counted as empty instead, the chosen tiles take 1.039 times the best ones' time where these take 1.025 (220 products,
// the worst 1.65 and 1.28), with uneven loads 1.044 and 1.034; us up (2 of 8 experts of 2,816, width 2,048): 700 rows and an expert for every row 68 -> 59,
// 2,048 over nine outputs 110 -> 103, 1,200 87 -> 92.
// 2,048 rows, 2 of 8 experts of 2,816 and one of 2,816 for every row, width 2,048, gated (us up / down): 256x256 191 / 83, 256x192 211 / 120,
// 256x128 197 / 97, 128x128 179 / 106, 64x64 279 / 156; 128x128 alone, in the order of the columns and with the epilogue reading row by row, was 228 / 120.
// 1,750 rows, 2 of 8 experts of 2,816: 122 / 73, 128 / 62, 130 / 87, 120 / 72 and 178 / 101 against 170 / 113.
static int plan_experts(const ExpertArgs& g, bool down, int per) {
#ifdef MS_ELEM_HALF
    if (g.T <= 64) return TILE_64x64_DEEP;
    // Rows fall to the router's outputs (of which some may be no experts) nearly as if at random: an expert has `mean` rows, give or take `spread`, and
    // its tiles are counted as the chances that it has more rows than each of them begins with.  `spread` is chance's and 3 % of the mean: routers do not share
    // out their rows quite as evenly as chance.  Over 220 products a line (110 sizes, 65 to 4,096 rows, 1 to 6 of 4 to 64 experts), the chosen tile's time
    // over the best one's on average, with 0, 3 and 10 %: loads as chance has them 1.025 1.026 1.030 and 1.033 1.041 1.049, wider by 2 to 3 % of the mean
    // 1.035 1.031 1.031 and 1.037 1.036 1.038, by 9 % 1.038 1.032 1.028.  (The down product of 2,048 rows over nine outputs, eight of them experts: 256x128 tiles are a round if
    // no expert has more than 512 rows and two if one has, 43 and 86 us; 256x192 53 to 59.)
    const int outputs = max(g.E, g.ld_gates - (g.shared ? 1 : 0));  // (a gate of the expert for every row is none of them)
    const double mean = (double)g.T * g.top / outputs, spread = sqrt(mean * (1.0 - 1.0 / outputs)) + 0.03 * mean + 1e-3;
    int best = TILE_64x64;
    float least = INFINITY;
    for (int i = 0; i < TILE_COUNT; ++i) {
        const TileCost& t = kTiles[i];
        if (i == TILE_256x256 && !down && per == 1) continue;  // every sum in its own activation: too many registers
        // (and their deviation with them: blocks that come to just a round in the mean are often a round and one)
        double tiles = 0.0, variance = 0.0;
        for (long at = 0; at < g.T && at < mean + 4.0 * spread; at += t.bm) {
            const double p = 0.5 * erfc((at + 0.5 - mean) / (spread * 1.4142135623730951));
            tiles += p * g.E;
            variance += p * (1.0 - p) * g.E;
        }
        const long routed = max(1L, lround(tiles + sqrt(variance))), all = g.shared ? ceil_div(g.T, t.bm) : 0;
        const long blocks = down ? (routed + all) * ceil_div(g.width, t.bn) : routed * ceil_div(per * g.ff, t.bn) + all * ceil_div(per * g.shared, t.bn);
        const long depth = down ? (routed * g.ff + all * g.shared) / (routed + all) : g.width;
        const float us = tile_time(t, blocks, (int)depth, down);
        if (us < least) {
            least = us;
            best = i;
        }
    }
    return best;
#else
    (void)g; (void)down; (void)per;
    return TILE_64x64_DEEP;
#endif
}

static long expert_routed_tiles(int T, int E, int top, long bm) {
    if (T <= 64) return E;
    return min((long)T * top / bm + min((long)E, (long)T * top), (long)E * ceil_div((long)T, bm));
}

// Rows of the activations before those of the expert that every row uses: with lists every expert's begin at a multiple of 64; without, as
// many as the step has rows are set aside for each (of one row and 1,024 experts of 2,048 columns 4 MB in two bytes, where 64 an expert were 268).
static long expert_routed_slots(int T, int E, int top) { return T <= 64 ? (long)E * T : expert_routed_tiles(T, E, top, 64) * 64; }

static int check_experts(const char* what, const ExpertArgs& g) {
    MS_REQUIRE(g.T > 0 && g.E > 0 && g.E <= MAX_EXPERTS && g.top >= 1 && g.top <= 64, "%s: %d rows, %d of %d experts", what, g.T, g.top, g.E);
    MS_REQUIRE(g.width > 0 && g.width % 64 == 0 && g.ff > 0 && g.ff % 64 == 0 && g.shared >= 0 && g.shared % 64 == 0,
               "%s: width %d, experts of %d and %d for every row: multiples of 64 are taken", what, g.width, g.ff, g.shared);
    MS_REQUIRE(g.plane && g.gates && g.ld_gates >= g.E + (g.shared_gate ? 1 : 0), "%s: %d weights a row for %d experts", what, g.ld_gates, g.E);
    MS_REQUIRE(g.act >= 0 && g.act <= 2, "%s: activation %d", what, g.act);
    MS_REQUIRE((g.T <= 64) == (g.rows == nullptr) && (g.T <= 64) == (g.counts == nullptr), "%s: lists of rows go with more than 64 of them", what);
    return 0;
}

template <int EPI>
static int launch_experts(const void* a, const void* w, void* out, ExpertArgs g, hipStream_t stream) {
    MS_REQUIRE((reinterpret_cast<uintptr_t>(a) & 15) == 0 && (reinterpret_cast<uintptr_t>(w) & 15) == 0, "experts: operands must be 16-byte aligned");
    constexpr bool DOWN = EPI == EPI_EXPERT_DOWN;
    constexpr int PER = EPI == EPI_EXPERT_GATED ? 2 : 1;
    const TileCost& tile = kTiles[plan_experts(g, DOWN, PER)];
    g.routed_tiles = (int)expert_routed_tiles(g.T, g.E, g.top, tile.bm);
    g.shared_tiles = g.shared ? ceil_div(g.T, tile.bm) : 0;
    g.routed_slots = (int)expert_routed_slots(g.T, g.E, g.top);
    const long cols_one = ceil_div(DOWN ? g.width : PER * g.ff, tile.bn), cols_all = ceil_div(DOWN ? g.width : PER * g.shared, tile.bn);
    const long nb = g.rows ? 8 * (ceil_div(g.routed_tiles * cols_one, 8L) + ceil_div(g.shared_tiles * cols_all, 8L))
                           : (long)(g.routed_tiles + g.shared_tiles) * max(cols_one, cols_all);
#define MS_EXPERTS(BM_, BN_, WM_, WN_, BK_, ST_)                                                                                    \
    do {                                                                                                                            \
        hipLaunchKernelGGL((expert_gemm_kernel<BM_, BN_, WM_, WN_, BK_, EPI, ST_>), dim3((unsigned)nb), dim3(64 * WM_ * WN_), 0,    \
                           stream, (const elem_t*)a, (const elem_t*)w, out, g);                                                     \
        return check_launch("experts " #BM_ "x" #BN_ "x" #BK_);                                                                     \
    } while (0)
#ifdef MS_ELEM_HALF
    if (g.T <= 32 && (DOWN ? min(g.ff, g.shared ? g.shared : g.ff) : g.width) >= 64 * FEW_WAVES) {
#define MS_EXPERTS_FEW(MT_, NT_, ST_)                                                                                                       \
    do {                                                                                                                                    \
        const long blocks = (long)(g.routed_tiles + g.shared_tiles) * ceil_div(DOWN ? g.width : PER * max(g.ff, g.shared), 16 * NT_);        \
        hipLaunchKernelGGL((expert_few_kernel<MT_, NT_, ST_, EPI>), dim3((unsigned)blocks), dim3(64 * FEW_WAVES), 0, stream, (const elem_t*)a, \
                           (const elem_t*)w, out, g);                                                                                        \
        return check_launch("experts, few rows");                                                                                            \
    } while (0)
        if (g.T <= 16) MS_EXPERTS_FEW(1, 2, 3);
        MS_EXPERTS_FEW(2, 2, 2);
#undef MS_EXPERTS_FEW
    }
    switch ((int)(&tile - kTiles)) {
        case TILE_256x256:
            if constexpr (EPI != EPI_EXPERT_PLAIN) MS_EXPERTS(256, 256, 2, 4, 64, GEMM_PIPED);
        case TILE_256x192: MS_EXPERTS(256, 192, 4, 2, 64, GEMM_PIPED);
        case TILE_256x128: MS_EXPERTS(256, 128, 4, 2, 64, GEMM_PIPED);
        case TILE_128x128: MS_EXPERTS(128, 128, 2, 4, 64, GEMM_PIPED);
        case TILE_64x64: MS_EXPERTS(64, 64, 2, 2, 64, GEMM_PIPED);
        default: MS_EXPERTS(64, 64, 2, 2, 64, 4);
    }
#else
    MS_EXPERTS(64, 64, 2, 2, 32, 3);
#endif
#undef MS_EXPERTS
}

}  // namespace ms

using namespace ms;

extern "C" int ms_route_max_experts() { return MAX_EXPERTS; }

// w [E + extra, d]; gates [T, E + extra]: the weights of the E outputs to choose from, then `extra` gates of every row.  With `plane`
// [T, real] (else null) the experts that each row uses among the first `real` outputs are numbered, and the rows of sums [top, T, d] that
// no expert will write are zeroed.
extern "C" int ms_route(const void* x, const float* w, const float* bias, float* gates, int T, int d, int E, int top, int scoring,
                        const float* correction, int extra, int* plane, float* sums, int real, hipStream_t stream) {
    MS_REQUIRE(scoring >= SOFTMAX_CHOSEN && scoring <= SIGMOID, "route: scoring %d", scoring);
    MS_REQUIRE(extra >= 0 && extra <= MAX_EXPERTS && (extra == 0 || (scoring != SOFTMAX_ALL && !bias)),
               "route: %d gates of every row (none with scores over all outputs or a bias)", extra);
    MS_REQUIRE(T > 0 && d > 0 && E > 0 && E <= MAX_EXPERTS, "route: %d rows of %d over %d experts (at most %d)", T, d, E, MAX_EXPERTS);
    MS_REQUIRE(top >= 1 && top <= E && top <= 64, "route: %d of %d experts a row (at most 64)", top, E);
    MS_REQUIRE((plane == nullptr) == (sums == nullptr) && (!plane || (real > 0 && real <= E)), "route: %d of %d outputs are experts", real, E);
    const RouteSums rs{plane, sums, real, d, T};
#define MS_ROUTE(R_, V_, EW_, A_)                                                                                                                     \
    hipLaunchKernelGGL((route_kernel<R_, V_, EW_, A_>), dim3(ceil_div(T, R_)), dim3(256), 0, stream, (const elem_t*)x, w, bias, gates, d, E, top, scoring, \
                       correction, extra, rs)
    // four columns a load where every row begins at a multiple of them; four rows a block where that leaves every CU a block
    const bool fours = d % 4 == 0 && (reinterpret_cast<uintptr_t>(w) & 15) == 0 && (reinterpret_cast<uintptr_t>(x) & (4 * sizeof(elem_t) - 1)) == 0;
    const bool many = T >= 4 * compute_units();
    // up to four outputs: one a wave, which asks for nothing twice (four outputs of 2,048, three a wave / one / an output in turn: 16 rows 5.0 / 4.2 / 4.9 us,
    // 1,000 rows 7.8 / 5.6 / 6.6; five outputs, three a wave / in turn: 5.0 / 5.7 and 7.9 / 7.5)
    const bool one = E + extra <= 4;
    // Steps asked for at once: eight, four where a row has four at most, two of two and of four rows, as long as the last round asks for few steps that the row does not have
    // (us, plain loop and so, 64 rows over 64 outputs: 1,536 columns, two of eight, 14.2 and 13.3; 2,304 columns, seven of sixteen, 17.0 and 18.8): a quarter at most; none of
    // four rows (2,048 rows of 768 columns over 9 outputs, one of four, 5.8 and 6.1); and one of eight, in one round, where two rows share a CU (300 rows:
    // 1,792 columns over 64 outputs, one of eight, 17.5 and 15.5; 1,536 over 9, two, 5.4 and 5.7; 3,584 over 9, two of sixteen, 7.2 and 7.6).  With more than two rows a CU
    // the blocks beside each other hide the loads, and the registers count (1,000 rows over 64 outputs: 1,280 columns 18.4 and 27, 2,048 columns 26.4 and 27.8).
    // An output a wave of four rows has fewer loads a step, of which the loop asks for four: two are enough up to 1,536 columns (2,048 rows over 2 outputs 4.8 and 4.4; one output of 4,096,
    // 1,024 rows 4.9 and 5.3), and with a column a load nowhere (one output of 3,001 6.6 and 8.6, 128 in 32-bit 137 and 147).
    const int steps = ceil_div(d, 64 * 4), most = many || steps <= 2 ? 2 : steps <= 4 ? 4 : 8, surplus = ceil_div(steps, most) * most - steps;
    const bool straight = many                     ? surplus == 0 && (!one || steps <= 6)
                          : T <= compute_units()     ? surplus * 4 <= steps + surplus
                          : T <= 2 * compute_units() ? surplus * 8 <= most && steps <= 8
                                                     : false;
    const int ahead = straight ? most : 1;
#define MS_ROUTE_FOURS(EW_)                              \
    do {                                                 \
        if (many && ahead == 2) MS_ROUTE(4, 4, EW_, 2);  \
        else if (many) MS_ROUTE(4, 4, EW_, 1);           \
        else if (ahead == 8) MS_ROUTE(1, 4, EW_, 8);     \
        else if (ahead == 4) MS_ROUTE(1, 4, EW_, 4);     \
        else if (ahead == 2) MS_ROUTE(1, 4, EW_, 2);     \
        else MS_ROUTE(1, 4, EW_, 1);                     \
    } while (0)
    if (one && fours) MS_ROUTE_FOURS(1);
    else if (fours) MS_ROUTE_FOURS(3);
    else if (one && many) MS_ROUTE(4, 1, 1, 1);
    else if (one) MS_ROUTE(1, 1, 1, 1);
    else if (many) MS_ROUTE(4, 1, 3, 1);
    else MS_ROUTE(1, 1, 3, 1);
#undef MS_ROUTE_FOURS
#undef MS_ROUTE
    return check_launch("route");
}

// n: columns of the output; with `gated`, up has 2 n columns.  ld_gates: numbers a row of gates has (>= E).
extern "C" int ms_expert_act(const float* up, const float* gates, void* out, int T, int n, int E, int ff, int act, int ld_gates, int gated,
                             int weigh_input, int shared_gate, int interleaved, hipStream_t stream) {
    MS_REQUIRE(!interleaved || (gated && n % 16 == 0 && ff % 4 == 0), "expert_act: %d gated columns in blocks of 16", n);
    MS_REQUIRE(T > 0 && n > 0 && E >= 0 && ff > 0 && (long)E * ff <= n && ld_gates >= E, "expert_act: %d columns for %d experts of %d", n, E, ff);
    MS_REQUIRE(act >= 0 && act <= 2, "expert_act: activation %d", act);
    MS_REQUIRE(!weigh_input || gated, "expert_act: weights inside experts that are not gated");
    MS_REQUIRE(!shared_gate || ld_gates > E, "expert_act: %d weights a row for %d experts and a gate", ld_gates, E);
    const dim3 grid(T, ceil_div(n, ACT_COLS));
    if (n % 4 == 0 && ff % 4 == 0) hipLaunchKernelGGL(expert_act_kernel<4>, grid, dim3(256), 0, stream, up, gates, (elem_t*)out, n, E, ff, act, ld_gates, gated,
                                                       weigh_input, shared_gate, interleaved);
    else hipLaunchKernelGGL(expert_act_kernel<1>, grid, dim3(256), 0, stream, up, gates, (elem_t*)out, n, E, ff, act, ld_gates, gated,
                                                       weigh_input, shared_gate, interleaved);
    return check_launch("expert_act");
}

extern "C" int ms_add_scaled_rows(float* x, const void* h, const float* weights, int ld_w, int first, int count, int T, int d,
                                  hipStream_t stream) {
    MS_REQUIRE(T > 0 && d > 0 && first >= 0 && count >= 1 && first + count <= ld_w, "add_scaled_rows: weights %d .. %d of %d", first,
               first + count, ld_w);
    hipLaunchKernelGGL(add_scaled_rows_kernel, dim3(T, ceil_div(d, 1024)), dim3(256), 0, stream, x, (const elem_t*)h, weights, ld_w, first,
                       count, d);
    return check_launch("add_scaled_rows");
}

// Rows of the activations that ms_experts_up leaves and ms_experts_down reads: the experts' one behind the other, then those of the expert
// that every row uses.
extern "C" long ms_experts_slots(int T, int E, int top, int shared) {
    if (T <= 0 || E <= 0 || top <= 0) return 0;
    return expert_routed_slots(T, E, top) + (shared > 0 ? T : 0);
}

// rows [E, T], counts [E]: the rows that use each expert, in ascending order.
extern "C" int ms_expert_rows(const int* plane, int* rows, int* counts, int T, int E, hipStream_t stream) {
    MS_REQUIRE(plane && rows && counts && T > 0 && E > 0 && E <= MAX_EXPERTS, "expert rows: %d rows of %d experts", T, E);
    hipLaunchKernelGGL(expert_rows_kernel, dim3(E), dim3(1024), 0, stream, plane, rows, counts, T, E);
    return check_launch("expert_rows");
}

// x [T, width]; w: the experts' matrices one behind the other and then that of the expert every row uses (`shared` columns, 0: none), each
// [cols, width], or with `gated` [2 cols, width] with gate and up rows interleaved in blocks of 16; out [slots, max(ff, shared)].
static int experts_up(const void* x, const void* w, void* out, const int* plane, const float* gates, const int* rows, const int* counts,
                             int T, int E, int ld_gates, int top, int ff, int shared, int width, int gated, int shared_gate, int weigh_input,
                             int act, hipStream_t stream, int past) {
    const ExpertArgs g{plane, gates, rows, counts, T, E, ld_gates, top, 0, 0, 0, ff, shared, width, shared_gate, weigh_input, act, past};
    if (int rc = check_experts("experts up", g)) return rc;
    MS_REQUIRE(!weigh_input || gated, "experts up: weights inside experts that are not gated");
    return gated ? launch_experts<EPI_EXPERT_GATED>(x, w, out, g, stream) : launch_experts<EPI_EXPERT_PLAIN>(x, w, out, g, stream);
}
extern "C" int ms_experts_up(const void* x, const void* w, void* out, const int* plane, const float* gates, const int* rows, const int* counts,
                             int T, int E, int ld_gates, int top, int ff, int shared, int width, int gated, int shared_gate, int weigh_input,
                             int act, hipStream_t stream) {
    return experts_up(x, w, out, plane, gates, rows, counts, T, E, ld_gates, top, ff, shared, width, gated, shared_gate, weigh_input, act, stream, 0);
}
extern "C" int ms_experts_up_past(const void* x, const void* w, void* out, const int* plane, const float* gates, const int* rows, const int* counts,
                             int T, int E, int ld_gates, int top, int ff, int shared, int width, int gated, int shared_gate, int weigh_input,
                             int act, hipStream_t stream) {
    return experts_up(x, w, out, plane, gates, rows, counts, T, E, ld_gates, top, ff, shared, width, gated, shared_gate, weigh_input, act, stream, 1);
}

// a [slots, max(ff, shared)] as ms_experts_up leaves it; w [width, E * ff + shared]: the experts' down matrices side by side,
// then the shared one's; sums [top (+ 1), T, width]: plane k of row t is the k-th expert that it uses, the last plane the shared one's.
static int experts_down(const void* a, const void* w, float* sums, const int* plane, const float* gates, const int* rows, const int* counts,
                               int T, int E, int ld_gates, int top, int ff, int shared, int width, hipStream_t stream, int past) {
    const ExpertArgs g{plane, gates, rows, counts, T, E, ld_gates, top, 0, 0, 0, ff, shared, width, 0, 0, 0, past};
    if (int rc = check_experts("experts down", g)) return rc;
    return launch_experts<EPI_EXPERT_DOWN>(a, w, sums, g, stream);
}
extern "C" int ms_experts_down(const void* a, const void* w, float* sums, const int* plane, const float* gates, const int* rows, const int* counts,
                               int T, int E, int ld_gates, int top, int ff, int shared, int width, hipStream_t stream) {
    return experts_down(a, w, sums, plane, gates, rows, counts, T, E, ld_gates, top, ff, shared, width, stream, 0);
}
extern "C" int ms_experts_down_past(const void* a, const void* w, float* sums, const int* plane, const float* gates, const int* rows, const int* counts,
                               int T, int E, int ld_gates, int top, int ff, int shared, int width, hipStream_t stream) {
    return experts_down(a, w, sums, plane, gates, rows, counts, T, E, ld_gates, top, ff, shared, width, stream, 1);
}
