// Gated linear attention (see gated_state.cuh): the decays, the walk over many rows, and its entry points.
#include "gated_state.cuh"

namespace ms {

// ---- gated linear attention's decays ------------------------------------------------------------------------
// alpha[t, c] = sigmoid(z)^(1 / tau) with z = b[c] + sum_r wt[r, c] low[t, r], low = R columns of `in` from col on; `wt` is the
// projection transposed, [R, C].  A block takes ROWS rows and 256 channels: a weight is read once for all of its rows.
// (the two-byte builds take the hardware's 32-bit exponential and logarithm: off by units of the last place of a decay)
__device__ __forceinline__ float key_decay_of(float z, float inv_tau) {
#ifdef MS_ELEM_HALF
    const float sp = z < -20.f ? -z : __logf(1.0f + __expf(-z));
    return __expf(-inv_tau * sp);
#else
    return expf(-inv_tau * softplus_f(-z));
#endif
}

template <int ROWS>
__global__ __launch_bounds__(256) void key_decay_kernel(Sums in, int col, const float* __restrict__ wt, const float* __restrict__ b,
                                                        float inv_tau, float* __restrict__ alpha, int T, int C, int R) {
    extern __shared__ float low[];  // [ROWS][R]
    const int t0 = blockIdx.x * ROWS, c = blockIdx.y * 256 + threadIdx.x;
    const int nr = min(ROWS, T - t0);
    for (int i = threadIdx.x; i < nr * R; i += 256) low[i] = sum_at(in, t0 + i / R, col + i % R);
    __syncthreads();
    if (c >= C) return;
    float acc[ROWS];
    const float bias = b[c];
#pragma unroll
    for (int k = 0; k < ROWS; ++k) acc[k] = bias;
#pragma unroll 8
    for (int r = 0; r < R; ++r) {
        const float w = wt[(size_t)r * C + c];
#pragma unroll
        for (int k = 0; k < ROWS; ++k) acc[k] += w * low[(k < nr ? k : 0) * R + r];
    }
#pragma unroll
    for (int k = 0; k < ROWS; ++k)
        if (k < nr) alpha[(size_t)(t0 + k) * C + c] = key_decay_of(acc[k], inv_tau);
}

// ---- gated linear attention over many rows ---------------------------------------------------------------------
// A thread is a value channel and holds its column of S in registers (DP of them; the rows beyond d stay zero).  Tokens come
// WALK_BATCH at a time through LDS; the next batch's numbers are asked for before the current batch is walked.  seg_len 0: a
// block walks all of a request's rows.  Else, if any request has more than `least` rows, those of more than `whole` are cut into segments (the requests' first ones are the first S blocks,
// cut_segment has the others): LOCAL walks each from zero and leaves what it adds (carry [places, H, d, dvp]) and the product of its decays (cdec [places, H, d]),
// the carry kernel replaces what it adds by the state that comes into it, and the second walk makes the outputs.  The other requests are
// walked by a block each in that launch, whatever comes with them: a row takes 1.27 us of a walk (64 x 128), three kernels over segments 78 us and more (100 rows alone
// 132 us walked, 79 in segments of 32; 64 rows 87 and 78; 60 single rows beside a prompt of 2,000 2,477 and 150) and more than twice the rows' work, which counts where the step's rows fill the
// chip as they are: `least` goes by how many come (us, walked and in segments: 16 requests of 70 rows, 8 heads of 128 x 256, 222 and 280, 32 of 100 314 and 621; 64 of 128, 16 heads of
// 64 x 128, 211 and 401, 16 of 200 258 and 187).  `whole` is less: beside one that is cut a walk stands behind the other two kernels (953 rows and 71, 16 heads of 64 x 128: the last launch
// 109 us with the 71 walked whole, 58 in segments).
// (The lengths are on the device: a step that may hold a request to be cut and holds none pays for two launches that find nothing, 4 us: 64 requests of 17 rows 44 and 48, of 2 rows 17.6 and 23.5.)
constexpr int WALK_BATCH = 8;
struct WalkArgs {
    StateArgs a;
    int seg_len, whole, least;  // (seg_len <= whole <= least)
    float* carry;
    float* cdec;
};
// The place of request s's first segment.  Only requests that are cut have places: such a one has more than `whole` rows, so that the request cut next begins at
// least that many rows further on, which makes up for the last segment's missing rows.  T / seg_len + min(T / whole, S) places hold all of a step's, however many
// single rows come with it (a place for each request beside took 0.3 GB for 512 single rows and a portion of 100, 16 heads of 64 x 128).
__device__ __forceinline__ int carry_base(const WalkArgs& w, int s) {
    const int q0 = w.a.seq_q_start[s];
    return q0 / w.seg_len + min(q0 / w.whole, s);
}

// Whether a request of the step is long enough for requests to be cut; every wave looks for itself, 64 a step.
__device__ __forceinline__ bool step_is_cut(const WalkArgs& w) {
    for (int s0 = threadIdx.x % WAVE; s0 - (int)(threadIdx.x % WAVE) < w.a.S; s0 += WAVE)
        if (__any(s0 < w.a.S && w.a.seq_q_len[s0] > w.least)) return true;
    return false;
}
__device__ __forceinline__ bool is_whole(const WalkArgs& w, int len) { return len <= w.whole || (len <= w.least && !step_is_cut(w)); }

// The requests that are cut, by number; behind the last S.
__device__ __forceinline__ int cut_request(const WalkArgs& w, int number) {
    if (!step_is_cut(w)) return w.a.S;
    const int lane = threadIdx.x % WAVE;
    for (int s0 = 0; s0 < w.a.S; s0 += WAVE) {
        const bool cut = s0 + lane < w.a.S && w.a.seq_q_len[s0 + lane] > w.whole;
        const uint64_t all = __ballot(cut), it = __ballot(cut && __popcll(all & ((1ull << lane) - 1)) == number);
        if (it) return s0 + __builtin_ctzll(it);
        number -= __popcll(all);
    }
    return w.a.S;
}

// Segments of the requests that are cut, by number without gaps, all but the one of each that LOCAL leaves out (the last: nobody needs what it passes on) or that has a block among the first
// S (the first); requests behind the last number are S.  Every wave adds the requests up for itself, 64 a step.  Numbers with gaps, every request's own from its first row / L on, left the blocks that
// walk unevenly over the chip's dies, which blocks go to in turn: 64 requests of 128 rows in segments (16 heads of 64 x 128) 504 us, now 401.
template <bool LOCAL>
__device__ __forceinline__ Piece cut_segment(const WalkArgs& w, int number) {
    if (!step_is_cut(w)) return Piece{w.a.S, 0};
    const int lane = threadIdx.x % WAVE;
    int before = 0;
    for (int s0 = 0; s0 < w.a.S; s0 += WAVE) {
        const int len = s0 + lane < w.a.S ? w.a.seq_q_len[s0 + lane] : 0, own = len > w.whole ? (len - 1) / w.seg_len : 0;
        int upto = own;
#pragma unroll
        for (int o = 1; o < WAVE; o <<= 1) {
            const int v = __shfl_up(upto, o, WAVE);
            if (lane >= o) upto += v;
        }
        const uint64_t behind = __ballot(before + upto > number);
        if (behind) {
            const int at = __builtin_ctzll(behind);
            return Piece{s0 + at, (number - before - __shfl(upto - own, at, WAVE) + (LOCAL ? 0 : 1)) * w.seg_len};
        }
        before += __shfl(upto, WAVE - 1, WAVE);
    }
    return Piece{w.a.S, 0};
}

template <int DP, int NT, bool LOCAL>
__global__ __launch_bounds__(NT) void state_walk_kernel(WalkArgs w) {
    constexpr int TB = WALK_BATCH, NW = NT / 64, KPT = TB * DP / NT;
    const StateArgs& a = w.a;
    __shared__ __align__(16) float qs[LOCAL ? 1 : TB][DP], ks[TB][DP], ws[TB][DP];
    __shared__ float vs[TB][NT], os[LOCAL ? 1 : TB][NT], part[TB][NW];
    // (heads innermost: the blocks that find nothing are the grid's last)
    const int number = blockIdx.x / a.H, h = blockIdx.x - number * a.H, j = threadIdx.x, d = a.d;
    Piece pc{number, 0};
    if (LOCAL) pc = cut_segment<true>(w, number);
    else if (w.seg_len && number >= a.S) pc = cut_segment<false>(w, number - a.S);
    if (pc.s >= a.S) return;  // the same for the whole block
    const int left = a.seq_q_len[pc.s] - pc.first;
    if (left <= 0) return;
    const bool whole = !LOCAL && (w.seg_len == 0 || (number < a.S && is_whole(w, left)));
    const int n = whole ? left : min(left, w.seg_len);
    const bool last = n == left;
    const int q0 = a.seq_q_start[pc.s] + pc.first, kh = h / (a.H / a.G);
    const bool live = j < a.dv;
    const size_t head = (size_t)d * a.dvp;
    float* st = a.state + ((size_t)a.seq_slot[pc.s] * a.H + h) * head + j;
    const size_t at = whole ? 0 : (size_t)(carry_base(w, pc.s) + pc.first / w.seg_len) * a.H + h;
    float* pass = whole ? nullptr : w.carry + at * head + j;
    float S[DP];
    {
        const float* from = whole ? st : pass;
#pragma unroll
        for (int i = 0; i < DP; ++i) S[i] = (!LOCAL && live && i < d) ? from[(size_t)i * a.dvp] : 0.f;
    }
    float pq[LOCAL ? 1 : KPT], pk[KPT], pw[KPT], pv[TB], pg[LOCAL ? 1 : TB];
    const float nw = live ? a.norm[j] : 0.f;
    auto fetch = [&](int j0) {  // tokens j0 .. j0 + TB - 1 (the last one again beyond the end)
        // all of one partial sum's loads go out on one straight path, then the next sum's
#pragma unroll
        for (int u = 0; u < KPT; ++u) {
            const int idx = j + u * NT, b = idx / DP, c = idx % DP;
            const int t = q0 + min(j0 + b, n - 1);
            pw[u] = a.decay[((size_t)t * a.H + h) * d + min(c, d - 1)];
        }
        for (int part_sum = 0; part_sum < a.k.n; ++part_sum) {
            const size_t off = part_sum * a.k.stride;  // (q, k, v and gate are columns of the same rows)
#pragma unroll
            for (int u = 0; u < KPT; ++u) {
                const int idx = j + u * NT, b = idx / DP, c = idx % DP;
                const size_t row = off + (size_t)(q0 + min(j0 + b, n - 1)) * a.k.ld + kh * d + min(c, d - 1);
                const float kv = a.k.p[row + a.k_col];
                pk[u] = part_sum ? pk[u] + kv : kv;
                if (!LOCAL) {
                    const float qv = a.k.p[row + a.q_col];
                    pq[u] = part_sum ? pq[u] + qv : qv;
                }
            }
#pragma unroll
            for (int b = 0; b < TB; ++b) {
                const size_t row = off + (size_t)(q0 + min(j0 + b, n - 1)) * a.k.ld + h * a.dv + (live ? j : 0);
                const float vv = a.k.p[row + a.v_col];
                pv[b] = part_sum ? pv[b] + vv : vv;
                if (!LOCAL) {
                    const float gv = a.k.p[row + a.g_col];
                    pg[b] = part_sum ? pg[b] + gv : gv;
                }
            }
        }
    };
    float prod[LOCAL ? (DP + NT - 1) / NT : 1];  // LOCAL: the product of the decays of key channels j, j + NT, ...
#pragma unroll
    for (int u = 0; u < (LOCAL ? (DP + NT - 1) / NT : 1); ++u) prod[u] = 1.f;
    fetch(0);
    for (int j0 = 0; j0 < n; j0 += TB) {
        const int nb = min(TB, n - j0);
        __syncthreads();  // the batch before has been walked by everyone
#pragma unroll
        for (int u = 0; u < KPT; ++u) {
            const int idx = j + u * NT, b = idx / DP, c = idx % DP;
            const bool in = c < d;
            ks[b][c] = in ? pk[u] : 0.f;
            ws[b][c] = in ? pw[u] : 0.f;
            if (!LOCAL) qs[b][c] = in ? pq[u] * a.q_scale : 0.f;
        }
        float gv[LOCAL ? 1 : TB];
#pragma unroll
        for (int b = 0; b < TB; ++b) {
            vs[b][j] = live ? pv[b] : 0.f;
            if (!LOCAL) gv[b] = pg[b];
        }
        __syncthreads();
        if (j0 + TB < n) fetch(j0 + TB);
        if constexpr (LOCAL) {
#pragma unroll
            for (int u = 0; u < (DP + NT - 1) / NT; ++u) {
                const int c = j + u * NT;
                if (c < DP)
                    for (int b = 0; b < nb; ++b) prod[u] *= ws[b][c];
            }
        }
        // the batch's outputs wait in LDS, each in its thread's own place: their norms are worked out together behind the walk
#pragma unroll 1
        for (int b = 0; b < nb; ++b) {
            const float vj = vs[b][j];
            float o0 = 0.f, o1 = 0.f, o2 = 0.f, o3 = 0.f;  // four chains of sums side by side
#pragma unroll
            for (int i = 0; i < DP; i += 4) {
                const float4 k4 = *reinterpret_cast<const float4*>(&ks[b][i]);
                const float4 w4 = *reinterpret_cast<const float4*>(&ws[b][i]);
                S[i] = fmaf(w4.x, S[i], k4.x * vj);
                S[i + 1] = fmaf(w4.y, S[i + 1], k4.y * vj);
                S[i + 2] = fmaf(w4.z, S[i + 2], k4.z * vj);
                S[i + 3] = fmaf(w4.w, S[i + 3], k4.w * vj);
                if (!LOCAL) {
                    const float4 q4 = *reinterpret_cast<const float4*>(&qs[b][i]);
                    o0 = fmaf(q4.x, S[i], o0);
                    o1 = fmaf(q4.y, S[i + 1], o1);
                    o2 = fmaf(q4.z, S[i + 2], o2);
                    o3 = fmaf(q4.w, S[i + 3], o3);
                }
            }
            if (!LOCAL) os[b][j] = (o0 + o1) + (o2 + o3);
        }
        if constexpr (!LOCAL) {
            float ob[TB], ss[TB];
#pragma unroll
            for (int b = 0; b < TB; ++b) {
                ob[b] = (live && b < nb) ? os[b][j] : 0.f;
                ss[b] = wave_sum(ob[b] * ob[b]);
            }
            if constexpr (NW > 1) {  // the head's other waves
                if ((j & 63) == 0) {
#pragma unroll
                    for (int b = 0; b < TB; ++b) part[b][j >> 6] = ss[b];
                }
                __syncthreads();
#pragma unroll
                for (int b = 0; b < TB; ++b) {
                    ss[b] = part[b][0];
#pragma unroll
                    for (int q = 1; q < NW; ++q) ss[b] += part[b][q];
                }
            }
#pragma unroll
            for (int b = 0; b < TB; ++b) {
                const int t = q0 + j0 + b;
                if (b >= nb) continue;
                if (live) a.out[(size_t)t * a.ld_out + h * a.dv + j] = from_f32<elem_t>(ob[b] / sqrtf(ss[b] / (float)a.dv + a.eps) * nw * silu_f(gv[b]));
                if (h == 0) zero_tail(a, t);
            }
        }
    }
    if (LOCAL) {
#pragma unroll
        for (int u = 0; u < (LOCAL ? (DP + NT - 1) / NT : 1); ++u)
            if (j + u * NT < d) w.cdec[at * d + j + u * NT] = prod[u];
    }
    if (j >= a.dvp) return;  // the columns that fill dv up hold zeros
    if (LOCAL) {
#pragma unroll
        for (int i = 0; i < DP; ++i)
            if (i < d) pass[(size_t)i * a.dvp] = S[i];
    } else if (last) {
#pragma unroll
        for (int i = 0; i < DP; ++i)
            if (i < d) st[(size_t)i * a.dvp] = S[i];
    }
}

// Between the two walks: S_in(next) = diag(product of the segment's decays) S_in + what the segment adds, from the slot's state.  A thread has four neighbouring
// value channels of a row; what CARRY_AHEAD segments add is asked for together (one after the other each was a trip to memory: 64 segments 25 us, now 15).
constexpr int CARRY_AHEAD = 8;
__global__ __launch_bounds__(256) void state_carry_kernel(WalkArgs w) {
    const StateArgs& a = w.a;
    const int s = cut_request(w, blockIdx.x), h = blockIdx.y, idx = (blockIdx.z * 256 + threadIdx.x) * 4, head = a.d * a.dvp;
    if (s >= a.S || idx >= head) return;
    const int i = idx / a.dvp, base = carry_base(w, s);
    const int nseg = (a.seq_q_len[s] + w.seg_len - 1) / w.seg_len;
    f32x4 Sin = *reinterpret_cast<const f32x4*>(a.state + ((size_t)a.seq_slot[s] * a.H + h) * head + idx);
    for (int seg0 = 0; seg0 < nseg; seg0 += CARRY_AHEAD) {
        f32x4 add[CARRY_AHEAD];
        float dec[CARRY_AHEAD];
#pragma unroll
        for (int u = 0; u < CARRY_AHEAD; ++u) {  // (what the last segment would pass on is never written: the one before is read in its place, and not used)
            const size_t at = (size_t)(base + max(min(seg0 + u, nseg - 2), 0)) * a.H + h;
            dec[u] = w.cdec[at * a.d + i];
            add[u] = *reinterpret_cast<const f32x4*>(w.carry + at * head + idx);
        }
#pragma unroll
        for (int u = 0; u < CARRY_AHEAD; ++u) {
            if (seg0 + u >= nseg) break;
            *reinterpret_cast<f32x4*>(w.carry + ((size_t)(base + seg0 + u) * a.H + h) * head + idx) = Sin;
            Sin = dec[u] * Sin + add[u];
        }
    }
}

}  // namespace ms

using namespace ms;

extern "C" int ms_gated_state_max_dim() { return MAX_DIM; }
extern "C" int ms_gated_state_max_rank() { return 1536; }  // eight rows of it lie in LDS

extern "C" int ms_key_decay(const float* in, int n_partials, int ld, int col, const float* wt, const float* b, float tau, float* alpha, int T,
                            int C, int R, hipStream_t stream) {
    MS_REQUIRE(T > 0 && C > 0 && R > 0 && n_partials > 0 && col >= 0 && col + R <= ld, "key decay: T=%d C=%d, %d columns at %d of %d", T, C, R, col, ld);
    MS_REQUIRE(R <= ms_gated_state_max_rank(), "key decay: a bottleneck of %d, at most %d", R, ms_gated_state_max_rank());
    MS_REQUIRE(tau > 0.f && in && wt && b && alpha, "key decay: tau %g, or a buffer is missing", (double)tau);
    const Sums rows{in, n_partials, (size_t)T * ld, ld};
    if (T >= 128)
        hipLaunchKernelGGL(key_decay_kernel<8>, dim3(ceil_div(T, 8), ceil_div(C, 256)), dim3(256), (size_t)8 * R * sizeof(float), stream, rows, col,
                           wt, b, 1.0f / tau, alpha, T, C, R);
    else
        hipLaunchKernelGGL(key_decay_kernel<1>, dim3(T, ceil_div(C, 256)), dim3(256), (size_t)R * sizeof(float), stream, rows, col, wt, b, 1.0f / tau,
                           alpha, T, C, R);
    return check_launch("key decay");
}

// Gated linear attention.  rows: float [n_partials, T, ld] with q [H, d], k [H, d], v [H, dv] and gate [H, dv] at their columns;
// alpha float [T, H * d].  single: every request has one row.  seg_len > 0: requests of more than `whole` rows, if one has more than `least`, in segments side by side with carry
// float [places, H, d, dvp] and cdec float [places, H, d] as workspace, places = T / seg_len + min(T / whole, S) (carry_base).
extern "C" int ms_gated_linear(const float* rows, int n_partials, int ld, int q_col, int k_col, int v_col, int g_col, float q_scale,
                               const float* alpha, const float* norm, float eps, float* state, const int* seq_q_start, const int* seq_q_len,
                               const int* seq_slot, int S, void* out, int ld_out, int T, int H, int d, int dv, int dvp, int single,
                               int seg_len, int whole, int least, float* carry, float* cdec, hipStream_t stream) {
    const Sums in{rows, n_partials, (size_t)T * ld, ld};
    const StateArgs a{in, in, in, q_col, k_col, v_col, q_scale, alpha, nullptr, in, g_col, norm, eps, state, seq_q_start, seq_q_len, seq_slot, S,
                      (elem_t*)out, ld_out, T, H, H, d, dv, dvp};
    MS_REQUIRE(n_partials > 0, "gated linear: no rows");
    if (int rc = check_state(a, "gated linear")) return rc;
    if (single) return launch_step<false>(a, stream);
    MS_REQUIRE(seg_len == 0 || (seg_len > 0 && whole >= seg_len && least >= whole && carry && cdec), "gated linear: segments of %d of requests above %d rows need their workspace", seg_len, whole);
    const WalkArgs w{a, seg_len, whole, least, carry, cdec};
#define MS_WALK(DP, NT, LOCAL, X) hipLaunchKernelGGL((state_walk_kernel<DP, NT, LOCAL>), dim3((unsigned)(X) * H), dim3(NT), 0, stream, w)
#define MS_WALK_N(DP, LOCAL, X)                   \
    do {                                          \
        if (dv <= 64) MS_WALK(DP, 64, LOCAL, X);  \
        else if (dv <= 128) MS_WALK(DP, 128, LOCAL, X); \
        else MS_WALK(DP, 256, LOCAL, X);          \
    } while (0)
#define MS_WALK_D(LOCAL, X)                       \
    do {                                          \
        if (d <= 32) MS_WALK_N(32, LOCAL, X);     \
        else if (d <= 64) MS_WALK_N(64, LOCAL, X); \
        else if (d <= 128) MS_WALK_N(128, LOCAL, X); \
        else MS_WALK_N(256, LOCAL, X);            \
    } while (0)
    if (seg_len == 0) {
        MS_WALK_D(false, S);
        return check_launch("gated linear");
    }
    const int cuts = T / seg_len;  // (a request of n rows has (n - 1) / seg_len of those that are numbered)
    MS_WALK_D(true, cuts);
    if (int rc = check_launch("gated linear, segments from zero")) return rc;
    hipLaunchKernelGGL(state_carry_kernel, dim3(min(S, T / (whole + 1)), H, ceil_div(d * dvp, 1024)), dim3(256), 0, stream, w);
    if (int rc = check_launch("gated linear, states between segments")) return rc;
    MS_WALK_D(false, S + cuts);
#undef MS_WALK_D
#undef MS_WALK_N
#undef MS_WALK
    return check_launch("gated linear, segments");
}
