// The second Mamba layer's recurrence (state-space duality) and the gated norm behind it.
//
// Per request, head h and token t, with x [P] the head's value channels, B and C [N] those of the head's group, all
// behind a convolution (32-bit rows) and SiLU, which is applied here where they are read:
//     dt = softplus(raw_dt[t, h] + dt_bias[h]);   a = exp(-exp(A_log[h]) dt)
//     S <- a S + dt B x^T   (S is N x P, 32-bit, carried in the request's slot);   y = S^T C + D[h] x
// Steps of few rows a request are walked token by token; long portions go in chunks whose sums over tokens and states are
// products on the matrix cores (32-bit operands and sums).  Everything is 32-bit in every build.
#include "recurrence.cuh"

namespace ms {

typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int SSD_TOK = 8;      // tokens whose B, C, dt and decay a walking block holds in LDS at a time
constexpr int SSD_CHUNK = 128;  // most tokens of a chunk
constexpr int SSD_HEADS = 4;    // most heads that a block takes one after the other
constexpr int SSD_PT = 2;       // tiles of 32 value channels that a block takes
constexpr float SSD_NOT_FINITE = 0x1.fffffep127f, SSD_LARGEST = 0x1.fffffcp127f;

struct SsdArgs {
    const float* xbc;      // [T, ld_xbc]: x [H, P], B [G, N], C [G, N] before their SiLU
    int ld_xbc;
    const float* proj;     // [T, ld_proj]: column dt_col + h is head h's raw step size
    int ld_proj, dt_col;
    const float* dt_bias;  // [H]
    const float* a_log;    // [H]
    const float* d_skip;   // [H]
    float* state;          // [slots, H, N, P]
    const int* seq_q_start;
    const int* seq_q_len;
    const int* seq_slot;
    int S;
    float* y;              // [T, H * P]
    int H, P, N, G;
    int chunk;             // tokens of a chunk (0: requests are walked)
    int heads;             // heads of a block, all of one group
    int h0, hw, g0, gw;    // the heads h0 .. h0 + hw that a launch takes, whole groups or part of one, and their groups
    int np, pz;            // states filled up to 64, 128 or 256; blocks of 64 value channels
    // what the chunks' kernels pass on, piece by piece, of the launch's hw heads and gw groups (see ssd_work)
    float* states;         // [pieces, hw, pz, np, 64]: what a chunk adds from zero, then the state that comes into it
    float* x;              // [pieces, hw, pz, 128, 64]: x behind its SiLU; what is not finite as SSD_NOT_FINITE, nothing else as large
    float* odd;            // [pieces, hw, pz, 4]: whether a quarter of those tokens (a wave's) has any such
    float* scores;         // [pieces, gw, 10, 4, 64, 4]: tiles of B C^T on and below the diagonal, as the lanes hold them
    float* c;              // [pieces, gw, 4, np / 8, 64, 4]: C behind its SiLU, as the lanes hold it
    float* cdec;           // [pieces, hw]: the product of a chunk's decays
};

// One request and head, token by token: a thread owns one value channel and keeps its column of the state in registers;
// the tokens' B, C, step sizes and decays come through LDS a few tokens at a time, so every thread reads them as
// broadcasts, four states at once.
template <int NMAX>
__global__ __launch_bounds__(256) void ssd_scan_kernel(SsdArgs a) {
    extern __shared__ __align__(16) float lds[];  // B [TOK, NMAX], C [TOK, NMAX] (zeros beyond N), dt [TOK], decay [TOK]
    float* Bs = lds;
    float* Cs = lds + SSD_TOK * NMAX;
    float* dts = Cs + SSD_TOK * NMAX;
    float* decs = dts + SSD_TOK;
    const int s = blockIdx.x, h = blockIdx.y, p = threadIdx.x;
    const int n_rows = a.seq_q_len[s];
    if (n_rows <= 0) return;  // the same for the whole block
    const int row0 = a.seq_q_start[s], slot = a.seq_slot[s];
    const int g = h / (a.H / a.G);
    const bool live = p < a.P;
    const int inner = a.H * a.P;
    float* st = a.state + ((size_t)slot * a.H + h) * a.N * a.P + p;
    float S[NMAX];
#pragma unroll
    for (int n = 0; n < NMAX; ++n) S[n] = (live && n < a.N) ? st[(size_t)n * a.P] : 0.f;
    const float rate = expf(a.a_log[h]), bias = a.dt_bias[h], skip = a.d_skip[h];
    for (int i = threadIdx.x; i < 2 * SSD_TOK * NMAX; i += blockDim.x) lds[i] = 0.f;  // the columns beyond N stay zeros
    for (int t0 = 0; t0 < n_rows; t0 += SSD_TOK) {
        const int nt = min(SSD_TOK, n_rows - t0);
        float xv[SSD_TOK];
#pragma unroll
        for (int k = 0; k < SSD_TOK; ++k)
            xv[k] = (live && k < nt) ? silu_f(a.xbc[(size_t)(row0 + t0 + k) * a.ld_xbc + h * a.P + p]) : 0.f;
        __syncthreads();  // the tile before has been read
        for (int i = threadIdx.x; i < nt * a.N; i += blockDim.x) {
            const int k = i / a.N, n = i - k * a.N;
            const float* src = a.xbc + (size_t)(row0 + t0 + k) * a.ld_xbc + inner + g * a.N + n;
            Bs[k * NMAX + n] = silu_f(src[0]);
            Cs[k * NMAX + n] = silu_f(src[(size_t)a.G * a.N]);
        }
        if (threadIdx.x < nt) {
            const float dt = softplus_f(a.proj[(size_t)(row0 + t0 + threadIdx.x) * a.ld_proj + a.dt_col + h] + bias);
            dts[threadIdx.x] = dt;
            decs[threadIdx.x] = expf(-rate * dt);
        }
        __syncthreads();
        for (int k = 0; k < nt; ++k) {
            const float dec = decs[k], dx = dts[k] * xv[k];
            const float4* Bk = reinterpret_cast<const float4*>(Bs + k * NMAX);
            const float4* Ck = reinterpret_cast<const float4*>(Cs + k * NMAX);
            float acc0 = 0.f, acc1 = 0.f, acc2 = 0.f, acc3 = 0.f;
#pragma unroll
            for (int n = 0; n < NMAX; n += 4) {
                const float4 b = Bk[n >> 2];
                S[n] = dec * S[n] + dx * b.x;
                S[n + 1] = dec * S[n + 1] + dx * b.y;
                S[n + 2] = dec * S[n + 2] + dx * b.z;
                S[n + 3] = dec * S[n + 3] + dx * b.w;
                const float4 c = Ck[n >> 2];
                acc0 += S[n] * c.x;
                acc1 += S[n + 1] * c.y;
                acc2 += S[n + 2] * c.z;
                acc3 += S[n + 3] * c.w;
            }
            if (live) a.y[(size_t)(row0 + t0 + k) * inner + h * a.P + p] = (acc0 + acc1) + (acc2 + acc3) + skip * xv[k];
        }
    }
    if (live) {
#pragma unroll
        for (int n = 0; n < NMAX; ++n)
            if (n < a.N) st[(size_t)n * a.P] = S[n];
    }
}

// ---- long portions in chunks of up to 128 tokens.  With L_t the sum of the tokens' log decays from the chunk's start,
//     y_t = exp(L_t) S_in^T C_t + sum_{s <= t} (B_s . C_t) exp(L_t - L_s) dt_s x_s + D x_t
//     S_out = exp(L_end) S_in + sum_s exp(L_end - L_s) dt_s B_s x_s^T
// in three kernels: what every chunk adds from zero (and, beside it, the scores B_s . C_t, which a group's heads share), the
// states chained from chunk to chunk, the chunks' outputs.  All products are mfma_f32_32x32x2 (32-bit operands and sums), and a
// product's result is the next one's operand where it lies: B C^T comes with a lane's token t in the column, which is the
// layout the product with x wants its right operand in.
//
// Differences of two sums L are wanted, and a sum over 128 decays can be hundreds while the difference is small: L is
// added up in 64 bits and kept as the sum of two 32-bit numbers, so that L_t - L_s is as exact as one decay is.
//
// A walk is a serial chain of tokens in vector arithmetic (2 us a token with 128 states of 64 channels).  64 such heads, walked in segments
// of 64 tokens side by side before / in chunks: a prompt of 2,048 358 / 150 us, of 256 246 / 53, of 877,
// 585 and 293 at once 351 / 124 (inside the model, operands cold: 71 + 17 + 74 in the three kernels).  The matrix instructions are 53,000 cycles of a SIMD's 120,000 in the last kernel; what is left is
// a block's start (gates, C, scores: 5 us of 18 for a single head), vector instructions (25,000) and memory: 250 MB pass between the kernels.
// Tried: operands straight from memory into registers, every wave with its own SiLU 237 us; one or four heads a block 147 and 162.
//
// Rows of 64 numbers in LDS, unpadded: lanes 32 .. 63 read the row four below that of lanes 0 .. 31, so column p of row r
// lies at p ^ 32 where bit 2 of r is set, and the two halves of a wave read different banks.

// e^x for x <= 0 (what lies below -150 counts as -150): the hardware's 2^p, and the part of x log2(e) that p lost to first order.
__device__ __forceinline__ float exp_near(float x) {
    x = fmaxf(x, -150.0f);
    const float p = x * 0x1.715476p+0f, rest = __builtin_fmaf(x, 0x1.4ae0bep-26f, __builtin_fmaf(x, 0x1.715476p+0f, -p));
    const float e = __builtin_amdgcn_exp2f(p);
    return __builtin_fmaf(e, rest * 0x1.62e430p-1f, e);
}

// Per (chunk, head) in LDS, tokens in order.
struct SsdGates {
    __align__(16) float dt[SSD_HEADS][SSD_CHUNK];  // zeros behind the chunk's rows
    float hi[SSD_HEADS][SSD_CHUNK], lo[SSD_HEADS][SSD_CHUNK];
    float out[SSD_HEADS][SSD_CHUNK];  // dt times the decays behind the token
    float skip[SSD_HEADS];
    __align__(16) float odd[SSD_HEADS][4];  // of the outputs' kernel: SsdArgs::odd
};

// The request's rows that a block of chunk kernels has: false if there are none.
struct SsdRows {
    int s, piece, row0, n, h0, heads, g;
};
__device__ __forceinline__ bool ssd_rows_of(const SsdArgs& a, int head_block, SsdRows& r) {
    r.piece = blockIdx.x;
    const Piece pc = piece_of(r.piece, a.chunk, a.seq_q_start, a.S);
    r.s = pc.s;
    const int left = a.seq_q_len[pc.s] - pc.first;
    if (left <= 0) return false;
    r.n = min(left, a.chunk);
    r.row0 = a.seq_q_start[pc.s] + pc.first;
    const int per = a.hw / a.gw, blocks = ceil_div(per, a.heads), group = head_block / blocks;  // (of the launch)
    const int first = (head_block - group * blocks) * a.heads;
    r.g = a.g0 + group;
    r.h0 = a.h0 + group * per + first;
    r.heads = min(a.heads, per - first);
    return true;
}

// A wave a head: lane l has the tokens 2l and 2l + 1.
__device__ __forceinline__ void ssd_gates(const SsdArgs& a, const SsdRows& r, SsdGates& gates) {
    const int hh = threadIdx.x / WAVE, l = threadIdx.x % WAVE;
    if (hh < r.heads) {
        const int h = r.h0 + hh;
        const float rate = expf(a.a_log[h]), bias = a.dt_bias[h];
        if (l == 0) gates.skip[hh] = a.d_skip[h];
        float dt[2];
        double sum[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const int t = 2 * l + e;
            const float raw = a.proj[(size_t)(r.row0 + min(t, r.n - 1)) * a.ld_proj + a.dt_col + h];
            dt[e] = t < r.n ? softplus_f(raw + bias) : 0.f;
            sum[e] = t < r.n ? (double)fmaxf(-rate * dt[e], -1e30f) : 0.0;  // finite, so that differences are
        }
        double upto = sum[0] + sum[1];
#pragma unroll
        for (int o = 1; o < WAVE; o <<= 1) {
            const double other = __shfl_up(upto, o, WAVE);
            if (l >= o) upto += other;
        }
        const double before = __shfl_up(upto, 1, WAVE);
        const double at[2] = {(l ? before : 0.0) + sum[0], upto}, end = __shfl(upto, WAVE - 1, WAVE);
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const int t = 2 * l + e;
            gates.dt[hh][t] = dt[e];
            gates.hi[hh][t] = (float)at[e];
            gates.lo[hh][t] = (float)(at[e] - (double)(float)at[e]);
            gates.out[hh][t] = dt[e] * exp_near((float)(end - at[e]));
        }
    }
    __syncthreads();
}

__device__ __forceinline__ f32x16 zero16() {
    f32x16 z;
#pragma unroll
    for (int i = 0; i < 16; ++i) z[i] = 0.f;
    return z;
}
// Row of a 32x32 result that register i of a lane holds (its column is lane % 32); also the token that step i of a tile of 32
// tokens stands for in that half of the lanes, where tokens are summed over.
__device__ __forceinline__ int row_of(int i, int half) { return 8 * (i >> 2) + 4 * half + (i & 3); }


// Loads from memory straight into LDS: 64 lanes of 16 bytes, one behind the other from `to` on.
__device__ __forceinline__ void to_lds(const float* from, unsigned to) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(from), "s"(to) : "memory", "m0");
}
template <int LEFT>  // every load is there but the wave's last LEFT
__device__ __forceinline__ void wait_and_meet() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(LEFT) : "memory");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
}

// Number i behind `base` (a chunk's first row, the same for the wave): less than 2^30, so that the place is one 32-bit register.
__device__ __forceinline__ float near(const float* base, unsigned i) { return *reinterpret_cast<const float*>(reinterpret_cast<const char*>(base) + i * 4u); }

// Scores of a chunk's tokens and their C, one group's: a wave has one of the ten tiles of 32 tokens t (columns) by 32 tokens s up to
// them, the diagonal ones write C as well.
constexpr int SSD_TILES = 10, SSD_SCORE_BLOCKS = (SSD_TILES + 3) / 4;
template <int NT>
__device__ __forceinline__ void ssd_scores(const SsdArgs& a, int g, int tile, const SsdRows& r) {
    const int l = threadIdx.x % WAVE, half = l / 32, col = l % 32;
    const int w = tile >= 6 ? 3 : tile >= 3 ? 2 : tile >= 1 ? 1 : 0, st = tile - w * (w + 1) / 2;
    if (tile >= SSD_TILES || 32 * w >= r.n) return;
    const float* rows = a.xbc + (size_t)r.row0 * a.ld_xbc + a.H * a.P + g * a.N;
    const unsigned mine = min(32 * w + col, r.n - 1) * a.ld_xbc + a.G * a.N, row = min(32 * st + col, r.n - 1) * a.ld_xbc;
    float* c_out = a.c + (((size_t)r.piece * a.gw + g - a.g0) * 4 + w) * (a.np / 8) * 256 + 4 * l;
    float* s_out = a.scores + (((size_t)r.piece * a.gw + g - a.g0) * SSD_TILES + tile) * 1024 + 4 * l;
    f32x16 sum = zero16();
    constexpr int PARTS = NT < 4 ? NT : 4;  // 32 states each, asked for at once
#pragma unroll 1
    for (int part0 = 0; part0 < NT; part0 += PARTS) {
        float C[PARTS][16], B[PARTS][16];
#pragma unroll
        for (int e = 0; e < PARTS; ++e)
#pragma unroll
            for (int i = 0; i < 16; ++i) {  // register 4q + i of a part stands for its state 8q + 4 half + i
                const unsigned n = min(32 * (part0 + e) + row_of(i, half), a.N - 1);
                C[e][i] = near(rows, mine + n);
                B[e][i] = near(rows, row + n);
            }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int e = 0; e < PARTS; ++e) {
#pragma unroll
            for (int i = 0; i < 16; ++i) C[e][i] = 32 * (part0 + e) + row_of(i, half) < a.N ? silu_f(C[e][i]) : 0.f;
            if (st == w) {
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    *reinterpret_cast<f32x4*>(c_out + (4 * (part0 + e) + q) * 256) = f32x4{C[e][4 * q], C[e][4 * q + 1], C[e][4 * q + 2], C[e][4 * q + 3]};
            }
            f32x16 acc = zero16();
#pragma unroll
            for (int i = 0; i < 16; ++i) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(silu_f(B[e][i]), C[e][i], acc, 0, 0, 0);
#pragma unroll
            for (int i = 0; i < 16; ++i) sum[i] += acc[i];
        }
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) *reinterpret_cast<f32x4*>(s_out + q * 256) = f32x4{sum[4 * q], sum[4 * q + 1], sum[4 * q + 2], sum[4 * q + 3]};
}

// What a chunk adds to the state, from zero: a wave has 32 of the block's 128 states, B of all the chunk's tokens in registers,
// and goes through the block's heads, whose x the block brings into LDS behind SiLU, step size and the decays to come, and leaves
// in memory without those for the outputs.  The first blocks work out the scores.
template <int NT>
__global__ __launch_bounds__(256, 2) void ssd_chunk_add_kernel(SsdArgs a) {
    __shared__ SsdGates gates;
    __shared__ __align__(16) float xs[SSD_CHUNK * 64];
    SsdRows r;
    const int head_block = (int)blockIdx.y - a.gw * SSD_SCORE_BLOCKS;
    if (!ssd_rows_of(a, max(head_block, 0), r)) return;
    if (head_block < 0) {
        if (blockIdx.z == 0) ssd_scores<NT>(a, a.g0 + blockIdx.y / SSD_SCORE_BLOCKS, __builtin_amdgcn_readfirstlane(blockIdx.y % SSD_SCORE_BLOCKS * 4 + threadIdx.x / WAVE), r);
        return;
    }
    const int pz = blockIdx.z % a.pz, n0 = blockIdx.z / a.pz * 128;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE), l = threadIdx.x % WAVE;
    const bool busy = n0 + w * 32 < a.N;  // the same for the whole wave
    const float* rows = a.xbc + (size_t)r.row0 * a.ld_xbc;
    float B[SSD_CHUNK / 2], x[SSD_CHUNK / 4];
    // a thread's x: one channel of the tokens w + 4k
    auto ask = [&](int h) {
        const unsigned at = h * a.P + min(pz * 64 + l, a.P - 1);
        int now = w;
        asm volatile("" : "+s"(now));  // rows are found anew for each head as well
#pragma unroll
        for (int k = 0; k < SSD_CHUNK / 4; ++k) x[k] = near(rows + (size_t)(unsigned)(min(now + 4 * k, r.n - 1) * a.ld_xbc), at);
    };
    const unsigned at = a.H * a.P + r.g * a.N + min(n0 + w * 32 + l % 32, a.N - 1);
#pragma unroll
    for (int j = 0; j < SSD_CHUNK / 2; ++j) B[j] = near(rows, min(32 * (j / 16) + row_of(j % 16, l / 32), r.n - 1) * a.ld_xbc + at);
    __builtin_amdgcn_sched_barrier(0);
    ask(r.h0);
    ssd_gates(a, r, gates);
    if ((int)threadIdx.x < r.heads && blockIdx.z == 0)
        a.cdec[(size_t)r.piece * a.hw + r.h0 - a.h0 + threadIdx.x] = expf(gates.hi[threadIdx.x][SSD_CHUNK - 1] + gates.lo[threadIdx.x][SSD_CHUNK - 1]);
#pragma unroll
    for (int j = 0; j < SSD_CHUNK / 2; ++j) {
        if (j % 8 == 0) __builtin_amdgcn_sched_barrier(0);
        B[j] = silu_f(B[j]);
    }
    for (int hh = 0; hh < r.heads; ++hh) {
        const int h = r.h0 + hh;
        const size_t at_head = ((size_t)r.piece * a.hw + h - a.h0) * a.pz + pz;
        float* keep = a.x + at_head * SSD_CHUNK * 64;
        const int lane = opaque(l);  // places are worked out for each head anew: kept over the loop they would fill the registers
        bool odd = false;
        __syncthreads();  // the head before has been read
#pragma unroll
        for (int k0 = 0; k0 < SSD_CHUNK / 4; k0 += 8)
            if (4 * k0 < r.n) {
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int k = k0; k < k0 + 8; ++k) {
                    x[k] = silu_f(x[k]);
                    xs[(w + 4 * k) * 64 + (lane ^ (k % 2 * 32))] = x[k] * gates.out[hh][w + 4 * k];
                }
                if (n0 == 0) {  // in the outputs a later token meets a factor of zero: finite, so that its overflow stays out of earlier ones
#pragma unroll
                    for (int k = k0; k < k0 + 8; ++k) {
                        const bool finite = fabsf(x[k]) < INFINITY;
                        odd |= !finite;
                        keep[(w + 4 * k) * 64 + (lane ^ (k % 2 * 32))] = finite ? __builtin_amdgcn_fmed3f(x[k], -SSD_LARGEST, SSD_LARGEST) : SSD_NOT_FINITE;
                    }
                }
            }
        const float any_odd = __ballot(odd) ? 1.f : 0.f;
        if (n0 == 0 && l == 0) a.odd[at_head * 4 + w] = any_odd;
        ask(min(h + 1, r.h0 + r.heads - 1));
        __syncthreads();
        if (!busy) continue;
        const int half = lane / 32, c = lane % 32;
        f32x16 acc[SSD_PT];
#pragma unroll
        for (int pt = 0; pt < SSD_PT; ++pt) acc[pt] = zero16();
#pragma unroll
        for (int st = 0; st < SSD_CHUNK / 32; ++st)
            if (32 * st < r.n) {
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int i = 0; i < 16; ++i)
#pragma unroll
                    for (int pt = 0; pt < SSD_PT; ++pt)
                        acc[pt] = __builtin_amdgcn_mfma_f32_32x32x2f32(B[16 * st + i], xs[(32 * st + row_of(i, half)) * 64 + 32 * (pt ^ half) + c], acc[pt], 0, 0, 0);
            }
        float* out = a.states + (at_head * a.np + n0 + w * 32) * 64;
#pragma unroll
        for (int pt = 0; pt < SSD_PT; ++pt)
#pragma unroll
            for (int i = 0; i < 16; ++i) out[row_of(i, half) * 64 + 32 * (pt ^ half) + c] = acc[pt][i];
    }
}

// S_in(chunk + 1) = (product of the chunk's decays) * S_in(chunk) + what the chunk adds, from the slot's state, which takes
// what comes out of the request's last chunk; zeros in the places of states and channels that are not there.
__global__ __launch_bounds__(256) void ssd_carry_kernel(SsdArgs a) {
    const int s = blockIdx.x, h = a.h0 + blockIdx.y, i = (blockIdx.z * 256 + threadIdx.x) * 4;
    const int n_pieces = ceil_div(a.seq_q_len[s], a.chunk), size = a.pz * a.np * 64;
    if (i >= size || n_pieces <= 0) return;
    const size_t piece0 = piece_base(s, a.chunk, a.seq_q_start), hop = (size_t)a.hw * size;
    const int n = i / 64 % a.np, p = i / (64 * a.np) * 64 + (i % 64 ^ (n & 4) * 8);
    float* slot = a.state + (((size_t)a.seq_slot[s] * a.H + h) * a.N + n) * a.P + p;
    float* at = a.states + (piece0 * a.hw + blockIdx.y) * size + i;
    const float* cd = a.cdec + piece0 * a.hw + blockIdx.y;
    f32x4 Sin;
    bool there[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        there[e] = n < a.N && p + e < a.P;
        Sin[e] = there[e] ? slot[e] : 0.f;
    }
    constexpr int BATCH = 8;  // chunks asked for at a time: the chain itself is one multiply-add a chunk
    for (int k0 = 0; k0 < n_pieces; k0 += BATCH) {
        f32x4 add[BATCH];
        float dec[BATCH];
#pragma unroll
        for (int k = 0; k < BATCH; ++k) {
            const int piece = min(k0 + k, n_pieces - 1);
            add[k] = *reinterpret_cast<const f32x4*>(at + piece * hop);
            dec[k] = cd[(size_t)piece * a.hw];
        }
#pragma unroll
        for (int k = 0; k < BATCH; ++k)
            if (k0 + k < n_pieces) {
                *reinterpret_cast<f32x4*>(at + (k0 + k) * hop) = Sin;
#pragma unroll
                for (int e = 0; e < 4; ++e) Sin[e] = there[e] ? dec[k] * Sin[e] + add[k][e] : 0.f;
            }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e)
        if (there[e]) slot[e] = Sin[e];
}

// A chunk's outputs: a wave has 32 tokens (columns of every product), their C and their scores in registers, and goes through the
// block's heads, whose incoming state and x come straight into LDS: the next head's state while x is multiplied, its x while
// its state is.  Sums of 32 products are made from zero and then added: as exact as the walk.
template <int NT, bool QUADS>
__global__ __launch_bounds__(256, NT <= 4 ? 2 : 1) void ssd_chunk_out_kernel(SsdArgs a) {
    constexpr int NP = NT * 32;
    __shared__ SsdGates gates;
    __shared__ __align__(16) float xs[SSD_CHUNK * 64], ss[NP * 64];
    SsdRows r;
    if (!ssd_rows_of(a, blockIdx.y, r)) return;
    const int l = threadIdx.x % WAVE;
    // wave 3's tokens have four tiles of scores, wave 0's one: every other block the other way round, so that a SIMD with waves of two blocks has both
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE), w = (blockIdx.y & 1) ? 3 - wave : wave;
    const unsigned xs_at = (unsigned)(uintptr_t)(__attribute__((address_space(3))) float*)xs, ss_at = (unsigned)(uintptr_t)(__attribute__((address_space(3))) float*)ss;
    const size_t first = (size_t)r.piece * a.hw * a.pz + blockIdx.z;
    auto ask_state = [&](int h) {
        const float* from = a.states + (first + (size_t)(h - a.h0) * a.pz) * NP * 64 + threadIdx.x * 4;
#pragma unroll
        for (int i = 0; i < NP / 16; ++i) to_lds(from + i * 1024, ss_at + i * 4096 + wave * 1024);
    };
    auto ask_x = [&](int h) {
        const float* from = a.x + (first + (size_t)(h - a.h0) * a.pz) * SSD_CHUNK * 64 + threadIdx.x * 4;
#pragma unroll
        for (int i = 0; i < SSD_CHUNK / 16; ++i) to_lds(from + i * 1024, xs_at + i * 4096 + wave * 1024);
    };
    const bool busy = 32 * w < r.n;  // the same for the whole wave
    float C[NT * 16];
    f32x16 scores[4];
#pragma unroll
    for (int j = 0; j < NT * 16; ++j) C[j] = 0.f;
    {
        const float* c_in = a.c + (((size_t)r.piece * a.gw + r.g - a.g0) * 4 + w) * (NP / 8) * 256 + 4 * l;
        const float* s_in = a.scores + (((size_t)r.piece * a.gw + r.g - a.g0) * SSD_TILES + w * (w + 1) / 2) * 1024 + 4 * l;
        if (busy) {
#pragma unroll
            for (int q = 0; q < NT * 4; ++q) {
                const f32x4 v = *reinterpret_cast<const f32x4*>(c_in + q * 256);
#pragma unroll
                for (int i = 0; i < 4; ++i) C[4 * q + i] = v[i];
            }
        }
#pragma unroll
        for (int st = 0; st < 4; ++st) {
            scores[st] = zero16();
            if (busy && st <= w) {
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const f32x4 v = *reinterpret_cast<const f32x4*>(s_in + st * 1024 + q * 256);
#pragma unroll
                    for (int i = 0; i < 4; ++i) scores[st][4 * q + i] = v[i];
                }
            }
        }
    }
    if ((int)threadIdx.x < 4 * r.heads)
        gates.odd[threadIdx.x / 4][threadIdx.x % 4] = a.odd[(first + (size_t)(r.h0 - a.h0 + threadIdx.x / 4) * a.pz) * 4 + threadIdx.x % 4];
    ssd_gates(a, r, gates);
    // C and the scores have arrived: a wait of the compiler's for them inside the loop would be one for the loads into LDS as well
#pragma unroll
    for (int j = 0; j < NT * 16; ++j) asm volatile("" : "+v"(C[j]));
#pragma unroll
    for (int st = 0; st < 4; ++st) asm volatile("" : "+v"(scores[st]));
    __builtin_amdgcn_sched_barrier(0);
    ask_state(r.h0);
    ask_x(r.h0);
    const int inner = a.H * a.P, p0 = blockIdx.z * 64;
    for (int hh = 0; hh < r.heads; ++hh) {
        const int h = r.h0 + hh, next = min(h + 1, r.h0 + r.heads - 1);
        const int half = opaque(l / 32), c = opaque(l % 32), t = 32 * w + c;  // worked out for each head anew: kept over the loop the places would fill the registers
        f32x16 y[SSD_PT];
#pragma unroll
        for (int pt = 0; pt < SSD_PT; ++pt) y[pt] = zero16();
        wait_and_meet<SSD_CHUNK / 16>();  // the state is there (x, asked for after it, may still come)
        if (busy) {
#pragma unroll
            for (int part = 0; part < NT; ++part) {
                __builtin_amdgcn_sched_barrier(0);
                f32x16 acc[SSD_PT];
#pragma unroll
                for (int pt = 0; pt < SSD_PT; ++pt) acc[pt] = zero16();
#pragma unroll
                for (int i = 0; i < 16; ++i)
#pragma unroll
                    for (int pt = 0; pt < SSD_PT; ++pt)
                        acc[pt] = __builtin_amdgcn_mfma_f32_32x32x2f32(ss[(32 * part + row_of(i, half)) * 64 + 32 * (pt ^ half) + c], C[16 * part + i], acc[pt], 0, 0, 0);
#pragma unroll
                for (int pt = 0; pt < SSD_PT; ++pt)
#pragma unroll
                    for (int i = 0; i < 16; ++i) y[pt][i] += acc[pt][i];
            }
        }
        wait_and_meet<0>();  // x is there, the state has been read
        ask_state(next);
        if (busy) {
            const float hi = gates.hi[hh][t], lo = gates.lo[hh][t], skip = gates.skip[hh];
            const float in = exp_near(hi + lo);
#pragma unroll
            for (int pt = 0; pt < SSD_PT; ++pt)
#pragma unroll
                for (int i = 0; i < 16; ++i) y[pt][i] *= in;
#pragma unroll
            for (int st = 0; st < 4; ++st)
                if (st <= w) {
                    f32x16 acc[SSD_PT];
#pragma unroll
                    for (int pt = 0; pt < SSD_PT; ++pt) acc[pt] = zero16();
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        __builtin_amdgcn_sched_barrier(0);
                        const int s0 = 32 * st + 8 * q + 4 * half;
                        const f32x4 dt4 = *reinterpret_cast<const f32x4*>(&gates.dt[hh][s0]);
                        const f32x4 hi4 = *reinterpret_cast<const f32x4*>(&gates.hi[hh][s0]);
                        const f32x4 lo4 = *reinterpret_cast<const f32x4*>(&gates.lo[hh][s0]);
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            const float d = dt4[i] * exp_near((hi - hi4[i]) + (lo - lo4[i]));
                            float m = scores[st][4 * q + i] * d;
                            if (st == w) m = s0 + i < t ? m : s0 + i == t ? m + skip : 0.f;
#pragma unroll
                            for (int pt = 0; pt < SSD_PT; ++pt)
                                acc[pt] = __builtin_amdgcn_mfma_f32_32x32x2f32(xs[(s0 + i) * 64 + 32 * (pt ^ half) + c], m, acc[pt], 0, 0, 0);
                        }
                    }
#pragma unroll
                    for (int pt = 0; pt < SSD_PT; ++pt)
#pragma unroll
                        for (int i = 0; i < 16; ++i) y[pt][i] += acc[pt][i];
                }
            const f32x4 odd = *reinterpret_cast<const f32x4*>(gates.odd[hh]);
            if (__builtin_amdgcn_readfirstlane((int)(odd[0] + odd[1] + odd[2] + odd[3])) != 0) {  // a channel is not finite from such an x on, as in a walk
                for (int s = 0; s <= min(t, r.n - 1); ++s)
#pragma unroll
                    for (int pt = 0; pt < SSD_PT; ++pt)
#pragma unroll
                        for (int i = 0; i < 16; ++i)
                            if (xs[s * 64 + ((32 * pt + row_of(i, half)) ^ ((s & 4) * 8))] == SSD_NOT_FINITE) y[pt][i] = NAN;
            }
            if (t < r.n) {
                float* out = a.y + (size_t)(r.row0 + t) * inner + h * a.P;
#pragma unroll
                for (int pt = 0; pt < SSD_PT; ++pt)
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const int p = p0 + 32 * pt + row_of(4 * q, half);
                        if constexpr (QUADS) {
                            if (p < a.P) *reinterpret_cast<f32x4*>(out + p) = f32x4{y[pt][4 * q], y[pt][4 * q + 1], y[pt][4 * q + 2], y[pt][4 * q + 3]};
                        } else {
#pragma unroll
                            for (int i = 0; i < 4; ++i)
                                if (p + i < a.P) out[p + i] = y[pt][4 * q + i];
                        }
                    }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();  // x has been read
        __builtin_amdgcn_sched_barrier(0);
        ask_x(next);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // what was asked for behind the last head
}

// out[t, c] = (y[t, c] silu(z[t, c])) / sqrt(mean over c's part of the same squared + eps) * w[c], in the element type;
// the row has `parts` equal parts, each normed by itself; columns n .. ld_out of the output are zeros.
__global__ __launch_bounds__(256) void gated_group_norm_kernel(const float* __restrict__ y, const float* __restrict__ z, int ld_z,
                                                               const float* __restrict__ w, elem_t* __restrict__ out, int ld_out, int n,
                                                               int parts, float eps) {
    __shared__ float scratch[4];
    const int t = blockIdx.x, part = blockIdx.y, m = n / parts, c0 = part * m;
    const float* yr = y + (size_t)t * n + c0;
    const float* zr = z + (size_t)t * ld_z + c0;
    float ss = 0.f;
    for (int c = threadIdx.x; c < m; c += 256) {
        const float v = yr[c] * silu_f(zr[c]);
        ss += v * v;
    }
    ss = block_sum<256>(ss, scratch);
    const float inv = 1.0f / sqrtf(ss / (float)m + eps);
    for (int c = threadIdx.x; c < m; c += 256)
        out[(size_t)t * ld_out + c0 + c] = from_f32<elem_t>(yr[c] * silu_f(zr[c]) * inv * w[c0 + c]);
    if (part == 0)
        for (int c = n + threadIdx.x; c < ld_out; c += 256) out[(size_t)t * ld_out + c] = from_f32<elem_t>(0.f);
}

}  // namespace ms

using namespace ms;

constexpr int SSD_MAX_STATES = 256, SSD_MAX_HEAD = 256;
extern "C" int ms_ssd_max_states() { return SSD_MAX_STATES; }
extern "C" int ms_ssd_max_head() { return SSD_MAX_HEAD; }

static void launch_walk(const SsdArgs& a, hipStream_t stream) {
    const dim3 grid(a.S, a.H), block(ceil_div(a.P, 64) * 64);
#define MS_SSD(NMAX) hipLaunchKernelGGL(ssd_scan_kernel<NMAX>, grid, block, (size_t)(2 * SSD_TOK * NMAX + 2 * SSD_TOK) * sizeof(float), stream, a)
    if (a.N <= 16) MS_SSD(16);
    else if (a.N <= 32) MS_SSD(32);
    else if (a.N <= 64) MS_SSD(64);
    else if (a.N <= 128) MS_SSD(128);
    else MS_SSD(256);
#undef MS_SSD
}

template <int NT>
static int launch_chunks(const SsdArgs& a, int pieces, hipStream_t stream) {
    const int head_blocks = a.gw * ceil_div(a.hw / a.gw, a.heads);
    hipLaunchKernelGGL(ssd_chunk_add_kernel<NT>, dim3(pieces, a.gw * SSD_SCORE_BLOCKS + head_blocks, a.pz * ceil_div(a.N, 128)), dim3(256), 0, stream, a);
    if (int rc = check_launch("ssd_scan, chunks from zero")) return rc;
    hipLaunchKernelGGL(ssd_carry_kernel, dim3(a.S, a.hw, ceil_div(a.pz * a.np * 16, 256)), dim3(256), 0, stream, a);
    if (int rc = check_launch("ssd_scan, states between chunks")) return rc;
    const dim3 grid(pieces, head_blocks, a.pz);
    // four numbers a store where every head's channels start at a multiple of four
    if (a.P % 4 == 0 && (uintptr_t)a.y % 16 == 0) hipLaunchKernelGGL((ssd_chunk_out_kernel<NT, true>), grid, dim3(256), 0, stream, a);
    else hipLaunchKernelGGL((ssd_chunk_out_kernel<NT, false>), grid, dim3(256), 0, stream, a);
    return check_launch("ssd_scan, chunks");
}

// Places of the chunks' parts in their workspace, in floats; every part is a multiple of four.
struct SsdWork {
    size_t states, x, scores, c, odd, cdec, end;
};
static int ssd_states(int N) { return N <= 64 ? 64 : N <= 128 ? 128 : 256; }
static SsdWork ssd_work(int T, int S, int H, int P, int N, int G, int chunk) {
    const size_t pieces = T / chunk + S, np = ssd_states(N), pz = ceil_div(P, 64);
    SsdWork w{};
    w.x = pieces * H * pz * np * 64;
    w.scores = w.x + pieces * H * pz * SSD_CHUNK * 64;
    w.c = w.scores + pieces * G * SSD_TILES * 1024;
    w.odd = w.c + pieces * G * 4 * (np / 8) * 256;
    w.cdec = w.odd + pieces * H * pz * 4;
    w.end = w.cdec + pieces * H;
    return w;
}

// Heads that go through the chunks' kernels at a time (heads are independent, and their groups' scores are worked out by every launch that has heads of
// them): all, or as many whole groups, or of one group as many heads, as a workspace of `floats` and a grid hold, and at least one.
static int ssd_heads_at_a_time(int T, int S, int H, int P, int N, int G, int chunk, size_t floats) {
    constexpr int MOST = 65535;
    const int per = H / G;
    if (ssd_work(T, S, H, P, N, G, chunk).end <= floats && H + SSD_SCORE_BLOCKS * G <= MOST) return H;
    const size_t group = ssd_work(T, S, per, P, N, 1, chunk).end, head = ssd_work(T, S, 2, P, N, 1, chunk).end - ssd_work(T, S, 1, P, N, 1, chunk).end;
    const size_t groups = min(floats / group, (size_t)(MOST / (per + SSD_SCORE_BLOCKS)));
    const auto evenly = [](int all, int most) { return ceil_div(all, ceil_div(all, most)); };
    if (groups >= 1) return evenly(G, (int)min(groups, (size_t)G)) * per;
    const size_t scores = ssd_work(T, S, 1, P, N, 1, chunk).end - head, left = floats > scores ? floats - scores : 0;
    return evenly(per, (int)max(min(left / head, (size_t)min(per, MOST - SSD_SCORE_BLOCKS)), (size_t)1));
}

// floats of a workspace of ms_ssd_scan in chunks: what all heads take, or if that is more than `most`, what as many of them take as need no more (one at least).
extern "C" long ms_ssd_chunk_floats(int T, int S, int H, int P, int N, int G, int chunk, long most) {
    if (T <= 0 || S <= 0 || H <= 0 || P <= 0 || N <= 0 || G <= 0 || H % G || chunk <= 0 || most <= 0) return 0;
    const int heads = ssd_heads_at_a_time(T, S, H, P, N, G, chunk, (size_t)most);
    return (long)ssd_work(T, S, heads, P, N, max(1, heads / (H / G)), chunk).end;
}

// chunk 0: every request's rows in one walk.  Else chunks of that many tokens, numbered as pieces of a step are (T / chunk + S of
// them); `work` is float [work_floats], 16-byte aligned: what ms_ssd_chunk_floats says for any limit.
extern "C" int ms_ssd_scan(const float* xbc, int ld_xbc, const float* proj, int ld_proj, int dt_col, const float* dt_bias, const float* a_log,
                           const float* d_skip, float* state, const int* seq_q_start, const int* seq_q_len, const int* seq_slot, int S, float* y,
                           int T, int H, int P, int N, int G, int chunk, float* work, long work_floats, hipStream_t stream) {
    MS_REQUIRE(T > 0 && S > 0 && H > 0 && G > 0 && H % G == 0, "ssd_scan: %d rows of %d requests, %d heads in %d groups", T, S, H, G);
    MS_REQUIRE(P >= 1 && P <= SSD_MAX_HEAD && N >= 1 && N <= SSD_MAX_STATES, "ssd_scan: heads of %d (at most %d) with %d states (at most %d)", P,
               SSD_MAX_HEAD, N, SSD_MAX_STATES);
    MS_REQUIRE(ld_xbc >= H * P + 2 * G * N && ld_proj >= dt_col + H && dt_col >= 0, "ssd_scan: rows of %d and %d numbers for %d heads", ld_xbc,
               ld_proj, H);
    MS_REQUIRE(H <= 65535, "ssd_scan: %d heads", H);
    SsdArgs a{xbc, ld_xbc, proj, ld_proj, dt_col, dt_bias, a_log, d_skip, state, seq_q_start, seq_q_len, seq_slot, S, y, H, P, N, G};
    if (chunk == 0) {
        launch_walk(a, stream);
        return check_launch("ssd_scan");
    }
    MS_REQUIRE(chunk > 0 && chunk <= SSD_CHUNK && work && (uintptr_t)work % 16 == 0, "ssd_scan: chunks of %d rows (at most %d) or without their workspace",
               chunk, SSD_CHUNK);
    MS_REQUIRE((long)ld_xbc * SSD_CHUNK < (1L << 30), "ssd_scan: rows of %d numbers", ld_xbc);
    const int per = H / G, together = ssd_heads_at_a_time(T, S, H, P, N, G, chunk, (size_t)max(work_floats, 0L));
    const SsdWork at = ssd_work(T, S, together, P, N, max(1, together / per), chunk);
    MS_REQUIRE((size_t)work_floats >= at.end, "ssd_scan: a workspace of %ld numbers, %zu are needed", work_floats, at.end);
    const int pieces = T / chunk + S;
    a.chunk = chunk;
    a.np = ssd_states(N);
    a.pz = ceil_div(P, 64);
    a.states = work + at.states;
    a.x = work + at.x;
    a.scores = work + at.scores;
    a.c = work + at.c;
    a.odd = work + at.odd;
    a.cdec = work + at.cdec;
    for (int h = 0; h < H; h += a.hw) {
        a.h0 = h;
        a.hw = min(together, together >= per ? H - h : per - h % per);
        a.g0 = h / per;
        a.gw = max(1, a.hw / per);
        // a block's heads share its B, C and scores: as many heads as leave two blocks for every CU
        a.heads = 1;
        while (a.heads < SSD_HEADS && (long)pieces * a.hw * a.pz / (2 * a.heads) >= 2 * compute_units()) a.heads *= 2;
        if (int rc = a.np == 64 ? launch_chunks<2>(a, pieces, stream) : a.np == 128 ? launch_chunks<4>(a, pieces, stream) : launch_chunks<8>(a, pieces, stream))
            return rc;
    }
    return 0;
}

extern "C" int ms_gated_group_norm(const float* y, const float* z, int ld_z, const float* w, void* out, int ld_out, int T, int n, int parts,
                                   float eps, hipStream_t stream) {
    MS_REQUIRE(T > 0 && n > 0 && parts >= 1 && n % parts == 0 && ld_out >= n && ld_z >= n, "gated_group_norm: %d rows of %d in %d parts", T, n, parts);
    MS_REQUIRE(parts <= 65535, "gated_group_norm: %d parts", parts);
    hipLaunchKernelGGL(gated_group_norm_kernel, dim3(T, parts), dim3(256), 0, stream, y, z, ld_z, w, (elem_t*)out, ld_out, n, parts, eps);
    return check_launch("gated_group_norm");
}
