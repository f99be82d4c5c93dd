// Causal grouped-query attention of a mixed batch over a paged cache, on the matrix cores.
//
// Role in the reference: attn_paged_tiled_*_gqa and *_gqa_runs
// (crates/mach-model/src/kernels.rs:1367-1496, 1650-1885): K/V tiles staged in LDS and
// shared by the query heads of one KV head, online softmax with
// m' = max(m, tile_max), acc = acc * exp(m - m') + sum exp(s - m') V.
//
// One block = 64 "flat rows" of one request and one KV head.  Flat row r of a request is
// (token r / g, query head kvh * g + r % g), g = heads per KV head: a prompt portion of n
// tokens has n * g rows, a decoded token g rows, and any g works the same way.  Each of the
// four waves owns 16 flat rows.  Scores are computed transposed, S^T = K Q^T, so that a lane
// holds four consecutive keys of one query row: row maxima and sums stay in the lane (plus
// two cross-lane steps), and the probabilities are already laid out as the B operand of
// O^T = V^T P^T.  V is stored transposed in its pages ([head_dim][page_size]) so that V^T
// tiles load with contiguous 16-byte reads.
//
// Key tiles start at absolute multiples of BKV from key 0, whatever the portion, so a
// row's result does not depend on how its request was cut into steps.
//
// Compiled once per MS_ATTN_ND (tile head size / 16); a smaller head size runs in the next
// larger tile with the unused columns zero.
#include <algorithm>
#include <mutex>
#include <type_traits>

#include "common.cuh"
#include "no_alloc.h"

#ifndef MS_ATTN_ND
#error "MS_ATTN_ND: head-size tile in units of 16"
#endif

namespace ms {

constexpr int ND = MS_ATTN_ND;
constexpr int HDT = ND * 16;             // head size of the tile
constexpr int NKS = (HDT + 31) / 32;     // K steps of 32 over the head size
#ifdef MS_ELEM_HALF
constexpr int BKV = ND <= 8 ? 64 : 32;
constexpr int EPC = 8;
// LDS has 64 banks of 4 bytes: the 16-byte reads of K fragments (row l % 16, chunk l / 16) are free of
// conflicts at a row pitch of 32 modulo 64 bytes, the 8-byte reads of V^T fragments at 16 modulo 32.
constexpr int KPAD = (ND * 16 * 2) % 64 == 0 ? 16 : 0, VPAD = 8;
#else
constexpr int BKV = ND <= 4 ? 64 : (ND <= 8 ? 32 : 16);
constexpr int EPC = 4;
constexpr int KPAD = 4, VPAD = 4;
#endif
constexpr int NT = BKV / 16;             // 16-key score tiles per key tile
constexpr int NTP = (NT + 1) / 2;        // pairs of score tiles = K steps of the PV product
constexpr int K_LD = HDT + KPAD, V_LD = BKV + VPAD;
// Flat rows of a work item (two-byte elements and a head size of 64: two blocks of 64 rows share an item).
#if defined(MS_ELEM_HALF) && (MS_ATTN_ND == 4 || MS_ATTN_ND == 8)
#define MS_HAS_ROWS32 1
#endif
#if defined(MS_ELEM_HALF) && MS_ATTN_ND == 4
constexpr int ROWS_PER_BLOCK = 128;
#else
constexpr int ROWS_PER_BLOCK = 64;
#endif
constexpr int SUB_BLOCKS = ROWS_PER_BLOCK / 64;  // blocks of the general kernel per work item
constexpr float NEG_BIG = -1e30f;
#ifdef MS_ELEM_HALF
constexpr int MAX_KEY_GROUPS = ND <= 4 ? 4 : 2;  // groups of four waves that may share a block's keys
#else
constexpr int MAX_KEY_GROUPS = 2;
#endif

struct AttnArgs {
    const elem_t* q;         // [T, H, hd]
    const elem_t* kpool;     // [pages, KV, ps, hd]
    const elem_t* vpool;     // [pages, KV, hd, ps]
    elem_t* out;             // [T, H * hd]
    const int* block_table;  // [S, table_stride]
    const int* seq_q_start;  // [S] first row of the request in this step
    const int* seq_q_len;    // [S] rows of the request in this step
    const int* seq_pos0;     // [S] position of its first row
    const int* work;         // [W, 2] (request index, first flat row), best with the longest contexts first
    int table_stride, H, KV, hd, ps, window;
    float scale;
    int n_work;     // W
    int pair_span;  // work items per round of blocks over the chip when two blocks share a CU, else 0
    // the keys of a block cut over gridDim.y blocks (few blocks of rows, long contexts): each writes
    // its unnormalised output and (max, sum) per row, and decode_merge_kernel adds them up
    int nsplit;
    float* part_o;   // [T, H, nsplit, hd]
    float* part_ml;  // [T, H, nsplit, 2]
    // [H] or null: a softmax sink per head, an extra term exp(sink) of the denominator, to which no key or value belongs
    // (natural-logarithm units of the scaled scores)
    const float* sinks;
    // [T, H] or null: what the output of (row, head) is multiplied by (a gate), in the same pass as the softmax's division
    const float* out_gate;
    // chunk > 0: a row at position p sees only the keys from floor(p / chunk) * chunk on (chunks counted from the
    // request's position 0), beside whatever the window leaves
    int chunk;
    // softcap > 0: the scaled score s becomes softcap * tanh(s / softcap) before the softmax
    float softcap;
    // tiles of 32 rows: the reference of a row's exponentials follows its maximum when that has risen by more (in powers of two)
    float rise;
    // what the kernels behind this one will read from memory (weights), in units of 16 bytes: blocks from `n_blocks` on bring it into the last-level cache
    int n_blocks;
    uint32_t n_ahead[2];
    const u32x4* ahead[2];
};

// A block beside the attention's own: its share of the bytes that are read ahead.  An attention over a prompt is bound by its instructions and leaves the memory idle, and
// products in tiles whose weights are in the last-level cache take less of a layer than with weights from memory (the loads of cold weights bound
// their loops): 2,048 rows, us, 896 x 4,864 in slices 26.6 and 20.5, 9,728 x 896 gated 36.8 and 32.5, 1,536 x 8,960 80 and 58, 2,048 x 2,048 22.8 and 18.6.
__device__ __forceinline__ void read_ahead(const AttnArgs& a, int block, int blocks) {
    constexpr uint32_t AT_ONCE = 16;
    u32x4 seen = {0u, 0u, 0u, 0u};
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        const uint32_t n = a.n_ahead[r], turn = blockDim.x * AT_ONCE;
        for (uint32_t at = (uint32_t)block * turn + threadIdx.x; at < n; at += (uint32_t)blocks * turn) {
            u32x4 v[AT_ONCE];
#pragma unroll
            for (uint32_t u = 0; u < AT_ONCE; ++u) v[u] = a.ahead[r][min(at + u * blockDim.x, n - 1)];
#pragma unroll
            for (uint32_t u = 0; u < AT_ONCE; ++u) seen ^= v[u];
        }
    }
    asm volatile("" ::"v"(seen));
}

// The first key a row at `pos` sees under a window and a chunked mask (either 0: none).
__device__ __forceinline__ int first_visible_key(int pos, int window, int chunk) {
    int lo = window > 0 ? pos - window + 1 : 0;
    if (chunk > 0) lo = max(lo, pos / chunk * chunk);
    return lo;
}

// A raw score under the cap, still in the units that the softmax's scale multiplies: scale * result = cap * tanh(scale * s / cap).
__device__ __forceinline__ float capped_raw(float s, float scale, float softcap) {
    return softcap / scale * tanhf(s * (scale / softcap));
}

__device__ __forceinline__ float exp_f(float x) {
#ifdef MS_ELEM_HALF
    return __expf(x);
#else
    return expf(x);
#endif
}

__device__ __forceinline__ float exp2_f(float x) {
#ifdef MS_ELEM_HALF
    return __builtin_amdgcn_exp2f(x);
#else
    return exp2f(x);
#endif
}

// What a row's unnormalised output is multiplied by at the end: 1 / l, or with a sink 1 / (l + exp(sink - m)), for a
// running sum l taken relative to the maximum m (scaled scores, natural logarithm); a row without keys gives 0.
// `gate`, if given, is the factor of this (row, head) on top of that.
__device__ __forceinline__ float softmax_norm(float m, float l, const float* __restrict__ sinks, int head,
                                              const float* __restrict__ gate, size_t row_head) {
    const float g = gate ? gate[row_head] : 1.0f;
    if (sinks == nullptr) return l > 0.f ? g / l : 0.f;
    const float sk = sinks[head], top = fmaxf(m, sk);
    const float c = l > 0.f ? exp_f(m - top) : 0.f;
    return g * c / (l * c + exp_f(sk - top));
}

// KG "key groups" of four waves each share a block: group kg takes the key tiles whose absolute
// index is kg modulo KG, with its own staging buffers, and the groups' running (max, sum, output)
// are merged through LDS at the end.  A block's time is the length of its serial chain of tiles,
// and a causal prompt's last rows see every key: more groups cut that chain.
// Waves per SIMD the compiler has to leave room for: with the small bfloat16 tiles two blocks of a CU
// overlap one's LDS traffic with the other's arithmetic, if the registers allow them.
#ifdef MS_ELEM_HALF
template <int KG> constexpr int attention_waves_per_simd() { return ND <= 4 ? (KG == 1 ? 3 : 4) : 1; }
#else
template <int KG> constexpr int attention_waves_per_simd() { return 1; }
#endif

template <int KG>
__global__ __launch_bounds__(256 * KG, attention_waves_per_simd<KG>()) void paged_attention_kernel(AttnArgs a) {
    if (a.n_blocks > 0 && (int)blockIdx.x >= a.n_blocks) {
        if (blockIdx.y == 0) read_ahead(a, blockIdx.x - a.n_blocks, gridDim.x - a.n_blocks);
        return;
    }
    constexpr int KS_ELEMS = BKV * K_LD, VS_ELEMS = HDT * V_LD;
    constexpr int STAGE_BYTES = (KS_ELEMS + VS_ELEMS) * (int)sizeof(elem_t);
    constexpr int MERGE_FLOATS = 4 * 64 * (4 * ND + 2);  // per group: four waves, per lane the output and (max, sum)
    // two stages per group: a tile is multiplied out of one while the next is written into the other
    constexpr int SMEM_BYTES = 2 * KG * STAGE_BYTES > (KG - 1) * MERGE_FLOATS * 4 ? 2 * KG * STAGE_BYTES : (KG - 1) * MERGE_FLOATS * 4;
    static_assert(SMEM_BYTES <= 160 * 1024, "the tiles of a block exceed the LDS of a CU");
    __shared__ __attribute__((aligned(16))) unsigned char smem[SMEM_BYTES];

    const int kg = threadIdx.x >> 8, tid = threadIdx.x & 255, lane = tid & 63, wave = tid >> 6;
    auto stage_k = [&](int b) { return reinterpret_cast<elem_t*>(smem + (2 * kg + b) * STAGE_BYTES); };
    auto stage_v = [&](int b) { return stage_k(b) + KS_ELEMS; };
    const int r16 = lane & 15, grp = lane >> 4;
    // Blocks are numbered item by item, the KV heads of an item side by side.  A block's work grows
    // with its context, and blocks go to the CUs in turn: with two blocks a CU, block b shares its
    // CU with block b + (number of CUs).  So the list's heaviest `pair_span` items come first, then
    // its lightest ones, lightest first (each beside one of the heaviest), then the middle.
    // (a work item of ROWS_PER_BLOCK rows is SUB_BLOCKS blocks of 64 rows here, side by side)
    const int kvh = blockIdx.x % a.KV, sub = (blockIdx.x / a.KV) % SUB_BLOCKS, turn = blockIdx.x / (a.KV * SUB_BLOCKS);
    int item = turn;
    if (a.pair_span > 0 && turn >= a.pair_span)
        item = turn < 2 * a.pair_span ? a.n_work - 1 - (turn - a.pair_span) : turn - a.pair_span;
    const int s = a.work[item * 2], r0 = a.work[item * 2 + 1] + 64 * sub;
    if (s < 0) return;  // an item that only fills the list up to a size that many steps share (the same for the whole block)
    const int g = a.H / a.KV;
    const int q_start = a.seq_q_start[s], q_len = a.seq_q_len[s], pos0 = a.seq_pos0[s];
    const int R = q_len * g;
    if (r0 >= R) return;  // the item's rows end in the block beside this one (the same for the whole block)
    const int hd = a.hd, ps = a.ps;
    const int* table = a.block_table + (size_t)s * a.table_stride;

    // this lane's query row
    const int row = r0 + wave * 16 + r16;
    const bool valid = row < R;
    const int tok = valid ? row / g : 0;
    const int head = kvh * g + (valid ? row % g : 0);
    const int pos = pos0 + tok;
    const bool wave_active = r0 + wave * 16 < R;

    // keys any row of the block may see, and of those the rounds of tiles that are this split's
    constexpr int ROUND = KG * BKV;  // keys per round of the block
    const int last_row = min(r0 + 64, R) - 1;
    int kv_hi = pos0 + last_row / g + 1;
    int kv_lo = 0;
    if (a.window > 0 || a.chunk > 0) kv_lo = max(0, first_visible_key(pos0 + r0 / g, a.window, a.chunk));
    const int lo_key = first_visible_key(pos, a.window, a.chunk);
    const int sp = blockIdx.y;
    if (a.nsplit > 1) {
        const int first = (kv_lo / ROUND) * ROUND;
        const int per = ceil_div(ceil_div(kv_hi - first, ROUND), a.nsplit) * ROUND;
        kv_lo = max(kv_lo, first + sp * per);
        kv_hi = min(kv_hi, first + (sp + 1) * per);
    }
    // a row's partial result of this split (group 0 writes, after the groups have been merged)
    auto write_partial = [&](const f32x4* o, float m, float l) {
        const size_t base = (((size_t)(q_start + tok)) * a.H + head) * a.nsplit + sp;
        float* po = a.part_o + base * hd;
#pragma unroll
        for (int dt = 0; dt < ND; ++dt) {
            const int d0 = dt * 16 + grp * 4;
            if (d0 < hd) {
#pragma unroll
                for (int i = 0; i < 4; ++i) po[d0 + i] = o[dt][i];
            }
        }
        // the merge takes maxima in natural-logarithm units of the scaled scores
        if (grp == 0) { a.part_ml[base * 2] = m * a.scale; a.part_ml[base * 2 + 1] = l; }
    };
    if (kv_lo >= kv_hi) {  // nothing for this split (the same for every thread of the block)
        if (a.nsplit > 1 && threadIdx.x < 256 && valid) {
            f32x4 zero[ND];
#pragma unroll
            for (int dt = 0; dt < ND; ++dt) zero[dt] = (f32x4){0.f, 0.f, 0.f, 0.f};
            write_partial(zero, NEG_BIG, 0.f);
        }
        return;
    }

    Frag qf[NKS];
    {
        const elem_t* qrow = a.q + ((size_t)(q_start + tok) * a.H + head) * hd;
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks) {
            const int d0 = ks * 32 + grp * 8;
            qf[ks] = (valid && d0 < hd) ? frag_load(qrow + d0) : frag_zero();
        }
    }

    f32x4 acc_o[ND];
#pragma unroll
    for (int i = 0; i < ND; ++i) acc_o[i] = (f32x4){0.f, 0.f, 0.f, 0.f};
    // running maximum in units of the raw score; exponentials are taken in base 2 with the scale
    // folded in: exp(scale * (s - m)) = exp2(s * sl - m * sl)
    float m_run = NEG_BIG, l_run = 0.f;
    const float sl = a.scale * 1.4426950408889634f;

    // Tiles go global -> registers -> LDS.  PF tiles per group are in flight at any time: a tile's
    // loads are requested PF rounds before it is multiplied, which covers the memory latency even
    // when few blocks share a CU.  Where a tile's 16-key groups lie in the pools is looked up once
    // per tile by NT threads and shared through LDS (offsets in units of 16 elements).
    constexpr int CPRK = HDT / EPC, CPRV = BKV / EPC;
    constexpr int NCK = (BKV * CPRK + 255) / 256, NCV = (HDT * CPRV + 255) / 256;
    constexpr int PF = KG == 1 ? (ND <= 4 ? 4 : (ND <= 8 ? 2 : 1)) : (ND <= 8 ? 2 : 1);
    constexpr unsigned ABSENT = 0xffffffffu;
    __shared__ unsigned kofs[KG][PF][NT], vofs[KG][PF][NT];
    u32x4 rk[PF][NCK], rv[PF][NCV];
    // what does not change from tile to tile: where in a 16-key group this thread's chunks lie (an
    // unused chunk, beyond the head size or the tile, reads the start of the pool)
    const elem_t* k_base[NCK];
    const elem_t* v_base[NCV];
    bool k_on[NCK], v_on[NCV];
#pragma unroll
    for (int i = 0; i < NCK; ++i) {
        const int c = tid + i * 256, kl = c / CPRK, d0 = (c % CPRK) * EPC;
        k_on[i] = c < BKV * CPRK && d0 < hd;
        k_base[i] = a.kpool + (k_on[i] ? (kl % 16) * hd + d0 : 0);
    }
#pragma unroll
    for (int i = 0; i < NCV; ++i) {
        const int c = tid + i * 256, d = c / CPRV, k0 = (c % CPRV) * EPC;
        v_on[i] = c < HDT * CPRV && d < hd;
        v_base[i] = a.vpool + (v_on[i] ? d * ps + (k0 % 16) : 0);
    }
    // Every load below is unconditional (an absent or unused chunk reads the start of the pool and is
    // zeroed when it is stored to LDS, PF rounds later): with loads on one straight path, and no use
    // of the loaded values before that, the compiler counts the loads and waits only for the tile it
    // is about to use, and the younger tiles stay in flight.  The page of a tile's 16-key group is
    // read one round before its offsets are needed; which logical page that is, is stepped from
    // round to round rather than divided out.
    const int tsub = tid % NT;
    const int round_pages = ROUND / ps, round_rem = ROUND % ps;
    int key_next, lp_next, off_next;  // this thread's 16-key group of the next tile to look up
    auto start_lookup = [&](int kt0) {
        key_next = kt0 + tsub * 16;
        lp_next = key_next / ps;
        off_next = key_next % ps;
    };
    struct Entry { int page, off; };
    auto lookup = [&]() {  // page (or -1) and offset in it of the group; moves on by one round
        Entry e{table[min(lp_next, a.table_stride - 1)] | (key_next < kv_hi ? 0 : -1), off_next};
        key_next += ROUND;
        lp_next += round_pages;
        off_next += round_rem;
        if (off_next >= ps) {
            off_next -= ps;
            ++lp_next;
        }
        return e;
    };
    auto fill_offsets = [&](int slot, Entry e) {
        if (tid < NT) {
            const size_t pk = (size_t)max(e.page, 0) * a.KV + kvh;
            kofs[kg][slot][tid] = e.page >= 0 ? (unsigned)(((pk * ps + e.off) * hd) >> 4) : ABSENT;
            vofs[kg][slot][tid] = e.page >= 0 ? (unsigned)((pk * hd * ps + e.off) >> 4) : ABSENT;
        }
    };
    unsigned live[PF];  // bit i: chunk i of the slot's tile was really read (K chunks first, then V)
    auto load_tile = [&](int slot, u32x4* pk, u32x4* pv) {
        unsigned bits = 0;
#pragma unroll
        for (int i = 0; i < NCK; ++i) {
            const int kl = (tid + i * 256) / CPRK;
            const unsigned o = kofs[kg][slot][(kl / 16) % NT];
            const bool on = k_on[i] && o != ABSENT;
            pk[i] = *reinterpret_cast<const u32x4*>(k_base[i] + ((size_t)(on ? o : 0u) << 4));
            bits |= (on ? 1u : 0u) << i;
        }
#pragma unroll
        for (int i = 0; i < NCV; ++i) {
            const int k0 = ((tid + i * 256) % CPRV) * EPC;
            const unsigned o = vofs[kg][slot][(k0 / 16) % NT];
            const bool on = v_on[i] && o != ABSENT;
            pv[i] = *reinterpret_cast<const u32x4*>(v_base[i] + ((size_t)(on ? o : 0u) << 4));
            bits |= (on ? 1u : 0u) << (NCK + i);
        }
        live[slot] = bits;
    };
    auto store_tile = [&](int slot, int b, const u32x4* pk, const u32x4* pv) {
        elem_t* Ks = stage_k(b);
        elem_t* Vs = stage_v(b);
        const unsigned bits = live[slot];
        // nearly always every chunk of every thread was really read: then nothing is masked
        if (__all(bits == (1u << (NCK + NCV)) - 1)) {
#pragma unroll
            for (int i = 0; i < NCK; ++i) {
                const int c = tid + i * 256;
                if (c < BKV * CPRK) *reinterpret_cast<u32x4*>(&Ks[(c / CPRK) * K_LD + (c % CPRK) * EPC]) = pk[i];
            }
#pragma unroll
            for (int i = 0; i < NCV; ++i) {
                const int c = tid + i * 256;
                if (c < HDT * CPRV) *reinterpret_cast<u32x4*>(&Vs[(c / CPRV) * V_LD + (c % CPRV) * EPC]) = pv[i];
            }
            return;
        }
#pragma unroll
        for (int i = 0; i < NCK; ++i) {
            const int c = tid + i * 256;
            const unsigned keep = (bits >> i & 1) ? 0xffffffffu : 0u;
            if (c < BKV * CPRK)
                *reinterpret_cast<u32x4*>(&Ks[(c / CPRK) * K_LD + (c % CPRK) * EPC]) = pk[i] & (u32x4){keep, keep, keep, keep};
        }
#pragma unroll
        for (int i = 0; i < NCV; ++i) {
            const int c = tid + i * 256;
            const unsigned keep = (bits >> (NCK + i) & 1) ? 0xffffffffu : 0u;
            if (c < HDT * CPRV)
                *reinterpret_cast<u32x4*>(&Vs[(c / CPRV) * V_LD + (c % CPRV) * EPC]) = pv[i] & (u32x4){keep, keep, keep, keep};
        }
    };
    // rows of this wave: the first and the last position decide which tiles need no mask at all
    const int pos_first = pos0 + (r0 + wave * 16) / g;
    const int pos_last = pos0 + min(r0 + wave * 16 + 15, max(R - 1, 0)) / g;
    const int lo_last = first_visible_key(pos_last, a.window, a.chunk);

    // Round r: group kg has the tile of absolute index round_first * KG + r * KG + kg.  Its loads are
    // asked for PF rounds ahead into register slot r % PF, it is written into LDS stage r % 2 while
    // round r - 1 is multiplied out of the other stage, and one barrier a round separates the two.
    const int kt_first = (kv_lo / ROUND) * ROUND;
    start_lookup(kt_first + kg * BKV);
#pragma unroll
    for (int j = 0; j < PF; ++j) fill_offsets(j, lookup());
    Entry ahead = lookup();
    __syncthreads();
#pragma unroll
    for (int j = 0; j < PF; ++j) load_tile(j, rk[j], rv[j]);
    __syncthreads();  // slot 0's offsets have been read by everyone
    fill_offsets(0, ahead);  // of round PF, which the first round asks for
    ahead = lookup();
    store_tile(0, 0, rk[0], rv[0]);
    __syncthreads();
    constexpr int UNROLL = PF > 2 ? PF : 2;
    for (int kt_base = kt_first; kt_base < kv_hi; kt_base += UNROLL * ROUND) {
#pragma unroll
      for (int u = 0; u < UNROLL; ++u) {
        if (kt_base + u * ROUND >= kv_hi) break;  // the same for every thread of the block
        const int j = u % PF, jn = (u + 1) % PF, b = u & 1;
        const int kt0 = kt_base + u * ROUND + kg * BKV;
        const elem_t* Ks = stage_k(b);
        const elem_t* Vs = stage_v(b);
        load_tile(j, rk[j], rv[j]);  // round r + PF into the slot that round r left
        const bool busy = wave_active && kt0 < kv_hi;

        // S^T = K Q^T: lane holds keys grp * 4 + i of tile nt for query row r16
        f32x4 sc[NT];
        if (busy) {
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                sc[nt] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int ks = 0; ks < NKS; ++ks) {
                    const int d0 = ks * 32 + grp * 8;
                    Frag kf = (d0 < HDT) ? frag_load(&Ks[(nt * 16 + r16) * K_LD + d0]) : frag_zero();
                    mma_16x16x32(sc[nt], kf, qf[ks]);
                }
            }
        }
        // the next round's tile goes into the other stage, which the round before this one has left
        if (kt_base + (u + 1) * ROUND < kv_hi) {
            store_tile(jn, b ^ 1, rk[jn], rv[jn]);
            fill_offsets(jn, ahead);
            ahead = lookup();
        }
        if (busy) {
        if (a.softcap > 0.f) {
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                for (int i = 0; i < 4; ++i) sc[nt][i] = capped_raw(sc[nt][i], a.scale, a.softcap);
        }
        // a tile that every row of the wave sees whole needs no mask
        const bool whole = kt0 + BKV - 1 <= pos_first && kt0 >= lo_last;
        float tmax = NEG_BIG;
        if (whole) {
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                for (int i = 0; i < 4; ++i) tmax = fmaxf(tmax, sc[nt][i]);
        } else {
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int key = kt0 + nt * 16 + grp * 4 + i;
                    const bool ok = valid && key <= pos && key >= lo_key;
                    const float v = ok ? sc[nt][i] : -INFINITY;
                    sc[nt][i] = v;
                    tmax = fmaxf(tmax, v);
                }
        }
        tmax = fmaxf(tmax, __shfl_xor(tmax, 16, WAVE));
        tmax = fmaxf(tmax, __shfl_xor(tmax, 32, WAVE));
        const float m_new = fmaxf(m_run, tmax);
        const float mb = m_new * sl;
        float psum = 0.f;
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float p = exp2_f(fmaf(sc[nt][i], sl, -mb));
                sc[nt][i] = p;
                psum += p;
            }
        psum += __shfl_xor(psum, 16, WAVE);
        psum += __shfl_xor(psum, 32, WAVE);
        // where no row's maximum rose the factor is exactly one: after the first tiles that is the rule
        if (__any(m_new > m_run)) {
            const float alpha = exp2_f((m_run - m_new) * sl);
            l_run *= alpha;
#pragma unroll
            for (int dt = 0; dt < ND; ++dt)
#pragma unroll
                for (int i = 0; i < 4; ++i) acc_o[dt][i] *= alpha;
        }
        l_run += psum;
        m_run = m_new;

        // O^T += V^T P^T: the probabilities of two score tiles form one B fragment
#pragma unroll
        for (int pp = 0; pp < NTP; ++pp) {
            Frag pf;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                pf.v[i] = from_f32<elem_t>(sc[2 * pp][i]);
                pf.v[4 + i] = from_f32<elem_t>((2 * pp + 1 < NT) ? sc[(2 * pp + 1) % NT][i] : 0.f);
            }
#pragma unroll
            for (int dt = 0; dt < ND; ++dt) {
                Frag vf;
                const elem_t* v0 = &Vs[(dt * 16 + r16) * V_LD + (2 * pp) * 16 + grp * 4];
#pragma unroll
                for (int i = 0; i < 4; ++i) vf.v[i] = v0[i];
                if (2 * pp + 1 < NT) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) vf.v[4 + i] = v0[16 + i];
                } else {
#pragma unroll
                    for (int i = 0; i < 4; ++i) vf.v[4 + i] = from_f32<elem_t>(0.f);
                }
                mma_16x16x32(acc_o[dt], vf, pf);
            }
        }
        }
        __syncthreads();  // this round's stage has been read, the next round's written
      }
    }

    if constexpr (KG > 1) {
        // groups 1.. hand (output, max, sum) to group 0 through LDS, which adds them in group order
        // (the rounds end with a barrier: the stages are free)
        float* mg = reinterpret_cast<float*>(smem);
        if (kg > 0) {
            float* mine = mg + ((size_t)(kg - 1) * 4 + wave) * 64 * (4 * ND + 2);
#pragma unroll
            for (int dt = 0; dt < ND; ++dt)
#pragma unroll
                for (int i = 0; i < 4; ++i) mine[(dt * 4 + i) * 64 + lane] = acc_o[dt][i];
            mine[(4 * ND) * 64 + lane] = m_run;
            mine[(4 * ND + 1) * 64 + lane] = l_run;
        }
        __syncthreads();
        if (kg > 0) return;
#pragma unroll
        for (int o = 0; o < KG - 1; ++o) {
            const float* other = mg + ((size_t)o * 4 + wave) * 64 * (4 * ND + 2);
            const float m_o = other[(4 * ND) * 64 + lane], l_o = other[(4 * ND + 1) * 64 + lane];
            const float m_new = fmaxf(m_run, m_o);
            const float c0 = exp2_f((m_run - m_new) * sl), c1 = exp2_f((m_o - m_new) * sl);
            l_run = l_run * c0 + l_o * c1;
            m_run = m_new;
#pragma unroll
            for (int dt = 0; dt < ND; ++dt)
#pragma unroll
                for (int i = 0; i < 4; ++i) acc_o[dt][i] = acc_o[dt][i] * c0 + other[(dt * 4 + i) * 64 + lane] * c1;
        }
    }

    if (valid && a.nsplit > 1) {
        write_partial(acc_o, m_run, l_run);
    } else if (valid) {
        const float inv = softmax_norm(m_run * a.scale, l_run, a.sinks, head, a.out_gate, (size_t)(q_start + tok) * a.H + head);
        elem_t* orow = a.out + ((size_t)(q_start + tok) * a.H + head) * hd;
#pragma unroll
        for (int dt = 0; dt < ND; ++dt) {
            const int d0 = dt * 16 + grp * 4;
            if (d0 < hd) {
#pragma unroll
                for (int i = 0; i < 4; ++i) orow[d0 + i] = from_f32<elem_t>(acc_o[dt][i] * inv);
            }
        }
    }
}


// ---------------------------------------------------------------------------------------
// The same attention in tiles of 32 query rows by 32 keys (`mfma_f32_32x32x16`), for the two-byte element
// types and head sizes of 64 and 128.  The counters of the kernel above say that it spends fifteen vector instructions
// on every matrix instruction.  Here a lane holds sixteen keys of one query row (one step across lanes instead of two) and a
// fragment read from LDS feeds twice the arithmetic; tiles go from memory straight into one of two LDS stages, a round before they are multiplied (no
// staging registers, no stores); and the block's share of the block table is copied into LDS once, so that no round waits
// for a page number.  A block is 64 flat rows, two waves of 32 rows under each of two key groups: three blocks (head size
// 64; two with 128) share a CU, where one's exponentials overlap another's products and a causal prompt's long blocks lie beside its short
// ones; what bounds it is that overlap (a tile is about as many cycles of vector as of matrix instructions) and, in one prompt, the longest block's
// chain of rounds.  Key tiles start at absolute multiples of 32, tile t belongs to group t mod 2, and every decision is a
// row's own, so a row's result depends neither on the step's cut nor on the rows beside it.
//
// Blocks measured (us; rows x key groups x stages, of 32 rows, 32 keys; general: the kernel above), prompts of 512, 2,048 and 4,096 tokens, eight of 200, 32 rows
// behind 1,500 keys beside a prompt of 512, all with the reference left 2^8 behind (see below; 2x2x2 then: 11.3, 30.6, 64, 8.7, 18.9; 15.3, 65, 200,
// 20.6, 31.1; 14.3, 44, 124, 12.1, 29.4):
//   head size 64, 14 over 2 heads    general 14.1  42.5   111  12.5  31.9;  2x2x2 10.5  29.1  61  8.3  18.2;  2x2x4 11.1  30.4  73  8.7  -;
//                                    2x4x2   12.5  32.8    83  12.8  -;     4x2x4 14.1  36.9  71  11.3  -;    4x4x4 14.8  32.9  66  12.8  -
//   head size 128, 28 over 4 heads   general 17.5   101   318  28.7  34.1;  2x2x2 13.8  58   184  20.4  28.7; 2x4x2 14.5  75.6  218  30.2  -
//   head size 128, 16 over 4 heads   general 16.4    57   181  19.5  33.6;  2x2x2 13.2  39   117  11.6  27.3; 2x4x2 13.4  40.3  124  19.9  -
//
// How far a row's maximum may rise before the reference of its exponentials follows it, and its sums are rescaled (`rise`): not at all, as in
// the kernel above, so that the largest probability is one, which rounds exactly.  Where it is left up to 2^8 behind this is 4 %
// faster (up to 12 %: heads of 128, 1,024 rows behind 16,000 keys 232 us against 254), but every probability is rounded, and rows that few
// keys decide are further off: 2.26e-3 of the result against 64 bits where following gives 1.78e-3 (bfloat16, scores of deviation
// two; half precision alike).  Heads of 64 behind tables of 2,048 keys and more have always been left behind; 2^6 it is there: 2.13e-3,
// where blocks of 128 rows under four key groups and 2^8 gave 2.22e-3 (128 rows behind 4,000 keys: 21.0 us; 2^8 20.2, not at all 22.3).
//
// Operands (K = 16): A is 32 rows x 16, lane l holds row l % 32, elements (l / 32) * 8 .. + 8; B likewise by
// column; the result has column l % 32 and, in register v, row 8 * (v / 4) + 4 * (l / 32) + v % 4.  With
// S^T = K Q^T a lane's registers 8c .. 8c + 7 are therefore rows 16c + {0..3, 8..11} + 4 * (l / 32) of the key
// tile: if row R of the tile holds key R with bits 2 and 3 exchanged, they are the eight consecutive keys
// 16c + 8 * (l / 32) .., which is a B fragment of P^T as it stands and one 16-byte read of V^T.
//
// A tile that is loaded straight into LDS cannot be zeroed on its way: sixteen keys that are not there (beyond the
// block's rows, in pages given back behind a window, in tiles past the block's range) read the rest of the block's last page or the start of the
// pool instead, are masked in the scores, and their values are overwritten with zeros (a caller's pool may hold anything in a page
// that no request of the step owns).  Of sixteen keys that are there in part the others' values are what the page's last owner left:
// finite, as every writer of a page sees to (cache_value), and met by probabilities of zero.
#ifdef MS_HAS_ROWS32
namespace r32 {
constexpr int TK = 32;                  // keys of a group's tile
constexpr int NC = HDT / 16;            // steps of the score product
constexpr int NDT = HDT / 32;           // 32-row tiles of the output's head dimension
// LDS rows are unpadded; 16-byte chunk q of row r sits at q ^ f(r), with f such that the rows a fragment read takes
// in one pass (0..7 with 16..23, 8..15 with 24..31) fall on different banks.
constexpr int K_BYTES = TK * HDT * 2, V_BYTES = HDT * TK * 2;
constexpr int STAGE = K_BYTES + V_BYTES;
constexpr int PER_LANE = 16 * NDT + 2;  // what a group hands over per lane: the output, the reference, the sum
constexpr int MAX_TABLE = 2048;  // pages of a block's share of the block table (in LDS)
constexpr int RW = 2, KG = 2, NS = 2;   // waves of rows, key groups, LDS stages: a tile is asked for a round before it is multiplied
constexpr int GT = RW * 64;             // threads of a key group
constexpr int ROUND = KG * TK;          // keys of a round of the block
constexpr int MERGE_BYTES = (KG - 1) * RW * 64 * PER_LANE * 4;
constexpr int SMEM = NS * KG * STAGE > MERGE_BYTES ? NS * KG * STAGE : MERGE_BYTES;
constexpr int SUB = ROWS_PER_BLOCK / (RW * 32);  // blocks of a work item
constexpr int LOADS = STAGE / 16 / GT;           // of a lane per tile
constexpr int PER_CU = HDT == 64 ? 3 : 2;        // blocks that share a CU: by the registers
static_assert(PER_CU * (SMEM + MAX_TABLE * 4 + 1024) <= 160 * 1024, "the tiles of a CU's blocks exceed its LDS");
typedef float f32x16 __attribute__((ext_vector_type(16)));

__device__ __forceinline__ void mma_32x32x16(f32x16& acc, const Frag& a, const Frag& b) {
#if defined(MS_ELEM_BF16)
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.v, b.v, acc, 0, 0, 0);
#else
    acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(a.v, b.v, acc, 0, 0, 0);
#endif
}
// The largest of three, as one instruction (from `fmaxf` the compiler makes two for every operand it cannot prove to be
// no signalling NaN; scores are sums of products of finite values, or -inf where masked).
__device__ __forceinline__ float max3(float a, float b, float c) {
    float r;
    asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}
// The larger of a lane's number and its counterpart's in the wave's other half, in registers (`__shfl_xor` goes through LDS).
__device__ __forceinline__ float max_of_halves(float v) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return max3(__uint_as_float(r[0]), __uint_as_float(r[1]), __uint_as_float(r[1]));
}
__device__ __forceinline__ int swap_bits_2_3(int r) { return (r & ~12) | ((r & 4) << 1) | ((r & 8) >> 1); }
__device__ __forceinline__ int k_swizzle(int r) {
    if constexpr (HDT == 64) return ((r >> 1) & 3) | (((r >> 4) & 1) << 2);  // rows of 8 chunks
    else return (r & 7) | (((r >> 4) & 1) << 3);                             // rows of 16
}
__device__ __forceinline__ int v_swizzle(int d) { return ((d >> 2) & 1) | (((d >> 4) & 1) << 1); }  // rows of 4 chunks
}  // namespace r32

// ONE_PAGE: the page size is a multiple of a tile's 32 keys
template <bool ONE_PAGE>
__global__ __launch_bounds__(r32::KG * r32::GT, r32::KG * r32::RW * r32::PER_CU / 4) void paged_attention_rows32_kernel(AttnArgs a) {
    if (a.n_blocks > 0 && (int)blockIdx.x >= a.n_blocks) {
        if (blockIdx.y == 0) read_ahead(a, blockIdx.x - a.n_blocks, gridDim.x - a.n_blocks);
        return;
    }
    using namespace r32;
    static_assert((HDT == 64 || HDT == 128) && TK == 32 && RW == 2 && NS == 2, "the swizzles, the tiles' split over a group's waves and the rounds are written for these shapes");
    __shared__ __attribute__((aligned(1024))) unsigned char smem[SMEM];
    __shared__ uint32_t tab[MAX_TABLE + 1];

    const int kg = threadIdx.x / GT, tg = threadIdx.x % GT, lane = tg & 63, rw = tg >> 6;
    const int n32 = lane & 31, h = lane >> 5;
    // the order of the blocks: as the general kernel's
    const int kvh = blockIdx.x % a.KV, sub = blockIdx.x / a.KV % SUB, turn = blockIdx.x / (a.KV * SUB);
    int item = turn;
    if (a.pair_span > 0 && turn >= a.pair_span)
        item = turn < 2 * a.pair_span ? a.n_work - 1 - (turn - a.pair_span) : turn - a.pair_span;
    const int s = a.work[item * 2], r0 = a.work[item * 2 + 1] + RW * 32 * sub;
    if (s < 0) return;  // an item that only fills the list up (the same for the whole block)
    const int g = a.H / a.KV;
    const int q_start = a.seq_q_start[s], q_len = a.seq_q_len[s], pos0 = a.seq_pos0[s];
    const int R = q_len * g;
    if (r0 >= R) return;  // the item's rows end in the block beside this one (the same for the whole block)
    constexpr int hd = HDT;
    const int ps = a.ps;
    const int* table = a.block_table + (size_t)s * a.table_stride;

    // this lane's query row (both halves of the wave hold the same 32 rows)
    const int row = r0 + rw * 32 + n32;
    const bool valid = row < R;
    const int tok = valid ? row / g : 0;
    const int head = kvh * g + (valid ? row % g : 0);
    const int pos = pos0 + tok;
    const bool wave_active = __builtin_amdgcn_readfirstlane((int)(r0 + rw * 32 < R)) != 0;  // the same for the whole wave

    const int last_row = min(r0 + RW * 32, R) - 1;
    int kv_hi = pos0 + last_row / g + 1;
    int kv_lo = 0;
    if (a.window > 0 || a.chunk > 0) kv_lo = max(0, first_visible_key(pos0 + r0 / g, a.window, a.chunk));
    const int lo_key = first_visible_key(pos, a.window, a.chunk);
    const int sp = blockIdx.y;
    if (a.nsplit > 1) {
        const int first = (kv_lo / ROUND) * ROUND;
        const int per = ceil_div(ceil_div(kv_hi - first, ROUND), a.nsplit) * ROUND;
        kv_lo = max(kv_lo, first + sp * per);
        kv_hi = min(kv_hi, first + (sp + 1) * per);
    }
    // a row's partial result of this split: d = 32 dt + 8 (v / 4) + 4 h + v % 4 in register v of tile dt
    auto write_partial = [&](const f32x16* o, float m, float l) {
        const size_t base = (((size_t)(q_start + tok)) * a.H + head) * a.nsplit + sp;
        float* po = a.part_o + base * hd;
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
            for (int qd = 0; qd < 4; ++qd) {
                const int d0 = 32 * dt + 8 * qd + 4 * h;
#pragma unroll
                for (int i = 0; i < 4; ++i) po[d0 + i] = o[dt][4 * qd + i];
            }
        if (h == 0) { a.part_ml[base * 2] = m * a.scale; a.part_ml[base * 2 + 1] = l; }
    };
    if (kv_lo >= kv_hi) {  // nothing for this split (the same for every thread of the block)
        if (a.nsplit > 1 && kg == 0 && valid) {
            f32x16 zero[NDT];
#pragma unroll
            for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
                for (int i = 0; i < 16; ++i) zero[dt][i] = 0.f;
            write_partial(zero, NEG_BIG, 0.f);
        }
        return;
    }
    // the pages of the block's keys, once: those of [kt_first, kv_hi), at most MAX_TABLE of them (the launcher sees to it)
    kv_lo = __builtin_amdgcn_readfirstlane(kv_lo);
    kv_hi = __builtin_amdgcn_readfirstlane(kv_hi);
    const int kt_first = __builtin_amdgcn_readfirstlane((kv_lo / ROUND) * ROUND);
    const int page_first = kt_first / ps, n_tab = max(min(ceil_div(kv_hi, ps), a.table_stride) - page_first, 0);
    // (as where the head's keys, and values, of a page begin in the pool, in units of sixteen numbers; a page that was given back, and the place behind the
    // last one, which stands for all that are not in the table: the pool's start)
    const uint32_t page_units = (uint32_t)(a.KV * ps * HDT) >> 4, head_units = (uint32_t)(kvh * ps * HDT) >> 4;
    for (int i = threadIdx.x; i < n_tab; i += KG * GT) {
        const int page = table[page_first + i];
        tab[i] = page >= 0 ? (uint32_t)page * page_units + head_units : 0u;
    }
    if (threadIdx.x == 0) tab[n_tab] = 0u;

    Frag qf[NC];
    {
        const elem_t* qrow = a.q + ((size_t)(q_start + tok) * a.H + head) * hd;
#pragma unroll
        for (int c = 0; c < NC; ++c) qf[c] = valid ? frag_load(qrow + c * 16 + h * 8) : frag_zero();
    }
    f32x16 acc[NDT];
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[dt][i] = 0.f;
    float m_run = NEG_BIG, l_run = 0.f;
    const float sl = a.scale * 1.4426950408889634f;

    // A group's waves bring the group's tile, an equal share of K and of V^T each: a wave's load lands at the
    // wave's LDS base + 16 * lane, so the chunk that belongs at place p of the K tile (row p / (HDT / 8),
    // chunk p % (HDT / 8) ^ swizzle) is the one this lane asks for; likewise the V^T tile (row p / 4; GT / 4 rows further on its
    // swizzle is the same).  Where a tile lies in one page its addresses are a scalar each for K and V^T and a lane's constant offsets;
    // else a load of K has the scalar of its rows' 16-key group, and a lane of V^T that of its chunk's.
    constexpr int KL = LOADS / 2;  // loads of K, and of V^T
    const int p_own = 64 * rw + lane;
    uint32_t k_off[KL], v_off[KL];
    auto k_group = [](int i) { return i * GT / (HDT / 8) / 16; };
    const int dv = p_own >> 2, vq = (p_own & 3) ^ v_swizzle(dv);  // keys 8 vq .. + 8 of row dv of V^T
    const int v_grp = vq >> 1;
#pragma unroll
    for (int i = 0; i < KL; ++i) {
        const int p = i * GT + p_own, Rk = p / (HDT / 8), kq = (p % (HDT / 8)) ^ k_swizzle(Rk), kl = swap_bits_2_3(Rk);  // row Rk of the tile holds key kl
        k_off[i] = ((ONE_PAGE ? kl : kl & 15) * hd + kq * 8) * (uint32_t)sizeof(elem_t);
        v_off[i] = ((dv + i * (GT / 4)) * ps + (ONE_PAGE ? vq : vq & 1) * 8) * (uint32_t)sizeof(elem_t);
    }
    // Where the tiles lie: every wave looks its group's tile up for itself, in scalars.  `look_up` asks LDS for the next tile's page (or its two 16-key groups'
    // pages), stepped from tile to tile rather than divided out; `resolve`, a round later, makes addresses of it.  (Two threads that did it for their group
    // through LDS were a chain in every round.)  Behind the block's pages it is the pool's start, as for keys that are not there.
    const int kg_keys = __builtin_amdgcn_readfirstlane(kg * TK);
    int lp_next = (kt_first + kg_keys) / ps - page_first, off_next = (kt_first + kg_keys) % ps;
    const int round_pages = ROUND / ps, round_rem = ROUND % ps;
    constexpr int NG = ONE_PAGE ? 1 : 2;
    uint32_t entry[NG];
    int entry_off[NG];
    auto look_up = [&]() {
        entry[0] = tab[min(lp_next, n_tab)];
        entry_off[0] = off_next;
        if constexpr (!ONE_PAGE) {
            const bool over = off_next + 16 >= ps;
            entry[1] = tab[min(lp_next + (over ? 1 : 0), n_tab)];
            entry_off[1] = off_next + 16 - (over ? ps : 0);
        }
        lp_next += round_pages;
        off_next += round_rem;
        if (off_next >= ps) {
            off_next -= ps;
            ++lp_next;
        }
    };
    const char *keys_at[NG], *values_at[NG], *next_values_at[NG];  // of the tile whose loads go out next
    auto resolve = [&]() {
#pragma unroll
        for (int u = 0; u < NG; ++u) {
            const size_t page = (size_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)entry[u]) * (16 * sizeof(elem_t));
            values_at[u] = next_values_at[u];
            keys_at[u] = reinterpret_cast<const char*>(a.kpool) + page + (uint32_t)entry_off[u] * (uint32_t)(HDT * sizeof(elem_t));
            next_values_at[u] = reinterpret_cast<const char*>(a.vpool) + page + (uint32_t)entry_off[u] * (uint32_t)sizeof(elem_t);
        }
    };
    // a tile straight into stage `B` (in assembly: of a load that it knows to write LDS the
    // compiler would make every later LDS read wait; the waits are written by hand at the rounds' ends)
    const uint32_t lds_own = __builtin_amdgcn_readfirstlane(
        (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const unsigned char*)(smem + kg * STAGE + 1024 * rw));
    auto load_keys = [&](auto stage_of, const char* const (&from)[NG]) {
#pragma unroll
        for (int i = 0; i < KL; ++i) {
            const uint32_t off = k_off[i], to = lds_own;
            const char* base = from[ONE_PAGE ? 0 : k_group(i)];
            asm volatile("s_add_i32 m0, %2, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "s"(to),
                         "n"(decltype(stage_of)::value * (KG * STAGE) + i * GT * 16) : "memory", "m0", "scc");
        }
    };
    auto load_values = [&](auto stage_of, const char* const (&from)[NG]) {
#pragma unroll
        for (int i = 0; i < KL; ++i) {
            constexpr int at = decltype(stage_of)::value * (KG * STAGE) + K_BYTES;
            const uint32_t off = v_off[i], to = lds_own;
            const char* base = v_grp && !ONE_PAGE ? from[NG - 1] : from[0];
            if constexpr (ONE_PAGE)
                asm volatile("s_add_i32 m0, %2, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "s"(to), "n"(at + i * GT * 16)
                             : "memory", "m0", "scc");
            else
                asm volatile("s_add_i32 m0, %1, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(base + off), "s"(to), "n"(at + i * GT * 16)
                             : "memory", "m0", "scc");
        }
    };
    // rows of this wave: the first and the last position decide which tiles need no mask at all
    const int first_row = __builtin_amdgcn_readfirstlane(r0 + rw * 32);
    const int pos_first = pos0 + first_row / g;
    const int pos_last = pos0 + min(first_row + 31, max(R - 1, 0)) / g;
    const int lo_last = first_visible_key(pos_last, a.window, a.chunk);
    // where this lane reads its fragments in a stage: row n32 of the K tile, row 32 dt + n32 of V^T, chunk 2c + h
    const int k_row = n32 * (HDT * 2), k_sw = k_swizzle(n32), v_row = K_BYTES + n32 * (TK * 2), v_sw = v_swizzle(n32);

    // Round r: group kg has the tile of absolute index (kt_first / 32) + r * KG + kg.  Its scores are multiplied a round ahead, between round r - 1's
    // exponentials, so that a wave's matrix and vector instructions run beside each other and not in turn; so its keys run a round ahead of its values and
    // take the place of the last round's but one, whose scores are done.  Pages are looked up a round before the keys' loads go out, loads go out a round
    // before what they bring is multiplied, and one barrier a round separates the steps.  A round is bound by what a wave does one after the other, scalar
    // instructions included (a prompt of 2,048, 14 heads of 64, 31.0 us: with the scores ahead and two lookups in scalars 29.1, with
    // one page a tile and a table of offsets in place of pages 28.0, and with two rounds in the loop's body, so that stages are constants and the scores
    // change places without moves, 22.9; 4,096 tokens 61 -> 47; heads of 128, 28 over 4, 60 -> 54; loads two or three rounds ahead, tiles of 64 keys,
    // and two blocks a CU in place of three gain nothing).
    // (the same for the whole block: kept in scalar registers, so that the rounds' branches are scalar ones)
    const int n_rounds = __builtin_amdgcn_readfirstlane(ceil_div(kv_hi - kt_first, ROUND));
    using Stage0 = std::integral_constant<int, 0>;
    using Stage1 = std::integral_constant<int, 1>;
    // the queries and the table are here before the first tile is asked for, so that no later wait of the compiler's
    // for them takes the tiles' loads with it
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
    for (int c = 0; c < NC; ++c) asm volatile("" : "+v"(qf[c].v));
    __syncthreads();  // the table is in LDS
    look_up();
    resolve();
    load_keys(Stage0{}, keys_at);
    load_values(Stage0{}, next_values_at);
    look_up();
    resolve();
    load_keys(Stage1{}, keys_at);
    look_up();
    // End of a round: this wave's loads have landed and its LDS accesses are done; then everybody's.
    auto round_end = [&]() {
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
    };
    round_end();
    // S^T = K Q^T of the group's tile: register v of this lane is key kt0 + 16 (v / 8) + 8 h + v % 8 for query row n32.
    f32x16 sc0, sc1;
    const unsigned char* own = smem + kg * STAGE;
    auto k_frag = [&](int b, int c) { return frag_load(reinterpret_cast<const elem_t*>(own + b * (KG * STAGE) + k_row + (((2 * c + h) ^ k_sw) << 4))); };
#pragma unroll
    for (int i = 0; i < 16; ++i) sc0[i] = 0.f;
#pragma unroll
    for (int c = 0; c < NC; ++c) mma_32x32x16(sc0, k_frag(0, c), qf[c]);
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();  // everybody has round 0's keys
    __builtin_amdgcn_sched_barrier(0);
    int kt0 = kt_first + kg_keys;
    // the round with its scores in `sc` and its tile's values in stage B, which leaves the next round's scores in `next`
    auto round_of = [&](int r, auto stage_of, f32x16& sc, f32x16& next) {
        constexpr int B = decltype(stage_of)::value;
        resolve();
        if (r + 2 < n_rounds) load_keys(std::integral_constant<int, B>{}, keys_at);  // into the places that the last round has left
        if (r + 1 < n_rounds) load_values(std::integral_constant<int, B ^ 1>{}, values_at);
        look_up();
        if (r == 0 || r + 1 == n_rounds) {
            // (the same for the whole block) values of sixteen keys that are not there: zero
            const int key = kt0 + 16 * v_grp;
            if (key + 16 <= kv_lo || key >= kv_hi) {
#pragma unroll
                for (int i = 0; i < KL; ++i)
                    *reinterpret_cast<u32x4*>(smem + (B * KG + kg) * STAGE + K_BYTES + (i * GT + p_own) * 16) = (u32x4){0, 0, 0, 0};
            }
            __builtin_amdgcn_sched_barrier(0);
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_s_barrier();
            __builtin_amdgcn_sched_barrier(0);
        }
        if (wave_active && kt0 < kv_hi) {
            // the values of the first sixteen keys, which the step after next multiplies by: asked for before the exponentials
            auto v_frag = [&](int c, int dt) {
                return frag_load(reinterpret_cast<const elem_t*>(own + B * (KG * STAGE) + v_row + dt * (32 * TK * 2) + (((2 * c + h) ^ v_sw) << 4)));
            };
            Frag vf[NDT];
#pragma unroll
            for (int dt = 0; dt < NDT; ++dt) vf[dt] = v_frag(0, dt);
            Frag kf[2] = {k_frag(B ^ 1, 0), k_frag(B ^ 1, 1)};  // two fragments in flight
            if (a.softcap > 0.f) {
#pragma unroll
                for (int i = 0; i < 16; ++i) sc[i] = capped_raw(sc[i], a.scale, a.softcap);
            }
            const bool whole = kt0 + TK - 1 <= pos_first && kt0 >= lo_last;
            if (!whole) {
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const int key = kt0 + 16 * (i / 8) + 8 * h + (i % 8);
                    const bool ok = valid && key <= pos && key >= lo_key;
                    sc[i] = ok ? sc[i] : -INFINITY;
                }
            }
            // this lane's half of the row's keys
            const float tmax = max3(max3(max3(sc[0], sc[1], sc[2]), max3(sc[3], sc[4], sc[5]), max3(sc[6], sc[7], sc[8])),
                                    max3(max3(sc[9], sc[10], sc[11]), sc[12], sc[13]), max3(sc[14], sc[15], sc[15]));
            // (the two lanes of a row keep the same reference; for a row that stays the factor is exactly one)
            if (__any((tmax - m_run) * sl > a.rise)) {
                const float row_max = max_of_halves(tmax);
                const float m_new = (row_max - m_run) * sl > a.rise ? row_max : m_run;
                const float alpha = exp2_f((m_run - m_new) * sl);
                l_run *= alpha;
#pragma unroll
                for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
                    for (int i = 0; i < 16; ++i) acc[dt][i] *= alpha;
                m_run = m_new;
            }
            const float mb = m_run * sl;
            // the exponentials, and between them the next tile's scores (behind the last tile of what the places hold, and not used)
#pragma unroll
            for (int i = 0; i < 16; ++i) next[i] = 0.f;
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                mma_32x32x16(next, kf[c & 1], qf[c]);
                if (c + 2 < NC) kf[c & 1] = k_frag(B ^ 1, c + 2);
#pragma unroll
                for (int i = 16 / NC * c; i < 16 / NC * (c + 1); ++i) sc[i] = exp2_f(fmaf(sc[i], sl, -mb));
                __builtin_amdgcn_sched_barrier(0);
            }
            float t8[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) t8[i] = sc[i] + sc[i + 8];
            l_run += ((t8[0] + t8[1]) + (t8[2] + t8[3])) + ((t8[4] + t8[5]) + (t8[6] + t8[7]));  // of this lane's half of the keys
            // O^T += V^T P^T: registers 8c .. 8c + 7 are the probabilities of keys 16c + 8h .. + 8, a B fragment as they stand
            Frag pf[2];
#pragma unroll
            for (int c = 0; c < 2; ++c)
#pragma unroll
                for (int i = 0; i < 8; ++i) pf[c].v[i] = from_f32<elem_t>(sc[8 * c + i]);
#pragma unroll
            for (int c = 0; c < 2; ++c)
#pragma unroll
                for (int dt = 0; dt < NDT; ++dt) {
                    mma_32x32x16(acc[dt], vf[dt], pf[c]);
                    if (c == 0) vf[dt] = v_frag(1, dt);
                }
        }
        kt0 += ROUND;
        round_end();
    };
    for (int r = 0; r < n_rounds; r += 2) {
        round_of(r, Stage0{}, sc0, sc1);
        if (r + 1 < n_rounds) round_of(r + 1, Stage1{}, sc1, sc0);
    }

    l_run += __shfl_xor(l_run, 32, WAVE);  // the row's two halves (they were scaled alike all along)
    // groups 1.. hand (output, reference, sum) to group 0 through LDS, which adds them in group order
    float* mg = reinterpret_cast<float*>(smem);
    if (kg > 0) {
        float* mine = mg + ((size_t)(kg - 1) * RW + rw) * 64 * PER_LANE;
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
            for (int i = 0; i < 16; ++i) mine[(dt * 16 + i) * 64 + lane] = acc[dt][i];
        mine[(16 * NDT) * 64 + lane] = m_run;
        mine[(16 * NDT + 1) * 64 + lane] = l_run;
    }
    __syncthreads();
    if (kg > 0) return;
    for (int o = 0; o < KG - 1; ++o) {
        const float* other = mg + ((size_t)o * RW + rw) * 64 * PER_LANE;
        const float m_o = other[(16 * NDT) * 64 + lane], l_o = other[(16 * NDT + 1) * 64 + lane];
        const float m_new = fmaxf(m_run, m_o);
        const float c0 = exp2_f((m_run - m_new) * sl), c1 = exp2_f((m_o - m_new) * sl);
        l_run = l_run * c0 + l_o * c1;
        m_run = m_new;
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[dt][i] = acc[dt][i] * c0 + other[(dt * 16 + i) * 64 + lane] * c1;
    }
    if (valid && a.nsplit > 1) {
        write_partial(acc, m_run, l_run);
    } else if (valid) {
        const float inv = softmax_norm(m_run * a.scale, l_run, a.sinks, head, a.out_gate, (size_t)(q_start + tok) * a.H + head);
        elem_t* orow = a.out + ((size_t)(q_start + tok) * a.H + head) * hd;
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
            for (int qd = 0; qd < 4; ++qd) {
                const int d0 = 32 * dt + 8 * qd + 4 * h;
                half4_t o4 = {from_f32<elem_t>(acc[dt][4 * qd] * inv), from_f32<elem_t>(acc[dt][4 * qd + 1] * inv),
                              from_f32<elem_t>(acc[dt][4 * qd + 2] * inv), from_f32<elem_t>(acc[dt][4 * qd + 3] * inv)};
                *reinterpret_cast<half4_t*>(orow + d0) = o4;
            }
    }
}
#endif  // MS_HAS_ROWS32

// ---------------------------------------------------------------------------------------
// Decode attention: every request of the step has one row.  The g query heads of one KV
// head are the rows of one MFMA tile (g <= 16), so each key and value is read once per KV
// head.  The keys of a request are cut into `nsplit` contiguous ranges (grid z), and inside
// a block each of the four waves takes every fourth key tile, reading K and V^T straight
// from the pages into fragments (nothing is shared between waves, so nothing is staged in
// LDS).  Waves combine through LDS; blocks write (max, sum, unnormalised output) per split,
// and a second kernel merges the splits.
// Role in the reference: attn_decode_batched_f16_gqa (crates/mach-model/src/kernels.rs:2905-3036).

struct DecodeArgs {
    const elem_t* q;         // [S, H, hd]
    const elem_t* kpool;
    const elem_t* vpool;
    elem_t* out;             // [S, H * hd] (written when nsplit == 1)
    float* part_o;           // [S, H, nsplit, hd]
    float* part_ml;          // [S, H, nsplit, 2]
    const int* block_table;  // [S, table_stride]
    const int* seq_pos0;     // [S] position of the row = number of keys before it
    int table_stride, H, KV, hd, ps, window, nsplit;
    float scale;
    // fused form: q, k, v of the step come as partial sums of the projection; the kernel adds
    // them and the bias, rotates q and k, writes k and v into their page and merges the splits
    const float* qkv;        // [n_partials, S, stride]: q heads, k heads, v heads
    const float* bias;       // [stride] or null
    const float* inv_freq;   // [hd / 2] or null: no rotation
    const int* slot_map;     // [S] page * ps + offset of the row's key
    int n_partials, stride;
    const float* sinks;      // [H] or null: see AttnArgs
    const float* out_gate;   // [S, H] or null: see AttnArgs
    int chunk;               // see AttnArgs
    float softcap;           // see AttnArgs
};

constexpr int MAX_SPLITS = 64;
// The decode kernel's key tile: a wave holds two tiles in registers (one being multiplied, one in
// flight), and smaller tiles leave room for more waves on a CU, which is what keeps memory busy.
#ifndef MS_DECODE_BKV
#define MS_DECODE_BKV (BKV >= 32 ? 32 : BKV)
#endif
constexpr int DBKV = MS_DECODE_BKV;
constexpr int DNT = DBKV / 16, DNTP = (DNT + 1) / 2;

// Fragments of one key tile for one lane: keys (K rows) for the scores, V^T groups for the output.
struct DecodeTile {
    Frag kf[DNT][NKS];
    Frag vf[DNTP][ND];
};

// MANY (fused): the q/k/v product left more than two partial sums, of which up to eight are then asked for first of all.  CUT (fused): the keys are cut over several blocks.
// WIDE (fused): a KV head's share of the row is more than 1,024 columns, five a thread.
template <bool FUSED, bool MANY = false, bool CUT = false, bool WIDE = false>
__global__ __launch_bounds__(256) void decode_attention_kernel(DecodeArgs a) {
    arguments_now(a.q, a.kpool, a.vpool, a.out, a.part_o, a.part_ml, a.block_table, a.seq_pos0, a.table_stride, a.H, a.KV, a.hd,
                  a.ps, a.window, a.nsplit, a.scale, a.qkv, a.bias, a.inv_freq, a.slot_map, a.n_partials, a.stride);
    __shared__ __align__(32) float sm_o[3][HDT][16];  // also the staging area of the fused prologue: (g + 2) * hd sums and g * hd elements
    __shared__ float sm_m[3][16], sm_l[3][16];
    __shared__ float cs[HDT / 2], sn[HDT / 2], knew[HDT], vnew[HDT];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int r16 = lane & 15, grp = lane >> 4;
    const int s = blockIdx.x, kvh = blockIdx.y, sp = blockIdx.z;
    const int g = a.H / a.KV, hd = a.hd, ps = a.ps;
    const int pos = a.seq_pos0[s];
    // keys read from the pages: all of them, or (fused) those before the row's own position,
    // whose key and value are still in registers and enter as one extra term
    const int kv_len = FUSED ? pos : pos + 1;
    const int lo_key = max(0, first_visible_key(pos, a.window, a.chunk));
    const int* table = a.block_table + (size_t)s * a.table_stride;
    const bool valid = r16 < g;
    const int head = kvh * g + (valid ? r16 : 0);

    const int t_lo = lo_key / DBKV, t_hi = ceil_div(kv_len, DBKV);
    const int tps = max(1, ceil_div(t_hi - t_lo, a.nsplit));
    const int t0 = t_lo + sp * tps, t1 = min(t_hi, t0 + tps);

    // Where the keys of a tile sit in the MFMA rows is free, as long as the probabilities meet the
    // values of the same keys.  With an even number of 16-key score tiles, the pair (2pp, 2pp + 1)
    // covers 32 keys so that the lane of key group `grp` ends up with the probabilities of the eight
    // consecutive keys pp * 32 + grp * 8 ..: its V^T fragment is then one contiguous read.  Row r16 of
    // score tile 2pp + j holds key pp * 32 + (r16 / 4) * 8 + j * 4 + r16 % 4.
    constexpr bool PAIRED = DNT % 2 == 0;
    auto k_row = [&](int nt) { return PAIRED ? (nt / 2) * 32 + (r16 >> 2) * 8 + (nt & 1) * 4 + (r16 & 3) : nt * 16 + r16; };
    auto score_key = [&](int nt, int i) { return PAIRED ? (nt / 2) * 32 + grp * 8 + (nt & 1) * 4 + i : nt * 16 + grp * 4 + i; };
    // Loads are unconditional and on one straight path, so that the compiler counts them and a wait
    // for one tile leaves the next in flight: a key that is not there (beyond the row, in a page
    // given back, in a tile past the split) is read from the start of the pool instead and masked in
    // the scores.  The pools hold finite values everywhere (cache_value), so a value that meets a zero probability
    // adds nothing.  The pages of a tile's 16-key groups are looked up one tile ahead.
    const float inv_gpp = 1.0f / (float)(ps >> 4);  // 1 / (16-key groups per page)
    // of this lane's groups: page as the table has it, -1 if the group is not to be read (else 0), offset in the page
    struct Pages { int kp[DNTP], kx[DNTP], ko[DNTP], vp[DNTP], vx[DNTP], vo[DNTP]; };
    auto lookup = [&](int t) {
        Pages pg;
        const int kt0 = t * DBKV;
#pragma unroll
        for (int pp = 0; pp < DNTP; ++pp) {
            // 16-key groups of this lane: of its K rows of score tiles 2pp and 2pp + 1, and of its V keys
            const int gk = (kt0 >> 4) + (PAIRED ? 2 * pp + (r16 >> 3) : pp), gv = (kt0 >> 4) + (PAIRED ? 2 * pp + (grp >> 1) : pp);
            const int lk = (int)(((float)gk + 0.5f) * inv_gpp), lv = (int)(((float)gv + 0.5f) * inv_gpp);
            const int pk = table[min(lk, a.table_stride - 1)], pv = table[min(lv, a.table_stride - 1)];
            // The loaded pages are not touched here (a use would wait for them), and are later "or"-ed with
            // a mask the compiler cannot see through: it would turn a select (and an "or" with a known
            // 0 / -1, which it reads as one) into a branch around the load.
            pg.kp[pp] = pk;
            pg.kx[pp] = opaque((t < t1 && gk * 16 < kv_len) ? 0 : -1);
            pg.ko[pp] = gk * 16 - lk * ps;
            pg.vp[pp] = pv;
            pg.vx[pp] = opaque((t < t1 && gv * 16 < kv_len) ? 0 : -1);
            pg.vo[pp] = gv * 16 - lv * ps;
        }
        return pg;
    };
    const size_t page_elems = (size_t)ps * hd;
    auto load_tile = [&](const Pages& pg, DecodeTile& td) {
#pragma unroll
        for (int nt = 0; nt < DNT; ++nt) {
            // the row of (page, kvh, offset of the row's 16-key group + place in the group) in [pages, KV, ps, hd]
            const int pp = PAIRED ? nt / 2 : nt;
            const int page = pg.kp[pp] | pg.kx[pp], off = pg.ko[pp] + (k_row(nt) & 15);
            const elem_t* krow = page >= 0 ? a.kpool + ((size_t)page * a.KV + kvh) * page_elems + (size_t)off * hd : a.kpool;
#pragma unroll
            for (int ks = 0; ks < NKS; ++ks) {
                const int d0 = ks * 32 + grp * 8;
                td.kf[nt][ks] = frag_load(krow + (d0 < hd ? d0 : 0));  // beyond the head size q is zero
            }
        }
#pragma unroll
        for (int pp = 0; pp < DNTP; ++pp) {
            const int page = pg.vp[pp] | pg.vx[pp], off = pg.vo[pp] + (PAIRED ? (grp & 1) * 8 : grp * 4);
            const elem_t* vcol = page >= 0 ? a.vpool + ((size_t)page * a.KV + kvh) * page_elems + off : a.vpool;
#pragma unroll
            for (int dt = 0; dt < ND; ++dt) {
                const int d = dt * 16 + r16;
                const elem_t* v0 = vcol + (page >= 0 && d < hd ? (size_t)d * ps : 0);
                if constexpr (PAIRED) {
                    td.vf[pp][dt] = frag_load(v0);
                } else {
                    Frag vf = frag_zero();
#pragma unroll
                    for (int i = 0; i < 4; ++i) vf.v[i] = v0[i];
                    td.vf[pp][dt] = vf;
                }
            }
        }
    };
    // The fused prologue stages this KV head's share of the step's row: its g query heads, its key, its
    // value, (g + 2) * hd columns, four per thread at a time, of more than 1,024 columns five (1,280: seven heads of 128 beside key and value are 1,152).  What the
    // first of them need from memory (the bias and the first partial sums) is asked for here, before anything else: nothing of it
    // depends on the row's position, and the row's query is what the block waits for in the end.  (Seven sums of 1,152 columns, 28 heads
    // over 4 of 128, 16 requests: two first, five more and the last 128 columns behind them 13.8 us, all at once 11.5.)
    const int width = FUSED ? (g + 2) * hd : 0;
    const size_t pstride = FUSED ? (size_t)gridDim.x * a.stride : 0;
    const float* row0 = FUSED ? a.qkv + (size_t)s * a.stride : nullptr;
    const float* bias = FUSED && a.bias ? a.bias : row0;  // without a bias: finite values, times zero
    const float bias_on = FUSED && a.bias ? 1.f : 0.f;
    auto column = [&](int c) {
        c = min(c, width - 1);
        const int qcol = kvh * g * hd, kcol = a.H * hd + kvh * hd, vcol = (a.H + a.KV) * hd + kvh * hd;
        return c < g * hd ? qcol + c : (c < (g + 1) * hd ? kcol + c - g * hd : vcol + c - (g + 1) * hd);
    };
    constexpr int COLS = WIDE ? 5 : 4, EARLY = MANY ? 8 : 2;
    int col_e[COLS];
    float bias_e[COLS], part_e[EARLY][COLS], freq_e = 0.f;
    int slot = -1;
    if constexpr (FUSED) {
#pragma unroll
        for (int u = 0; u < COLS; ++u) {
            col_e[u] = column(tid + u * 256);
            bias_e[u] = bias[col_e[u]];
            if constexpr (!MANY) {  // a column's bias and sums side by side: 8 requests behind 2,048 tokens 0.8851 -> 0.8835 ms a step (24 layers)
                part_e[0][u] = row0[col_e[u]];
                part_e[1][u] = row0[(size_t)min(1, a.n_partials - 1) * pstride + col_e[u]];
            }
        }
        if constexpr (MANY) {
#pragma unroll
            for (int q = 0; q < EARLY; ++q) {
                const size_t po = (size_t)min(q, a.n_partials - 1) * pstride;
#pragma unroll
                for (int u = 0; u < COLS; ++u) part_e[q][u] = row0[po + col_e[u]];
            }
        }
        freq_e = (a.inv_freq ? a.inv_freq : row0)[min(tid, hd / 2 - 1)];
        slot = a.slot_map[s];
        __builtin_amdgcn_sched_barrier(0);  // the loads stay up here
    }

    // The first tile depends on nothing the prologue computes: it is requested before the prologue
    // so that its latency hides behind it.
    DecodeTile next;
    Pages ahead = lookup(t0 + wave);
    load_tile(ahead, next);
    ahead = lookup(t0 + wave + 4);

    Frag qf[NKS];
    if constexpr (FUSED) {
        const int half = hd / 2;
        float* rowv = &sm_o[0][0][0];                                   // (g + 2) * hd sums, then ...
        elem_t* qrot = reinterpret_cast<elem_t*>(rowv + (g + 2) * hd);  // ... the g rotated queries, rounded
        // the angles, while the sums are on their way
        if (tid < half) {
            float c = 1.f, sv = 0.f;
            if (a.inv_freq) sincosf((float)pos * freq_e, &sv, &c);
            cs[tid] = c;
            sn[tid] = sv;
        }
        int page = 0, off = 0;
        auto find_slot = [&] {
            page = slot >= 0 ? slot / ps : 0;
            off = slot >= 0 ? slot % ps : 0;
        };
        if constexpr (!CUT) find_slot();  // (divisions: while the sums are on their way)
        // Further partial sums, eight at a time, all of their loads asked for before the first is added: the
        // sums were written by the kernel before this one, and one load after the other would be as many trips
        // to them (beyond the last partial sum: the last one again, not added).
        auto add_partials = [&](int first, const int (&col)[COLS], float (&v)[COLS]) {
            constexpr int NB = 8;
            for (int p0 = first; p0 < a.n_partials; p0 += NB) {
                float t[NB][COLS];
#pragma unroll
                for (int q = 0; q < NB; ++q) {
                    const size_t po = (size_t)min(p0 + q, a.n_partials - 1) * pstride;
#pragma unroll
                    for (int u = 0; u < COLS; ++u) t[q][u] = row0[po + col[u]];
                }
#pragma unroll
                for (int q = 0; q < NB; ++q)
                    if (p0 + q < a.n_partials) {
#pragma unroll
                        for (int u = 0; u < COLS; ++u) v[u] += t[q][u];
                    }
            }
        };
        {
            float v[COLS];
#pragma unroll
            for (int u = 0; u < COLS; ++u) {
                v[u] = bias_e[u] * bias_on + part_e[0][u];
#pragma unroll
                for (int q = 1; q < EARLY; ++q) v[u] += q < a.n_partials ? part_e[q][u] : 0.f;
            }
            add_partials(EARLY, col_e, v);
#pragma unroll
            for (int u = 0; u < COLS; ++u)
                if (tid + u * 256 < width) rowv[tid + u * 256] = v[u];
        }
        for (int c0 = tid + COLS * 256; c0 < width; c0 += COLS * 256) {  // more columns: many large heads
            int col[COLS];
            float v[COLS];
#pragma unroll
            for (int u = 0; u < COLS; ++u) {
                col[u] = column(c0 + u * 256);
                v[u] = bias[col[u]] * bias_on;
            }
            add_partials(0, col, v);
#pragma unroll
            for (int u = 0; u < COLS; ++u)
                if (c0 + u * 256 < width) rowv[c0 + u * 256] = v[u];
        }
        __syncthreads();
        // Rotation, one pair (d, d + hd / 2) of a query head or of the key per thread at a time; the row's
        // own key and value are rounded as the page holds them, and one block writes them there (nobody
        // reads them in this launch).
        {
            if constexpr (CUT) find_slot();
            const bool writes = sp == 0 && slot >= 0;
            elem_t* kdst = const_cast<elem_t*>(a.kpool) + (((size_t)page * a.KV + kvh) * ps + off) * hd;
            elem_t* vdst = const_cast<elem_t*>(a.vpool) + ((size_t)page * a.KV + kvh) * hd * ps + off;
            const float inv_half = 1.0f / (float)half;
            for (int i = tid; i < (g + 1) * half; i += 256) {
                const int row = (int)(((float)i + 0.5f) * inv_half), j = i - row * half;  // i < 17 * 128: exact
                const float x0 = rowv[row * hd + j], x1 = rowv[row * hd + j + half];
                const elem_t r0 = from_f32<elem_t>(x0 * cs[j] - x1 * sn[j]), r1 = from_f32<elem_t>(x0 * sn[j] + x1 * cs[j]);
                if (row < g) {
                    qrot[row * hd + j] = r0;
                    qrot[row * hd + j + half] = r1;
                } else {
                    knew[j] = to_f32(r0);
                    knew[j + half] = to_f32(r1);
                    if (writes) {
                        kdst[j] = r0;
                        kdst[j + half] = r1;
                    }
                }
            }
            const float* vv_ = rowv + (g + 1) * hd;
            for (int d = tid; d < hd; d += 256) {
                const elem_t ve = cache_value(vv_[d]);
                vnew[d] = to_f32(ve);
                if (writes) vdst[(size_t)d * ps] = ve;
            }
        }
        __syncthreads();
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks) {
            const int d0 = ks * 32 + grp * 8;
            qf[ks] = (valid && d0 < hd) ? frag_load(qrot + r16 * hd + d0) : frag_zero();
        }
        __syncthreads();  // the staging area is free again: the waves hand their results over through it
    } else {
        const elem_t* qrow = a.q + ((size_t)s * a.H + head) * hd;
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks) {
            const int d0 = ks * 32 + grp * 8;
            qf[ks] = (valid && d0 < hd) ? frag_load(qrow + d0) : frag_zero();
        }
    }

    f32x4 acc_o[ND];
#pragma unroll
    for (int i = 0; i < ND; ++i) acc_o[i] = (f32x4){0.f, 0.f, 0.f, 0.f};
    float m_run = NEG_BIG, l_run = 0.f;

    auto process = [&](const DecodeTile& cur, int t) {
        const int kt0 = t * DBKV;
        f32x4 sc[DNT];
#pragma unroll
        for (int nt = 0; nt < DNT; ++nt) {
            sc[nt] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int ks = 0; ks < NKS; ++ks) mma_16x16x32(sc[nt], cur.kf[nt][ks], qf[ks]);
        }
        float tmax = NEG_BIG;
#pragma unroll
        for (int nt = 0; nt < DNT; ++nt)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int key = kt0 + score_key(nt, i);
                const bool ok = valid && key < kv_len && key >= lo_key;
                float sv = sc[nt][i] * a.scale;
                if (a.softcap > 0.f) sv = a.softcap * tanhf(sv / a.softcap);
                const float v = ok ? sv : -INFINITY;
                sc[nt][i] = v;
                tmax = fmaxf(tmax, v);
            }
        tmax = fmaxf(tmax, __shfl_xor(tmax, 16, WAVE));
        tmax = fmaxf(tmax, __shfl_xor(tmax, 32, WAVE));
        // A tile's probabilities refer to its own maximum (the largest is one, which rounds exactly) and its sums join the others' in 32 bits: a wave's
        // tiles give what they would each in a wave of its own, so uncut keys are as exact as keys cut over blocks (with the running
        // maximum: 1 % further off at 129 to 256 keys).  Fresh accumulators for a tile are also the faster way, 1 to 3 % (heads of 256
        // 21 %): its products wait for no rescaling.
        const float m_new = fmaxf(m_run, tmax);
        const float alpha = exp_f(m_run - m_new), beta = exp_f(tmax - m_new);
        float psum = 0.f;
#pragma unroll
        for (int nt = 0; nt < DNT; ++nt)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float p = exp_f(sc[nt][i] - tmax);
                sc[nt][i] = p;
                psum += p;
            }
        psum += __shfl_xor(psum, 16, WAVE);
        psum += __shfl_xor(psum, 32, WAVE);
        l_run = l_run * alpha + psum * beta;
        m_run = m_new;
        f32x4 pv[ND];
#pragma unroll
        for (int dt = 0; dt < ND; ++dt) pv[dt] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int pp = 0; pp < DNTP; ++pp) {
            Frag pf;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                pf.v[i] = from_f32<elem_t>(sc[2 * pp][i]);
                pf.v[4 + i] = from_f32<elem_t>((2 * pp + 1 < DNT) ? sc[(2 * pp + 1) % DNT][i] : 0.f);
            }
#pragma unroll
            for (int dt = 0; dt < ND; ++dt) mma_16x16x32(pv[dt], cur.vf[pp][dt], pf);
        }
#pragma unroll
        for (int dt = 0; dt < ND; ++dt)
#pragma unroll
            for (int i = 0; i < 4; ++i) acc_o[dt][i] = fmaf(pv[dt][i], beta, acc_o[dt][i] * alpha);
    };
    // Two tile buffers take turns, so that no tile is copied.  The loads of the tile after next are
    // issued before the current tile is multiplied, and the scheduler may not move them below it:
    // it would, to keep fewer registers live, and the loads' latency would then lie open.
    DecodeTile other;
    for (int t = t0 + wave; t < t1; t += 8) {
        load_tile(ahead, other);  // of tile t + 4; past the split it reads one line of the pool's start
        ahead = lookup(t + 8);
        __builtin_amdgcn_sched_barrier(0);
        process(next, t);
        if (t + 4 >= t1) break;
        load_tile(ahead, next);
        ahead = lookup(t + 12);
        __builtin_amdgcn_sched_barrier(0);
        process(other, t + 4);
    }

    if constexpr (FUSED) {
        // The row's own key: one more term of the online softmax, in split 0.  Where the keys are not cut it is the last wave's, which has no more tiles than
        // the others (with up to 192 keys none): in wave 0, behind its tile, it took 1.1 of a block's 7.6 us behind 33 keys.  Where they are cut the waves' tiles
        // are many as a rule, and which wave has it made no difference.
        if (sp == 0 && wave == (CUT ? 0 : 3)) {
            float dot = 0.f;
#pragma unroll
            for (int ks = 0; ks < NKS; ++ks) {
                const int d0 = ks * 32 + grp * 8;
                if (d0 < hd) {
#pragma unroll
                    for (int e = 0; e < 8; ++e) dot += to_f32(qf[ks].v[e]) * knew[d0 + e];
                }
            }
            dot += __shfl_xor(dot, 16, WAVE);
            dot += __shfl_xor(dot, 32, WAVE);
            const float sv = valid ? dot * a.scale : -INFINITY;
            const float m_new = fmaxf(m_run, sv);
            const float alpha = exp_f(m_run - m_new), p = exp_f(sv - m_new);
            l_run = l_run * alpha + p;
            m_run = m_new;
#pragma unroll
            for (int dt = 0; dt < ND; ++dt)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int d = dt * 16 + grp * 4 + i;
                    acc_o[dt][i] = acc_o[dt][i] * alpha + (d < hd ? p * vnew[d] : 0.f);
                }
        }
    }

    // waves 1..3 hand their state to wave 0
    if (wave > 0) {
        if (grp == 0) { sm_m[wave - 1][r16] = m_run; sm_l[wave - 1][r16] = l_run; }
#pragma unroll
        for (int dt = 0; dt < ND; ++dt)
#pragma unroll
            for (int i = 0; i < 4; ++i) sm_o[wave - 1][dt * 16 + grp * 4 + i][r16] = acc_o[dt][i];
    }
    __syncthreads();
    if (wave > 0) return;
    float m_all = m_run;
#pragma unroll
    for (int w = 0; w < 3; ++w) m_all = fmaxf(m_all, sm_m[w][r16]);
    const float c0 = exp_f(m_run - m_all);
    float l_all = l_run * c0;
#pragma unroll
    for (int dt = 0; dt < ND; ++dt)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc_o[dt][i] *= c0;
#pragma unroll
    for (int w = 0; w < 3; ++w) {
        const float c = exp_f(sm_m[w][r16] - m_all);
        l_all += sm_l[w][r16] * c;
#pragma unroll
        for (int dt = 0; dt < ND; ++dt)
#pragma unroll
            for (int i = 0; i < 4; ++i) acc_o[dt][i] += sm_o[w][dt * 16 + grp * 4 + i][r16] * c;
    }
    if (!valid) return;
    if (a.nsplit == 1) {
        const float inv = softmax_norm(m_all, l_all, a.sinks, head, a.out_gate, (size_t)s * a.H + head);
        elem_t* orow = a.out + ((size_t)s * a.H + head) * hd;
#pragma unroll
        for (int dt = 0; dt < ND; ++dt) {
            const int d0 = dt * 16 + grp * 4;
            if (d0 < hd) {
#pragma unroll
                for (int i = 0; i < 4; ++i) orow[d0 + i] = from_f32<elem_t>(acc_o[dt][i] * inv);
            }
        }
    } else {
        const size_t base = ((size_t)s * a.H + head) * a.nsplit + sp;
        float* po = a.part_o + base * hd;
#pragma unroll
        for (int dt = 0; dt < ND; ++dt) {
            const int d0 = dt * 16 + grp * 4;
            if (d0 < hd) {
#pragma unroll
                for (int i = 0; i < 4; ++i) po[d0 + i] = acc_o[dt][i];
            }
        }
        if (grp == 0) { a.part_ml[base * 2] = m_all; a.part_ml[base * 2 + 1] = l_all; }
    }
}

// out[row, :] = sum_sp o_sp exp(m_sp - m) / sum_sp l_sp exp(m_sp - m), splits in order.
// One wave per (request, head); lane = element of the head (in chunks of 64).  The splits' outputs of all chunks are
// asked for BATCH at a time, the first together with the (max, sum) pairs and before anything
// is computed from those: with as many as there are splits the kernel waits for memory once.  A split's coefficient is read
// from its lane into a scalar.
constexpr int MERGE_CHUNKS = (HDT + 63) / 64;
template <int BATCH>
__device__ __forceinline__ void merge_row(const float* __restrict__ part_o, const float* __restrict__ part_ml, elem_t* __restrict__ out, int hd, int nsplit,
                                          const float* __restrict__ sinks, int H, const float* __restrict__ out_gate) {
    const size_t row = blockIdx.x;  // (request, head)
    const int lane = threadIdx.x;
    const float* ml = part_ml + row * nsplit * 2;
    const float* po = part_o + row * nsplit * hd;
    float v[BATCH][MERGE_CHUNKS];
    auto fetch = [&](int sp0) {
#pragma unroll
        for (int u = 0; u < BATCH; ++u)
#pragma unroll
            for (int c = 0; c < MERGE_CHUNKS; ++c) v[u][c] = po[(size_t)min(sp0 + u, nsplit - 1) * hd + min(lane + 64 * c, hd - 1)];
    };
    fetch(0);
    // every lane holds one split's (max, sum); nsplit <= 64
    const int own = min(lane, nsplit - 1);
    const float m_ld = ml[own * 2], l_ld = ml[own * 2 + 1];
    const float m_own = lane < nsplit ? m_ld : NEG_BIG;
    const float l_own = lane < nsplit ? l_ld : 0.f;
    const float m = wave_max(m_own);
    const float c_own = lane < nsplit ? exp_f(m_own - m) : 0.f;
    auto of_lane = [](float x, int from) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), from)); };
    float l = 0.f;
    for (int sp = 0; sp < nsplit; ++sp) l += of_lane(l_own * c_own, sp);  // in split order
    const float inv = softmax_norm(m, l, sinks, sinks ? (int)(row % (size_t)H) : 0, out_gate, row);
    const float coef = c_own * inv;  // of split `lane`; zero beyond the last split
    float o[MERGE_CHUNKS] = {};
    for (int sp0 = 0; sp0 < nsplit; sp0 += BATCH) {
        if (sp0) fetch(sp0);
#pragma unroll
        for (int u = 0; u < BATCH; ++u) {
            const float of = of_lane(coef, min(sp0 + u, 63));  // zero beyond the last split
#pragma unroll
            for (int c = 0; c < MERGE_CHUNKS; ++c) o[c] += v[u][c] * of;
        }
    }
#pragma unroll
    for (int c = 0; c < MERGE_CHUNKS; ++c)
        if (lane + 64 * c < hd) out[row * hd + lane + 64 * c] = from_f32<elem_t>(o[c]);
}
__global__ __launch_bounds__(64) void decode_merge_kernel(const float* __restrict__ part_o, const float* __restrict__ part_ml,
                                                          elem_t* __restrict__ out, int hd, int nsplit,
                                                          const float* __restrict__ sinks, int H,
                                                          const float* __restrict__ out_gate) {
    arguments_now(part_o, part_ml, out, hd, nsplit, sinks, H, out_gate);
    constexpr int MOST = 64 / MERGE_CHUNKS / 16 * 16;  // splits whose outputs fit the registers at once: 64, 32 or 16
    if (nsplit <= 4) merge_row<4>(part_o, part_ml, out, hd, nsplit, sinks, H, out_gate);
    else if (nsplit <= 8) merge_row<8>(part_o, part_ml, out, hd, nsplit, sinks, H, out_gate);
    else if (nsplit <= 16 || MOST == 16) merge_row<16>(part_o, part_ml, out, hd, nsplit, sinks, H, out_gate);
    else if (nsplit <= 24 || MOST < 64) merge_row<MOST == 64 ? 24 : MOST>(part_o, part_ml, out, hd, nsplit, sinks, H, out_gate);
    else merge_row<32>(part_o, part_ml, out, hd, nsplit, sinks, H, out_gate);
}

}  // namespace ms

using namespace ms;

#define MS_CAT2(a, b) a##b
#define MS_CAT(a, b) MS_CAT2(a, b)

// Attention of a mixed batch.  `work` lists (request index, first flat row) for every ROWS_PER_BLOCK
// flat rows of a request (ms_attention_rows_per_block_nd<N>() tells the caller the number; the general kernel
// takes an item as SUB_BLOCKS blocks of 64 rows, the kernel of 32-row tiles as r32::SUB); an item of
// request -1 only fills a list up and is skipped; see the file comment.  window = 0 means all keys.  max_key_groups = 0 lets the
// launcher choose how many key groups share a block (1, 2 or 4) from the width of the block tables;
// a positive value asks for that many (as far as this tile has them).  nsplit > 1 cuts every block's
// keys over that many blocks (few blocks of rows over long contexts would leave most of the chip idle
// and run as long as their chain of tiles); T is the number of rows, part_o [T, H, nsplit, hd] and
// part_ml [T, H, nsplit, 2] are float workspaces.
//
// Whether a launch with these sizes runs in the kernel of 32-row tiles: where the head size is the tile's and a block's share of the
// block table fits its place in LDS (asked for by name with max_key_groups = 32; 1, 2 and 4 ask for the general kernel).  It was
// the faster one at every size measured (its comment has some): one prompt of 17 to 8,192 tokens, requests of 40 to 877, decode rows
// behind 1,500 to 16,000 keys beside a prompt, windows of 512 and 1,024; with blocks of 128 rows, one a CU, it had been the slower one below 2,048 keys.
static bool takes_rows32(int hd, int ps, int table_stride, int window, int max_key_groups) {
#ifdef MS_HAS_ROWS32
    const long pages_of_span = window > 0 ? ((long)window + 2 * ROWS_PER_BLOCK + r32::ROUND) / ps + 2 : (long)table_stride;
    return hd == HDT && pages_of_span <= r32::MAX_TABLE && (max_key_groups == 32 || max_key_groups == 0);
#else
    (void)hd; (void)ps; (void)table_stride; (void)window; (void)max_key_groups;
    return false;
#endif
}

static int attention_compute_units() {
    static int cus = 0;
    if (cus == 0) {
        int dev = 0, n = 0;
        if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n < 1) n = 256;
        (void)hipGetLastError();
        cus = n;
    }
    return cus;
}

// Into how many blocks ms_paged_attention should cut the keys of every block of rows (its `nsplit`) when the caller
// leaves the choice to the library: n_work items of the work list, T rows in the step.  Few blocks of rows over long
// contexts leave most of the chip idle and run as long as their chain of tiles; cutting the chain fills the chip, at
// the price of the partial results' trip through memory and the merge's launch.  Block tables no wider than twice the
// step's rows are (or may be) those of prompts that run whole, whose blocks walk half the keys on average and whose
// longest block decides: cutting those only adds (0.5B heads, one prompt of 1,024 tokens 18.9 us uncut, 22.8 in two,
// 31.9 in four; 1,536 tokens 24.4 / 32.3 / 36.8).
// Heads of 64 in the kernel of 32-row tiles, whose items are two blocks, three to a CU: two blocks a CU in all, at least 1,024 keys a split, and three
// where that leaves 1,664 keys a split; where the items alone are more than that and yet no whole round of the chip, as many splits of 1,664 keys and
// more as fill its rounds best.  us (0.5B heads unless said; splits by the first clause alone -> by all; in brackets the kernel of 128-row
// blocks that the first clause was made for): 1,024 rows behind 4,000 keys 46.9 -> 43.5 (44.6), 16,000 keys 125 -> 108 (105); 2,048 rows behind
// 16,000 keys 225 -> 208 (195); 512 rows behind 16,000 keys 66 -> 60 (62); 8 over 8 heads, 32 requests of two rows behind 8,000 keys 129 -> 109
// (112).  Over 165 cases (17 to 2,048 rows behind 1,500 to 32,000 keys, 14 over 2, 8 over 8 and 4 over 2 heads) 0.91 of the time of those blocks, 1.06 at
// most.  256 rows and fewer would gain by more and shorter splits (64 rows behind 4,000 keys: 19.8 in four, 13.5 in sixteen; those blocks 22.7).
// Other heads, among them those of 128 in the kernel of 32-row tiles, go by the rule of the general kernel's 64-row blocks, two to a CU: three quarters of
// a round and more stay whole, fewer are cut into a round and a half, at least 512 keys a split.  With heads of 128 all of 163 cases are faster by it
// than in the general kernel (0.72 of its time), and 1.09 of the best cut; the furthest from it are 1,024 rows of 12 over 2 heads behind 32,000 keys (473
// whole, 285 in eight).
// The cut depends on the batch, so results differ in rounding between batches.
extern "C" int MS_CAT(ms_attention_splits_nd, MS_ATTN_ND)(int n_work, int KV, int T, int hd, int ps, int table_stride, int window) {
    if (n_work < 1 || KV < 1 || ps < 1 || table_stride < 1) return 1;
    const long blocks = (long)n_work * KV;
    long span = (long)table_stride * ps;
    if (window > 0 && span > (long)window + 64) span = (long)window + 64;
    if (span <= 2L * T) return 1;
    long n;
    if (HDT == 64 && span >= 2048 && takes_rows32(hd, ps, table_stride, window, 0)) {
        const long cus = attention_compute_units();
        n = std::min(cus / blocks, span / 1024);
#ifdef MS_HAS_ROWS32
        const long places = cus * r32::PER_CU, small = blocks * r32::SUB, full = places / small;
        if (n >= 2 && full > n && span / 1664 >= full) n = full;
        if (n < 2) {
            n = 1;
            if (small < places)
                for (long s = 2; s <= span / 1664; ++s)  // the chip's rounds times the length of a split
                    if (ceil_div(small * s, places) * n < ceil_div(small * n, places) * s) n = s;
        }
#endif
    } else {
        if (blocks >= 192) return 1;
        n = std::min((384 + blocks - 1) / blocks, span / 512);
    }
    return (int)std::max(1L, std::min(n, (long)MAX_SPLITS));
}

// `sinks`: null, or one number per head that the softmax's denominator also holds as exp(sink); `out_gate`: null, or
// float [T, H] that the output of each (row, head) is multiplied by.
// `chunk`, `softcap`: see AttnArgs (0: none).  What a row can reach back (`reach`: the window, the chunk, or the smaller of
// both) is what the choice of the kernel and of its key groups goes by.
// How many blocks read `bytes` ahead beside the `blocks` of a kernel of which the chip holds `places`: those that fill the CUs up to equally many, which cost
// the attention nothing, or if they are too few to be done in its time a block more on every CU; none where the attention is more than a round.  us of an attention over
// 2,048 tokens (14 over 2 heads of 64, 452 blocks) that reads 26 MB ahead, by blocks beside: none 25.1, 16 40.6, 32 24.8, 48 24.9, 60 25.2, 64 28.6, 96 27.3, 128 26.9, 316 26.7.
// ms with 32 MB ahead at most and without, 0.5B: 100 tokens 1.14 and 1.20, 400 1.53 and 1.62, 700 1.69 and 1.81, 1,000 2.06 and 2.06, 2,048 3.01 and 3.15; 1.5B: 200
// tokens 2.31 and 2.48, 500 3.02 and 3.06, 2,000 7.20 and 7.20.
static int blocks_ahead(long bytes, long blocks, long places, int threads) {
    constexpr long LEAST = 48, MOST = 256;
    if (bytes < 16) return 0;
    const long cus = attention_compute_units();
    long n = ceil_div(blocks, cus) * cus - blocks;
    if (n < LEAST) n += cus;
    return (int)std::max(0L, std::min({n, places - blocks, MOST, ceil_div(bytes, (long)threads * 256)}));
}

extern "C" int MS_CAT(ms_paged_attention_ahead_nd, MS_ATTN_ND)(
    const void* q, const void* kpool, const void* vpool, void* out, const int* block_table, int table_stride,
    const int* seq_q_start, const int* seq_q_len, const int* seq_pos0, const int* work, int n_work, int H, int KV,
    int hd, int ps, int n_pages, int window_of_mask, float scale, int max_key_groups, int T, int nsplit, float* part_o,
    float* part_ml, const float* sinks, const float* out_gate, int chunk, float softcap, const void* ahead0, long bytes0, const void* ahead1,
    long bytes1, hipStream_t stream) {
    MS_REQUIRE(n_work > 0, "attention: no work");
    MS_REQUIRE(chunk >= 0 && softcap >= 0.f && (softcap == 0.f || scale != 0.f), "attention: chunk %d, score cap %g", chunk, (double)softcap);
    const int window = window_of_mask > 0 && chunk > 0 ? (window_of_mask < chunk ? window_of_mask : chunk) : (window_of_mask > 0 ? window_of_mask : chunk);
    MS_REQUIRE(nsplit >= 1 && nsplit <= MAX_SPLITS && (nsplit == 1 || (part_o && part_ml && T > 0)),
               "attention: %d key splits (at most %d, with their workspaces)", nsplit, MAX_SPLITS);
    MS_REQUIRE(hd % 16 == 0 && hd > 0 && hd <= HDT, "attention: head size %d does not fit this tile of %d", hd, HDT);
    MS_REQUIRE(KV > 0 && H % KV == 0, "attention: %d heads are not a multiple of %d key/value heads", H, KV);
    MS_REQUIRE(ps % 16 == 0 && ps > 0, "attention: page size %d must be a multiple of 16", ps);
    MS_REQUIRE(window >= 0, "attention: window %d", window);
    MS_REQUIRE((double)n_pages * KV * ps * hd < 68719476736.0, "attention: a pool of %d pages exceeds 2^36 elements", n_pages);
    AttnArgs a{(const elem_t*)q, (const elem_t*)kpool, (const elem_t*)vpool, (elem_t*)out, block_table, seq_q_start,
               seq_q_len, seq_pos0, work, table_stride, H, KV, hd, ps, window_of_mask, scale, n_work, 0, nsplit, part_o, part_ml, sinks, out_gate,
               chunk, softcap};
    MS_REQUIRE(bytes0 >= 0 && bytes1 >= 0 && bytes0 < 1L << 35 && bytes1 < 1L << 35 && (bytes0 < 16 || ahead0) && (bytes1 < 16 || ahead1) &&
                   ((reinterpret_cast<uintptr_t>(ahead0) | reinterpret_cast<uintptr_t>(ahead1)) & 15) == 0,
               "attention: what is read ahead must begin at 16 bytes");
    a.ahead[0] = (const u32x4*)ahead0, a.ahead[1] = (const u32x4*)ahead1;
    a.n_ahead[0] = (uint32_t)(bytes0 / 16), a.n_ahead[1] = (uint32_t)(bytes1 / 16);
    // key groups per block by the longest context the block tables allow (the lengths themselves
    // are on the device): short contexts have no chain worth cutting
    const long span = window > 0 ? (long)window + BKV : (long)table_stride * ps;
    // measured at 512 to 8,192 keys: two groups beat one by a quarter, four gain nothing over two
    int groups = 2;
    if (max_key_groups > 0) {
        groups = max_key_groups < MAX_KEY_GROUPS ? max_key_groups : MAX_KEY_GROUPS;
    } else if (span < 4 * BKV) {
        groups = 1;
    }
    MS_REQUIRE((long)n_work * KV * SUB_BLOCKS < 2147483647L, "attention: %d blocks of rows times %d key/value heads", n_work, KV);
    dim3 grid((unsigned)(n_work * KV * SUB_BLOCKS), (unsigned)nsplit);
    // how many blocks of each variant a CU holds, and how many CUs there are: asked once
    static int cus = 0, resident[4] = {0, 0, 0, 0};
    if (cus == 0) {
        int dev = 0, n = 0;
        if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n < 1)
            n = 256;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&resident[0], paged_attention_kernel<1>, 256, 0) != hipSuccess) resident[0] = 1;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&resident[1], paged_attention_kernel<2>, 512, 0) != hipSuccess) resident[1] = 1;
        if constexpr (MAX_KEY_GROUPS >= 4) {
            if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&resident[2], paged_attention_kernel<4>, 1024, 0) != hipSuccess) resident[2] = 1;
        }
        (void)hipGetLastError();
        cus = n;
    }
    auto span_for = [&](int variant) { return resident[variant] == 2 ? (cus / (KV * SUB_BLOCKS) > 0 ? cus / (KV * SUB_BLOCKS) : 1) : 0; };
#ifdef MS_HAS_ROWS32
    {
        if (takes_rows32(hd, ps, table_stride, window, max_key_groups)) {
            a.pair_span = r32::PER_CU == 2 ? std::max(cus / (KV * r32::SUB), 1) : 0;
            a.rise = HDT == 64 && span >= 2048 ? 6.0f : 0.0f;  // see the kernel
            const long own = (long)n_work * KV * r32::SUB;
            const int beside = blocks_ahead(bytes0 + bytes1, own * nsplit, (long)cus * r32::PER_CU, r32::KG * r32::GT);
            if (beside > 0) a.n_blocks = (int)own;
            const dim3 grid32((unsigned)(own + beside), (unsigned)nsplit);
            if (ps % r32::TK == 0) hipLaunchKernelGGL(paged_attention_rows32_kernel<true>, grid32, dim3(r32::KG * r32::GT), 0, stream, a);
            else hipLaunchKernelGGL(paged_attention_rows32_kernel<false>, grid32, dim3(r32::KG * r32::GT), 0, stream, a);
            int rc32 = check_launch("paged_attention (32-row tiles)");
            if (rc32 || nsplit == 1) return rc32;
            hipLaunchKernelGGL(decode_merge_kernel, dim3((unsigned)((size_t)T * H)), dim3(64), 0, stream, part_o, part_ml, (elem_t*)out, hd, nsplit, a.sinks, H, a.out_gate);
            return check_launch("attention_merge");
        }
    }
#endif
    const int variant = groups >= 4 && MAX_KEY_GROUPS >= 4 ? 2 : groups >= 2 ? 1 : 0;
    if (const int beside = blocks_ahead(bytes0 + bytes1, (long)grid.x * nsplit, (long)cus * resident[variant], 256 << variant)) {
        a.n_blocks = (int)grid.x;
        grid.x += (unsigned)beside;
    }
    if (groups >= 4 && MAX_KEY_GROUPS >= 4) {
        // sixteen waves leave each 128 registers, which only the small bfloat16 tiles fit into
        a.pair_span = span_for(2);
        if constexpr (MAX_KEY_GROUPS >= 4) hipLaunchKernelGGL(paged_attention_kernel<4>, grid, dim3(1024), 0, stream, a);
    } else if (groups >= 2) {
        a.pair_span = span_for(1);
        hipLaunchKernelGGL(paged_attention_kernel<2>, grid, dim3(512), 0, stream, a);
    } else {
        a.pair_span = span_for(0);
        hipLaunchKernelGGL(paged_attention_kernel<1>, grid, dim3(256), 0, stream, a);
    }
    int rc = check_launch("paged_attention");
    if (rc || nsplit == 1) return rc;
    hipLaunchKernelGGL(decode_merge_kernel, dim3((unsigned)((size_t)T * H)), dim3(64), 0, stream, part_o, part_ml, (elem_t*)out, hd, nsplit, a.sinks, H, a.out_gate);
    return check_launch("attention_merge");
}

extern "C" int MS_CAT(ms_paged_attention_mask_nd, MS_ATTN_ND)(
    const void* q, const void* kpool, const void* vpool, void* out, const int* block_table, int table_stride,
    const int* seq_q_start, const int* seq_q_len, const int* seq_pos0, const int* work, int n_work, int H, int KV,
    int hd, int ps, int n_pages, int window, float scale, int max_key_groups, int T, int nsplit, float* part_o,
    float* part_ml, const float* sinks, const float* out_gate, int chunk, float softcap, hipStream_t stream) {
    return MS_CAT(ms_paged_attention_ahead_nd, MS_ATTN_ND)(q, kpool, vpool, out, block_table, table_stride, seq_q_start, seq_q_len,
                                                             seq_pos0, work, n_work, H, KV, hd, ps, n_pages, window, scale,
                                                             max_key_groups, T, nsplit, part_o, part_ml, sinks, out_gate, chunk, softcap,
                                                             nullptr, 0, nullptr, 0, stream);
}

extern "C" int MS_CAT(ms_paged_attention_ex_nd, MS_ATTN_ND)(
    const void* q, const void* kpool, const void* vpool, void* out, const int* block_table, int table_stride,
    const int* seq_q_start, const int* seq_q_len, const int* seq_pos0, const int* work, int n_work, int H, int KV,
    int hd, int ps, int n_pages, int window, float scale, int max_key_groups, int T, int nsplit, float* part_o,
    float* part_ml, const float* sinks, const float* out_gate, hipStream_t stream) {
    return MS_CAT(ms_paged_attention_mask_nd, MS_ATTN_ND)(q, kpool, vpool, out, block_table, table_stride, seq_q_start, seq_q_len,
                                                            seq_pos0, work, n_work, H, KV, hd, ps, n_pages, window, scale,
                                                            max_key_groups, T, nsplit, part_o, part_ml, sinks, out_gate, 0, 0.f, stream);
}

extern "C" int MS_CAT(ms_paged_attention_nd, MS_ATTN_ND)(
    const void* q, const void* kpool, const void* vpool, void* out, const int* block_table, int table_stride,
    const int* seq_q_start, const int* seq_q_len, const int* seq_pos0, const int* work, int n_work, int H, int KV,
    int hd, int ps, int n_pages, int window, float scale, int max_key_groups, int T, int nsplit, float* part_o,
    float* part_ml, hipStream_t stream) {
    return MS_CAT(ms_paged_attention_ex_nd, MS_ATTN_ND)(q, kpool, vpool, out, block_table, table_stride, seq_q_start, seq_q_len,
                                                          seq_pos0, work, n_work, H, KV, hd, ps, n_pages, window, scale,
                                                          max_key_groups, T, nsplit, part_o, part_ml, nullptr, nullptr, stream);
}

extern "C" int MS_CAT(ms_attention_rows_per_block_nd, MS_ATTN_ND)() { return ROWS_PER_BLOCK; }

// Attention of a step in which every request has exactly one row (row s = request s).
// part_o [S, H, nsplit, hd] and part_ml [S, H, nsplit, 2] are float workspaces (unused when
// nsplit == 1).  Needs H / KV <= 16.
extern "C" int MS_CAT(ms_decode_attention_mask_nd, MS_ATTN_ND)(
    const void* q, const void* kpool, const void* vpool, void* out, float* part_o, float* part_ml, const int* block_table,
    int table_stride, const int* seq_pos0, int S, int H, int KV, int hd, int ps, int window, int nsplit, float scale,
    const float* sinks, const float* out_gate, int chunk, float softcap, hipStream_t stream) {
    MS_REQUIRE(S > 0, "decode attention: no rows");
    MS_REQUIRE(chunk >= 0 && softcap >= 0.f, "decode attention: chunk %d, score cap %g", chunk, (double)softcap);
    MS_REQUIRE(hd % 16 == 0 && hd > 0 && hd <= HDT, "decode attention: head size %d does not fit this tile of %d", hd, HDT);
    MS_REQUIRE(KV > 0 && H % KV == 0 && H / KV <= 16, "decode attention: %d heads over %d key/value heads (at most 16 each)", H, KV);
    MS_REQUIRE(ps % 16 == 0 && ps > 0, "decode attention: page size %d must be a multiple of 16", ps);
    MS_REQUIRE(nsplit >= 1 && nsplit <= MAX_SPLITS && (nsplit == 1 || (part_o && part_ml)), "decode attention: %d splits (at most %d)", nsplit, MAX_SPLITS);
    DecodeArgs a{(const elem_t*)q, (const elem_t*)kpool, (const elem_t*)vpool, (elem_t*)out, part_o, part_ml, block_table,
                 seq_pos0, table_stride, H, KV, hd, ps, window, nsplit, scale, nullptr, nullptr, nullptr, nullptr, 0, 0, sinks, out_gate,
                 chunk, softcap};
    hipLaunchKernelGGL(decode_attention_kernel<false>, dim3((unsigned)S, (unsigned)KV, (unsigned)nsplit), dim3(256), 0, stream, a);
    int rc = check_launch("decode_attention");
    if (rc || nsplit == 1) return rc;
    hipLaunchKernelGGL(decode_merge_kernel, dim3((unsigned)(S * H)), dim3(64), 0, stream, part_o, part_ml, (elem_t*)out, hd, nsplit, a.sinks, H, a.out_gate);
    return check_launch("decode_merge");
}

extern "C" int MS_CAT(ms_decode_attention_ex_nd, MS_ATTN_ND)(
    const void* q, const void* kpool, const void* vpool, void* out, float* part_o, float* part_ml, const int* block_table,
    int table_stride, const int* seq_pos0, int S, int H, int KV, int hd, int ps, int window, int nsplit, float scale,
    const float* sinks, const float* out_gate, hipStream_t stream) {
    return MS_CAT(ms_decode_attention_mask_nd, MS_ATTN_ND)(q, kpool, vpool, out, part_o, part_ml, block_table, table_stride, seq_pos0,
                                                             S, H, KV, hd, ps, window, nsplit, scale, sinks, out_gate, 0, 0.f, stream);
}

extern "C" int MS_CAT(ms_decode_attention_nd, MS_ATTN_ND)(
    const void* q, const void* kpool, const void* vpool, void* out, float* part_o, float* part_ml, const int* block_table,
    int table_stride, const int* seq_pos0, int S, int H, int KV, int hd, int ps, int window, int nsplit, float scale,
    hipStream_t stream) {
    return MS_CAT(ms_decode_attention_ex_nd, MS_ATTN_ND)(q, kpool, vpool, out, part_o, part_ml, block_table, table_stride, seq_pos0,
                                                           S, H, KV, hd, ps, window, nsplit, scale, nullptr, nullptr, stream);
}

// Scratch memory of ms_decode_attention_noalloc_nd*: the splits' partial outputs, then their (max, sum)
// pairs.  Each GPU on which the library runs holds its own copy of this array, at its own address, until
// the process ends.  In host code the name is only a handle for hipGetSymbolAddress; the address that
// kernels and copies take is looked up once per device and kept in g_scratch_ptr.
constexpr size_t NOALLOC_SCRATCH_FLOATS = (size_t)1 << 20;  // 4 MiB
static __device__ __align__(256) float scratch[NOALLOC_SCRATCH_FLOATS];
constexpr int NOALLOC_MAX_DEVICES = 64;
static float* g_scratch_ptr[NOALLOC_MAX_DEVICES] = {};
static std::mutex g_scratch_mutex;

// The device address of `scratch` on the current device (null and an error message if it cannot be had).
static float* scratch_of_current_device() {
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess || dev < 0 || dev >= NOALLOC_MAX_DEVICES) {
        ms::set_error("decode attention (no allocation): device %d (%s); at most %d devices", dev, hipGetErrorString(e),
                      NOALLOC_MAX_DEVICES);
        return nullptr;
    }
    std::lock_guard<std::mutex> hold(g_scratch_mutex);
    if (!g_scratch_ptr[dev]) {
        float* ptr = nullptr;
        e = hipGetSymbolAddress((void**)&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !ptr) {
            ms::set_error("decode attention (no allocation): hipGetSymbolAddress on device %d: %s", dev, hipGetErrorString(e));
            return nullptr;
        }
        g_scratch_ptr[dev] = ptr;
    }
    return g_scratch_ptr[dev];
}

// ms_decode_attention_nd* for callers that cannot allocate (declared in no_alloc.h): the same kernels, with the
// workspace of the splits in `scratch` instead of two buffers of the caller.  It calls no hipMalloc, hipFree or
// allocating library routine.  S * H * nsplit * (hd + 2) floats must fit NOALLOC_SCRATCH_FLOATS.  Nothing in
// the scratch has to start at zero (every block writes its split's partial result, an empty split a sum
// of zero); it keeps the last call's contents, and all calls on one GPU share it, so two calls that
// overlap on one GPU (two streams, two threads) race: the caller orders them.
extern "C" int MS_CAT(ms_decode_attention_noalloc_nd, MS_ATTN_ND)(
    const void* q, const void* kpool, const void* vpool, void* out, const int* block_table, int table_stride,
    const int* seq_pos0, int S, int H, int KV, int hd, int ps, int window, int nsplit, float scale, hipStream_t stream) {
    MS_REQUIRE(S > 0 && H > 0 && hd > 0 && nsplit >= 1, "decode attention (no allocation): %d rows, %d heads, head size %d, %d splits",
               S, H, hd, nsplit);
    float* part_o = nullptr;
    float* part_ml = nullptr;
    if (nsplit > 1) {
        const double need = (double)S * H * nsplit * (hd + 2);
        MS_REQUIRE(need <= (double)NOALLOC_SCRATCH_FLOATS,
                   "decode attention (no allocation): %d rows x %d heads x %d splits x (%d + 2) floats = %.0f exceed the scratch of %zu floats",
                   S, H, nsplit, hd, need, NOALLOC_SCRATCH_FLOATS);
        float* base = scratch_of_current_device();
        if (!base) return 1;
        part_o = base;
        part_ml = base + (size_t)S * H * nsplit * hd;
    }
    return MS_CAT(ms_decode_attention_nd, MS_ATTN_ND)(q, kpool, vpool, out, part_o, part_ml, block_table, table_stride,
                                                      seq_pos0, S, H, KV, hd, ps, window, nsplit, scale, stream);
}
// The most floats of scratch a step may need.  The call also looks up the scratch's address on the current device
// (the set-up that the entry point would otherwise do at its first call there): a caller that is about to capture
// a stream calls this first, on each device it uses, and the entry point itself then makes nothing but launches.
extern "C" long MS_CAT(ms_decode_attention_noalloc_max_floats_nd, MS_ATTN_ND)() {
    (void)scratch_of_current_device();
    return (long)NOALLOC_SCRATCH_FLOATS;
}

// The same from the partial sums of the q/k/v projection: adds them and the bias, rotates q and k
// by the row's position, writes k and v into the row's page, and attends; a second launch merges
// the splits.  (Merging in the block that finishes last needs a device-wide fence in every block,
// which on this chip writes back a whole L2 and costs more than the launch it saves.)
// qkv is float [n_partials, S, stride] with the q heads, then the k heads, then the v heads.
extern "C" int MS_CAT(ms_decode_attention_fused_nd, MS_ATTN_ND)(
    const float* qkv, int n_partials, int stride, const float* bias, const float* inv_freq, const int* slot_map,
    void* kpool, void* vpool, void* out, float* part_o, float* part_ml, const int* block_table,
    int table_stride, const int* seq_pos0, int S, int H, int KV, int hd, int ps, int window, int nsplit, float scale,
    hipStream_t stream) {
    MS_REQUIRE(S > 0 && n_partials >= 1, "decode attention: no rows");
    MS_REQUIRE(hd % 16 == 0 && hd > 0 && hd <= HDT, "decode attention: head size %d does not fit this tile of %d", hd, HDT);
    MS_REQUIRE(KV > 0 && H % KV == 0 && H / KV <= 16, "decode attention: %d heads over %d key/value heads (at most 16 each)", H, KV);
    MS_REQUIRE(ps % 16 == 0 && ps > 0, "decode attention: page size %d must be a multiple of 16", ps);
    MS_REQUIRE(stride >= (H + 2 * KV) * hd, "decode attention: row stride %d too small", stride);
    MS_REQUIRE(nsplit >= 1 && nsplit <= MAX_SPLITS && (nsplit == 1 || (part_o && part_ml)), "decode attention: %d splits (at most %d)", nsplit, MAX_SPLITS);
    MS_REQUIRE(slot_map && kpool && vpool, "decode attention: the fused form writes the cache");
    DecodeArgs a{nullptr, (const elem_t*)kpool, (const elem_t*)vpool, (elem_t*)out, part_o, part_ml, block_table, seq_pos0,
                 table_stride, H, KV, hd, ps, window, nsplit, scale, qkv, bias, inv_freq, slot_map, n_partials, stride, nullptr, nullptr};
    const bool many = n_partials > 2, cut = nsplit > 1;
    auto form = [&](auto wide) {
        constexpr bool W = decltype(wide)::value;
        return many ? (cut ? decode_attention_kernel<true, true, true, W> : decode_attention_kernel<true, true, false, W>)
                    : (cut ? decode_attention_kernel<true, false, true, W> : decode_attention_kernel<true, false, false, W>);
    };
    auto kernel = form(std::false_type{});
    if constexpr (ND > 4)  // (of at most 1,024 columns the fifth is one that nobody uses: us, 12 heads over 2 of 128, one sum, five and four: 8 requests behind 33 keys 8.39 and 8.27,
                           // behind 2,048 12.62 and 12.45, 64 behind 120 10.53 and 10.43)
        if ((H / KV + 2) * hd > 1024) kernel = form(std::true_type{});
    hipLaunchKernelGGL(kernel, dim3((unsigned)S, (unsigned)KV, (unsigned)nsplit), dim3(256), 0, stream, a);
    int rc = check_launch("decode_attention_fused");
    if (rc || nsplit == 1) return rc;
    hipLaunchKernelGGL(decode_merge_kernel, dim3((unsigned)(S * H)), dim3(64), 0, stream, part_o, part_ml, (elem_t*)out, hd, nsplit, a.sinks, H, a.out_gate);
    return check_launch("decode_merge");
}

extern "C" int MS_CAT(ms_attention_key_tile_nd, MS_ATTN_ND)() { return DBKV; }  // of the decode kernel
