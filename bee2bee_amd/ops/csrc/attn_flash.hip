// Causal prompt attention: whole packed prompts, and query chunks against the
// paged history (query row j of sequence b stands at hist + j, hist =
// seq_lens[b] - its query length; the chunk's own keys are in the pages).
//
// What bounds it is the CU: the matrix cores, the exponentials beside them
// and the LDS reads that feed them, about equal in time.
//  * A workgroup takes the query rows of ALL heads that share a key head: row
//    = position * group + head, so that any group size and any chunk length
//    fill the 32-row tiles, and a key tile is read once for the group.
//  * Scores are computed transposed, S^T = K Q^T on 32x32x16 tiles: a lane
//    holds 16 keys of ONE query row, so that the row's maximum and sum are
//    in-lane (one exchange with lane + 32), and its weights are, as they
//    stand, the right operand of O^T = V^T P^T: no trip through LDS. That
//    product takes its 16 keys in the order the score tile holds them, which
//    the transposing LDS read of V follows.
//  * Keys and values are staged in LDS row-major (two buffers), 16-byte chunks
//    xor-ed by the key, the next tile's global reads in flight over the
//    current tile's products.
//  * 256 rows at head size 128 (TURNS): eight waves, two a SIMD, that take
//    turns: while one multiplies (O of the last tile, S of the next), the other
//    takes its maximum, weights and sum, with a barrier at each change. Left to
//    themselves both multiply, then both wait for the vector units: the sum of
//    the two times was 4400 clocks a tile of 64 keys, where each takes 2000 of
//    both waves; in turns it is 3400. Fragments are read two groups of products
//    ahead, tiles go straight to one of four LDS buffers two and three tiles
//    ahead (no registers, no divisions by the page size in the loop).
//  * At head size 128 the running maximum is raised only by a score FL_SLACK
//    powers of two above it: most tiles leave the sums as they are. Sums are
//    fp32, of the weights as rounded for the product, so that most of what
//    rounding does cancels.
// Scores are scaled in fp32 (queries enter the product unrounded). The kernel
// before it (16-row tiles, weights and V transposed through LDS by 2-byte
// writes) reached 97-170 TFLOP/s on the same shapes; this one: 4096 queries
// of 28 heads on 16384 keys 728 us (1155 TFLOP/s; 890 without turns), four
// prompts of 512 to 4096 tokens of 28 heads 215 (284 as 128 rows without
// turns), 2048 tokens of 32 heads 55 (59), nine prompts of 112 to 901 tokens
// 35. Without s_setprio for the multiplying waves 1 to 2% are lost.
#include "common.h"

#include <type_traits>

typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) short short4v;
typedef __attribute__((address_space(3))) short4v lds_short4v;

constexpr int FL_KT = 64;   // keys per staged tile
// a row's running maximum is raised only by a score this far (in powers of
// two) above it. A row's largest weight is then rounded like the others instead
// of being 1: of rows that few keys dominate the error grows (random scores of
// deviation 4, 300 keys, relative to 64 bits, before the output's rounding:
// 0.0005 without slack, 0.0008 with it). The kernel before, which rounded the
// scaled queries to bf16 and summed the unrounded weights, had 0.0033 at head
// size 128, but 0.0005 at 64, where the scale is a power of two: slack at 128
// only. It is worth 3 to 6% there (4096 queries on 16384 keys 918 us against
// 945, 700 on 7700 160 against 171), 1 to 3% at 64.
template <int HD> constexpr float FL_SLACK = HD == 128 ? 8.f : 0.f;

// 8 cache elements as they lie, widened when they are stored
DEV_INLINE bf16x8 fl_raw(const unsigned short* p) { return load_kv8_bf16(p); }
DEV_INLINE uint2v fl_raw(const unsigned char* p) {
    return *reinterpret_cast<const uint2v*>(p);
}
DEV_INLINE bf16x8 fl_bf16(bf16x8 r) { return r; }
DEV_INLINE bf16x8 fl_bf16(uint2v r) {
    return load_kv8_bf16(reinterpret_cast<const unsigned char*>(&r));
}

// 16 bytes a lane to LDS at `to` + lane * 16, from base + off. The compiler
// does not see these loads: the kernel waits for them itself.
DEV_INLINE void fl_load(const char* base, unsigned off, unsigned to) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\t"
                 "global_load_lds_dwordx4 %0, %1"
                 ::"v"(off), "s"(base), "s"(to) : "memory", "m0");
}

// A block: a sequence, its first query and their number, the tokens that it has
// with them, and which of its rows of tiles
struct FlBlock {
    int seq, s0, QL, L, tile;
};

// The order of a key head's blocks, those with many keys first (figures at
// attn_flash_order): row of tiles by row of tiles, the sequences as they stand, or
// turned by one from each row to the next, or by one more every `nseq` rows; or by the
// number of keys, which each workgroup works out, of up to 64 sequences.
enum { FL_STRAIGHT = 0, FL_TURNED = 1, FL_TURNED_MORE = 2, FL_BY_KEYS = 3 };

// The j-th block in that order, of sequences of up to `most` blocks of `rows` query
// rows; false: there is none
DEV_INLINE bool fl_block(const int* cu, const int* seq_lens, int nseq, int G,
                         int rows, int j, int most, int order, FlBlock& b) {
    if (order != FL_BY_KEYS) {
        const int up = j / nseq;
        const int turn = order == FL_STRAIGHT ? 0
                         : order == FL_TURNED ? up : up + up / nseq;
        b.tile = most - 1 - up;
        b.seq = (j + turn) % nseq;
        b.s0 = cu[b.seq];
        b.QL = cu[b.seq + 1] - b.s0;
        b.L = seq_lens ? seq_lens[b.seq] : b.QL;
        return b.tile * rows < b.QL * G;
    }
    const int lane = threadIdx.x & 63, at = min(lane, nseq - 1);
    const int s0 = cu[at], len = cu[at + 1] - s0;
    const int L = seq_lens ? seq_lens[at] : len;
    const int mine =
        lane < nseq ? min((max(len, 0) * G + rows - 1) / rows, most) : 0;
    // a block's level: rows of tiles before it, as if the history were queries
    const int low = max(L - len, 0) * G / rows;
    // blocks at level x and above, a lane a level: 64 at a time
    auto from = [&](int x) {
        int n = 0;
        for (int i = 0; i < nseq; ++i) {
            const int m = __builtin_amdgcn_readlane(mine, i);
            n += min(max(m + __builtin_amdgcn_readlane(low, i) - x, 0), m);
        }
        return n;
    };
    // (as many blocks behind as much history each: the search is 0.5 us more)
    const auto first_of = [](int x) { return __builtin_amdgcn_readfirstlane(x); };
    if (!__ballot(lane < nseq &&
                  (mine != first_of(mine) || low != first_of(low)))) {
        b.seq = j % nseq;
        b.s0 = __builtin_amdgcn_readlane(s0, b.seq);
        b.QL = __builtin_amdgcn_readlane(len, b.seq);
        b.L = __builtin_amdgcn_readlane(L, b.seq);
        b.tile = first_of(mine) - 1 - j / nseq;
        return b.tile >= 0;
    }
    int span = 1, lo = 0, above = 0;
    for (int i = 0; i < nseq; ++i)
        span = max(span, __builtin_amdgcn_readlane(mine + low, i));
    for (bool first = true; first || span > 1; first = false) {
        const int step = (span + 63) / 64, n = from(lo + lane * step);
        const unsigned long higher = __ballot(n > j);
        if (!higher) return false;             // (the first time)
        const int last = 63 - __builtin_clzl(higher);
        if (last < 63) above = __builtin_amdgcn_readlane(n, last + 1);
        lo += last * step;
        span = step;
    }
    // the (j - above)-th sequence that has one there
    const bool has = lo >= low && lo < low + mine;
    const unsigned long all = __ballot(has);
    const int before = __builtin_amdgcn_mbcnt_hi(
        (unsigned)(all >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)all, 0));
    b.seq = __builtin_ctzl(__ballot(has && before == j - above));
    b.s0 = __builtin_amdgcn_readlane(s0, b.seq);
    b.QL = __builtin_amdgcn_readlane(len, b.seq);
    b.L = __builtin_amdgcn_readlane(L, b.seq);
    b.tile = lo - __builtin_amdgcn_readlane(low, b.seq);
    return true;
}

// What one sequence's blocks beyond whole rounds of 256 workgroups are shared by
struct FlShare {
    int from;                  // the first of the 256 workgroups that share them
    float *o, *ml;             // [pieces, 256, 128], [pieces, 256, 2]
};
constexpr int FL_SHARERS = 256;

// Workgroup w of a key head's has tiles of its block t: from one such pair to the
// next w + t grows, so that this many places hold the pieces of `rest` blocks
__host__ __device__ constexpr long fl_pieces(long rest) {
    return FL_SHARERS + rest;
}
DEV_INLINE long fl_piece(int w, int t, int nkv, int kvh) {
    return (long)(w + t) * nkv + kvh;
}

// Whether `rest` blocks of a sequence of L tokens are shared: what it saves is half
// of the chip's idle part of a last round, as long as a block of all keys; pieces
// and their sums cost 50 us. us, whole / shared, 32/8 heads: 2100 on 2200 147 / 154
// (264 blocks), on 4000 232 / 206, on 8000 418 / 310, on 16000 808 / 555; 2500 (320) on 2600
// 185 / 188, on 8000 442 / 381; 28/4: 3150 (348) on 3200 228 / 252, on 8000 459 / 435, 5000
// (548) on 14000 1246 / 1035; 4096 (448) on 12288 779 / 845.
__host__ __device__ inline bool fl_worth(int rest, long L) {
    return rest > 0 && rest <= 96 && (256 - rest) * L >= 5800L * 256;
}

// tiles of 64 keys that the block `tile` of a sequence has
DEV_INLINE int fl_tiles(int tile, int rows, int G, int QL, int hist) {
    if (tile * rows >= QL * G) return 0;
    return (hist + min((tile + 1) * rows - 1, QL * G - 1) / G + FL_KT) / FL_KT;
}

// SHARE: one sequence; workgroups from share.from on take parts of the last blocks
template <int HD, int RW, int KSP, bool PAGED, bool TURNS, bool SHARE,
          typename KVT>
__global__ __launch_bounds__(RW * KSP * 64, 2) void attn_flash_kernel(
    const unsigned short* __restrict__ q, const KVT* __restrict__ k,
    const KVT* __restrict__ v, const int* __restrict__ cu,
    const int* __restrict__ block_table, const int* __restrict__ seq_lens,
    unsigned short* __restrict__ out, int blocks, int order, int nq, int nkv,
    long s_q, long s_k, long s_v, int W, int bs, int pairs, float scale_log2,
    const FlShare share) {
    constexpr int NW = RW * KSP;           // waves
    constexpr int ROWS = RW * 32;          // query rows of a workgroup
    constexpr int NF = 2 / KSP;            // 32-key tiles of a wave's step
    constexpr int KS = HD / 16;            // k steps of a score tile
    constexpr int DT = HD / 32;            // output tiles of 32 coordinates
    constexpr int CPR = HD / 8;            // 16-byte chunks of a key row
    constexpr int RB = HD * 2;             // bytes of a key row
    constexpr int RPT = NW * 64 / CPR;     // key rows staged at once
    constexpr int NST = FL_KT / RPT;       // staging steps of a tile
    constexpr int TILE = FL_KT * RB;       // bytes of a K or V tile
    static_assert(!TURNS || (HD == 128 && RW == 8 && KSP == 1), "");
    static_assert(FL_KT % RPT == 0, "whole staging steps");

    extern __shared__ __attribute__((aligned(16))) char smem[];
    // two buffers, or four, of a K and a V tile each
    // (numbers that are scalars, or what depends on them would be vectors: up to 9%
    // of a step)
    auto same = [](int x) { return __builtin_amdgcn_readfirstlane(x); };
    const int G = nq / nkv, kvh = blockIdx.x % nkv;

    // The tiles t0 .. t1 - 1 (t1 0: all) of a block; piece: where its sums go, -1:
    // they are the result
    auto block = [&](const int seq, const int s0, const int QL, const int L,
                     const int tile, const int t0, const int t1,
                     const int piece) __attribute__((always_inline)) {
    const int hist = L - QL;
    const int row0 = tile * ROWS;
    const int* bt = PAGED ? block_table + (long)seq * W : nullptr;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lr = lane & 31, hi = lane >> 5;
    const int rw = KSP == 1 ? wid : wid % RW;     // row block of the wave
    const int f0 = KSP == 1 ? 0 : wid / RW;       // its first 32-key tile

    // ---- this lane's query row
    const int R = row0 + rw * 32 + lr;
    const bool row_ok = R < QL * G;
    const int pos = row_ok ? R / G : QL - 1;       // chunk position
    const int head = kvh * G + (row_ok ? R % G : G - 1);
    bf16x8 bq[KS];
    {
        const unsigned short* qr = q + (long)(s0 + pos) * s_q + (long)head * HD;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
            bq[ks] = *reinterpret_cast<const bf16x8*>(qr + ks * 16 + hi * 8);
    }
    const int see = hist + pos;                    // last key this row sees
    // of the wave: the earliest row's last key, and the end of all its keys
    const int wr0 = row0 + rw * 32;
    const int w_first =
        __builtin_amdgcn_readfirstlane(hist + min(wr0, QL * G - 1) / G);
    const int w_end = __builtin_amdgcn_readfirstlane(
        wr0 < QL * G ? hist + min(wr0 + 31, QL * G - 1) / G + 1 : 0);
    const int kv_end = __builtin_amdgcn_readfirstlane(
        hist + min(row0 + ROWS - 1, QL * G - 1) / G + 1);

    // Chunks of a staged row are xor-ed so that no two lanes served together
    // meet in a bank. LDS serves 256 bytes a clock: 16 lanes of a 16-byte read
    // (16 keys, one chunk), 32 lanes of a transposing read (4 keys, two pairs
    // of chunks). With patterns made for 128 bytes a clock, 44% of the LDS
    // cycles were conflicts and 8192 tokens of 32 heads took 578 us, not 561.
    auto k_swz = [](int row) { return HD == 128 ? row & 15 : (row >> 1) & 7; };
    auto v_swz = [](int row) {
        return HD == 128 ? 4 * (row & 3) : 4 * ((row >> 1) & 1);
    };
    // ---- staging: thread -> (key row, chunk)
    const int st_row = tid / CPR, st_c = tid % CPR;
    typedef decltype(fl_raw((const KVT*)nullptr)) Raw;
    Raw rk[NST], rv[NST];
    // Tiles are loaded in order. Pages of whole tiles: a tile's page is one
    // scalar look-up, made a tile ahead.
    const bool whole_pages = PAGED && bs % FL_KT == 0;
    int page = 0, in_page = 0, page_at = 0;
    if (whole_pages && kv_end > 0) page = bt[0];
    auto load_tile = [&](int kb) {
        if (PAGED && !whole_pages) {
#pragma unroll
            for (int i = 0; i < NST; ++i) {
                const int key = min(kb + st_row + i * RPT, kv_end - 1);
                const long off = (((long)bt[key / bs] * nkv + kvh) * bs +
                                  key % bs) * HD + st_c * 8;
                rk[i] = fl_raw(k + off);
                rv[i] = fl_raw(v + off);
            }
            return;
        }
        const long off = PAGED ? (((long)page * nkv + kvh) * bs + in_page) * HD
                               : (long)kvh * HD;
        const KVT* kt = k + (PAGED ? off : off + (long)(s0 + kb) * s_k);
        const KVT* vt = v + (PAGED ? off : off + (long)(s0 + kb) * s_v);
#pragma unroll
        for (int i = 0; i < NST; ++i) {
            const int row = min(st_row + i * RPT, kv_end - 1 - kb);
            rk[i] = fl_raw(kt + (unsigned)(row * (PAGED ? HD : (int)s_k) +
                                           st_c * 8));
            rv[i] = fl_raw(vt + (unsigned)(row * (PAGED ? HD : (int)s_v) +
                                           st_c * 8));
        }
        if (PAGED && kb + FL_KT < kv_end && (in_page += FL_KT) == bs) {
            in_page = 0;
            page = bt[++page_at];
        }
    };
    auto store_tile = [&](int buf) {
        char* kd = smem + buf * 2 * TILE;
        char* vd = kd + TILE;
#pragma unroll
        for (int i = 0; i < NST; ++i) {
            const int row = st_row + i * RPT;
            *reinterpret_cast<bf16x8*>(
                kd + row * RB + ((st_c ^ k_swz(row)) << 4)) = fl_bf16(rk[i]);
            *reinterpret_cast<bf16x8*>(
                vd + row * RB + ((st_c ^ v_swz(row)) << 4)) = fl_bf16(rv[i]);
        }
    };

    // ---- fragment addresses
    // K (rows = keys): lane reads key lr of a 32-key tile, chunk 2 ks + hi
    const int k_base = lr * RB;
    const int k_sw = k_swz(lr);
    // V^T (rows = coordinates) through the transposing read: the 16 lanes of
    // a group address 4 keys x 16 coordinates
    const int v_key = 4 * hi + ((lane >> 2) & 3);
    const int v_c0 = ((lane >> 4) & 1) * 2 + ((lane & 3) >> 1);
    const int v_sw = v_swz(v_key);
    int v_off[DT];
#pragma unroll
    for (int d = 0; d < DT; ++d)
        v_off[d] = TILE + v_key * RB + (((d * 4 + v_c0) ^ v_sw) << 4) +
                   (lane & 1) * 8;

    f32x16 o[DT];
#pragma unroll
    for (int d = 0; d < DT; ++d)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[d][r] = 0.f;
    float m = -1e30f, l = 0.f;

    // ---- S^T = K Q^T: column = query row, rows = keys
    f32x16 s[NF];
    auto scores = [&](const char* base) {
#pragma unroll
        for (int f = 0; f < NF; ++f) {
#pragma unroll
            for (int r = 0; r < 16; ++r) s[f][r] = 0.f;
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
                const bf16x8 ak = *reinterpret_cast<const bf16x8*>(
                    base + (f0 + f) * 32 * RB + k_base +
                    (((ks * 2 + hi) ^ k_sw) << 4));
                s[f] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ak, bq[ks],
                                                               s[f], 0, 0, 0);
            }
        }
    };
    // ---- online softmax, in powers of two, of the tile at key kb
    bf16x8 bp[NF * 2];
    auto maximum = [&](int kb) {
        if (kb + FL_KT - 1 > w_first) {
#pragma unroll
            for (int f = 0; f < NF; ++f)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int key =
                        kb + (f0 + f) * 32 + (r & 3) + 8 * (r >> 2) + 4 * hi;
                    if (key > see) s[f][r] = -INFINITY;
                }
        }
        float mx = s[0][0];
#pragma unroll
        for (int f = 0; f < NF; ++f)
#pragma unroll
            for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[f][r]);
        mx = pair_max(mx) * scale_log2;
        if (__any(mx > m + FL_SLACK<HD>)) {
            const float mn = fmaxf(m, mx);
            const float alpha = __builtin_amdgcn_exp2f(m - mn);
            m = mn;
            l *= alpha;
#pragma unroll
            for (int d = 0; d < DT; ++d)
#pragma unroll
                for (int r = 0; r < 16; ++r) o[d][r] *= alpha;
        }
    };
    auto weight = [&](int st, int e) {
        bp[st][e] = (__bf16)__builtin_amdgcn_exp2f(
            fmaf(s[st / 2][st % 2 * 8 + e], scale_log2, -m));
    };
    auto weights = [&](int kb) {
        maximum(kb);
#pragma unroll
        for (int st = 0; st < NF * 2; ++st)
#pragma unroll
            for (int e = 0; e < 8; ++e) weight(st, e);
        // the sum that divides is of the weights as they are multiplied
#pragma unroll
        for (int st = 0; st < NF * 2; ++st) l = add_bf16x8(bp[st], l);
    };
    // ---- O^T += V^T P^T; the keys of a step in the order the score tile holds
    // them: 4 hi + {0..3}, then 8 + 4 hi + {0..3}
    auto outputs = [&](const char* base) {
#pragma unroll
        for (int st = 0; st < NF * 2; ++st)
#pragma unroll
            for (int d = 0; d < DT; ++d) {
                const char* va = base + v_off[d] + (f0 * 2 + st) * 16 * RB;
                const short4v a0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                    (lds_short4v*)va);
                const short4v a1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                    (lds_short4v*)(va + 8 * RB));
                const short8 av = __builtin_shufflevector(a0, a1, 0, 1, 2, 3,
                                                          4, 5, 6, 7);
                o[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                    __builtin_bit_cast(bf16x8, av), bp[st], o[d], 0, 0, 0);
            }
    };

    if constexpr (TURNS) {
        // Two waves a SIMD: while one multiplies, O of the last tile and S of
        // this one, the other takes its weights.
        constexpr bool DIRECT = sizeof(KVT) == 2;
        // The first 32 keys' weights are taken before the turn ends, and kept from
        // moving to where they are multiplied. Against pages the other 32 keys'
        // follow two after each product of the first, in its shadow: 4096 queries
        // of 28 heads on 16384 keys 743 -> 728 us (fp8 776 -> 762), two portions
        // of 700 on 8400 198 -> 190, 512 of 32 heads on 8512 197 -> 188. Whole
        // prompts are faster with them before the turn's end, as far as the
        // compiler leaves them there (four of 512 to 4096 236, against 242).
        constexpr bool SHADOW = PAGED;
        auto turn = [&]() {
            __builtin_amdgcn_sched_barrier(0);
            asm volatile("s_barrier" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
        };
        auto tile_at = [&](int t) { return smem + (t & 3) * 2 * TILE; };
        // bf16 goes straight to LDS: a wave's loads are 4 rows of 256 bytes,
        // lane l the 16 bytes that belong at l * 16
        const int nt = (kv_end + FL_KT - 1) / FL_KT, te = SHARE ? t1 : nt;
        unsigned off[2][2][NST];               // K, V; a whole tile, the last
#pragma unroll
        for (int i = 0; i < NST; ++i) {
            const int row = (i * 8 + wid) * 4 + (lane >> 4);
            const int left = kv_end - 1 - (nt - 1) * FL_KT;
            const int kc = ((lane & 15) ^ k_swz(row)) << 4;
            const int vc = ((lane & 15) ^ v_swz(row)) << 4;
            const int ks = PAGED ? RB : (int)s_k * 2;
            const int vs = PAGED ? RB : (int)s_v * 2;
            off[0][0][i] = row * ks + kc;
            off[1][0][i] = row * vs + vc;
            // (rows past the last: its)
            off[0][1][i] = min(row, left) * ks + kc;
            off[1][1][i] = min(row, left) * vs + vc;
        }
        const unsigned lds =
            (unsigned)(unsigned long)(__attribute__((address_space(3)))
                                          const char*)smem + wid * 1024;
        // Tiles are asked for in order, K's one ahead of V's: where the next
        // ones lie in memory and in LDS, and what is left of K's page.
        const char *k_src = nullptr, *v_src = nullptr, *v_next = nullptr;
        int k_to = (t0 & 3) * 2 * TILE, v_to = k_to + TILE, k_left = 0, k_at = 0;
        auto page_of = [&](const KVT* pool, int b) {
            return reinterpret_cast<const char*>(
                pool + ((long)b * nkv + kvh) * bs * HD);
        };
        if (DIRECT && nt > 0) {
            if (PAGED) {
                k_at = t0 * FL_KT / bs;
                const int b = bt[k_at], in = t0 * FL_KT - k_at * bs;
                k_src = page_of(k, b) + in * RB;
                v_src = page_of(v, b) + in * RB;
                k_left = bs - in;
            } else {
                k_src = reinterpret_cast<const char*>(
                    k + (long)s0 * s_k + (long)kvh * HD);
                v_src = reinterpret_cast<const char*>(
                    v + (long)s0 * s_v + (long)kvh * HD);
            }
            v_next = v_src;
        }
        int new_page = 0;                      // asked for a turn ahead
        auto load_k = [&](int t) {
            if (t >= te) return;
            if (t + 1 == nt)
#pragma unroll
                for (int i = 0; i < NST; ++i) off[0][0][i] = off[0][1][i];
            if (PAGED && k_left == 0) {
                k_src = page_of(k, new_page);
                v_next = page_of(v, new_page);
                k_left = bs;
            }
#pragma unroll
            for (int i = 0; i < NST; ++i)
                fl_load(k_src, off[0][0][i], lds + k_to + i * 8192);
            k_to = (k_to + 2 * TILE) & (8 * TILE - 1);
            k_src += PAGED ? FL_KT * RB : s_k * FL_KT * 2;
            if (PAGED && (k_left -= FL_KT) == 0 && t + 1 < nt)
                new_page = bt[++k_at];
        };
        auto load_v = [&](int t) {
            if (t >= te) return;
            if (t + 1 == nt)
#pragma unroll
                for (int i = 0; i < NST; ++i) off[1][0][i] = off[1][1][i];
            v_src = v_next;
#pragma unroll
            for (int i = 0; i < NST; ++i)
                fl_load(v_src, off[1][0][i], lds + v_to + i * 8192);
            v_to = (v_to + 2 * TILE) & (8 * TILE - 1);
            v_next = v_src + (PAGED ? FL_KT * RB : s_v * FL_KT * 2);
        };
        // Fragments: four groups of V for the products of O, then KS / 2 of K
        // for S, each read two groups ahead.
        bf16x8 fr[3][4];
        auto read_v = [&](const char* base, int g) {
#pragma unroll
            for (int d = 0; d < DT; ++d) {
                const char* va = base + v_off[d] + g * 16 * RB;
                const short4v a0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                    (lds_short4v*)va);
                const short4v a1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                    (lds_short4v*)(va + 8 * RB));
                fr[g % 3][d] = __builtin_bit_cast(
                    bf16x8, __builtin_shufflevector(a0, a1, 0, 1, 2, 3, 4, 5,
                                                    6, 7));
            }
        };
        auto read_k = [&](const char* base, int g) {
#pragma unroll
            for (int e = 0; e < 4; ++e)        // two steps of both key tiles
                fr[(g + 4) % 3][e] = *reinterpret_cast<const bf16x8*>(
                    base + (e & 1) * 32 * RB + k_base +
                    (((g * 4 + e / 2 * 2 + hi) ^ k_sw) << 4));
        };
        auto make_o = [&](const char* vb, auto more, const char* kb_) {
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                if (g < 2) read_v(vb, g + 2);
                else if (decltype(more)::value) read_k(kb_, g - 2);
#pragma unroll
                for (int d = 0; d < DT; ++d) {
                    o[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                        fr[g % 3][d], bp[g], o[d], 0, 0, 0);
                    if (!SHADOW) continue;
                    if (g < 2) {
                        weight(g + 2, d * 2);
                        weight(g + 2, d * 2 + 1);
                    } else if (d == 0) {
                        l = add_bf16x8(bp[g], l);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        auto make_s = [&](const char* kb_) {
#pragma unroll
            for (int g = 0; g < KS / 2; ++g) {
                if (g + 2 < KS / 2) read_k(kb_, g + 2);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    f32x16 z;
#pragma unroll
                    for (int r = 0; r < 16; ++r) z[r] = 0.f;
                    s[e & 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                        fr[(g + 4) % 3][e], bq[g * 2 + e / 2],
                        g == 0 && e < 2 ? z : s[e & 1], 0, 0, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        auto first_weights = [&](int kb) {
            maximum(kb);
#pragma unroll
            for (int st = 0; st < (SHADOW ? 2 : 4); ++st)
#pragma unroll
                for (int e = 0; e < 8; ++e) weight(st, e);
#pragma unroll
            for (int st = 0; st < 2; ++st) {
                f32x4 u = __builtin_bit_cast(f32x4, bp[st]);
                asm volatile("" : "+v"(u));
                bp[st] = __builtin_bit_cast(bf16x8, u);
            }
#pragma unroll
            for (int st = 0; st < (SHADOW ? 2 : 4); ++st)
                l = add_bf16x8(bp[st], l);
        };
        if (nt > 0) {
            if (DIRECT) {
                load_k(t0);
                load_v(t0);
                load_k(t0 + 1);
                load_v(t0 + 1);
                load_k(t0 + 2);
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            } else {
                load_tile(0);
                store_tile(0);
                if (nt > 1) {
                    load_tile(FL_KT);
                    store_tile(1);
                }
                if (nt > 2) load_tile(2 * FL_KT);
                __builtin_amdgcn_s_waitcnt(0xc07f);
            }
            turn();
            if (wid >= 4) turn();
            read_k(tile_at(t0), 0);
            read_k(tile_at(t0), 1);
            make_s(tile_at(t0));
            turn();
            for (int t = t0; t + 1 < te; ++t) {
                // V of tile t + 2 takes the place of t - 2's, K of t + 3 that
                // of t - 1's: their last readers were in the turn before. What
                // the last such turn asked for has come by the end of this.
                if (DIRECT) {
                    load_v(t + 2);
                    load_k(t + 3);
                } else {
                    if (t + 2 < nt) store_tile((t + 2) & 3);
                    if (t + 3 < nt) load_tile((t + 3) * FL_KT);
                }
                first_weights(t * FL_KT);
                if (!DIRECT) __builtin_amdgcn_s_waitcnt(0xc07f);
                read_v(tile_at(t), 0);
                read_v(tile_at(t), 1);
                if (DIRECT) {
                    if (t + 3 < te)
                        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * NST)
                                     : "memory");
                    else
                        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                }
                turn();
                __builtin_amdgcn_s_setprio(1);
                make_o(tile_at(t), std::true_type(), tile_at(t + 1));
                make_s(tile_at(t + 1));
                __builtin_amdgcn_s_setprio(0);
                turn();
            }
            first_weights((te - 1) * FL_KT);
            read_v(tile_at(te - 1), 0);
            read_v(tile_at(te - 1), 1);
            make_o(tile_at(te - 1), std::false_type(), nullptr);
            if (wid < 4) turn();
        }
    } else {
        if (kv_end > 0) {
            load_tile(0);
            store_tile(0);
        }
        int buf = 0;
        for (int kb = 0; kb < kv_end; kb += FL_KT, buf ^= 1) {
            __syncthreads();
            const bool more = kb + FL_KT < kv_end;
            if (more) load_tile(kb + FL_KT);
            if (kb < w_end) {
                const char* base = smem + buf * 2 * TILE;
                scores(base);
                weights(kb);
                outputs(base);
            }
            if (more) store_tile(buf ^ 1);
        }
    }

    l = pair_sum(l);
    if (KSP == 2) {
        // the halves' sums meet in LDS (over the tiles): [row block][lane]
        // columns of DT * 16 sums, then m and l
        float* mg = reinterpret_cast<float*>(smem) + rw * (DT * 16 + 2) * 64 +
                    lane;
        __syncthreads();
        if (f0 == 1) {
#pragma unroll
            for (int d = 0; d < DT; ++d)
#pragma unroll
                for (int r = 0; r < 16; ++r) mg[(d * 16 + r) * 64] = o[d][r];
            mg[DT * 16 * 64] = m;
            mg[(DT * 16 + 1) * 64] = l;
        }
        __syncthreads();
        if (f0 == 1) return;
        const float m1 = mg[DT * 16 * 64];
        const float mn = fmaxf(m, m1);
        const float a0 = __builtin_amdgcn_exp2f(m - mn);
        const float a1 = __builtin_amdgcn_exp2f(m1 - mn);
        l = l * a0 + mg[(DT * 16 + 1) * 64] * a1;
#pragma unroll
        for (int d = 0; d < DT; ++d)
#pragma unroll
            for (int r = 0; r < 16; ++r)
                o[d][r] = o[d][r] * a0 + mg[(d * 16 + r) * 64] * a1;
    }
    if (SHARE && piece >= 0) {
        const int row = rw * 32 + lr;
        float* to = share.o + ((long)piece * ROWS + row) * HD;
#pragma unroll
        for (int d = 0; d < DT; ++d)
#pragma unroll
            for (int r4 = 0; r4 < 4; ++r4)
                *reinterpret_cast<f32x4*>(to + d * 32 + r4 * 8 + hi * 4) =
                    f32x4{o[d][r4 * 4], o[d][r4 * 4 + 1], o[d][r4 * 4 + 2],
                          o[d][r4 * 4 + 3]};
        if (hi == 0) {
            share.ml[((long)piece * ROWS + row) * 2] = m;
            share.ml[((long)piece * ROWS + row) * 2 + 1] = l;
        }
        return;
    }
    if (!row_ok) return;
    const float inv = l == 0.f ? 0.f : 1.f / l;
    unsigned short* orow = out + ((long)(s0 + pos) * nq + head) * HD;
#pragma unroll
    for (int d = 0; d < DT; ++d)
#pragma unroll
        for (int r4 = 0; r4 < 4; ++r4) {
            short4v w;
#pragma unroll
            for (int e = 0; e < 4; ++e)
                w[e] = (short)f2bf(o[d][r4 * 4 + e] * inv);
            *reinterpret_cast<short4v*>(orow + d * 32 + r4 * 8 + hi * 4) = w;
        }
    };

    const bool shared =
        SHARE && fl_worth(blocks - share.from, seq_lens[0]);
    if (SHARE && !shared && blockIdx.x >= (unsigned)blocks) return;
    if (!shared || blockIdx.x < (unsigned)share.from) {
        // workgroups go round the 8 dies in turn: heads fastest, so that a key
        // head stays on few of them, and long rows of tiles first
        FlBlock at;
        if (SHARE) {
            at.seq = 0;
            at.s0 = cu[0];
            at.QL = cu[1] - at.s0;
            at.L = seq_lens[0];
            at.tile = blocks / nkv - 1 - blockIdx.x / nkv;
            if (at.tile * ROWS >= at.QL * G) return;
        } else if (!fl_block(cu, PAGED ? seq_lens : nullptr, pairs / nkv, G, ROWS,
                             blockIdx.x / nkv, blocks / pairs, order, at)) {
            return;
        }
        const int QL = same(at.QL), L = same(at.L), tile = same(at.tile);
        const int hist = L - QL;
        block(same(at.seq), same(at.s0), QL, L, tile, 0,
              SHARE ? fl_tiles(tile, ROWS, G, QL, hist) : 0, -1);
        return;
    }
    if constexpr (SHARE) {
        const int s0 = cu[0], QL = cu[1] - s0, L = seq_lens[0], hist = L - QL;
        const int rest = (blocks - share.from) / nkv;
        const int sharers = FL_SHARERS / nkv;
        const int mine = (blockIdx.x - share.from) / nkv;
        int total = 0;
        for (int t = 0; t < rest; ++t) total += fl_tiles(t, ROWS, G, QL, hist);
        const int lo = (long)total * mine / sharers;
        const int hi_ = (long)total * (mine + 1) / sharers;
        int before = 0;
        for (int t = 0; t < rest && before < hi_; ++t) {
            const int n = fl_tiles(t, ROWS, G, QL, hist);
            const int a = max(lo - before, 0), b = min(hi_ - before, n);
            before += n;
            if (a >= b) continue;
            block(0, s0, QL, L, t, a, b,
                  a == 0 && b == n ? -1 : (int)fl_piece(mine, t, nkv, kvh));
            __syncthreads();                   // the tiles are read
        }
    }
}

// The pieces of shared blocks: workgroup = (block, 8 of its rows), 32 threads a
// row, 4 coordinates each
__global__ __launch_bounds__(256) void attn_flash_join_kernel(
    const FlShare share, const int* __restrict__ cu,
    const int* __restrict__ seq_lens, unsigned short* __restrict__ out, int nq,
    int nkv, int blocks) {
    constexpr int ROWS = 256, HD = 128;
    const int G = nq / nkv;
    if (!fl_worth(blocks - share.from, seq_lens[0])) return;
    const int s0 = cu[0], QL = cu[1] - s0, hist = seq_lens[0] - QL;
    const int kvh = blockIdx.x / 32 % nkv, tile = blockIdx.x / 32 / nkv;
    const int rest = (blocks - share.from) / nkv, sharers = FL_SHARERS / nkv;
    int total = 0, before = 0;
    for (int t = 0; t < rest; ++t) {
        if (t == tile) before = total;
        total += fl_tiles(t, ROWS, G, QL, hist);
    }
    const int n = fl_tiles(tile, ROWS, G, QL, hist);
    const int row = blockIdx.x % 32 * 8 + threadIdx.x / 32;
    const int c = threadIdx.x % 32 * 4, R = tile * ROWS + row;
    if (n == 0 || R >= QL * G) return;
    // who has the block's first tile
    int w = (long)before * sharers / total;
    while ((long)total * (w + 1) / sharers <= before) ++w;
    if ((long)total * (w + 1) / sharers >= before + n) return;   // and all others
    float M = -1e30f, sum = 0.f;
    f32x4 acc{0.f, 0.f, 0.f, 0.f};
    for (; (long)total * w / sharers < before + n; ++w) {
        if ((long)total * (w + 1) / sharers == (long)total * w / sharers)
            continue;                          // (fewer tiles than sharers)
        const long at = fl_piece(w, tile, nkv, kvh) * ROWS + row;
        const float m = share.ml[at * 2], l = share.ml[at * 2 + 1];
        const f32x4 o = *reinterpret_cast<const f32x4*>(share.o + at * HD + c);
        const float mn = fmaxf(M, m);
        const float old = __builtin_amdgcn_exp2f(M - mn);
        const float now = __builtin_amdgcn_exp2f(m - mn);
        M = mn;
        sum = sum * old + l * now;
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[e] = acc[e] * old + o[e] * now;
    }
    const float inv = sum == 0.f ? 0.f : 1.f / sum;
    short4v y;
#pragma unroll
    for (int e = 0; e < 4; ++e) y[e] = (short)f2bf(acc[e] * inv);
    *reinterpret_cast<short4v*>(
        out + ((long)(s0 + R / G) * nq + kvh * G + R % G) * HD + c) = y;
}

// ------------------------------------------------------------- launchers

static int flash_smem(int hd, int rw, int ksp, bool turns) {
    const int tiles = (turns ? 8 : 4) * FL_KT * hd * 2;
    const int merge = ksp == 2 ? rw * (hd / 2 + 2) * 64 * 4 : 0;
    return tiles > merge ? tiles : merge;
}

// Shape of a workgroup by how many of 256 rows the step fills (`full`,
// T * nq / 256; a CU holds one such workgroup at head size 128, two at 64):
// 256 rows read a key tile from memory least often, at head size 128 take
// turns at the matrix cores, and win where there are enough of them and their
// tiles are about as long as each other (one long prompt's, in falling order, or
// portions behind long histories); with fewer, 128 rows balance better, with
// less than a chip of those 64 rows, whose two wave pairs share a tile's keys.
// Prompts of different lengths leave tiles of every length to balance: 256 rows
// need more of them the more prompts there are, and, as measured, more again
// from eight prompts on where seven or eight heads share a key head. Three
// prompts, and few of one length (`level`), want more of them than two or four
// of different lengths.
// Measured (us, 256 / 128 / 64 rows; heads 32/8 unless stated), head size 128:
//   one prompt: full 150 35/34/30, 190 42/44/40, 230 50/53/56, 350 77/83/102,
//    600 192/212/261, 1000 466/553/687;
//   2 of an eighth to 1: 150 31/32/39, 600 233/286/399; of one length 150
//    22/20/18, 230 29/30/33, 450 62/74/88;
//   3: 229 33/31/30 (28/4: 37/35/34), 299 46/46/50 (45/46/49), 600 104/110/139;
//   4: 149 21/20/28 (28/4: 23/22/20), 189 27/28/36 (26/27/27), 299 50/52/71
//    (36/41/49), 1000 317/392/550; of one length 230 20/19/24, 300 26/24/34, 450
//    42/45/56;
//   9: 149 14/13.6/16, 449 39/34/46 (28/4: 53/45/69), 999 106/99/140, 1399
//    170/179/242 (28/4: 311/285/439, 64/8: 113/107/150; of one length 149/147/200,
//    28/4 157/162/224), 2000 322/349/470 (28/4: 590/582/833, 64/8: 207/197/276),
//    2800 581/664/871 (976/1106/1561, 346/361/492); 16: 2000 246/250/355 (28/4:
//    249/242/338, 64/8: 179/160/229), 2800 409/456/648 (429/460/618, 277/272/395);
//   30: 1000 65/59/78, 2000 165/156/220, 2800 267/263/375;
//   8000 cached: 120 206/206/187, 140 210/261/334, 256 287/330/393, 400
//    489/597/732, 1000 1372/1612/1999; 500 cached: 120 42/37/33, 140 45/44/40,
//    185 54/53/59, 300 82/84/106, 600 235/250/307; without turns (pages of 48):
//    8000 140 269/295/359, 300 534/517/596, 350 579/545/678, 400 605/655/827;
//    500 140 54/49/45, 185 66/59/68, 256 90/78/90, 300 95/91/118, 350
//    112/121/146, 600 272/269/354;
// head size 64:
//   one prompt: 300 53/47/44 (12/12: 139/121/106), 350 64/56/57, 600
//    134/128/144, 1000 306/313/373; 9 prompts: 300 17/15/16 (12/12: 34/30/26),
//    600 30/29/34, 1000 61/60/76 (12/12: 146/137/169); 2: 600 152/155/193;
//   8000 cached: 150 176/177/160, 230 193/192/216, 300 286/264/286, 400
//    328/357/386, 1000 843/914/1083.
static int flash_shape(int hd, long T, int nseq, int nq, int nkv, int max_qlen,
                       bool pages, bool turns) {
    const long full = T * nq / 256;
    const bool lone = !pages && nseq == 1;
    if (hd == 128 && pages) {
        if (full >= (turns ? 140 : 380)) return 0;
        return full >= 140 ? 1 : 2;
    }
    if (hd == 128) {
        const bool level = 4 * T >= 3L * nseq * max_qlen;
        long least = 150L * nseq;
        if (lone) least = 210;
        else if (nseq <= 4 && (level || nseq == 3)) least = 90 * nseq;
        else if (nseq <= 4) least = nseq == 2 ? 150 : 180;
        else if (nseq >= 8 && nq >= 7 * nkv && !level) {
            const long more = 240L * nseq < 2200 ? 240L * nseq : 2200;
            least = more > least ? more : least;
        }
        if (full >= least) return 0;
        return full >= 115 && !lone ? 1 : 2;
    }
    if (full >= (pages ? 400 : 700)) return 0;
    return full >= (lone ? 320 : pages ? 185 : 230) ? 1 : 2;
}

// whole tiles in a page, in pieces that go straight to LDS
static bool flash_turns(int hd, bool pages, int bs, bool aligned) {
    return hd == 128 && (!pages || (bs % FL_KT == 0 && aligned));
}

// What a step of these sizes runs on: the workgroup's rows (256, 128 or 64), + 1
// where its waves take turns. bs: keys of a page, 0 for packed prompts.
extern "C" int attn_flash_form(long T, int nseq, int nq, int nkv, int hd,
                               int max_qlen, int bs) {
    const bool turns = flash_turns(hd, bs > 0, bs, true);
    const int shape =
        flash_shape(hd, T, nseq, nq, nkv, max_qlen, bs > 0, turns);
    return (256 >> shape) + (shape == 0 && turns);
}

// The order of a step's blocks. The chip deals workgroups out to its eight dies in
// turn and a die's to its four parts, and one that finds its part full holds up those
// behind it: a long sequence's blocks should be on all parts, and a sequence's on one
// die, whose L2 then has its keys. From one row of tiles to the next a sequence moves
// on by nseq * nkv workgroups, turned by (nseq - 1) * nkv. Where that is an odd number
// of times 8, its die stays and its part changes: turned; an odd number of sequences of
// other sizes moves on by itself. Even ones are turned, where a row of tiles goes round
// all dies (nkv a multiple of 8) by one more each time round; of twelve and more, which
// share parts by threes, only in large steps.
// By keys, each workgroup looks at all sequences, 0.3 to 1 us of its time: two, four and
// six prompts of different lengths, for which turning is not enough, and portions, whose
// histories the host does not know, of up to eight sequences; not small steps, nor
// prompts of about one length.
// us, straight / turned (by one more) / by keys, an eighth of the longest up to it: 2
// prompts of up to 2500 tokens of 32/8 heads 94.9 / 67.7 / 67.4, 4 175 / 106 / 99, 6 157 / 149
// / 144, 8 of up to 1000 60.0 / 46.6 / 48.3, 12 80.6 / 67.9 / 71.5; 28/4, 9 of up to 1600 93 /
// 137 / 96, 7 of up to 700 27.3 / 25.2 / 26.0; 12/12 of 64, 7 of up to 2500 71.6 / 59.1 / 57.6,
// 5 56.1 / 62.5 / 53.1; small and level ones of 32/8, 4 of up to 64 6.1 / 6.2 / 6.6, 2 of 200
// 8.5 / 8.4 / 8.7; portions of 32/8, 1000 tokens on 0 to 4000, 3 168 / - / 135, 4 218 / 211 / 161, 4
// on 4000 269 / 269 / 271, 8 of 64 on 100 9.1 / 9.1 / 9.9.
extern "C" int attn_flash_order(long T, int nseq, int nq, int nkv, int max_qlen,
                                bool pages) {
    const long full = T * nq / 256;
    const bool level = 4 * T >= 3L * nseq * max_qlen;
    if (nseq == 1) return FL_STRAIGHT;
    if (pages ? nseq <= 8 && full >= 80
              : nseq % 2 == 0 && nseq <= 6 && !level && full >= 40)
        return FL_BY_KEYS;
    if (nkv % 8 == 0)
        return nseq % 2 || full < (nseq >= 12 ? 600 : pages ? 80 : 0)
                   ? FL_STRAIGHT : FL_TURNED_MORE;
    return nseq % 2 == 0 || (nseq - 1) * nkv % 16 == 8 ? FL_TURNED : FL_STRAIGHT;
}

// Workgroups of a step that take whole blocks where 256 more share the rest, 0:
// all take whole ones. One portion, of bf16 pages: its blocks are about as long as
// each other, and what is left over whole rounds of 256 takes as long as a round.
// W * bs: the most tokens that it may have; the kernel looks at those it has.
extern "C" int attn_flash_share(int nseq, int nq, int nkv, int hd, int max_qlen,
                                int W, int bs, int fp8, int shape256) {
    if (nseq != 1 || hd != 128 || fp8 || !shape256 || FL_SHARERS % nkv) return 0;
    const long blocks = ((long)max_qlen * (nq / nkv) + 255) / 256 * nkv;
    const long rest = blocks % 256;
    if (blocks < 256 || blocks > 1 << 20 || !fl_worth(rest, (long)W * bs))
        return 0;
    return (int)(blocks - rest);
}

// fp32 numbers that a step's pieces take, 0: it has none
extern "C" long attn_flash_pieces(long T, int nseq, int nq, int nkv, int hd,
                                  int max_qlen, int W, int bs, int fp8) {
    const bool turns = flash_turns(hd, true, bs, true);
    if (nseq != 1 || max_qlen < 1 || !turns) return 0;
    const int shape = flash_shape(hd, T, nseq, nq, nkv, max_qlen, true, turns);
    const int from =
        attn_flash_share(nseq, nq, nkv, hd, max_qlen, W, bs, fp8, shape == 0);
    const long blocks = ((long)max_qlen * (nq / nkv) + 255) / 256 * nkv;
    return from ? fl_pieces(blocks - from) * 256 * (128 + 2) : 0;
}

#define FL_ONE(HDV, RWV, KSPV, PG, TU, KVT)                                   \
    do {                                                                      \
        const int blocks = (rows + RWV * 32 - 1) / (RWV * 32) * pairs;        \
        hipLaunchKernelGGL(                                                   \
            (attn_flash_kernel<HDV, RWV, KSPV, PG, TU, false, KVT>),          \
            dim3((unsigned)blocks), dim3(RWV * KSPV * 64),                    \
            flash_smem(HDV, RWV, KSPV, TU), stream, q, (const KVT*)k,         \
            (const KVT*)v, cu, block_table, seq_lens, out, blocks, order, nq, \
            nkv, s_q, s_k, s_v, W, bs, pairs, scale * LOG2E, FlShare{});      \
    } while (0)
#define FL_HD(HDV, PG, KVT)                                                   \
    do {                                                                      \
        if (shape == 0 && HDV == 128 && turns)                                \
            FL_ONE(HDV, 8, 1, PG, HDV == 128, KVT);                           \
        else if (shape == 0) FL_ONE(HDV, 8, 1, PG, false, KVT);               \
        else if (shape == 1) FL_ONE(HDV, 4, 1, PG, false, KVT);               \
        else FL_ONE(HDV, 2, 2, PG, false, KVT);                               \
    } while (0)

constexpr float LOG2E = 1.44269504088896340736f;

// Whole packed prompts, or (block_table given) query chunks whose keys come
// from the pages only, bf16 or fp8 bytes. T: query tokens of the step. Head
// size 64 or 128 and a positive scale (a row's maximum is taken before it);
// keys and values of packed prompts 16-byte aligned, row strides multiples of 8
// below 2^24 (a tile's offsets are of 32 bits). Nonzero for any other.
extern "C" int launch_attn_flash(
    const unsigned short* q, const void* k, const void* v, const int* cu,
    const int* block_table, const int* seq_lens, unsigned short* out,
    float* pieces, long T, int nseq, int nq, int nkv, int hd, long s_q, long s_k,
    long s_v, int W, int bs, int max_qlen, float scale, int fp8,
    hipStream_t stream) {
    if ((hd != 64 && hd != 128) || !(scale > 0.f)) return 1;
    const bool aligned = ((unsigned long)k | (unsigned long)v) % 16 == 0;
    if (!block_table && (!aligned || s_k % 8 || s_v % 8 || s_k >= 1 << 24 ||
                         s_v >= 1 << 24))
        return 1;
    if (nseq == 0 || max_qlen <= 0) return 0;
    const int pairs = nseq * nkv;
    const long rows = (long)max_qlen * (nq / nkv);
    const bool turns = flash_turns(hd, block_table, bs, aligned);
    const int shape =
        flash_shape(hd, T, nseq, nq, nkv, max_qlen, block_table, turns);
    const int from = pieces ? attn_flash_share(nseq, nq, nkv, hd, max_qlen, W, bs,
                                               fp8, shape == 0 && turns)
                            : 0;
    if (from && block_table) {
        const int blocks = (int)((rows + 255) / 256 * pairs);
        const FlShare share{from, pieces + fl_pieces(blocks - from) * 256 * 2,
                            pieces};
        hipLaunchKernelGGL(
            (attn_flash_kernel<128, 8, 1, true, true, true, unsigned short>),
            dim3(from + FL_SHARERS), dim3(512), flash_smem(128, 8, 1, true),
            stream, q, (const unsigned short*)k, (const unsigned short*)v, cu,
            block_table, seq_lens, out, blocks, FL_STRAIGHT, nq, nkv, s_q, s_k,
            s_v, W, bs, pairs, scale * LOG2E, share);
        hipLaunchKernelGGL(attn_flash_join_kernel, dim3((blocks - from) * 32),
                           dim3(256), 0, stream, share, cu, seq_lens, out, nq,
                           nkv, blocks);
        return 0;
    }
    const int order =
        attn_flash_order(T, nseq, nq, nkv, max_qlen, block_table != nullptr);
    if (!block_table) {
        if (hd == 128) FL_HD(128, false, unsigned short);
        else FL_HD(64, false, unsigned short);
    } else if (fp8) {
        if (hd == 128) FL_HD(128, true, unsigned char);
        else FL_HD(64, true, unsigned char);
    } else {
        if (hd == 128) FL_HD(128, true, unsigned short);
        else FL_HD(64, true, unsigned short);
    }
    return 0;
}
#undef FL_HD
#undef FL_ONE
