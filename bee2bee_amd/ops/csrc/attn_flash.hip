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
//  * At head size 128 the running maximum is raised only by a score FL_SLACK
//    powers of two above it: most tiles leave the sums as they are. Sums are
//    fp32, of the weights as rounded for the product, so that most of what
//    rounding does cancels.
// Scores are scaled in fp32 (queries enter the product unrounded). The kernel
// before it (16-row tiles, weights and V transposed through LDS by 2-byte
// writes) reached 97-170 TFLOP/s on the same shapes; this one: 4096 queries
// of 28 heads on 16384 keys 860 us instead of 5240 (980 TFLOP/s), 2048 tokens
// of 32 heads 63 us instead of 386 (540), nine prompts of 112 to 901 tokens
// 38 us instead of 140. Neither fetching key fragments two steps ahead by hand
// nor computing the next tile's scores beside this one's exponentials (with
// or without a forced interleaving) made it faster: at 980 TFLOP/s the clock
// has come down to 1.75 GHz.
#include "common.h"

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

template <int HD, int RW, int KSP, bool PAGED, typename KVT>
__global__ __launch_bounds__(RW * KSP * 64, 2) void attn_flash_kernel(
    const unsigned short* __restrict__ q, const KVT* __restrict__ k,
    const KVT* __restrict__ v, const int* __restrict__ cu,
    const int* __restrict__ block_table, const int* __restrict__ seq_lens,
    unsigned short* __restrict__ out, int nq, int nkv, long s_q, long s_k,
    long s_v, int W, int bs, int pairs, float scale_log2) {
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
    static_assert(FL_KT % RPT == 0, "whole staging steps");

    // workgroups go round the 8 dies in turn: heads fastest, so that a key
    // head stays on few of them, long rows of tiles first, and the sequences
    // rotated from one tile to the next, so that a long one is on all
    const int nseq = pairs / nkv;
    const int up = blockIdx.x / pairs, tile = gridDim.x / pairs - 1 - up;
    const int seq =
        (blockIdx.x % pairs / nkv + (nkv % 8 ? up : 0)) % nseq;
    const int kvh = blockIdx.x % nkv;
    const int G = nq / nkv;
    const int s0 = cu[seq], QL = cu[seq + 1] - s0;
    const int L = PAGED ? seq_lens[seq] : QL;
    const int hist = L - QL;
    const int row0 = tile * ROWS;
    if (row0 >= QL * G) return;
    const int* bt = PAGED ? block_table + (long)seq * W : nullptr;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lr = lane & 31, hi = lane >> 5;
    const int rw = KSP == 1 ? wid : wid % RW;     // row block of the wave
    const int f0 = KSP == 1 ? 0 : wid / RW;       // its first 32-key tile

    extern __shared__ __attribute__((aligned(16))) char smem[];
    // two buffers of a K and a V tile each

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
    const int w_first = hist + min(wr0, QL * G - 1) / G;
    const int w_end =
        wr0 < QL * G ? hist + min(wr0 + 31, QL * G - 1) / G + 1 : 0;
    const int kv_end = hist + min(row0 + ROWS - 1, QL * G - 1) / G + 1;

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
    bf16x8 rk[NST], rv[NST];
    // pages of whole tiles: a tile's page is one scalar look-up
    const bool whole_pages = PAGED && bs % FL_KT == 0;
    auto load_tile = [&](int kb) {
        long tile_off = 0;
        if (whole_pages)
            tile_off =
                (((long)bt[kb / bs] * nkv + kvh) * bs + kb % bs) * HD;
#pragma unroll
        for (int i = 0; i < NST; ++i) {
            const int key = min(kb + st_row + i * RPT, kv_end - 1);
            if (PAGED) {
                const long off =
                    (whole_pages
                         ? tile_off + (long)(key - kb) * HD
                         : (((long)bt[key / bs] * nkv + kvh) * bs +
                            key % bs) * HD) +
                    st_c * 8;
                rk[i] = load_kv8_bf16(k + off);
                rv[i] = load_kv8_bf16(v + off);
            } else {
                rk[i] = load_kv8_bf16(k + (long)(s0 + key) * s_k +
                                      (long)kvh * HD + st_c * 8);
                rv[i] = load_kv8_bf16(v + (long)(s0 + key) * s_v +
                                      (long)kvh * HD + st_c * 8);
            }
        }
    };
    auto store_tile = [&](int buf) {
        char* kd = smem + buf * 2 * TILE;
        char* vd = kd + TILE;
#pragma unroll
        for (int i = 0; i < NST; ++i) {
            const int row = st_row + i * RPT;
            *reinterpret_cast<bf16x8*>(kd + row * RB +
                                       ((st_c ^ k_swz(row)) << 4)) = rk[i];
            *reinterpret_cast<bf16x8*>(
                vd + row * RB + ((st_c ^ v_swz(row)) << 4)) = rv[i];
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
            // ---- S^T = K Q^T: column = query row, rows = keys
            f32x16 s[NF];
#pragma unroll
            for (int f = 0; f < NF; ++f) {
#pragma unroll
                for (int r = 0; r < 16; ++r) s[f][r] = 0.f;
#pragma unroll
                for (int ks = 0; ks < KS; ++ks) {
                    const bf16x8 ak = *reinterpret_cast<const bf16x8*>(
                        base + (f0 + f) * 32 * RB + k_base +
                        (((ks * 2 + hi) ^ k_sw) << 4));
                    s[f] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                        ak, bq[ks], s[f], 0, 0, 0);
                }
            }
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
            // ---- online softmax, in powers of two
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
            bf16x8 bp[NF * 2];
#pragma unroll
            for (int f = 0; f < NF; ++f)
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    bp[f * 2 + r / 8][r % 8] = (__bf16)__builtin_amdgcn_exp2f(
                        fmaf(s[f][r], scale_log2, -m));
            // the sum that divides is of the weights as they are multiplied
#pragma unroll
            for (int st = 0; st < NF * 2; ++st) l = add_bf16x8(bp[st], l);
            // ---- O^T += V^T P^T; the keys of a step in the order the score
            // tile holds them: 4 hi + {0..3}, then 8 + 4 hi + {0..3}
#pragma unroll
            for (int st = 0; st < NF * 2; ++st)
#pragma unroll
                for (int d = 0; d < DT; ++d) {
                    const char* va =
                        base + v_off[d] + (f0 * 2 + st) * 16 * RB;
                    const short4v a0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                        (lds_short4v*)va);
                    const short4v a1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                        (lds_short4v*)(va + 8 * RB));
                    const short8 av = __builtin_shufflevector(
                        a0, a1, 0, 1, 2, 3, 4, 5, 6, 7);
                    o[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                        __builtin_bit_cast(bf16x8, av), bp[st], o[d], 0, 0, 0);
                }
        }
        if (more) store_tile(buf ^ 1);
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
}

// ------------------------------------------------------------- launchers

static int flash_smem(int hd, int rw, int ksp) {
    const int tiles = 4 * FL_KT * hd * 2;
    const int merge = ksp == 2 ? rw * (hd / 2 + 2) * 64 * 4 : 0;
    return tiles > merge ? tiles : merge;
}

// Shape of a workgroup by how many of 256 rows the step fills (`full`,
// T * nq / 256; a CU holds one such workgroup at head size 128, two at 64):
// 256 rows read a key tile from memory least often and win where there are
// enough of them and their tiles are about as long as each other (one long
// prompt's, in falling order, or portions behind long histories); with fewer,
// 128 rows balance better, with less than a chip of those 64 rows, whose two
// wave pairs share a tile's keys. Prompts of different lengths leave tiles of
// every length to balance: 256 rows need 256 fillings a prompt.
// Measured (us, 256 / 128 / 64 rows; heads 32/8 unless stated), head size 128:
//   one prompt: full 150 42/34/30, 256 70/57/63, 350 92/85/101, 400 107/108/127,
//    450 121/135/159, 600 218/214/268, 1000 534/549/709;
//   9 prompts of an eighth to 1: 100 12.9/12.3/10.4, 149 15/14/17, 450
//    38/34/46 (28/4: 59/45/71), 1000 116/102/141 (28/4: 215/167/248), 1400
//    191/183/247; 4 prompts: 124 22/19/24, 600 171/161/224, 1000 412/405/561,
//    2000 1525/1521/2078;
//   8000 cached: 100 263/220/186, 150 275/288/347, 256 322/346/421, 300
//    518/503/559, 350 548/527/619, 400 573/632/767, 600 946/930/1143, 1000
//    1537/1681/2123;
// head size 64:
//   one prompt: 300 54/46/45 (12/12: 140/117/107), 350 64/55/56, 600
//    135/132/147, 750 184/191/221; 9 prompts: 200 15.2/10.7/11 (12/12:
//    23/21/17), 600 31/30/34, 1000 59/60/72 (12/12: 151/146/180); 2: 600
//    157/171/202;
//   8000 cached: 150 193/187/169, 200 205/195/215, 300 297/272/303, 400
//    338/391/402, 520 491/476/543, 1000 863/951/1127.
static int flash_shape(int hd, long full, int nseq, bool pages) {
    const bool lone = !pages && nseq == 1;
    if (hd == 128) {
        if (full >= 400 && (pages || full >= 256L * nseq)) return 0;
        return full >= (lone ? 230 : pages ? 140 : 115) ? 1 : 2;
    }
    if (full >= (pages ? 400 : 700)) return 0;
    return full >= (lone ? 320 : pages ? 185 : 230) ? 1 : 2;
}

#define FL_ONE(HDV, RWV, KSPV, PG, KVT)                                       \
    hipLaunchKernelGGL(                                                       \
        (attn_flash_kernel<HDV, RWV, KSPV, PG, KVT>),                         \
        dim3((unsigned)((rows + RWV * 32 - 1) / (RWV * 32) * pairs)),         \
        dim3(RWV * KSPV * 64), flash_smem(HDV, RWV, KSPV), stream, q,         \
        (const KVT*)k, (const KVT*)v, cu, block_table, seq_lens, out, nq,     \
        nkv, s_q, s_k, s_v, W, bs, pairs, scale * LOG2E)
#define FL_HD(HDV, PG, KVT)                                                   \
    do {                                                                      \
        if (shape == 0) FL_ONE(HDV, 8, 1, PG, KVT);                           \
        else if (shape == 1) FL_ONE(HDV, 4, 1, PG, KVT);                      \
        else FL_ONE(HDV, 2, 2, PG, KVT);                                      \
    } while (0)

constexpr float LOG2E = 1.44269504088896340736f;

// Whole packed prompts, or (block_table given) query chunks whose keys come
// from the pages only, bf16 or fp8 bytes. T: query tokens of the step. Head
// size 64 or 128 and a positive scale (a row's maximum is taken before it);
// nonzero for any other.
extern "C" int launch_attn_flash(
    const unsigned short* q, const void* k, const void* v, const int* cu,
    const int* block_table, const int* seq_lens, unsigned short* out, long T,
    int nseq, int nq, int nkv, int hd, long s_q, long s_k, long s_v, int W,
    int bs, int max_qlen, float scale, int fp8, hipStream_t stream) {
    if ((hd != 64 && hd != 128) || !(scale > 0.f)) return 1;
    if (nseq == 0 || max_qlen <= 0) return 0;
    const int pairs = nseq * nkv;
    const long rows = (long)max_qlen * (nq / nkv);
    const int shape = flash_shape(hd, T * nq / 256, nseq, block_table);
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
