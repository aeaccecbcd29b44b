// Paged attention of a few query rows per sequence: decode steps, and the
// chunks of a few tokens that speculative decoding verifies.
//
// Bound by reading the cache once. A wave takes tiles of 32 keys on its own:
// whole 16-byte chunks of neighbouring rows into registers (1 KB a load, with
// the streaming hint where the block table has room for more than 6 MB of keys
// and values: 1536 sequences below 653 us without it; 8 of 500 tokens, 8 heads of
// 128, 8.8 against 10.0 where no cache holds them. One sequence of 300 or 1000
// tokens takes the same time with it, 6.4 to 7.5, but a step that finds its pages
// in a cache is slower: six layers of 12 heads of 64, 300 keys, 190 us against
// 187), on to its part of LDS, the next tile's loads on their way over the
// products of this one, no barrier before the end. Scores are S^T = K Q^T on 16x16x32
// matrix tiles (a column is a query row; the rows of all heads that share the
// key head, times the chunk's tokens), so that the weights are, as they
// stand, the right operand of O^T = V^T P^T, whose keys follow the score
// tile's order through the transposing LDS read. One pass over K and V: no
// weights written, no second kernel unless the context is split over
// workgroups (their fp32 sums, combined). fp8 rows are widened to bf16 on
// their way into LDS (decode queries are rounded to fp8 like them, chunks'
// are not).
// Measured against the kernels before it (scores, weights through memory,
// values, combine): 1536 sequences of 137..1100 tokens, 8 key heads of size
// 128: 595 us (6.55 TB/s) instead of 778; fp8 337 (5.8) instead of 588; 200
// sequences of up to 3000 fp8 120 instead of 228 (122.8 with 8 bytes a lane);
// one of 3000 8.5 instead of 15.3; 16 sequences' 5 tokens on 1500 24 instead
// of 166. Loads two tiles ahead gain nothing on fp8 rows (121) and spill on
// others. A CU draws 45 to 57 GB/s of what no cache holds, from 32 KB under way on,
// so that what is left to gain are CUs without work: longer contexts start first
// (figures at decode_plan). Whole pages are told at compile time: with the look-up of
// a key's page in the loop, for pages that tiles cross, a step of a wave was 697
// instructions, of which 300 are left (200 sequences of up to 3000 fp8 121 -> 118 us,
// 16 sequences' 5 tokens on 1500 23.8 -> 23.5, 8 of 4000 20.7 -> 20.0).
#include "common.h"

typedef __attribute__((ext_vector_type(4))) short short4v;
typedef __attribute__((address_space(3))) short4v lds_short4v;

// Eight waves of a context gain 3 to 16% in uneven batches that start in the order
// of their lengths, and lose elsewhere: such a workgroup has a CU to itself. us, four /
// eight waves, 8 key heads of size 128, 24, 40 and 64 sequences: of 250 to 2000 tokens
// by length 27.4 / 24.1, 38.6 / 35.4, 52.3 / 49.0; of 2000 38.2 / 40.5, 64.7 / 67.4,
// 82.5 / 83.8; of 200 10.1 / 11.8, 11.8 / 13.6, 13.6 / 16.4; of 5 to 40 6.1 / 6.0, 6.8 /
// 8.9, 7.4 / 10.4; fp8 pages, 17 of 2000 21.3 / 25.7, 20 of 200 9.8 / 12.4, 40 of 250 to
// 2000 by length 25.5 / 22.0. The lengths are on the GPU, so no rule tells them apart.
constexpr int ST_WAVES = 4;
constexpr int ST_KEYS = 32;                      // keys of a wave's tile
constexpr int ST_STEP = ST_WAVES * ST_KEYS;      // keys of a workgroup's step
constexpr float ST_LOG2E = 1.44269504088896340736f;

// 16 bytes of a row, as read
typedef __attribute__((ext_vector_type(4))) unsigned int st_raw;

DEV_INLINE short8 st_widen(uint2v x) {
    typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
    bf16x8 r;
    const unsigned int w[2] = {x[0], x[1]};
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const bf16x2 a =
            __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w[i], 1.f, false);
        const bf16x2 b =
            __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w[i], 1.f, true);
        r[i * 4] = a[0];
        r[i * 4 + 1] = a[1];
        r[i * 4 + 2] = b[0];
        r[i * 4 + 3] = b[1];
    }
    return __builtin_bit_cast(short8, r);
}

template <bool STREAM> DEV_INLINE st_raw st_load(const st_raw* p) {
    if constexpr (STREAM) return __builtin_nontemporal_load(p);
    else return *p;
}

// elements 8 p .. 8 p + 7 of a load, in bf16
template <typename KVT> DEV_INLINE short8 st_piece(st_raw x, int p) {
    if constexpr (sizeof(KVT) == 2) return __builtin_bit_cast(short8, x);
    else return st_widen(uint2v{x[p * 2], x[p * 2 + 1]});
}

// 8 queries times the score scale, rounded to fp8
DEV_INLINE bf16x8 st_round_fp8(bf16x8 x, float scale) {
    float f[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) f[e] = (float)(__bf16)((float)x[e] * scale);
    uint2v w;
#pragma unroll
    for (int i = 0; i < 2; ++i)
        w[i] = f2fp8x2(f[i * 4], f[i * 4 + 1]) |
               (unsigned int)f2fp8x2(f[i * 4 + 2], f[i * 4 + 3]) << 16;
    return __builtin_bit_cast(bf16x8, st_widen(w));
}

// keys per split, the same for every reader: a context in `even` parts of whole
// steps of a workgroup, none above `most` keys (whole steps too)
DEV_INLINE int split_keys(int L, int even, int most) {
    return min(((L + even - 1) / even + ST_STEP - 1) / ST_STEP * ST_STEP, most);
}

// WHOLE: bs is a multiple of ST_KEYS, so that no tile crosses pages
template <int HD, int QT, typename KVT, bool STREAM, bool WHOLE>
__global__ __launch_bounds__(ST_WAVES * 64, 2) void attn_stream_kernel(
    const unsigned short* __restrict__ q, const KVT* __restrict__ k_cache,
    const KVT* __restrict__ v_cache, const int* __restrict__ cu,
    const int* __restrict__ block_table, const int* __restrict__ seq_lens,
    const int* __restrict__ order, unsigned short* __restrict__ out,
    float* __restrict__ out_ml, float* __restrict__ part_o,
    float* __restrict__ part_ml, int nkv, int G, int W, int bs, int Z, int even,
    int most, int max_rows, long s_q, float scale) {
    constexpr int KS = HD / 32;          // k steps of a score tile
    constexpr int DT = HD / 16;          // output tiles of 16 coordinates
    constexpr int PC = 2 / sizeof(KVT);  // chunks of 8 elements of a load
    constexpr int CPR = HD / 8 / PC;     // loads of a key row
    constexpr int RB = HD * 2;           // bytes of a staged row
    constexpr int RPI = 64 / CPR;        // rows a wave loads at once
    constexpr int NL = ST_KEYS / RPI;    // loads of a tile
    constexpr int TILE = ST_KEYS * RB;
    // chunks of a staged row are xor-ed so that the lanes LDS serves together
    // (256 bytes a clock: 16 keys of one chunk; 8 keys of one pair of chunks)
    // meet in no bank
    auto k_swz = [](int row) { return HD == 128 ? row & 15 : (row >> 1) & 7; };
    auto v_swz = [](int row) {
        return 2 * (HD == 128 ? row & 7 : (row >> 1) & 3);
    };

    const int at = blockIdx.x / nkv, kvh = blockIdx.x % nkv;
    const int b = order ? order[at] : at;
    const int s0 = cu ? cu[b] : b;
    const int rows = (cu ? cu[b + 1] - s0 : 1) * G;
    const int row0 = blockIdx.z * QT * 16;
    // a chunk longer than the caller said has no room in the workspaces
    const int live = min(rows, max_rows);
    if (row0 >= live) return;
    const int L = min(seq_lens[b], W * bs);    // (what its pages hold)
    const int hist = L - rows / G;
    const int per = split_keys(L, even, most);
    const bool split = L > per;          // or the result itself is written
    const int k0 = blockIdx.y * per, k1 = min(L, k0 + per);
    if (k0 >= L && blockIdx.y > 0) return;
    const int* bt = block_table + (long)b * W;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int li = lane & 15, lg = lane >> 4;

    extern __shared__ __attribute__((aligned(16))) char smem[];
    char* kd = smem + wid * 2 * TILE;    // this wave's K tile, then its V tile

    // decoding on an 8-bit cache, scaled queries are of its type too
    const bool round_q = sizeof(KVT) == 1 && !cu;
    const float scale_log2 = round_q ? ST_LOG2E : scale * ST_LOG2E;

    // ---- query rows: column li of tile qt is row row0 + qt * 16 + li
    bf16x8 bq[QT][KS];
    int see[QT];                         // last key of the row
    long q_off[QT];                      // of the row's output
#pragma unroll
    for (int t = 0; t < QT; ++t) {
        const int r = min(row0 + t * 16 + li, rows - 1);
        const int pos = r / G, head = kvh * G + r % G;
        const unsigned short* qr =
            q + (long)(s0 + pos) * s_q + (long)head * HD;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
            bq[t][ks] =
                *reinterpret_cast<const bf16x8*>(qr + ks * 32 + lg * 8);
        see[t] = hist + pos;
        q_off[t] = (long)(s0 + pos) * nkv * G + head;
    }
    const int first_see = hist + row0 / G;

    // ---- loading: lane -> (row of RPI, PC chunks). Each row is read once on
    // the chip (query rows past 32 aside), so it is only streamed through L2.
    const int ld_row = lane / CPR, ld_c = lane % CPR * PC;
    st_raw rk[NL], rv[NL];
    auto load = [&](int i, const KVT* k, const KVT* v, long off) {
        rk[i] = st_load<STREAM>(reinterpret_cast<const st_raw*>(k + off));
        rv[i] = st_load<STREAM>(reinterpret_cast<const st_raw*>(v + off));
    };
    auto load_tile = [&](int kb) {
        if constexpr (WHOLE) {
            // a tile inside one page: the page is a scalar look-up, and a lane's
            // rows lie at 32-bit offsets from it
            const int page = bt[kb / bs];
            BB_KASSERT(page >= 0);
            const long base =
                (((long)page * nkv + kvh) * bs + kb % bs) * HD;
            const int most = k1 - 1 - kb;
#pragma unroll
            for (int i = 0; i < NL; ++i)
                load(i, k_cache + base, v_cache + base,
                     (unsigned)(min(ld_row + i * RPI, most) * HD + ld_c * 8));
        } else {
#pragma unroll
            for (int i = 0; i < NL; ++i) {
                const int key = min(kb + ld_row + i * RPI, k1 - 1);
                const int page = bt[key / bs];
                BB_KASSERT(page >= 0);
                load(i, k_cache, v_cache,
                     (((long)page * nkv + kvh) * bs + key % bs) * HD +
                         ld_c * 8);
            }
        }
    };

    // ---- fragment addresses: K row li (+ 16), chunk ks * 4 + lg; V through
    // the transposing read, 16 lanes on 4 keys x 16 coordinates
    const int k_base = li * RB, k_sw = k_swz(li);
    const int v_key = lg * 4 + (li >> 2);
    const int v_sw = v_swz(v_key);
    const int v_base = TILE + v_key * RB + (lane & 1) * 8;
    const int v_c = (lane & 3) >> 1;

    f32x4 o[DT][QT];
    float m[QT], l[QT];
#pragma unroll
    for (int t = 0; t < QT; ++t) {
        m[t] = -1e30f;
        l[t] = 0.f;
#pragma unroll
        for (int d = 0; d < DT; ++d) o[d][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    }

    int kb = k0 + wid * ST_KEYS;
    if (kb < k1) load_tile(kb);
    // (what the loop needs is worked out behind these loads, not before them: one
    // context of 2000 tokens 8.3 -> 8.0 us, 16 of 25 to 200 8.3 -> 7.8, 200 of 200 32.7
    // -> 29.7, fp8 one of 2000 8.3 -> 8.2)
    __builtin_amdgcn_sched_barrier(0);
    if (round_q && kb < k1)
#pragma unroll
        for (int t = 0; t < QT; ++t)
#pragma unroll
            for (int ks = 0; ks < KS; ++ks)
                bq[t][ks] = st_round_fp8(bq[t][ks], scale);
    for (; kb < k1; kb += ST_STEP) {
        // ---- registers -> LDS (16-byte chunks xor-ed by the key), and the
        // next tile's loads on their way over this tile's products
#pragma unroll
        for (int i = 0; i < NL; ++i) {
            const int row = ld_row + i * RPI;
#pragma unroll
            for (int p = 0; p < PC; ++p) {
                *reinterpret_cast<short8*>(
                    kd + row * RB + (((ld_c + p) ^ k_swz(row)) << 4)) =
                    st_piece<KVT>(rk[i], p);
                *reinterpret_cast<short8*>(
                    kd + TILE + row * RB + (((ld_c + p) ^ v_swz(row)) << 4)) =
                    st_piece<KVT>(rv[i], p);
            }
        }
        if (kb + ST_STEP < k1) load_tile(kb + ST_STEP);
        WAVE_LDS_SYNC();

        // ---- S^T = K Q^T: column = query row, rows = 16 keys
        f32x4 s[2][QT];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            bf16x8 ak[KS];
#pragma unroll
            for (int ks = 0; ks < KS; ++ks)
                ak[ks] = *reinterpret_cast<const bf16x8*>(
                    kd + h * 16 * RB + k_base +
                    (((ks * 4 + lg) ^ k_sw) << 4));
#pragma unroll
            for (int t = 0; t < QT; ++t) {
                s[h][t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int ks = 0; ks < KS; ++ks)
                    s[h][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                        ak[ks], bq[t][ks], s[h][t], 0, 0, 0);
            }
        }
        if (kb + ST_KEYS - 1 > first_see) {
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int t = 0; t < QT; ++t)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        if (kb + h * 16 + lg * 4 + r > see[t])
                            s[h][t][r] = -INFINITY;
        }

        // ---- online softmax, in powers of two
        bf16x8 bp[QT];
#pragma unroll
        for (int t = 0; t < QT; ++t) {
            float mx = s[0][t][0];
#pragma unroll
            for (int r = 0; r < 4; ++r)
                mx = fmaxf(fmaxf(mx, s[0][t][r]), s[1][t][r]);
            mx = rows_max(mx) * scale_log2;
            const float mn = fmaxf(m[t], mx);
            if (__any(mn > m[t])) {
                const float alpha = __builtin_amdgcn_exp2f(m[t] - mn);
                m[t] = mn;
                l[t] *= alpha;
#pragma unroll
                for (int d = 0; d < DT; ++d)
#pragma unroll
                    for (int r = 0; r < 4; ++r) o[d][t][r] *= alpha;
            }
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    bp[t][h * 4 + r] = (__bf16)__builtin_amdgcn_exp2f(
                        fmaf(s[h][t][r], scale_log2, -m[t]));
            // the sum that divides is of the weights as they are multiplied:
            // what rounding does to both cancels
            l[t] = add_bf16x8(bp[t], l[t]);
        }
        // ---- O^T += V^T P^T; keys in the order the score tiles hold them:
        // lane group lg has 4 lg + {0..3}, then 16 + 4 lg + {0..3}
#pragma unroll
        for (int d = 0; d < DT; ++d) {
            const char* va = kd + v_base + (((d * 2 + v_c) ^ v_sw) << 4);
            const short4v a0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                (lds_short4v*)va);
            const short4v a1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                (lds_short4v*)(va + 16 * RB));
            const bf16x8 av = __builtin_bit_cast(
                bf16x8, __builtin_shufflevector(a0, a1, 0, 1, 2, 3, 4, 5, 6,
                                                7));
#pragma unroll
            for (int t = 0; t < QT; ++t)
                o[d][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                    av, bp[t], o[d][t], 0, 0, 0);
        }
        WAVE_LDS_SYNC();
    }

    // ---- the four waves' sums meet in LDS: each leaves m, l and O in its
    // own tiles
    float* mine = reinterpret_cast<float*>(kd);
#pragma unroll
    for (int t = 0; t < QT; ++t) {
        l[t] = rows_sum(l[t]);
#pragma unroll
        for (int d = 0; d < DT; ++d)
            *reinterpret_cast<f32x4*>(mine + ((t * DT + d) * 64 + lane) * 4) =
                o[d][t];
    }
    float* ml_s = reinterpret_cast<float*>(smem + ST_WAVES * 2 * TILE);
    if (lg == 0) {
#pragma unroll
        for (int t = 0; t < QT; ++t) {
            ml_s[((t * 16 + li) * ST_WAVES + wid) * 2] = m[t];
            ml_s[((t * 16 + li) * ST_WAVES + wid) * 2 + 1] = l[t];
        }
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < QT; ++t) {
        if (row0 + t * 16 + li >= live) continue;
        float wm[ST_WAVES], M = -1e30f, lsum = 0.f;
#pragma unroll
        for (int w = 0; w < ST_WAVES; ++w) {
            wm[w] = ml_s[((t * 16 + li) * ST_WAVES + w) * 2];
            M = fmaxf(M, wm[w]);
        }
#pragma unroll
        for (int w = 0; w < ST_WAVES; ++w) {
            wm[w] = __builtin_amdgcn_exp2f(wm[w] - M);
            lsum += wm[w] * ml_s[((t * 16 + li) * ST_WAVES + w) * 2 + 1];
        }
        const long part =
            (((long)b * nkv + kvh) * Z + blockIdx.y) * max_rows + row0 +
            t * 16 + li;
        if (wid == 0 && lg == 0) {
            if (split) {
                part_ml[part * 2] = M;
                part_ml[part * 2 + 1] = lsum;
            } else if (out_ml) {
                out_ml[q_off[t] * 2] = M / ST_LOG2E;
                out_ml[q_off[t] * 2 + 1] = lsum;
            }
        }
        // (no keys: zeros; a NaN is neither less nor greater and stays one)
        const float inv = lsum == 0.f ? 0.f : 1.f / lsum;
        for (int d = wid; d < DT; d += ST_WAVES) {
            f32x4 a{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int w = 0; w < ST_WAVES; ++w) {
                const f32x4 x = *reinterpret_cast<const f32x4*>(
                    smem + w * 2 * TILE + ((t * DT + d) * 64 + lane) * 16);
#pragma unroll
                for (int r = 0; r < 4; ++r) a[r] += x[r] * wm[w];
            }
            if (split) {
                *reinterpret_cast<f32x4*>(part_o + part * HD + d * 16 +
                                          lg * 4) = a;
            } else {
                short4v w;
#pragma unroll
                for (int r = 0; r < 4; ++r) w[r] = (short)f2bf(a[r] * inv);
                *reinterpret_cast<short4v*>(out + q_off[t] * HD + d * 16 +
                                            lg * 4) = w;
            }
        }
    }
}

// The splits' sums of one row: workgroup = (sequence and key head, row). A
// chain of loads and nothing else, so each wave takes the at most 32 maxima
// and sums in one load, a lane a split, and P splits are read at once, 4
// coordinates a thread: every load is under way before the first is used. With
// a thread a coordinate and a loop over the splits 32 splits of 7 rows took
// 10.8 us, 8 groups of them, and 4.7 now; 6.2 and 4.8 with 4 rows. Up to 4
// splits take one wave a row (2 splits of 20 rows, 128 groups: 4.9, 5.6 with
// four).
template <int HD, int P, int I>
__global__ __launch_bounds__(HD / 4 * P) void attn_stream_combine_kernel(
    const float* __restrict__ part_o, const float* __restrict__ part_ml,
    const int* __restrict__ cu, const int* __restrict__ seq_lens,
    unsigned short* __restrict__ out, float* __restrict__ out_ml, int nkv,
    int G, int pages, int Z, int even, int most, int max_rows) {
    constexpr int C = HD / 4;                  // threads of a split
    const int b = blockIdx.x / nkv, kvh = blockIdx.x % nkv;
    const int s0 = cu ? cu[b] : b;
    const int row = blockIdx.y;
    if (row >= (cu ? cu[b + 1] - s0 : 1) * G) return;
    const int L = min(seq_lens[b], pages);
    const int per = split_keys(L, even, most);
    if (L <= per) return;                      // written by its workgroup
    const int nz = (L + per - 1) / per;
    const long p0 = (long)blockIdx.x * Z * max_rows + row;
    const int lane = threadIdx.x & 63, c = threadIdx.x % C;
    const int z0 = threadIdx.x / C;            // 0 .. P - 1
    f32x4 o[I];                                // P * I >= Z
#pragma unroll
    for (int i = 0; i < I; ++i) {
        o[i] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (z0 + i * P < nz)
            o[i] = *reinterpret_cast<const f32x4*>(
                part_o + (p0 + (long)(z0 + i * P) * max_rows) * HD + c * 4);
    }
    float m = -1e30f, l = 0.f;
    if (lane < nz) {
        const float2 ml = *reinterpret_cast<const float2*>(
            part_ml + (p0 + (long)lane * max_rows) * 2);
        m = ml.x;
        l = ml.y;
    }
    const float M = wave_max(m);
    const float w = __builtin_amdgcn_exp2f(m - M);
    const float lsum = wave_sum(w * l);
    f32x4 acc{};
#pragma unroll
    for (int i = 0; i < I; ++i) {
        const float wz = __shfl(w, z0 + i * P);
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[r] = fmaf(wz, o[i][r], acc[r]);
    }
    __shared__ f32x4 sums[P][C];
    sums[z0][c] = acc;
    __syncthreads();
    if (z0) return;
#pragma unroll
    for (int i = 1; i < P; ++i) {
        const f32x4 t = sums[i][c];
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[r] += t[r];
    }
    const long at = (long)(s0 + row / G) * nkv * G + kvh * G + row % G;
    short4v y;
#pragma unroll
    for (int r = 0; r < 4; ++r)
        y[r] = (short)f2bf(lsum == 0.f ? 0.f : acc[r] / lsum);
    *reinterpret_cast<short4v*>(out + at * HD + c * 4) = y;
    if (out_ml && c == 0) {
        out_ml[at * 2] = M / ST_LOG2E;
        out_ml[at * 2 + 1] = lsum;
    }
}

// Workgroups of a step that take one (sequence, key head) and up to 32 query
// rows each.
static long stream_groups(long pairs, long rows) {
    return pairs * ((rows + 31) / 32);
}

// Query chunks against the pages: this kernel, or attn_flash.hip's. This one
// fills the chip with splits of the context where there are few rows; the
// other reads a key once for 64 rows and more. They cross at about 500
// workgroups here (us, this / that, 8000 cached tokens, 8 key heads of size
// 128: 5 rows x 1 sequence 24 / 158; 128 rows x 4 67 / 163; 128 rows x 16
// 178 / 213; 256 rows x 16 365 / 243; 64 rows x 64 with 2000 cached 210 /
// 104). Up to 32 rows stay here at any batch (64 sequences, 2000 cached: 109
// / 101), so that verified tokens attend as decoded ones do in steps of more
// rows than decode_stack.hip takes; to the bit only the last token of each
// sequence, beside as many sequences in a table as wide (the splits' borders
// follow from them) and on bf16 pages (decoding rounds its queries on 8-bit
// ones).
extern "C" int attn_stream_takes(long pairs, long rows) {
    return rows <= 32 || stream_groups(pairs, rows) <= 448;
}

// Splits of the contexts of a step, of up to `keys` keys (what the block table
// holds; their lengths are on the GPU). `even`: about a workgroup a CU where
// there are few; more cost more in the combine than they hide (192 (sequence,
// key head) pairs of up to 2000 keys: 25.1 us with 2 splits, 26.4 with 6, 28.9
// with 16; 8 pairs of 3000: 35.7 with 1, 10.1 with 8, 8.6 with 32).
// `most`: a workgroup takes 12 ns a key, so with one or two splits the longest
// context of an uneven batch is read by a few CUs when the others are done.
// There, a context is cut into parts of 2048 keys and more, as many as keep the
// grid within ST_GRID workgroups (most leave at once). One long context among
// short ones of 60 keys (us, 8 key heads of size 128; even splits alone / with
// the limit / the three-stage kernels before, of 4096 workgroups): 4000 and 42
// short ones 45.7 / 26.5 / 35.5, 8000 and 42 86.5 / 29.4 / 48.7; of 4 key
// heads 8000 and 79 83 / 27 / 59, 30000 and 79 299 / 85 / 213. An even batch
// may pay for the combine: 16 of 900 to 7000 61.3 / 64.9 / 88.8, 64 of 500 to
// 4000 117.1 / 117.6 / 154, but 24 of 900 to 7000 89.9 / 82.4 / 105. From 768
// groups on nothing is cut (200 of 400 to 3000 would take 237.8, not 232.9),
// and the three stages had five workgroups a context or fewer, of 67 ns a key.
constexpr long ST_GRID = 1536;
extern "C" int attn_stream_splits(long pairs, long rows, long keys, int* even,
                                  int* most) {
    const long groups = pairs > 0 ? stream_groups(pairs, rows) : 1;
    const long steps = (keys + ST_STEP - 1) / ST_STEP;
    long e = (256 + groups - 1) / groups;
    if (e > 32) e = 32;                        // the combine's lanes
    if (e > steps) e = steps;
    if (e < 1) e = 1;
    long z = e;
    if (e <= 2) {
        z = (keys + 2047) / 2048;
        if (z > ST_GRID / groups) z = ST_GRID / groups;
        if (z > 32) z = 32;
        if (z < e) z = e;
    }
    *even = (int)e;
    // (a split of no more than its share of `keys`: never more than z)
    *most = z > e ? (int)((steps + z - 1) / z) * ST_STEP : 1 << 30;
    return (int)z;
}

// cu null: one row a sequence (decode). part_o [nseq * nkv, Z, max_rows, hd]
// and part_ml [.., 2] fp32 when Z > 1; out_ml (optional) [T, nq, 2]: natural-
// log (m, l) of every row. Head size 64 or 128 and a positive scale, nonzero
// for any other.
extern "C" int launch_attn_stream(
    const unsigned short* q, const void* k_cache, const void* v_cache,
    const int* cu, const int* block_table, const int* seq_lens,
    const int* order, unsigned short* out, float* out_ml, float* part_o,
    float* part_ml, int nseq, int nkv, int G, int W, int bs, int hd, int Z,
    int even, int most, int max_qlen, long s_q, float scale, int fp8,
    hipStream_t stream) {
    if ((hd != 64 && hd != 128) || !(scale > 0.f)) return 1;
    if (nseq == 0 || max_qlen <= 0) return 0;
    const int max_rows = max_qlen * G;
    const int qt = max_rows <= 16 ? 1 : 2;
    const dim3 grid(nseq * nkv, Z, (max_rows + qt * 16 - 1) / (qt * 16));
    const bool whole = bs % ST_KEYS == 0;
    const int smem = ST_WAVES * 2 * ST_KEYS * hd * 2 +
                     qt * 16 * ST_WAVES * 2 * (int)sizeof(float);
    const bool streamed =
        (long)nseq * nkv * W * bs * hd * (fp8 ? 2 : 4) > 6 << 20;
#define ST_ONE(HDV, QTV, KVT)                                                 \
    do {                                                                      \
        if (streamed && whole) ST_GO(HDV, QTV, KVT, true, true);              \
        else if (streamed) ST_GO(HDV, QTV, KVT, true, false);                 \
        else if (whole) ST_GO(HDV, QTV, KVT, false, true);                    \
        else ST_GO(HDV, QTV, KVT, false, false);                              \
    } while (0)
#define ST_GO(HDV, QTV, KVT, STR, WHOLE)                                      \
    hipLaunchKernelGGL(                                                       \
        (attn_stream_kernel<HDV, QTV, KVT, STR, WHOLE>), grid,                \
        dim3(ST_WAVES * 64), smem, stream, q, (const KVT*)k_cache,            \
        (const KVT*)v_cache, cu, block_table, seq_lens, order, out, out_ml,   \
        part_o, part_ml, nkv, G, W, bs, Z, even, most, max_rows, s_q, scale)
#define ST_COMBINE(HDV, P, I)                                                 \
    hipLaunchKernelGGL((attn_stream_combine_kernel<HDV, P, I>),               \
                       dim3(nseq * nkv, max_rows), dim3(HDV / 4 * (P)), 0,    \
                       stream, part_o, part_ml, cu, seq_lens, out, out_ml,    \
                       nkv, G, W * bs, Z, even, most, max_rows)
#define ST_HD(HDV)                                                            \
    do {                                                                      \
        if (fp8 && qt == 1) ST_ONE(HDV, 1, unsigned char);                    \
        else if (fp8) ST_ONE(HDV, 2, unsigned char);                          \
        else if (qt == 1) ST_ONE(HDV, 1, unsigned short);                     \
        else ST_ONE(HDV, 2, unsigned short);                                  \
        if (Z > 4) ST_COMBINE(HDV, 8, 4);                                     \
        else if (Z > 1) ST_COMBINE(HDV, 256 / HDV, HDV / 64);                 \
    } while (0)
    if (hd == 128) ST_HD(128);
    else ST_HD(64);
#undef ST_HD
#undef ST_COMBINE
#undef ST_ONE
#undef ST_GO
    return 0;
}
