// Projections of at most 16 rows (decode steps of small batches, the tokens
// speculative decoding verifies, the logits of a few prompts), with what
// stands before and after them: the norm of the input, and bias, activation,
// rotation and page store, or the residual add.
//
// Bound by reading the weights once, and by launches: at one row a launch
// costs as much as 20 MB of weights, and the small kernels between the
// projections cost as much again. So a decode layer is five launches here.
//  * y^T = W x^T on 16x16x32 tiles: 16 rows of W are the left operand as they
//    lie in memory (16 bytes a lane, no LDS), the input rows are the columns.
//    The waves of a workgroup share K and add up in LDS; there is no split
//    over workgroups, so a row's result depends neither on the other rows nor
//    on their number.
//  * TC 8: 8 rows of W at two places along K, 128 bytes of a row together (whole
//    lines), as one left operand, 8 input rows at both places as the other; the
//    two diagonal quarters of the product add up. Twice the workgroups where 16
//    columns each leave CUs without one, and better pieces to load elsewhere.
//    These loads carry the streaming hint (STREAM): weights that no cache holds
//    come 3 to 9% sooner (2x14336x4096 41 us without and 36.5 with, 4096x14336
//    24.2 and 22.1, 2048x2048 4.4 and 4.1), but those that the 256 MB memory-side
//    cache has kept since the last step 5 to 15% later, at the time of those that
//    it has not. So not where the sides are those of stacks of 768 (sides up to
//    768 and 4096), which fit there whole: distilgpt2, one row, repeated 199.6 us
//    with the hint on all and 187.2, a first step on new weights 230 and 218;
//    with three such stacks in turn, which do not fit, 205 and 213. 1024x1024
//    belongs to stacks that do not fit: 3.4 us with it and 3.8.
//  * Between two layers' projections the residual sum stays in fp32: the norm
//    after an add takes the sum before it is rounded, as the kernel that adds
//    and norms does. For an RMS norm the projection that adds leaves the sum
//    times the norm's weight, in bf16, and sums of squares (Sum, LR_SCALED):
//    reading fp32 rows instead cost 24 us of a step of 8 layers of 4096, one
//    row (965 to 989). The error of such a step against 64 bits went from
//    0.010 to 0.0053 of its norm. A layer norm reads the fp32 rows.
//  * RMS norm: the columns enter as bf16(x w), the sum of squares is taken on
//    the way and 1/rms multiplies the fp32 sum: one rounding, as if the normed
//    row had been written and read. Layer norm needs mean and deviation first:
//    each workgroup takes them from the rows itself (they are in L2).
//  * two batches of weight loads, LR_U tiles each, are on their way: with 8 or
//    16 the registers cost more waves than the loads gain (output head of
//    128256 x 4096, us: 4 tiles 182, 8 205, 16 230), and the streaming hint on
//    16-row tiles loses the half lines a 64-byte piece leaves (206 to 240). The
//    input asked for as early as the weights costs registers too (a step of 8
//    layers of 3584, two rows: 1220 to 1290 us; of 4096, one row: 1014 to 1034).
// Measured (us, one row, beside the library product alone): 6144x4096 13.8
// (14.5), 4096x4096 8.5 (15.6), 2x14336x4096 36.5 (64), 4096x14336 22.1 (27),
// 128256x4096 178 (194); bytes at 6.5 TB/s: 7.7, 5.2, 36, 18, 162. With 16 rows
// 15.5, 10.8, 52, 31, 188: the input's reads add up, so more rows, the longest
// gated projections and most output heads are linear_mid.hip's.
#include "common.h"

typedef __attribute__((ext_vector_type(4))) short short4v;

constexpr int LR_U = 4;     // weight tiles of a batch of loads

enum { LR_PLAIN = 0, LR_GLU = 1, LR_GELU = 2, LR_QKV = 3 };
// LR_SCALED: RMS norm of rows that come as what Sum below makes of them
enum { LR_NONE = 0, LR_RMS = 1, LR_LAYER = 2, LR_SCALED = 3 };

// What an LR_QKV epilogue reads and writes besides the rows: queries rotated
// into q [M, nq, hd]; keys rotated, and values, into the pages (bf16 or fp8).
struct QkvStore {
    const int* pos;           // null: no rotation
    const float* cos_t;       // [table, hd / 2]
    const float* sin_t;
    int table;
    const int* slots;
    void* k_cache;            // [nb, nkv, bs, hd]
    void* v_cache;
    int nq, nkv, hd, bs, fp8;
};

// What an LR_PLAIN epilogue adds, and what it leaves of the sum: bf16 or fp32
// rows, and for the RMS norm that reads them next (then_w its weight) the rows
// times that weight and the sums of squares of 8 columns each.
struct Sum {
    const void* resid;            // [M, N] bf16 or fp32, or null
    int resid32, y32;
    const unsigned short* then_w; // [N], or null
    unsigned short* scaled;       // [M, N]
    float* squares;               // [M, N / 8]
};

DEV_INLINE void load_x8(const unsigned short* p, float* v) {
    load_bf16x8(p, v);
}
DEV_INLINE void load_x8(const float* p, float* v) {
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const f32x4 u = reinterpret_cast<const f32x4*>(p)[q];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[q * 4 + e] = u[e];
    }
}

DEV_INLINE void store_row4(void* cache, long at, int fp8, const float* z) {
    if (fp8) {
        *reinterpret_cast<unsigned int*>(
            reinterpret_cast<unsigned char*>(cache) + at) =
            f2fp8x2(bf2f(f2bf(z[0])), bf2f(f2bf(z[1]))) |
            (unsigned int)f2fp8x2(bf2f(f2bf(z[2])), bf2f(f2bf(z[3]))) << 16;
    } else {
        *reinterpret_cast<short4v*>(
            reinterpret_cast<unsigned short*>(cache) + at) =
            short4v{(short)f2bf(z[0]), (short)f2bf(z[1]), (short)f2bf(z[2]),
                    (short)f2bf(z[3])};
    }
}

// (see above)
template <bool STREAM> DEV_INLINE bf16x8 lr_weights(const unsigned short* p) {
    if constexpr (STREAM)
        return __builtin_nontemporal_load(reinterpret_cast<const bf16x8*>(p));
    else
        return *reinterpret_cast<const bf16x8*>(p);
}

// EPI LR_PLAIN: y = n(x) W^T [+ bias] [+ resid]; LR_GLU: y = silu(g) u, g and
// u from the halves of W [2N, K]; LR_GELU: y = gelu_tanh(n(x) W^T + bias);
// LR_QKV: see QkvStore (W [N, K], bias optional). NT tiles of 16 columns of y
// per workgroup (LR_GLU, LR_QKV: of each half; LR_QKV's halves are those of a
// head).
// x is of type XT: bf16, or (LR_LAYER) fp32. squares: of LR_SCALED's rows.
template <int NW, int NT, int TC, int G, int NORM, int EPI, typename XT,
          bool STREAM>
__global__ __launch_bounds__(NW * 64) void linear_rows_kernel(
    const XT* __restrict__ x,
    const unsigned short* __restrict__ norm_w,
    const unsigned short* __restrict__ norm_b,
    const unsigned short* __restrict__ w,
    const unsigned short* __restrict__ bias,
    const float* __restrict__ squares, Sum add,
    unsigned short* __restrict__ y, int M, int N, int K, float eps,
    QkvStore st) {
    constexpr bool PAIR = EPI == LR_GLU || EPI == LR_QKV;
    constexpr int WT = PAIR ? 2 * NT : NT;
    constexpr int H = TC == 16 ? G : 1;        // tiles of W along K a step
    // (4 tiles: whole 128-byte lines of W a batch, as with fewer)
    constexpr int U = NT == 4 ? 2 : LR_U / (WT * H) > 0 ? LR_U / (WT * H) : 1;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int li = lane & 15, lg = lane >> 4;
    // TC 8: lanes 8..15 take the same weights' rows, and the same input rows,
    // 32 further along K; the off-diagonal quarters of the tile are not read.
    // G 2: TC 8: input rows 0-7 and 8-15; TC 16: K and K + 32, summed apart as
    // TC 8 does
    constexpr int KS = TC == 8 || G == 2 ? 64 : 32;    // K of a step
    constexpr int RG = TC == 8 ? 8 : 0;        // rows from acc[0] to acc[1]
    const int lj = li & (TC - 1), lk = (li - lj) * 4 + lg * 8;
    int n0 = blockIdx.x * NT * TC;             // first column of y
    int half = N;                              // to the pair's other tile
    if (EPI == LR_QKV) {
        const int per = st.hd / (2 * TC);      // workgroups of a head
        n0 = blockIdx.x / per * st.hd + blockIdx.x % per * TC;
        half = st.hd / 2;
    }
    const int steps = K / KS;                  // this wave's: s0 .. s1
    const int s0 = steps * wid / NW, s1 = steps * (wid + 1) / NW;

    const unsigned short* wp[WT];
#pragma unroll
    for (int t = 0; t < WT; ++t) {
        int n = n0 + (t % NT) * TC + lj;
        if (!PAIR) n = min(n, N - 1);
        wp[t] = w + (long)(t < NT ? n : half + n) * K + lk;
    }
    bf16x8 aw[2][U][H][WT];
    auto fetch = [&](int set, int s) {
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int h = 0; h < H; ++h)
#pragma unroll
                for (int t = 0; t < WT; ++t)
                    aw[set][u][h][t] = lr_weights<STREAM>(
                        wp[t] + (long)(s + u) * KS + h * 32);
    };
    int s = s0;
    if (s + U <= s1) fetch(0, s);

    float mean[G], dev[G];                     // LR_LAYER: of acc[g]'s row
    if (NORM == LR_LAYER) {
        __shared__ float stat[16][2];
        for (int m = wid; m < M; m += NW) {
            float sum = 0.f, sumsq = 0.f;
            for (int i = lane * 8; i < K; i += 512) {
                float v[8];
                load_x8(x + (long)m * K + i, v);
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    sum += v[e];
                    sumsq += v[e] * v[e];
                }
            }
            sum = wave_sum(sum) / (float)K;
            sumsq = wave_sum(sumsq) / (float)K;
            if (lane == 0) {
                stat[m][0] = sum;
                stat[m][1] = rsqrtf(sumsq - sum * sum + eps);
            }
        }
        __syncthreads();
#pragma unroll
        for (int g = 0; g < G; ++g) {
            mean[g] = stat[min(lj + RG * g, M - 1)][0];
            dev[g] = stat[min(lj + RG * g, M - 1)][1];
        }
    }

    long x_off[G];
    f32x4 acc[G][WT];
    float sq[G];                               // LR_RMS
#pragma unroll
    for (int g = 0; g < G; ++g) {
        x_off[g] = (long)min(lj + RG * g, M - 1) * K + lk;
        sq[g] = 0.f;
#pragma unroll
        for (int t = 0; t < WT; ++t) acc[g][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    auto products = [&](const bf16x8 (*a)[WT], int st_) {
        bf16x8 nw, nb;
#pragma unroll
        for (int g = 0; g < G; ++g) {
            const long k = (long)st_ * KS + (TC == 16 ? g * 32 : 0);
            if ((NORM == LR_RMS || NORM == LR_LAYER) && (g == 0 || TC == 16))
                nw = *reinterpret_cast<const bf16x8*>(norm_w + lk + k);
            if (NORM == LR_LAYER && (g == 0 || TC == 16))
                nb = *reinterpret_cast<const bf16x8*>(norm_b + lk + k);
            bf16x8 bx;
            if (NORM == LR_NONE || NORM == LR_SCALED) {
                bx = *reinterpret_cast<const bf16x8*>(x + x_off[g] + k);
            } else {
                float v[8];
                load_x8(x + x_off[g] + k, v);
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    if (NORM == LR_RMS) {
                        sq[g] = fmaf(v[e], v[e], sq[g]);
                        bx[e] = (__bf16)(v[e] * (float)nw[e]);
                    } else {
                        bx[e] = (__bf16)((v[e] - mean[g]) * dev[g] *
                                             (float)nw[e] +
                                         (float)nb[e]);
                    }
                }
            }
#pragma unroll
            for (int t = 0; t < WT; ++t)
                acc[g][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                    a[TC == 16 ? g : 0][t], bx, acc[g][t], 0, 0, 0);
        }
    };
    for (; s + 2 * U <= s1; s += 2 * U) {
        fetch(1, s + U);
#pragma unroll
        for (int u = 0; u < U; ++u) products(aw[0][u], s + u);
        if (s + 3 * U <= s1) fetch(0, s + 2 * U);
#pragma unroll
        for (int u = 0; u < U; ++u) products(aw[1][u], s + U + u);
    }
    if (s + U <= s1) {
#pragma unroll
        for (int u = 0; u < U; ++u) products(aw[0][u], s + u);
        s += U;
    }
    for (; s < s1; ++s) {
        bf16x8 a[H][WT];
#pragma unroll
        for (int h = 0; h < H; ++h)
#pragma unroll
            for (int t = 0; t < WT; ++t)
                a[h][t] = lr_weights<STREAM>(wp[t] + (long)s * KS + h * 32);
        products(a, s);
    }

    // LR_SCALED: 1/rms, a wave a row (at one row a shorter chain than 16
    // lanes: 3072x2048 6.4 us, not 6.8) or, of more rows than waves, 16 lanes.
    // (Before the loop it keeps the first wave from its weights: 2x14336x4096,
    // one row, 46.9 us, not 45.7.)
    __shared__ float scale_s[16];
    if (NORM == LR_SCALED) {
        const bool wide = M <= NW;
        const int m = wide ? wid : wid * 4 + lg;
        float sum = 0.f;
        if (m < M) {
            const float* sp = squares + (long)m * (K / 8);
#pragma unroll 4
            for (int i = (wide ? lane : li) * 4; i < K / 8;
                 i += wide ? 256 : 64) {
                const f32x4 v = *reinterpret_cast<const f32x4*>(sp + i);
                sum += (v[0] + v[1]) + (v[2] + v[3]);
            }
        }
#pragma unroll
        for (int o = 1; o < 16; o <<= 1) sum += __shfl_xor(sum, o);
        if (wide) sum = rows_sum(sum);
        if (m < M && li == 0) scale_s[m] = rsqrtf(sum / (float)K + eps);
    }

    // ---- the waves' sums; C layout: column li = row of x, rows lg * 4 + r =
    // columns of y
    __shared__ f32x4 part[NW][G][WT][64];
    __shared__ float sqp[NW][G][16];
#pragma unroll
    for (int g = 0; g < G; ++g) {
        if (NORM == LR_RMS) {
            sq[g] = rows_sum(sq[g]);
            if (lg == 0) sqp[wid][g][li] = sq[g];
        }
#pragma unroll
        for (int t = 0; t < WT; ++t) part[wid][g][t][lane] = acc[g][t];
    }
    __syncthreads();
    if (wid >= NT * (TC == 8 ? G : 1) ||
        (TC == 8 && (li >= 8 || lg >= 2))) return;
    const int g = wid / NT, tile = wid % NT, m = li + RG * g;
    if (m >= M) return;
    // the sums over K and over K + 32, each of all waves, then together
    constexpr bool TWO = KS == 64;
    const int g2 = TC == 8 ? g : G - 1, up = TC == 8 ? 8 : 0;   // li + 8, and
    const int up_lane = TC == 8 ? 40 : 0;                       // lg + 2
    float inv = 1.f;
    if (NORM == LR_RMS) {
        float v = 0.f;
#pragma unroll
        for (int k = 0; k < NW; ++k) {
            v += sqp[k][g][li];
            if (TWO) v += sqp[k][g2][li + up];
        }
        inv = rsqrtf(v / (float)K + eps);
    }
    if (NORM == LR_SCALED) inv = scale_s[m];
    auto total = [&](int t, float* z) {
        f32x4 v = part[0][g][t][lane];
#pragma unroll
        for (int k = 1; k < NW; ++k) {
            const f32x4 p = part[k][g][t][lane];
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] += p[r];
        }
        if (TWO) {
#pragma unroll
            for (int k = 0; k < NW; ++k) {
                const f32x4 p = part[k][g2][t][lane + up_lane];
#pragma unroll
                for (int r = 0; r < 4; ++r) v[r] += p[r];
            }
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) z[r] = v[r] * inv;
    };
    const int n = n0 + tile * TC + lg * 4;     // (NT * G <= NW)
    if (!PAIR && n >= N) return;
    float z[4];
    total(tile, z);
    if (EPI == LR_GLU) {
        float u[4];
        total(NT + tile, u);
#pragma unroll
        for (int r = 0; r < 4; ++r) z[r] = z[r] / (1.f + __expf(-z[r])) * u[r];
    } else if (EPI == LR_QKV) {
        float u[4];
        total(NT + tile, u);
        if (bias) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                z[r] += bf2f(bias[n + r]);
                u[r] += bf2f(bias[n + half + r]);
            }
        }
        const int head = n / st.hd, d = n % st.hd;
        if (st.pos && head < st.nq + st.nkv) {
            const long tab = turn_row(st.pos[m], st.table) * half + d;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float c = st.cos_t[tab + r], sn = st.sin_t[tab + r];
                const float a = z[r], b = u[r];
                z[r] = a * c - b * sn;
                u[r] = b * c + a * sn;
            }
        }
        if (head < st.nq) {
            const long at = ((long)m * st.nq + head) * st.hd + d;
            store_row4(y, at, 0, z);
            store_row4(y, at + half, 0, u);
            return;
        }
        const bool is_k = head < st.nq + st.nkv;
        const int kvh = head - st.nq - (is_k ? 0 : st.nkv);
        const int slot = st.slots[m];
        if (slot < 0) return;                  // no such position
        const long at = (((long)(slot / st.bs) * st.nkv + kvh) * st.bs +
                         slot % st.bs) * st.hd + d;
        void* cache = is_k ? st.k_cache : st.v_cache;
        store_row4(cache, at, st.fp8, z);
        store_row4(cache, at + half, st.fp8, u);
        return;
    } else {
        const long at = (long)m * N + n;
        if (EPI == LR_PLAIN && add.resid32 && N % 4 == 0) {
            const f32x4 v = *reinterpret_cast<const f32x4*>(
                reinterpret_cast<const float*>(add.resid) + at);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                if (bias) z[r] += bf2f(bias[n + r]);
                z[r] += v[r];
            }
        } else {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const bool in = n + r < N;
                if (bias && in) z[r] += bf2f(bias[n + r]);
                if (EPI == LR_GELU) {
                    const float c = 0.7978845608028654f *
                                    (z[r] + 0.044715f * z[r] * z[r] * z[r]);
                    z[r] = 0.5f * z[r] * (1.f + tanhf(c));
                }
                if (add.resid && in)
                    z[r] += add.resid32
                                ? reinterpret_cast<const float*>(
                                      add.resid)[at + r]
                                : bf2f(reinterpret_cast<const unsigned short*>(
                                      add.resid)[at + r]);
            }
        }
    }
    const long at = (long)m * N + n;
    if (EPI == LR_PLAIN && add.then_w) {       // (N % 8 == 0)
        const short4v tw = *reinterpret_cast<const short4v*>(add.then_w + n);
        float v[4], sq4 = 0.f;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            v[r] = z[r] * bf2f((unsigned short)tw[r]);
            sq4 += z[r] * z[r];
        }
        store_row4(add.scaled, at, 0, v);
        sq4 += __shfl_xor(sq4, 16);            // the next 4 columns'
        if (lg % 2 == 0) add.squares[(long)m * (N / 8) + n / 8] = sq4;
    }
    if (EPI == LR_PLAIN && add.y32) {
        float* y32 = reinterpret_cast<float*>(y) + at;
        if (N % 4 == 0) {
            *reinterpret_cast<f32x4*>(y32) = f32x4{z[0], z[1], z[2], z[3]};
        } else {
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (n + r < N) y32[r] = z[r];
        }
    } else if (N % 4 == 0) {
        store_row4(y, at, 0, z);
    } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
            if (n + r < N) y[at + r] = f2bf(z[r]);
    }
}

// x [M, K] and w rows of K, 1 <= M <= 16, K % 32 == 0, all contiguous and
// 16-byte aligned; x32: x is fp32 (norm 2); norm 0 none, 1 RMS, 2 layer norm, 3
// RMS with `squares` [M, K / 8]; epi as above (LR_GLU: N % 16 == 0, LR_QKV: hd %
// 32 == 0); resid32, y32: the residual, and LR_PLAIN's y, are fp32; then_w: see
// Sum (N % 8 == 0). Nonzero for anything else.
//
// The shape of a workgroup (waves x tiles x columns of a tile) depends on N and
// K only, or on M between shapes of the same sums: 16 columns with G 2 add as 8
// do. Measured (us) at 1 / 8 / 16 rows:
//   q, k, v: 3072x2048 8x1x8 6.5 / 7.1 / 8.3, 8x1x16 8.2 / 8.7 / 9.3 (96
//    workgroups); 2304x768 5.8 / 6.2 / 7.8 and 6.0 / 6.6 / 7.5; but 5120x3072
//    11.8 / 12.9 / 16.3 and 11.9 / 11.7 / 12.6, 6144x4096 15.2 / 17.0 / 20.3
//    and 15.4 / 16.4 / 17.2;
//   gated: 2x14336x4096 4x1x8 44 / 49 / 64, 4x1x16 50 / 52 / 57, 8x1x16 49 /
//    50 / 55; 2x18944x3584 53 / 59 / 76, 54 / 57 / 63, 54 / 57 / 63;
//    2x8192x2048 15.7 / 17.2 / 21.7, 16.0 / 16.2 / 17.4, 15.8 / 16.2 / 17.3;
//   up to 2048 columns: 2048x8192 8x1x8 10 / 11.7 / 15.4, 8x2x8 13 / 14.7 /
//    18.6, 16x1x16 14 / 16 / 18.7; 2048x2048 4.5 / 5.2 / 6.1, 5.3 / 5.9 / 6.8,
//    5.3 / 6.1 / 6.8; 768x3072 5.6 / 6.3 / 7.8, 6.3 / 7.2 / 8.7, 6.8 / 7.9 /
//    9.2;
//   up to 4096: 3072x8192 14.1 / 19 / 25, 14.0 / 16.6 / 19.2, 15.4 / 18 / 19.7;
//    4096x4096 8.6 / 10.9 / 14.4, 9.3 / 9.8 / 11.6, 9.2 / 10.4 / 11.9;
//    4096x14336 24.9 / 32 / 44, 24.9 / 26.5 / 34.5, 25.4 / 29.3 / 34.6;
//    3584x18944 31 / 41 / 56, 29 / 34 / 44, 32 / 40 / 46;
//   above: 128256x4096 8x2x8 174 / 204 / 272, 8x2x16 184 / 194 / 217;
//   from 16384 on, K below 8192 (output heads): of 9 rows and more the input,
//    read once for 32 columns, is half of what comes through L2, so 4 tiles;
//    4 waves leave the registers for whole lines of 4 tiles, and add as 4 waves
//    of 2 do (1 / 9 / 16 rows, 8x2x16 and 4x2x16 or 4x4x16): 128256x4096 186 /
//    193 / 210 and 175 / 190 / 192, 128256x3072 140 / 147 / 165 and 137 / 147 /
//    154, 152064x3584 189 / 207 / 224 and 184 / 198 / 207; 128256x8192 360 /
//    372 / 396 and 394 / 420 / 428; 4608x4096, too few workgroups, 17 / 18 / 18
//    and 17 / 24 / 26.
extern "C" int launch_linear_rows(
    const void* x, int x32, const unsigned short* norm_w,
    const unsigned short* norm_b, const unsigned short* w,
    const unsigned short* bias, const float* squares, const void* resid,
    int resid32, void* y, int y32, const unsigned short* then_w,
    unsigned short* scaled, float* squares_out, int M, int N, int K,
    float eps, int norm, int epi,
    const int* pos, const float* cos_t, const float* sin_t, int table,
    const int* slots, void* k_cache, void* v_cache, int nq, int nkv, int hd, int bs, int fp8,
    hipStream_t stream) {
    if (M < 1 || M > 16 || N < 1 || K < 32 || K % 32) return 1;
    if (epi == LR_GLU && N % 16) return 1;
    if ((x32 && norm != LR_LAYER) || (norm == LR_SCALED && !squares)) return 1;
    if ((y32 || then_w) && epi != LR_PLAIN) return 1;
    if (then_w && N % 8) return 1;
    const Sum add{resid, resid32, y32, then_w, scaled, squares_out};
    if (epi == LR_QKV && (hd % 32 || N != (nq + 2 * nkv) * hd)) return 1;
    const QkvStore st{pos,     cos_t, sin_t, table, slots, k_cache,
                      v_cache, nq,    nkv,   hd,    bs,    fp8};
    // (see above: stacks of more than 768)
    const int WN = epi == LR_GLU ? 2 * N : N;
    const bool streamed = (WN < K ? WN : K) > 768 || (WN < K ? K : WN) > 4096;
#define LR_COLS(NTV, TCV, EP) (NTV * TCV * (EP == LR_QKV ? 2 : 1))
#define LR_ONE(NWV, NTV, TCV, GV, NO, EP, XT, STR)                            \
    hipLaunchKernelGGL(                                                       \
        (linear_rows_kernel<NWV, NTV, TCV, GV, NO, EP, XT, STR>),             \
        dim3((N + LR_COLS(NTV, TCV, EP) - 1) / LR_COLS(NTV, TCV, EP)),        \
        dim3(NWV * 64), 0, stream, (const XT*)x, norm_w, norm_b, w, bias,     \
        squares, add, (unsigned short*)y, M, N, K, eps, st)
#define LR_GO(NWV, NTV, TCV, GV, NO, EP, XT)                                  \
    do {                                                                      \
        if (TCV == 8 && streamed)                                             \
            LR_ONE(NWV, NTV, TCV, GV, NO, EP, XT, TCV == 8);                  \
        else                                                                  \
            LR_ONE(NWV, NTV, TCV, GV, NO, EP, XT, false);                     \
    } while (0)
#define LR_NORMS(NWV, NTV, TCV, GV, EP)                                       \
    do {                                                                      \
        if (norm == LR_SCALED)                                                \
            LR_GO(NWV, NTV, TCV, GV, LR_SCALED, EP, unsigned short);          \
        else if (norm == LR_RMS)                                              \
            LR_GO(NWV, NTV, TCV, GV, LR_RMS, EP, unsigned short);             \
        else if (norm == LR_LAYER && x32)                                     \
            LR_GO(NWV, NTV, TCV, GV, LR_LAYER, EP, float);                    \
        else if (norm == LR_LAYER)                                            \
            LR_GO(NWV, NTV, TCV, GV, LR_LAYER, EP, unsigned short);           \
        else                                                                  \
            LR_GO(NWV, NTV, TCV, GV, LR_NONE, EP, unsigned short);            \
    } while (0)
#define LR_16(NWV, NTV, EP) LR_NORMS(NWV, NTV, 16, 1, EP)
#define LR_8(NWV, NTV, EP)                                                    \
    do {                                                                      \
        if (M > 8) LR_NORMS(NWV, NTV, 8, 2, EP);                              \
        else LR_NORMS(NWV, NTV, 8, 1, EP);                                    \
    } while (0)
    const bool t8 = K % 64 == 0;
    if (epi == LR_QKV && N <= 4096 && t8) LR_8(8, 1, LR_QKV);
    else if (epi == LR_QKV) LR_16(8, 1, LR_QKV);
    else if (epi == LR_GLU && t8 && M <= 8) LR_NORMS(4, 1, 8, 1, LR_GLU);
    else if (epi == LR_GLU && t8) LR_NORMS(4, 1, 16, 2, LR_GLU);
    else if (epi == LR_GLU) LR_16(4, 1, LR_GLU);
    else if (epi == LR_GELU) LR_16(8, 1, LR_GELU);
    else if (N >= 16384 && K < 8192 && M > 8) LR_16(4, 4, LR_PLAIN);
    else if (N >= 16384 && K < 8192) LR_16(4, 2, LR_PLAIN);
    else if (N > 4096) LR_16(8, 2, LR_PLAIN);
    else if (N > 2048 && t8) LR_8(8, 2, LR_PLAIN);
    else if (t8) LR_8(8, 1, LR_PLAIN);
    else LR_16(8, 1, LR_PLAIN);
#undef LR_8
#undef LR_16
#undef LR_NORMS
#undef LR_GO
#undef LR_ONE
#undef LR_COLS
    return 0;
}
