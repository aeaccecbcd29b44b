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
//  * RMS norm: the columns enter as bf16(x w), the sum of squares is taken on
//    the way and 1/rms multiplies the fp32 sum: one rounding, as if the normed
//    row had been written and read. Layer norm needs mean and deviation first:
//    each workgroup takes them from the rows itself (they are in L2).
//  * two batches of weight loads, LR_U tiles each, are on their way: with 8 or
//    16 the registers cost more waves than the loads gain (output head of
//    128256 x 4096, us: 4 tiles 182, 8 205, 16 230), and a streaming hint on
//    the loads loses the half lines a 64-byte piece leaves (206 to 240).
// Measured (us, one row, beside the library product alone): 6144x4096 14
// (14.5), 4096x4096 9 (15.6), 2x14336x4096 48 (64), 4096x14336 24 (27),
// 128256x4096 182 (190); floor at 5.9 TB/s and 4 us a launch: 12.5, 9.7, 44,
// 24, 182. With 16 rows 16, 11, 54, 31, 207: the input's reads add up, so
// more rows go to the library.
#include "common.h"

typedef __attribute__((ext_vector_type(4))) short short4v;

constexpr int LR_U = 4;     // weight tiles of a batch of loads

enum { LR_PLAIN = 0, LR_GLU = 1, LR_GELU = 2, LR_QKV = 3 };
enum { LR_NONE = 0, LR_RMS = 1, LR_LAYER = 2 };

// What an LR_QKV epilogue reads and writes besides the rows: queries rotated
// into q [M, nq, hd]; keys rotated, and values, into the pages (bf16 or fp8).
struct QkvStore {
    const int* pos;           // null: no rotation
    const float* cos_t;       // [max_len, hd / 2]
    const float* sin_t;
    const int* slots;
    void* k_cache;            // [nb, nkv, bs, hd]
    void* v_cache;
    int nq, nkv, hd, bs, fp8;
};

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

// EPI LR_PLAIN: y = n(x) W^T [+ bias] [+ resid]; LR_GLU: y = silu(g) u, g and
// u from the halves of W [2N, K]; LR_GELU: y = gelu_tanh(n(x) W^T + bias);
// LR_QKV: see QkvStore (W [N, K], bias optional). NT tiles of 16 columns of y
// per workgroup (LR_GLU, LR_QKV: of each half; LR_QKV's halves are those of a
// head).
template <int NW, int NT, int NORM, int EPI>
__global__ __launch_bounds__(NW * 64) void linear_rows_kernel(
    const unsigned short* __restrict__ x,
    const unsigned short* __restrict__ norm_w,
    const unsigned short* __restrict__ norm_b,
    const unsigned short* __restrict__ w,
    const unsigned short* __restrict__ bias,
    const unsigned short* __restrict__ resid, unsigned short* __restrict__ y,
    int M, int N, int K, float eps, QkvStore st) {
    constexpr bool PAIR = EPI == LR_GLU || EPI == LR_QKV;
    constexpr int WT = PAIR ? 2 * NT : NT;
    constexpr int U = LR_U / WT > 0 ? LR_U / WT : 1;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int li = lane & 15, lg = lane >> 4;
    int n0 = blockIdx.x * NT * 16;             // first column of y
    int half = N;                              // to the pair's other tile
    if (EPI == LR_QKV) {
        const int per = st.hd / 32;            // workgroups of a head
        n0 = blockIdx.x / per * st.hd + blockIdx.x % per * 16;
        half = st.hd / 2;
    }
    // this wave's steps of 32 along K
    const int steps = K / 32;
    const int s0 = steps * wid / NW, s1 = steps * (wid + 1) / NW;

    const unsigned short* wp[WT];
#pragma unroll
    for (int t = 0; t < WT; ++t) {
        int n = n0 + (t % NT) * 16 + li;
        if (!PAIR) n = min(n, N - 1);
        wp[t] = w + (long)(t < NT ? n : half + n) * K + lg * 8;
    }
    bf16x8 aw[2][U][WT];
    auto fetch = [&](int set, int s) {
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int t = 0; t < WT; ++t)
                aw[set][u][t] = *reinterpret_cast<const bf16x8*>(
                    wp[t] + (long)(s + u) * 32);
    };
    int s = s0;
    if (s + U <= s1) fetch(0, s);

    float mean = 0.f, dev = 1.f;               // LR_LAYER: of row li
    if (NORM == LR_LAYER) {
        __shared__ float stat[16][2];
        for (int m = wid; m < M; m += NW) {
            float sum = 0.f, sumsq = 0.f;
            for (int i = lane * 8; i < K; i += 512) {
                float v[8];
                load_bf16x8(x + (long)m * K + i, v);
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
        mean = stat[min(li, M - 1)][0];
        dev = stat[min(li, M - 1)][1];
    }

    const long x_off = (long)min(li, M - 1) * K + lg * 8;
    f32x4 acc[WT];
    float sq = 0.f;                            // LR_RMS
#pragma unroll
    for (int t = 0; t < WT; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto products = [&](const bf16x8* a, int st_) {
        const long k = (long)st_ * 32;
        bf16x8 bx = *reinterpret_cast<const bf16x8*>(x + x_off + k);
        if (NORM == LR_RMS) {
            const bf16x8 g =
                *reinterpret_cast<const bf16x8*>(norm_w + lg * 8 + k);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float v = (float)bx[e];
                sq = fmaf(v, v, sq);
                bx[e] = (__bf16)(v * (float)g[e]);
            }
        } else if (NORM == LR_LAYER) {
            const bf16x8 g =
                *reinterpret_cast<const bf16x8*>(norm_w + lg * 8 + k);
            const bf16x8 c =
                *reinterpret_cast<const bf16x8*>(norm_b + lg * 8 + k);
#pragma unroll
            for (int e = 0; e < 8; ++e)
                bx[e] = (__bf16)(((float)bx[e] - mean) * dev * (float)g[e] +
                                 (float)c[e]);
        }
#pragma unroll
        for (int t = 0; t < WT; ++t)
            acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[t], bx, acc[t],
                                                             0, 0, 0);
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
        bf16x8 a[WT];
#pragma unroll
        for (int t = 0; t < WT; ++t)
            a[t] = *reinterpret_cast<const bf16x8*>(wp[t] + (long)s * 32);
        products(a, s);
    }

    // ---- the waves' sums; C layout: column li = row of x, rows lg * 4 + r =
    // columns of y
    __shared__ f32x4 part[NW][WT][64];
    __shared__ float sqp[NW][16];
    if (NORM == LR_RMS) {
        sq = rows_sum(sq);
        if (lg == 0) sqp[wid][li] = sq;
    }
#pragma unroll
    for (int t = 0; t < WT; ++t) part[wid][t][lane] = acc[t];
    __syncthreads();
    const int m = li;
    if (wid >= NT || m >= M) return;
    float inv = 1.f;
    if (NORM == LR_RMS) {
        float v = 0.f;
#pragma unroll
        for (int k = 0; k < NW; ++k) v += sqp[k][m];
        inv = rsqrtf(v / (float)K + eps);
    }
    auto total = [&](int t, float* z) {
        f32x4 v = part[0][t][lane];
#pragma unroll
        for (int k = 1; k < NW; ++k) {
            const f32x4 p = part[k][t][lane];
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] += p[r];
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) z[r] = v[r] * inv;
    };
    const int n = n0 + wid * 16 + lg * 4;      // (wid: the tile; NT <= NW)
    if (!PAIR && n >= N) return;
    float z[4];
    total(wid, z);
    if (EPI == LR_GLU) {
        float u[4];
        total(NT + wid, u);
#pragma unroll
        for (int r = 0; r < 4; ++r) z[r] = z[r] / (1.f + __expf(-z[r])) * u[r];
    } else if (EPI == LR_QKV) {
        float u[4];
        total(NT + wid, u);
        if (bias) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                z[r] += bf2f(bias[n + r]);
                u[r] += bf2f(bias[n + half + r]);
            }
        }
        const int head = n / st.hd, d = n % st.hd;
        if (st.pos && head < st.nq + st.nkv) {
            const long tab = (long)st.pos[m] * half + d;
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
        const long at = (((long)(slot / st.bs) * st.nkv + kvh) * st.bs +
                         slot % st.bs) * st.hd + d;
        void* cache = is_k ? st.k_cache : st.v_cache;
        store_row4(cache, at, st.fp8, z);
        store_row4(cache, at + half, st.fp8, u);
        return;
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
            if (resid && in) z[r] += bf2f(resid[(long)m * N + n + r]);
        }
    }
    const long at = (long)m * N + n;
    if (N % 4 == 0) {
        store_row4(y, at, 0, z);
    } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
            if (n + r < N) y[at + r] = f2bf(z[r]);
    }
}

// x [M, K] and w rows of K, 1 <= M <= 16, K % 32 == 0, all contiguous and
// 16-byte aligned; norm 0 none, 1 RMS, 2 layer norm; epi as above (LR_GLU: N %
// 16 == 0, LR_QKV: hd % 32 == 0). Nonzero for anything else. The shape of a workgroup depends on N and K only. Measured (us, one
// row; 16 columns and 8 waves / 16 and 16 / 32 and 8): 4096x4096 9.4 / 8.7 /
// 12.3, 4096x14336 28.5 / 23.8 / 37, 3584x18944 33 / 30 / 42, 3072x2048 6.5 /
// 6.5 / 7.9, 768x3072 6.0 / 6.3 / 9.4; 6144x4096 15.6 / 17 / 13.8, 4608x3584
// 14.1 / 16 / 11.6, 128256x4096 198 / 260 / 182; gated, 2x14336x4096 48 with
// 8 waves, 50 with 4, 2x8192x2048 16.1 and 14.8.
extern "C" int launch_linear_rows(
    const unsigned short* x, const unsigned short* norm_w,
    const unsigned short* norm_b, const unsigned short* w,
    const unsigned short* bias, const unsigned short* resid,
    unsigned short* y, int M, int N, int K, float eps, int norm, int epi,
    const int* pos, const float* cos_t, const float* sin_t, const int* slots,
    void* k_cache, void* v_cache, int nq, int nkv, int hd, int bs, int fp8,
    hipStream_t stream) {
    if (M < 1 || M > 16 || N < 1 || K < 32 || K % 32) return 1;
    if (epi == LR_GLU && N % 16) return 1;
    if (epi == LR_QKV && (hd % 32 || N != (nq + 2 * nkv) * hd)) return 1;
    const QkvStore st{pos,     cos_t, sin_t, slots, k_cache,
                      v_cache, nq,    nkv,   hd,    bs, fp8};
#define LR_GO(NWV, NTV, NO, EP, COLS)                                         \
    hipLaunchKernelGGL((linear_rows_kernel<NWV, NTV, NO, EP>),                \
                       dim3((N + (COLS) - 1) / (COLS)), dim3(NWV * 64), 0,    \
                       stream, x, norm_w, norm_b, w, bias, resid, y, M, N, K, \
                       eps, st)
#define LR_NORMS(NWV, NTV, EP, COLS)                                          \
    do {                                                                      \
        if (norm == LR_RMS) LR_GO(NWV, NTV, LR_RMS, EP, COLS);                \
        else if (norm == LR_LAYER) LR_GO(NWV, NTV, LR_LAYER, EP, COLS);       \
        else LR_GO(NWV, NTV, LR_NONE, EP, COLS);                              \
    } while (0)
    if (epi == LR_QKV) LR_NORMS(8, 1, LR_QKV, 32);
    else if (epi == LR_GLU && K >= 3072) LR_NORMS(8, 1, LR_GLU, 16);
    else if (epi == LR_GLU) LR_NORMS(4, 1, LR_GLU, 16);
    else if (epi == LR_GELU) LR_NORMS(8, 1, LR_GELU, 16);
    else if (N > 4096) LR_NORMS(8, 2, LR_PLAIN, 32);
    else if (K >= 2048) LR_NORMS(16, 1, LR_PLAIN, 16);
    else LR_NORMS(8, 1, LR_PLAIN, 16);
#undef LR_NORMS
#undef LR_GO
    return 0;
}
