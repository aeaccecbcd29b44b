// Projections of 17 to 160 rows of up to 6144 outputs, or 3.5 times as deep as
// wide (q|k|v, attention output, feed-forward output; the last, where it is
// deep, to 256 rows): split over K, the splits' fp32 sums left to the kernel
// that reads them anyway (qkv_rope_store, add_norm_parts).
//
// Bound by reading the weights once, by a chip that 64 columns a workgroup
// would leave three quarters idle at 4096 of them (hence the split), and by
// the latency of a step. A workgroup takes 64 rows of W and a part of K: four
// waves of 16 rows, twice, for the two halves of that part. Weights go from
// memory into the left operand as they lie, three steps ahead, the input rows
// two steps ahead and then through LDS, shared by the four waves, xor-ed so
// that the 16 rows of a read meet in no bank (LDS serves 256 bytes a clock).
// Measured beside the library's product (us; 24 / 57 / 80 / 128 rows):
// 4096x14336 26 / 29 / 33 / 40 (32 / 41 / 43 / 76), 4096x4096 10.2 / 11.2 / 13
// / 16 (13.7 / 13.8 / 17 / 24), 6144x4096 14.7 / 17 / 19 / 24 (15 / 18 / 23 /
// 25); with the input one step ahead, and twice the workgroups to hide that,
// 27 / 31 / 34 / 42, 10.6 / 13 / 14 / 16, 15.4 / 18 / 20.5 / 24.5. Wide
// outputs stay with the library (2x14336x4096: 66 here against 56 at 24 rows).
// At 160 / 200 / 256 rows 4096x14336 46 / 54 / 62 (84 / 57 / 63), 6144x4096 26
// / 31 / 35 (28 / 26 / 40), 4096x4096 17.5 / 20.5 / 23 (27 / 22 / 22.5),
// 3072x8192 27 / 32 / 36 (28 / 31 / 34), 3072x2048 11.6 / 13.7 / 15.5 (12 / 13
// / 13), but 3584x18944 56 / 67 / 76 (107 / 123 / 127) and 2048x8192 18 / 21 /
// 24 (26 / 27.5 / 26.5): above 160 rows only products 3.5 times as deep as
// wide, and deeper. Where that line lies is the library's doing and not a
// property of the shapes: between 160 and 256 rows its products of 3584x18944
// and 2048x8192 are half as fast as those of 4096x14336, where the gain of a
// whole step is within 1%. Wider outputs (us, with the kernel that reads them;
// 17 / 48 / 80 / 128 / 160 rows, the library's in brackets): 10240x8192, K not
// split, 55 / 61 / 67 / 80 / 86 (43 / 48 / 80 / 64 / 72), 8192x8192 43 / 44 /
// 46 / 52 / 57 (36 / 40 / 44 / 56 / 61), 8192x4096 23 / 24 / 27 / 32 / 34 (22 /
// 24 / 30 / 33 / 35), 8192x28672 95 / 110 / 128 / 155 / 169 (99 / 179 / 198 /
// 210 / 224).
#include "common.h"

constexpr int LM_W = 4;     // steps of weights under way, and the current one's

template <int MT>
__global__ __launch_bounds__(512) void linear_mid_kernel(
    const unsigned short* __restrict__ x, const unsigned short* __restrict__ w,
    float* __restrict__ part, int M, int N, int K, int S) {
    constexpr int MP = MT * 16;
    constexpr int XB = 2 * MP * 128;       // bytes of a staged buffer: [half]
                                           // [row][64 of K]
    constexpr int NLD = MT / 2;            // 16-byte chunks a thread stages
    const int tid = threadIdx.x, lane = tid & 63;
    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int li = lane & 15, lg = lane >> 4;
    const int rw = wid & 3, kh = wid >> 2; // row tile, half of the K part
    const int n0 = blockIdx.x * 64 + rw * 16;
    // steps of 64 along K: of the workgroup, of its first half, of this wave
    const int CH = K / 64;
    const int c0 = CH * blockIdx.y / S, c1 = CH * (blockIdx.y + 1) / S;
    const int first = (c1 - c0 + 1) / 2;
    const int my0 = kh ? c0 + first : c0;
    const int mine = kh ? c1 - c0 - first : first;

    extern __shared__ __attribute__((aligned(16))) char smem[];

    const unsigned short* wp = w + (long)min(n0 + li, N - 1) * K + lg * 8;
    const unsigned short* xs[NLD];
    int xd[NLD], xlast[NLD];
#pragma unroll
    for (int j = 0; j < NLD; ++j) {
        const int i = tid + 512 * j, c = i & 7;
        const int row = (i >> 3) % MP, h = (i >> 3) / MP;
        xs[j] = x + (long)min(row, M - 1) * K +
                (long)(h ? c0 + first : c0) * 64 + c * 8;
        xlast[j] = (h ? c1 - c0 - first : first) - 1;
        xd[j] = (h * MP + row) * 128 + ((c ^ (row >> 1 & 7)) << 4);
    }
    // (a half without steps left loads, and ignores, a step of the other)
    bf16x8 xr[2][NLD];
    auto load_x = [&](int set, int it) {
#pragma unroll
        for (int j = 0; j < NLD; ++j)
            xr[set][j] = *reinterpret_cast<const bf16x8*>(
                xs[j] + (long)min(it, xlast[j]) * 64);
    };
    auto store_x = [&](int set) {          // into the buffer of its number
#pragma unroll
        for (int j = 0; j < NLD; ++j)
            *reinterpret_cast<bf16x8*>(smem + set * XB + xd[j]) = xr[set][j];
    };
    bf16x8 aw[LM_W][2];
    auto load_w = [&](int set, int it) {
        const long k = (long)min(my0 + it, CH - 1) * 64;
#pragma unroll
        for (int s = 0; s < 2; ++s)
            aw[set][s] = *reinterpret_cast<const bf16x8*>(wp + k + s * 32);
    };
    f32x4 acc[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[m] = f32x4{0.f, 0.f, 0.f, 0.f};

    load_x(0, 0);
#pragma unroll
    for (int i = 0; i < LM_W - 1; ++i) load_w(i, i);
    load_x(1, 1);
    store_x(0);
    __syncthreads();
    const char* xb = smem + kh * MP * 128 + li * 128;
    // step `it` with `it` % LM_W == j: the input of the step after the next
    // and weights of LM_W - 1 later ones set out, the next step's input goes
    // to LDS. No load stands under a condition: what is under way would have
    // to be waited for where the two ways meet.
    auto step = [&](int j, int it) {
        load_x(j & 1, it + 2);
        load_w((j + LM_W - 1) % LM_W, it + LM_W - 1);
        if (it < mine) {
            const char* b = xb + (j & 1) * XB;
#pragma unroll
            for (int s = 0; s < 2; ++s)
#pragma unroll
                for (int m = 0; m < MT; ++m) {
                    const bf16x8 bx = *reinterpret_cast<const bf16x8*>(
                        b + m * 16 * 128 +
                        (((s * 4 + lg) ^ (li >> 1)) << 4));
                    acc[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                        aw[j][s], bx, acc[m], 0, 0, 0);
                }
        }
        store_x((j + 1) & 1);
        __syncthreads();
    };
    for (int it = 0;;) {
#pragma unroll
        for (int j = 0; j < LM_W; ++j) {
            step(j, it);
            if (++it >= first) goto done;
        }
    }
done:
    // ---- the halves' sums meet in LDS
    f32x4* mg = reinterpret_cast<f32x4*>(smem) + rw * MT * 64 + lane;
    if (kh == 1) {
#pragma unroll
        for (int m = 0; m < MT; ++m) mg[m * 64] = acc[m];
    }
    __syncthreads();
    const int n = n0 + lg * 4;
    if (kh == 1 || n >= N) return;
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        const int row = m * 16 + li;
        if (row >= M) continue;
        const f32x4 p = mg[m * 64];
        f32x4 v;
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = acc[m][r] + p[r];
        *reinterpret_cast<f32x4*>(
            part + ((long)blockIdx.y * M + row) * N + n) = v;
    }
}

// Splits of K: up to a workgroup a CU, at least four steps of 64 a half. Two
// workgroups a CU: 4096x14336 at 80 rows 36 us against 32.6, 6144x4096 21.5
// against 18.9, 4096x4096 15.2 against 12.9, and the reader has twice the
// parts.
extern "C" int linear_mid_splits(int N, int K) {
    const int tiles = (N + 63) / 64;
    int S = 1;
    while (S < 8 && tiles * S * 2 <= 256 && K / 64 >= S * 16) S *= 2;
    return S;
}

// part [S, M, N] fp32: x [M, K] times rows of w [N, K] over S parts of K. x and
// w contiguous and 16-byte aligned, 1 <= M <= 256, N % 4 == 0, K % 64 == 0, S
// <= K / 64; nonzero for anything else.
extern "C" int launch_linear_mid(const unsigned short* x,
                                 const unsigned short* w, float* part, int M,
                                 int N, int K, int S, hipStream_t stream) {
    if (M < 1 || M > 256 || N < 4 || N % 4 || K < 64 || K % 64) return 1;
    if (S < 1 || S > K / 64) return 1;
    const dim3 grid((N + 63) / 64, S);
#define LM_GO(MTV)                                                            \
    hipLaunchKernelGGL((linear_mid_kernel<MTV>), grid, dim3(512),             \
                       2 * 2 * MTV * 16 * 128, stream, x, w, part, M, N, K, S)
    if (M <= 32) LM_GO(2);
    else if (M <= 64) LM_GO(4);
    else if (M <= 96) LM_GO(6);
    else if (M <= 128) LM_GO(8);
    else if (M <= 160) LM_GO(10);
    else if (M <= 192) LM_GO(12);
    else if (M <= 224) LM_GO(14);
    else LM_GO(16);
#undef LM_GO
    return 0;
}

// ----------------------------------------------------------- add_norm_parts
// resid_out = resid + sum of the parts [+ bias]; y = norm(resid_out) (RMS, or
// layer norm with norm_b), both from the fp32 sum; y null: the sum only. One
// workgroup a row; the row stays in registers between its two uses.
constexpr int ANP_T = 256;
template <int S>
__global__ __launch_bounds__(ANP_T) void add_norm_parts_kernel(
    const float* __restrict__ part, const unsigned short* __restrict__ bias,
    const unsigned short* __restrict__ resid,
    const unsigned short* __restrict__ norm_w,
    const unsigned short* __restrict__ norm_b,
    unsigned short* __restrict__ resid_out, unsigned short* __restrict__ y,
    int M, int H, float eps) {
    constexpr int MAXC = 4;                 // chunks of 8 a thread holds
    const long row = blockIdx.x;
    float v[MAXC][8], sum = 0.f, sumsq = 0.f;
#pragma unroll
    for (int c = 0; c < MAXC; ++c) {
        const int i = (c * ANP_T + threadIdx.x) * 8;
        if (i >= H) break;
        load_bf16x8(resid + row * H + i, v[c]);
        if (bias) {
            float b[8];
            load_bf16x8(bias + i, b);
#pragma unroll
            for (int e = 0; e < 8; ++e) v[c][e] += b[e];
        }
        // all parts on their way before the first is added
        f32x4 p[S][2];
#pragma unroll
        for (int s = 0; s < S; ++s)
#pragma unroll
            for (int q = 0; q < 2; ++q)
                p[s][q] = reinterpret_cast<const f32x4*>(
                    part + ((long)s * M + row) * H + i)[q];
#pragma unroll
        for (int s = 0; s < S; ++s)
#pragma unroll
            for (int e = 0; e < 8; ++e) v[c][e] += p[s][e / 4][e % 4];
        store_bf16x8(resid_out + row * H + i, v[c]);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            sum += v[c][e];
            sumsq += v[c][e] * v[c][e];
        }
    }
    if (!y) return;
    __shared__ float red[ANP_T / WAVE][2];
    sum = wave_sum(sum);
    sumsq = wave_sum(sumsq);
    if (threadIdx.x % WAVE == 0) {
        red[threadIdx.x / WAVE][0] = sum;
        red[threadIdx.x / WAVE][1] = sumsq;
    }
    __syncthreads();
    sum = sumsq = 0.f;
#pragma unroll
    for (int w = 0; w < ANP_T / WAVE; ++w) {
        sum += red[w][0];
        sumsq += red[w][1];
    }
    const float mean = norm_b ? sum / (float)H : 0.f;
    const float inv = rsqrtf(sumsq / (float)H - mean * mean + eps);
#pragma unroll
    for (int c = 0; c < MAXC; ++c) {
        const int i = (c * ANP_T + threadIdx.x) * 8;
        if (i >= H) break;
        float w[8], o[8];
        load_bf16x8(norm_w + i, w);
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = (v[c][e] - mean) * inv * w[e];
        if (norm_b) {
            float b[8];
            load_bf16x8(norm_b + i, b);
#pragma unroll
            for (int e = 0; e < 8; ++e) o[e] += b[e];
        }
        store_bf16x8(y + row * H + i, o);
    }
}

// H % 8 == 0, H <= 8192, S 1, 2, 4 or 8; nonzero otherwise
extern "C" int launch_add_norm_parts(
    const float* part, const unsigned short* bias, const unsigned short* resid,
    const unsigned short* norm_w, const unsigned short* norm_b,
    unsigned short* resid_out, unsigned short* y, int M, int H, int S,
    float eps, hipStream_t stream) {
    if (M < 1 || H % 8 || H > ANP_T * 32) return 1;
#define ANP_GO(SV)                                                            \
    case SV:                                                                  \
        hipLaunchKernelGGL((add_norm_parts_kernel<SV>), dim3(M), dim3(ANP_T), \
                           0, stream, part, bias, resid, norm_w, norm_b,      \
                           resid_out, y, M, H, eps);                          \
        return 0
    switch (S) {
        ANP_GO(1);
        ANP_GO(2);
        ANP_GO(4);
        ANP_GO(8);
    }
#undef ANP_GO
    return 1;
}
