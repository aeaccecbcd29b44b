// Projections of 17 to 256 rows, of wide stacks from 9 or 12 on, and of fewer the
// longest gated ones and most output heads: x [M, K] times rows of w [N, K]. Three forms of result:
//  parts   fp32 sums over S parts of K, left to the kernel that reads them
//          anyway (qkv_rope_store, add_norm_parts): narrow projections, which
//          would leave most of the chip idle unsplit;
//  gated   silu(gate) * value in bf16 from w's two halves: the row tiles of w
//          take 8 rows of each half, and lanes l and l + 32 hold a pair;
//  rows    bf16, with bias and tanh-gelu where wanted (the output head, the
//          feed-forward of the GPT-2 family).
//
// Bound by reading the weights once, up to about 128 rows; beyond, by the steps of
// the four waves that load the input: at 200 rows 2200 clocks, of which products 900;
// their seven loads wait up to 1000 for the memory pipe, and the other four waves at
// the barrier for them. So a step finds out as little as it can: the two kinds of
// waves have loops of their own, in which the number of loads under way is known (us,
// with both in one loop / as now: 2x14336x4096 68.6 / 63.4 at 200 rows, 81.8 / 72.5
// at 256, 51.2 / 50.3 at 128; 4096x14336 38.9 / 36.4 at 200; 2x18944x3584 122 / 107;
// fewer rows within 2%). Loads spread between the products changed nothing, nor did
// halves that read and multiply in turn, weights in registers and the input in all of
// LDS, or tiles of 128 rows of w in turns with three buffers of both. A workgroup a
// CU, with two rings in LDS: 64 of K by the workgroup's rows of w, and by all input
// rows. Four waves fill the one, four the other, straight from memory
// (global_load_lds: no registers), and all eight multiply: the fragments of the next
// half step are read while this one's products run. The weights carry the streaming
// hint, so that they do not push the input out of L2 (2x14336x4096 at 24 rows 40.8 us
// without, 36.8 with; 4096x14336 24.8 / 22.2). Rows of 128 bytes in LDS are xor-ed by
// half their number: no two of a read's 16 rows meet in a bank. Workgroups start at
// different places of K: in step they would all ask for the same few channels
// (2x14336x4096 44.8 -> 41.3 us at 24 rows, 53 -> 44.5 at 80). Rows of more than four
// tiles a workgroup, which output heads are, start 5 steps apart and not one:
// 128256x4096 167 -> 159 us at 24 rows, 193 -> 188 at 80, 32000x4096 43.5 -> 41.8 at
// 24, 32000x2048 23.6 -> 22.6 (gated 2 to 4% slower so, others the same). The rings
// of up to 8 tiles hold what covers the memory's latency and no more: four slots of
// weights, 32 KB up to 4 tiles and 64 above. With all of LDS for weights every CU
// asks for 100 KB at once, and the input that the first step waits for queues behind
// it (us, rings of 96 to 112 KB / as now: 2048x8192 9.6 / 8.5 at 24 rows, 11.1 / 9.5
// at 57; 4096x4096 11.6 / 10.4 at 80; 2x8192x2048 16.0 / 14.7 at 57; 2x14336x4096
// 45.0 / 43.2 at 80; with 48 and 24 KB a third to half more time). The input has six
// slots there, fewer from 129 rows on, down to the three that LDS has room for above
// 192 (with two 44 -> 61 us at 80 rows). Gated products of 9 to 12 tiles and those of
// scaled rows (LM_SCALED) still have the long rings, 96 to 144 KB of weights; shorter
// ones were not measured there. Input rows apart by an odd number of lines change
// nothing. A CU takes in 57 GB/s from memory, 50 to 60 of weights and input together,
// so what a slot has past the rows and tiles that there are is not loaded (loaded /
// not: 2x18944x3584 47.5 / 46.4 at 24 rows, 54.8 / 52.4 at 80, 103 / 96 at 200, 123 /
// 109 at 256; 2x14336x4096 40.2 / 39.2 at 57, 43.8 / 42.4 at 80, 63.0 / 62.2 at 200;
// 6144x4096 14.4 / 13.9 at 80; others within 1%).
//
// Measured (us, launch after launch with weights that no cache holds, 24 / 80 / 128
// / 200 / 256 rows; in brackets with one loop and the long rings):
//   4096x14336 20.9 / 25.0 / 28.8 / 36.1 / 42.9 (21.1 / 26.3 / 29.7 / 38.9 / 45.3)
//   4096x4096  8.3 / 10.4 / 12.4 / 16.8 / 19.1 (9.4 / 11.6 / 13.2 / 17.5 / 19.9)
//   6144x4096  11.3 / 14.8 / 17.3 / 22.8 / 26.1 (11.4 / 15.8 / 18.6 / 24.5 / 27.9)
//   3584x18944 23.5 / 29.0 / 33.5 / 43.1 / 50.0 (23.9 / 30.5 / 34.5 / 45.1 / 52.7)
//   2048x8192  8.5 / 10.5 / 12.5 / 16.7 / 19.5 (9.6 / 11.7 / 13.2 / 18.0 / 20.2)
// The library's figures are at the rules in ops/__init__.py.
#include "common.h"

#include <type_traits>

enum { LM_PARTS = 0, LM_GATED = 1, LM_ROWS = 2 };

DEV_INLINE unsigned lm_lds(const void* p) {
    return (unsigned)(unsigned long)(
        __attribute__((address_space(3))) const char*)p;
}
// 16 bytes a lane of `lanes` from base + off to LDS at `to` + lane * 16 (all lanes
// are active before and after). The compiler does not see these loads: lm_wait
// counts them, those of no lane too. (M0 is set where it is used.)
template <bool STREAM>
DEV_INLINE void lm_load(const void* base, unsigned off, unsigned to,
                        unsigned long lanes) {
    if constexpr (STREAM)
        asm volatile("s_mov_b32 m0, %2\n\ts_mov_b64 exec, %3\n\t"
                     "global_load_lds_dwordx4 %0, %1 nt\n\t"
                     "s_mov_b64 exec, -1"
                     ::"v"(off), "s"(base), "s"(to), "s"(lanes)
                     : "memory", "m0");
    else
        asm volatile("s_mov_b32 m0, %2\n\ts_mov_b64 exec, %3\n\t"
                     "global_load_lds_dwordx4 %0, %1\n\t"
                     "s_mov_b64 exec, -1"
                     ::"v"(off), "s"(base), "s"(to), "s"(lanes)
                     : "memory", "m0");
}
// until at most `left` stages, of LO to HI, of PER loads each are under way
template <int PER, int LO, int HI>
DEV_INLINE void lm_wait(int left) {
    if constexpr (HI <= LO) {
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(PER * (HI > 0 ? HI : 0))
                     : "memory");
    } else {
        constexpr int MID = (LO + HI + 1) / 2;
        if (left >= MID) lm_wait<PER, MID, HI>(left);
        else lm_wait<PER, LO, MID - 1>(left);
    }
}

// Waves: WN groups of TW tiles of 16 rows of w, by WM groups of MW tiles of 16
// input rows, by WK halves of a step. DW, DX: slots of the rings. `tiles` of
// the TW * WN are used. WK 1: a workgroup takes every gridDim.x-th group of
// tiles, loading the next one's first steps under this one's last. APART: the two
// halves of K's steps have sums of their own, as with WK 2.
template <int TW, int MW, int WN, int WM, int WK, int DW, int DX, int OUT,
          bool SCALED = false, bool APART = false>
__global__ __launch_bounds__(512) void linear_mid_kernel(
    const unsigned short* __restrict__ x, const unsigned short* __restrict__ w,
    const unsigned short* __restrict__ bias, void* __restrict__ out, int M,
    int N, int K, int S, int tiles, int gelu,
    const float* __restrict__ squares, float eps) {
    constexpr int T = TW * WN, MT = MW * WM;
    static_assert(WN * WM * WK == 8 && DW >= 2 && DX >= 2, "");
    static_assert(WK == 1 || !APART, "");
    constexpr int NLW = T / 2, NLX = (MT + 1) / 2;  // loads of a wave a step
    constexpr int WB = NLW * 4096, XB = NLX * 4096; // bytes of a slot
    const int tid = threadIdx.x, lane = tid & 63;
    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int li = lane & 15, lg = lane >> 4;
    const int wn = wid % WN, wm = wid / WN % WM, wk = wid / WN / WM;
    const int NT = OUT == LM_GATED ? N / 8 : (N + 15) / 16;
    const int NG = (NT + tiles - 1) / tiles;
    const int CH = K / 64;                     // steps of 64: of them
    const int c0 = CH * blockIdx.y / S, n = CH * (blockIdx.y + 1) / S - c0;
    // where it starts
    const int rot = blockIdx.x / 8 * (OUT == LM_ROWS && tiles > 4 ? 5 : 1) % n;
    int g = blockIdx.x;
    const int total = n * ((NG - 1 - g) / (int)gridDim.x + 1);
    extern __shared__ __attribute__((aligned(16))) char smem[];

    // ---- loads: a wave's load is 8 rows of 128 bytes, lane l the chunk of 16
    // bytes that belongs at l * 16
    const bool of_w = wid < 4;
    const int r8 = lane >> 3, p8 = lane & 7;
    unsigned off[NLW > NLX ? NLW : NLX];
    // of the tiles and rows that there are: others' places in LDS hold anything,
    // and only their own sums come of it
    unsigned lanes[NLW > NLX ? NLW : NLX][2];
    auto only = [&](int j, unsigned long of) {
        lanes[j][0] = __builtin_amdgcn_readfirstlane((unsigned)of);
        lanes[j][1] = __builtin_amdgcn_readfirstlane((unsigned)(of >> 32));
    };
    const char* src = reinterpret_cast<const char*>(of_w ? w : x);
    auto rows_of = [&](int grp) {              // (tiles past the last: its)
        const int t0 = grp * tiles;
        if (OUT != LM_GATED)
            src = reinterpret_cast<const char*>(w + (long)t0 * 16 * K);
#pragma unroll
        for (int j = 0; j < NLW; ++j) {
            const int i = wid * NLW + j;
            const int r = (i & 1) * 8 + r8;
            const int t = min(t0 + min(i >> 1, tiles - 1), NT - 1);
            only(j, (i >> 1) < tiles && t0 + (i >> 1) < NT ? ~0ul : 0ul);
            const long row = OUT == LM_GATED
                                 ? (long)t * 8 + r8 + (i & 1) * (long)N
                                 : min(t * 16 + r, N - 1) - t0 * 16;
            off[j] = (unsigned)((row * K + (p8 ^ (r >> 1 & 7)) * 8) * 2);
        }
    };
    if (of_w) {
        rows_of(g);
    } else {
#pragma unroll
        for (int j = 0; j < NLX; ++j) {
            const int r = ((wid - 4) * NLX + j) * 8 + r8;
            off[j] = (unsigned)(((long)min(r, M - 1) * K +
                                 (p8 ^ (r >> 1 & 7)) * 8) * 2);
            only(j, __ballot(r < M));
        }
    }
    const unsigned to0 = lm_lds(smem) +
                         (of_w ? wid * NLW * 1024
                               : DW * WB + (wid - 4) * NLX * 1024);
    const char* at = src + (long)(c0 + rot) * 128;     // the next stage's
    int lk = rot, lleft = n, lgrp = g, lslot = 0;
    auto issue = [&](auto of) {                // its loads
        constexpr bool W = decltype(of)::value;
        if (W || MT > 1 || wid < 6)            // (MT 1: two waves' are all)
#pragma unroll
            for (int j = 0; j < (W ? NLW : NLX); ++j)
                lm_load<W>(at, off[j], to0 + lslot * (W ? WB : XB) + j * 1024,
                           lanes[j][0] | (unsigned long)lanes[j][1] << 32);
        if (++lslot == (W ? DW : DX)) lslot = 0;
        at += 128;
        if (++lk == n) {
            lk = 0;
            at -= (long)n * 128;
        }
        if (W && WK == 1 && --lleft == 0) {
            lleft = n;
            lgrp += gridDim.x;
            if (lgrp < NG) {
                rows_of(lgrp);
                at = src + (long)(c0 + lk) * 128;
            }
        }
    };
    using Yes = std::true_type;
    using No = std::false_type;
    if (of_w)
        for (int i = 0; i < DW && i < total; ++i) issue(Yes());
    else
        for (int i = 0; i < DX && i < total; ++i) issue(No());
    // 1 / rms of each row, while the weights are on their way: the waves of
    // the input, whose few stages the compiler's wait may include
    __shared__ float inv_s[16];
    if (SCALED && !of_w) {
        for (int row = wid - 4; row < M; row += 4) {
            float v = 0.f;
            for (int c = lane * 4; c < K / 8; c += 256) {
                const f32x4 q = *reinterpret_cast<const f32x4*>(
                    squares + (long)row * (K / 8) + c);
                v += (q[0] + q[1]) + (q[2] + q[3]);
            }
            v = wave_sum(v);
            if (lane == 0) inv_s[row] = rsqrtf(v / (float)K + eps);
        }
    }

    // ---- products
    f32x4 acc[TW][MW], other[APART ? TW : 1][APART ? MW : 1];
    auto clear = [&]() {
#pragma unroll
        for (int t = 0; t < TW; ++t)
#pragma unroll
            for (int m = 0; m < MW; ++m) {
                acc[t][m] = f32x4{0.f, 0.f, 0.f, 0.f};
                if constexpr (APART) other[t][m] = acc[t][m];
            }
    };
    clear();
    bf16x8 fw[2][TW], fx[2][MW];
    const char* wf = smem + (wn * TW * 16 + li) * 128;
    const char* xf = smem + DW * WB + (wm * MW * 16 + li) * 128;
    int ws = 0, xs = 0;                        // slots read from
    auto read = [&](int set, int half) {
        const int pos = ((half * 4 + lg) ^ (li >> 1)) << 4;
#pragma unroll
        for (int t = 0; t < TW; ++t)
            fw[set][t] = *reinterpret_cast<const bf16x8*>(
                wf + ws * WB + pos + t * 2048);
#pragma unroll
        for (int m = 0; m < MW; ++m)
            fx[set][m] = *reinterpret_cast<const bf16x8*>(
                xf + xs * XB + pos + m * 2048);
    };
    auto products = [&](int set) {
#pragma unroll
        for (int m = 0; m < MW; ++m)
#pragma unroll
            for (int t = 0; t < TW; ++t) {
                f32x4& to = APART && set ? other[APART ? t : 0][APART ? m : 0]
                                         : acc[t][m];
                to = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                    fw[set][t], fx[set][m], to, 0, 0, 0);
            }
    };
    // (the builtin: the compiler has to know that nothing is under way, or it
    // waits for what was only just asked for)
    auto fragments_here = [&]() { __builtin_amdgcn_s_waitcnt(0xc07f); };
    auto finish = [&](int grp) {
        const float inv = SCALED ? inv_s[min(li, M - 1)] : 1.f;
#pragma unroll
        for (int t = 0; t < TW; ++t) {
            const int tt = wn * TW + t, tile = grp * tiles + tt;
            if (tt >= tiles || tile >= NT) continue;
            // C layout: column li = input row, rows lg * 4 + r = columns
            const int col = OUT == LM_GATED ? tile * 8 + lg * 4
                                            : tile * 16 + lg * 4;
#pragma unroll
            for (int m = 0; m < MW; ++m) {
                const int row = (wm * MW + m) * 16 + li;
                f32x4 z = acc[t][m];
                if (OUT == LM_GATED) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const float2v p = lane_pair(
                            SCALED ? acc[t][m][r] * inv : acc[t][m][r]);
                        z[r] = p.x / (1.f + __expf(-p.x)) * p.y;
                    }
                }
                if (row >= M || (OUT == LM_GATED ? lane >= 32 : col >= N))
                    continue;
                if (OUT == LM_PARTS) {
                    *reinterpret_cast<f32x4*>(
                        reinterpret_cast<float*>(out) +
                        ((long)blockIdx.y * M + row) * N + col) = z;
                    continue;
                }
                if (OUT == LM_ROWS) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        if (bias) z[r] += bf2f(bias[col + r]);
                        if (gelu) {
                            // (1 + tanh c) / 2 = 1 / (1 + exp(-2 c))
                            const float c = 0.7978845608028654f *
                                            (z[r] + 0.044715f * z[r] * z[r] *
                                                        z[r]);
                            z[r] = z[r] / (1.f + __expf(-2.f * c));
                        }
                    }
                }
                *reinterpret_cast<uint2v*>(
                    reinterpret_cast<unsigned short*>(out) + (long)row * N +
                    col) =
                    uint2v{f2bf(z[0]) | (unsigned)f2bf(z[1]) << 16,
                           f2bf(z[2]) | (unsigned)f2bf(z[3]) << 16};
            }
        }
    };
    if (of_w) lm_wait<NLW, 0, DW - 1>(min(total, DW) - 1);
    else lm_wait<NLX, 0, DX - 1>(min(total, DX) - 1);
    fragments_here();                          // (and inv_s is written)
    asm volatile("s_barrier" ::: "memory");
    read(0, WK == 2 ? wk : 0);
    // Step s of `total`: stages up to s + D - 1 have been asked for, and behind the
    // barrier all have read stage s, and stage s + 1 has come. fast: there is a
    // stage s + D, so nothing has to be found out.
    auto step = [&](auto of, auto fast, int set, int s) {
        constexpr bool W = decltype(of)::value, FAST = decltype(fast)::value;
        constexpr int D = W ? DW : DX, PER = W ? NLW : NLX;
        fragments_here();
        if (WK == 1) {
            read(1, 1);
            products(0);
            fragments_here();
        }
        if (FAST || s + 1 < total) {
            lm_wait<PER, FAST ? D - 2 : 0, D - 2>(min(total - 2 - s, D - 2));
            asm volatile("s_barrier" ::: "memory");
            if (++ws == DW) ws = 0;
            if (++xs == DX) xs = 0;
            read(WK == 2 ? set ^ 1 : 0, WK == 2 ? wk : 0);
            if (FAST || s + D < total) issue(of);
        }
        products(WK == 2 ? set : 1);
        // (products that moved into the next step would need registers for three
        // steps' fragments)
        __builtin_amdgcn_sched_barrier(0);
    };
    auto steps = [&](auto of, int s, int end) {    // (WK 2: all of them)
        const int fast = min(end, total - (decltype(of)::value ? DW : DX));
        if (WK == 1) {
            for (; s < fast; ++s) step(of, Yes(), 0, s);
            for (; s < end; ++s) step(of, No(), 0, s);
            return;
        }
        for (; s + 1 < fast; s += 2) {
            step(of, Yes(), 0, s);
            step(of, Yes(), 1, s + 1);
        }
        for (;;) {
            step(of, No(), 0, s);
            if (++s >= end) break;
            step(of, No(), 1, s);
            if (++s >= end) break;
        }
    };
    if constexpr (WK == 1) {
        for (int s = 0; s < total; s += n) {
            if (of_w) steps(Yes(), s, s + n);
            else steps(No(), s, s + n);
            if constexpr (APART)
#pragma unroll
                for (int t = 0; t < TW; ++t)
#pragma unroll
                    for (int m = 0; m < MW; ++m)
#pragma unroll
                        for (int r = 0; r < 4; ++r)
                            acc[t][m][r] += other[t][m][r];
            finish(g);
            g += gridDim.x;
            clear();
        }
        return;
    }
    // The halves' sums meet in LDS (every load has come, and been read). Waves 0-3
    // are the first half: the two go their own ways from here, or their sums would
    // need the same registers.
    f32x4* mg = reinterpret_cast<f32x4*>(smem) +
                wid % (WN * WM) * TW * MW * 64 + lane;
    if (of_w) {
        steps(Yes(), 0, total);
        __syncthreads();
        __syncthreads();
#pragma unroll
        for (int t = 0; t < TW; ++t)
#pragma unroll
            for (int m = 0; m < MW; ++m) {
                const f32x4 p = mg[(t * MW + m) * 64];
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[t][m][r] += p[r];
            }
        finish(g);
    } else {
        steps(No(), 0, total);
        __syncthreads();
#pragma unroll
        for (int t = 0; t < TW; ++t)
#pragma unroll
            for (int m = 0; m < MW; ++m) mg[(t * MW + m) * 64] = acc[t][m];
        __syncthreads();
    }
}

// Tiles of 16 rows of w in a workgroup, as few as a chip of 256 CUs leaves it
// with `S` parts of K; `most` of them at most (then more workgroups than CUs,
// or rounds).
static int lm_tiles(int NT, int S, int most) {
    const int cus = 256 / S;
    const int rounds = (NT + cus * most - 1) / (cus * most);
    return (NT + cus * rounds - 1) / (cus * rounds);
}

// Parts of K: as many as leave a workgroup at most 8 tiles and, of K, twice as
// many steps of 64 as it has tiles (and 6), so that the parts, written and read
// once more, stay well below the weights. Measured with the kernel that reads
// them (us, 24 / 200 rows, before the streaming hint): 6144x4096 2 parts of 3
// tiles 19.6 / 30.9, 4 of 6 17.6 / 28.5, 8 of 12 20.1 / 33.9; 4096x4096 2 16.7 /
// 27.7, 4 14.5 / 22.4, 8 15.3 / 24.5; 4096x14336 4 28.1 / 48.2, 8 28.4 / 43.1;
// 3072x8192 4 18.9 / 30.7, 8 17.2 / 28.1; 2048x2048 2 10.1 / 16.7, 4 8.4 / 14.8,
// 8 8.6 / 17.1.
extern "C" int linear_mid_splits(int N, int K) {
    const int NT = (N + 15) / 16;
    int S = 1;
    for (int s = 2; s <= 8; s *= 2) {
        const int tiles = (NT + 256 / s - 1) / (256 / s);
        const int n = K / 64 / s;
        if (tiles <= 8 && n >= 6 && n >= 2 * tiles) S = s;
    }
    return S;
}

// x [M, K] and w contiguous and 16-byte aligned, 1 <= M <= 256, K % 64 == 0.
// out: form LM_PARTS [S, M, N] fp32, 1 <= S <= K / 64; LM_GATED [M, N] bf16, w
// [2N, K], N % 8 == 0, S 1, no bias; LM_ROWS [M, N] bf16, S 1. N % 4 == 0.
// squares [M, K / 8] (LM_GATED, M <= 16; else null): RMS norm of
// rows that come multiplied by its weight, whose sums of squares these are.
// Nonzero for anything else.
extern "C" int launch_linear_mid(const unsigned short* x,
                                 const unsigned short* w,
                                 const unsigned short* bias, void* out, int M,
                                 int N, int K, int S, int form, int gelu,
                                 const float* squares, float eps,
                                 hipStream_t stream) {
    if (M < 1 || M > 256 || N < 4 || N % 4 || K < 64 || K % 64) return 1;
    if (S < 1 || S > K / 64 || (form != LM_PARTS && S != 1)) return 1;
    if (form == LM_GATED && N % 8) return 1;
    // offsets are of 32 bits
    if (form == LM_GATED && ((long)2 * N * K * 2) >> 32) return 1;
    const int NT = form == LM_GATED ? N / 8 : (N + 15) / 16;
    // 12 tiles and all rows' sums fit the registers of up to 160 rows
    const int most = form == LM_GATED && M <= 160 && NT > 2048 && NT <= 3072
                         ? 12 : 8;
    const int tiles = lm_tiles(NT, S, most);
    const int NG = (NT + tiles - 1) / tiles;
    const bool once = NG * S <= 256;           // no second group of tiles
#define LM_GO(TW, MW, WN, WM, WK, DW, DX, F)                                  \
    LM_SUMS(TW, MW, WN, WM, WK, DW, DX, F, false)
#define LM_SUMS(TW, MW, WN, WM, WK, DW, DX, F, APART)                         \
    do {                                                                      \
        constexpr int lds =                                                   \
            DW * (TW * WN / 2) * 4096 + DX * ((MW * WM + 1) / 2) * 4096;      \
        static_assert(lds <= 163840, "LDS of a CU");                          \
        static_assert(WK == 1 || TW * MW * 1024 * 4 <= lds, "halves");        \
        hipLaunchKernelGGL(                                                   \
            (linear_mid_kernel<TW, MW, WN, WM, WK, DW, DX, F, false, APART>), \
            dim3(WK == 1 && !once ? 256 / S : NG, S), dim3(512),              \
            lds, stream, x, w, bias, out, M, N, K, S, tiles, gelu, nullptr,   \
            0.f);                                                             \
        return 0;                                                             \
    } while (0)
#define LM_4(F)                                                               \
    do {                                                                      \
        if (M <= 32) LM_GO(1, 2, 4, 1, 2, 4, 6, F);                           \
        if (M <= 64) LM_GO(1, 4, 4, 1, 2, 4, 6, F);                           \
        if (M <= 96) LM_GO(2, 3, 2, 2, 2, 4, 6, F);                           \
        if (M <= 128) LM_GO(2, 4, 2, 2, 2, 4, 6, F);                          \
        if (M <= 160) LM_GO(2, 5, 2, 2, 2, 4, 6, F);                          \
        if (M <= 192) LM_GO(2, 6, 2, 2, 2, 4, 5, F);                          \
        if (M <= 224) LM_GO(2, 7, 2, 2, 2, 4, 4, F);                          \
        LM_GO(2, 8, 2, 2, 2, 4, 4, F);                                        \
    } while (0)
#define LM_8(F)                                                               \
    do {                                                                      \
        if (M <= 32) LM_GO(1, 2, 8, 1, 1, 4, 6, F);                           \
        if (M <= 64) LM_GO(1, 4, 8, 1, 1, 4, 6, F);                           \
        if (M <= 96 && once) LM_GO(2, 6, 4, 1, 2, 4, 6, F);                   \
        if (M <= 96) LM_GO(1, 6, 8, 1, 1, 4, 6, F);                           \
        if (M <= 128) LM_GO(2, 4, 4, 2, 1, 4, 6, F);                          \
        if (M <= 160) LM_GO(2, 5, 4, 2, 1, 4, 4, F);                          \
        if (M <= 192) LM_GO(2, 6, 4, 2, 1, 4, 4, F);                          \
        if (M <= 224) LM_GO(2, 7, 4, 2, 1, 4, 3, F);                          \
        LM_GO(2, 8, 4, 2, 1, 4, 3, F);                                        \
    } while (0)
#define LM_APART(F)                                                           \
    do {                                                                      \
        if (M <= 192) LM_SUMS(2, 6, 4, 2, 1, 4, 4, F, true);                  \
        LM_SUMS(2, 7, 4, 2, 1, 4, 3, F, true);                                \
    } while (0)
#define LM_SCALED(TW, MW, WN, WM, WK, DW, DX)                                 \
    do {                                                                      \
        constexpr int lds =                                                   \
            DW * (TW * WN / 2) * 4096 + DX * ((MW * WM + 1) / 2) * 4096;      \
        static_assert(lds + 64 <= 163840, "LDS of a CU");                     \
        hipLaunchKernelGGL(                                                   \
            (linear_mid_kernel<TW, MW, WN, WM, WK, DW, DX, LM_GATED, true>),  \
            dim3(WK == 1 && !once ? 256 : NG), dim3(512), lds, stream, x, w,  \
            nullptr, out, M, N, K, 1, tiles, 0, squares, eps);                \
        return 0;                                                             \
    } while (0)
    if (squares) {
        if (form != LM_GATED || M > 16) return 1;
        if (tiles > 8) LM_SCALED(3, 1, 4, 1, 2, 6, 3);
        if (tiles > 4) LM_SCALED(1, 1, 8, 1, 1, 8, 4);
        LM_SCALED(1, 1, 4, 1, 2, 12, 6);
    }
    if (form == LM_GATED && tiles > 8) {
        if (M <= 32) LM_GO(3, 2, 4, 1, 2, 6, 3, LM_GATED);
        if (M <= 64) LM_GO(3, 4, 4, 1, 2, 5, 3, LM_GATED);
        if (M <= 96) LM_GO(3, 3, 4, 2, 1, 5, 3, LM_GATED);
        if (M <= 128) LM_GO(3, 4, 4, 2, 1, 4, 3, LM_GATED);
        LM_GO(3, 5, 4, 2, 1, 4, 3, LM_GATED);
    }
    // Sums of all of K in one chain are half as far off again (parts of 4096x14336 from
    // 64 bits 2.5e-7 of their norm, in two chains 1.7e-7); where registers allow it they
    // are two. us, one chain / two, at 192 rows: 4096x14336 33.7 / 34.8, 2x14336x4096 58.2
    // / 58.7; 224: 36.4 / 36.7, 65.9 / 63.7.
    const bool apart = tiles > 4 && once && M > 160 && M <= 224;
    if (form == LM_GATED && tiles <= 4) LM_4(LM_GATED);
    if (form == LM_GATED && apart) LM_APART(LM_GATED);
    if (form == LM_GATED) LM_8(LM_GATED);
    if (form == LM_ROWS && tiles <= 4) LM_4(LM_ROWS);
    // (half the input: 128256x4096 168 -> 155 us at 1 row with the places of K,
    // 128256x2048 79.5 -> 77.9, 152064x3584 165 -> 163)
    if (form == LM_ROWS && M <= 16) LM_GO(1, 1, 8, 1, 1, 4, 6, LM_ROWS);
    if (form == LM_ROWS) LM_8(LM_ROWS);
    if (tiles <= 4) LM_4(LM_PARTS);
    if (apart) LM_APART(LM_PARTS);
    LM_8(LM_PARTS);
#undef LM_SCALED
#undef LM_APART
#undef LM_8
#undef LM_4
#undef LM_SUMS
#undef LM_GO
    return 1;
}

// ----------------------------------------------------------- add_norm_parts
// sum = resid + the parts [+ bias], either in bf16 or fp32; y = norm(sum) (RMS, or
// layer norm with norm_b), from the fp32 sum; y null: the sum only. One
// workgroup of T threads a row, which stays in registers between its two uses; a
// thread takes V columns at a time. Many rows are bound by their bytes; of few, a
// row's workgroup by the latency of its parts, which come from other XCDs: 1024
// threads that ask for all of them at once. Behind the product that makes them,
// us, with 256 threads of 8 columns / as now: 8 parts of 24x4096 5.2 / 4.6, of
// 80x4096 6.8 / 5.9, of 24x3072 4.8 / 3.9, 4 parts of 24x4096 4.0 / 3.5, of 57x2048
// 3.4 / 3.3; 2 of 1536x4096 14.6 and with 1024 threads 15.9.
constexpr int ANP_MOST = 8192;              // columns
template <int V> DEV_INLINE void anp_load(const unsigned short* p, float* to) {
    if constexpr (V == 8) {
        load_bf16x8(p, to);
    } else {
        const uint2v u = *reinterpret_cast<const uint2v*>(p);
#pragma unroll
        for (int e = 0; e < 4; ++e)
            to[e] = bf2f((unsigned short)(u[e / 2] >> e % 2 * 16));
    }
}
template <int V>
DEV_INLINE void anp_store(unsigned short* p, const float* from) {
    if constexpr (V == 8)
        store_bf16x8(p, from);
    else
        *reinterpret_cast<uint2v*>(p) =
            uint2v{f2bf(from[0]) | (unsigned)f2bf(from[1]) << 16,
                   f2bf(from[2]) | (unsigned)f2bf(from[3]) << 16};
}
template <int S, int T, int V>
__global__ __launch_bounds__(T) void add_norm_parts_kernel(
    const float* __restrict__ part, const unsigned short* __restrict__ bias,
    const void* __restrict__ resid, int resid32,
    const unsigned short* __restrict__ norm_w,
    const unsigned short* __restrict__ norm_b, void* __restrict__ sum_out,
    int sum32, unsigned short* __restrict__ y, int M, int H, float eps) {
    constexpr int MAXC = ANP_MOST / (T * V);    // chunks of V a thread holds
    const long row = blockIdx.x;
    __attribute__((aligned(16))) float v[MAXC][V];
    float sum = 0.f, sumsq = 0.f;
#pragma unroll
    for (int c = 0; c < MAXC; ++c) {
        const int i = (c * T + threadIdx.x) * V;
        if (i >= H) break;
        // all parts on their way before the first is added
        f32x4 p[S][V / 4];
#pragma unroll
        for (int s = 0; s < S; ++s)
#pragma unroll
            for (int q = 0; q < V / 4; ++q)
                p[s][q] = reinterpret_cast<const f32x4*>(
                    part + ((long)s * M + row) * H + i)[q];
        if (resid32) {
#pragma unroll
            for (int q = 0; q < V / 4; ++q)
                *reinterpret_cast<f32x4*>(v[c] + q * 4) =
                    reinterpret_cast<const f32x4*>(
                        reinterpret_cast<const float*>(resid) + row * H + i)[q];
        } else {
            anp_load<V>(reinterpret_cast<const unsigned short*>(resid) +
                            row * H + i, v[c]);
        }
        if (bias) {
            float b[V];
            anp_load<V>(bias + i, b);
#pragma unroll
            for (int e = 0; e < V; ++e) v[c][e] += b[e];
        }
#pragma unroll
        for (int s = 0; s < S; ++s)
#pragma unroll
            for (int e = 0; e < V; ++e) v[c][e] += p[s][e / 4][e % 4];
        if (sum32) {
#pragma unroll
            for (int q = 0; q < V / 4; ++q)
                reinterpret_cast<f32x4*>(reinterpret_cast<float*>(sum_out) +
                                         row * H + i)[q] =
                    *reinterpret_cast<const f32x4*>(v[c] + q * 4);
        } else {
            anp_store<V>(reinterpret_cast<unsigned short*>(sum_out) + row * H +
                             i, v[c]);
        }
#pragma unroll
        for (int e = 0; e < V; ++e) {
            sum += v[c][e];
            sumsq += v[c][e] * v[c][e];
        }
    }
    if (!y) return;
    __shared__ float red[T / WAVE][2];
    sum = wave_sum(sum);
    sumsq = wave_sum(sumsq);
    if (threadIdx.x % WAVE == 0) {
        red[threadIdx.x / WAVE][0] = sum;
        red[threadIdx.x / WAVE][1] = sumsq;
    }
    __syncthreads();
    sum = sumsq = 0.f;
#pragma unroll
    for (int w = 0; w < T / WAVE; ++w) {
        sum += red[w][0];
        sumsq += red[w][1];
    }
    const float mean = norm_b ? sum / (float)H : 0.f;
    const float inv = rsqrtf(sumsq / (float)H - mean * mean + eps);
#pragma unroll
    for (int c = 0; c < MAXC; ++c) {
        const int i = (c * T + threadIdx.x) * V;
        if (i >= H) break;
        float w[V], o[V];
        anp_load<V>(norm_w + i, w);
#pragma unroll
        for (int e = 0; e < V; ++e) o[e] = (v[c][e] - mean) * inv * w[e];
        if (norm_b) {
            float b[V];
            anp_load<V>(norm_b + i, b);
#pragma unroll
            for (int e = 0; e < V; ++e) o[e] += b[e];
        }
        anp_store<V>(y + row * H + i, o);
    }
}

// H % 8 == 0, H <= 8192, S 1, 2, 4 or 8; nonzero otherwise
extern "C" int launch_add_norm_parts(
    const float* part, const unsigned short* bias, const void* resid,
    int resid32, const unsigned short* norm_w, const unsigned short* norm_b,
    void* sum, int sum32, unsigned short* y, int M, int H, int S, float eps,
    hipStream_t stream) {
    if (M < 1 || H % 8 || H > ANP_MOST) return 1;
#define ANP_ONE(SV, T, V)                                                     \
    hipLaunchKernelGGL((add_norm_parts_kernel<SV, T, V>), dim3(M), dim3(T),   \
                       0, stream, part, bias, resid, resid32, norm_w, norm_b, \
                       sum, sum32, y, M, H, eps)
#define ANP_GO(SV)                                                            \
    case SV:                                                                  \
        if (M > 256) ANP_ONE(SV, 256, 8);                                     \
        else if (H > 2048) ANP_ONE(SV, 1024, 4);                              \
        else ANP_ONE(SV, 512, 4);                                             \
        return 0
    switch (S) {
        ANP_GO(1);
        ANP_GO(2);
        ANP_GO(4);
        ANP_GO(8);
    }
#undef ANP_ONE
#undef ANP_GO
    return 1;
}
