// Projections of many rows: x [M, K] times rows of w [N, K], in bf16 with fp32
// sums. Three forms of result:
//  rows    x w^T in bf16;
//  gated   silu(gate) * value from w's two halves, so that the pass that reads
//          both and writes their product is gone, and neither is rounded;
//  parts   fp32 sums over S parts of K, left to the kernel that reads them
//          anyway (qkv_rope_store, add_norm_parts): where whole tiles would
//          leave much of the chip idle.
//
// Bound by the matrix cores (at the clock that the power limit leaves them:
// 8192x8192x8192 704 to 729 us from card to card, 1510 to 1560 TFLOP/s). A
// workgroup a CU: 256 rows of x (or 128, 160, 192, 224: so many as fill the last
// round) by 256 of w, 64 of K at a time in one of two buffers of 64 KB, filled
// straight from memory. Eight waves, two a SIMD: 128 x 64 sums each, in four quarters of 64 x
// 32. Waves 0-3 read a quarter's fragments while 4-7 multiply, and the other way
// round, so that the matrix cores always have one of a SIMD's two waves; a
// barrier at each change keeps them apart. What a quarter has read is loaded
// again at once, for the step after next: 3500 clocks ahead, 6 of 8 regions
// always under way. An XCD's workgroups take neighbouring tiles (8 by 4 at a
// time), which share what its L2 holds. Where there are more tiles than CUs a
// workgroup takes several: the next one's first steps are loaded under the last
// ones of this, whose rows go out from the registers (2 to 4% of a gated product,
// 1% of others).
//
// Measured with weights that no cache holds (us, on a card of the slower kind; in
// brackets the library's product, and of gated ones its swiglu):
//   gated 9216x2x18944x3584 1715 (2059), 4096x2x18944x3584 788 (911),
//    4559x2x8192x3072 340 (481), 1536x2x14336x4096 278 (318), 500x 95 (112);
//   rows 9216x3584x18944 848 (845), 4096x3584x18944 393 (498), 4096x4608x3584
//    116 (129), 1536x6144x4096 68 (74), 1536x128256x4096 1150 (1268);
//   parts, or rows, with the norm that follows: 1536x4096x14336 164 (190), 1100x
//    137 (168), 500x 71 (102), 800x2048x8192 40 (53), 1536x4096x4096 62 (64).
// Tried and slower: an XCD's tiles as one stretch for its workgroups (3 to 6%: some
// have a round more), tiles split over K inside one launch, the last to come
// adding (256 KB a tile and part written and read: 40 to 80 us a product).
#include "common.h"

#include <type_traits>

enum { LW_ROWS = 0, LW_GATED = 1, LW_PARTS = 2 };

DEV_INLINE unsigned lw_lds(const void* p) {
    return (unsigned)(unsigned long)(
        __attribute__((address_space(3))) const char*)p;
}
// 16 bytes a lane from base + off to LDS at `to` + lane * 16. The compiler does
// not see these loads: lw_wait counts them.
DEV_INLINE void lw_load(const void* base, unsigned off, unsigned to) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\t"
                 "global_load_lds_dwordx4 %0, %1"
                 ::"v"(off), "s"(base), "s"(to) : "memory", "m0");
}
// the lane, as a value that is not kept in a register from one use to the next
DEV_INLINE int lw_lane() {
    int z = 0;
    asm volatile("" : "+v"(z));
    return __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, z));
}
template <int N> DEV_INLINE void lw_wait() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
DEV_INLINE void lw_barrier() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}

// Fewest loads of a wave in X regions of x that follow one another, the last of
// them of the second half, or of either
constexpr int lw_loads(int MA, int MB, int X, bool second) {
    int least = 1 << 30;
    for (int early = 0; early < 2; ++early)    // waves 0-3, 4-7
        for (int last = second; last < 2; ++last) {
            int sum = 0;
            for (int i = 0; i < X; ++i) {
                const int g = (last + i) % 2, mt = g ? MB : MA;
                sum += mt == 4 || (mt == 3 && (early == 0) == (g == 0)) ? 2 : 1;
            }
            least = sum < least ? sum : least;
        }
    return least;
}

constexpr int LW_REGION = 128 * 128;           // 128 rows of 64 of K
constexpr int LW_LDS = 8 * LW_REGION;

// MA, MB: tiles of 16 rows of x that a wave takes in either half of a tile's
// 32 * (MA + MB) rows
template <int FORM, int MA, int MB>
__global__ __launch_bounds__(512) void linear_wide_kernel(
    const unsigned short* __restrict__ x, const unsigned short* __restrict__ w,
    void* __restrict__ out, int M, int N, int K, int S, int TM, int TN,
    int strip, int stride) {
    constexpr int BM = (MA + MB) * 32, HM = MA * 32;   // rows, of the first half
    static_assert(MA >= MB && MB >= 2 && MA <= 4, "");
    auto MT = [](int g) { return g ? MB : MA; };
    constexpr int BN = FORM == LW_GATED ? 128 : 256;   // columns of a tile
    const int tid = threadIdx.x, lane = tid & 63;
    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int li = lane & 15, lg = lane >> 4;
    const int wm = wid >> 2, wn = wid & 3;
    extern __shared__ __attribute__((aligned(16))) char smem[];

    // ---- tiles: an XCD's workgroups (every eighth) take neighbours, in strips
    // of `strip` row tiles; workgroup b its XCD's b / 8, b / 8 + stride, ..
    const int total = TM * TN * S, xcd = blockIdx.x & 7;
    const int mine = (total >> 3) + (xcd < (total & 7));       // of this XCD
    const int t0 = (total >> 3) * xcd + min(xcd, total & 7);
    int idx = blockIdx.x >> 3;
    const int n = K / 64 / S;                  // steps of 64: even
    int part, m0, n0;
    auto tile = [&](int i) {
        int t = t0 + i;
        part = t / (TM * TN);
        t -= part * TM * TN;
        const int s0 = t / (strip * TN), h = min(strip, TM - s0 * strip);
        t -= s0 * strip * TN;
        m0 = (s0 * strip + t % h) * BM;
        n0 = t / h * BN;
    };
    tile(idx);

    // ---- loads: a wave's are 8 rows of 128 bytes, lane l the 16 bytes that
    // belong at l * 16 (xor-ed by half the row's number: no two of a read's 16
    // rows meet in a bank)
    const char *xb, *wb, *wb1;
    // Of each half of w's 256 rows a wave loads 16, of x's twice 8, or once (of
    // halves of 96 rows four waves twice: of the first half 0-3, of the other
    // 4-7).
    auto first = [&](int g) {                  // its first 8 rows of x's half
        return MT(g) == 4 ? wid * 2 : MT(g) == 2 ? wid
               : (wid < 4) == (g == 0) ? wid % 4 * 2 : 8 + wid % 4;
    };
    unsigned xo[2][2], wo[2][2];
    auto aim = [&]() {                         // at the tile
        xb = reinterpret_cast<const char*>(x + (long)m0 * K + part * n * 64);
        wb = reinterpret_cast<const char*>(w + (long)n0 * K + part * n * 64);
        wb1 = FORM == LW_GATED ? wb + (long)N * K * 2 : wb;
        const int l = lw_lane(), r8 = l >> 3;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const unsigned c = ((l & 7) ^ (r8 >> 1)) * 16, c1 = c ^ 64;
#pragma unroll
            for (int g = 0; g < 2; ++g) {
                const int f = first(g) + j, xr = g * HM + f * 8 + r8;
                xo[g][j] = (unsigned)min(xr, M - 1 - m0) * K * 2 +
                           (f & 1 ? c1 : c);
                // (rows past the last: its)
                const int wr = (FORM == LW_GATED ? 0 : g * 128) + wid * 16 +
                               j * 8 + r8;
                wo[g][j] = (unsigned)min(wr, N - 1 - n0) * K * 2 + (j ? c1 : c);
            }
        }
    };
    aim();
    const unsigned to = __builtin_amdgcn_readfirstlane(lw_lds(smem));
    // regions of a buffer: x's halves, w's halves
    auto load_x = [&](int buf, int g, int step) {
        const char* b = xb + (long)step * 128;
        const unsigned at = to + (buf * 4 + g) * LW_REGION + first(g) * 1024;
        lw_load(b, xo[g][0], at);
        if (MT(g) == 4 || (MT(g) == 3 && (wid < 4) == (g == 0)))
            lw_load(b, xo[g][1], at + 1024);
    };
    auto load_w = [&](int buf, int g, int step) {
        const char* b = (g ? wb1 : wb) + (long)step * 128;
        const unsigned at = to + (buf * 4 + 2 + g) * LW_REGION + wid * 2048;
        lw_load(b, wo[g][0], at);
        lw_load(b, wo[g][1], at + 1024);
    };
    // until at most R regions' loads are under way (in the order w, x 0, w, x 1
    // of a step; the last of them x 1 where AT 1, and either kind elsewhere: R is
    // 6 there; as the wave has it that issued fewest), and, behind a whole tile's
    // `stores`, those
    constexpr int STORES = (FORM == LW_GATED ? 1 : FORM == LW_ROWS ? 2 : 4) *
                           (MA + MB);
    bool stores = false;
    auto wait = [&](auto regions, auto at1) {
        constexpr int R = decltype(regions)::value;
        constexpr bool A = decltype(at1)::value;
        constexpr int W = A ? R / 2 : (R + 1) / 2, X = R - W;
        static_assert(A || R == 6, "");
        constexpr int L = W * 2 + lw_loads(MA, MB, X, A);
        if (!A && stores) lw_wait<L + STORES>();
        else lw_wait<L>();
    };

    f32x4 acc[2][2][MA][2];                    // half of x, of w, tiles
    auto clear = [&]() {
#pragma unroll
        for (int i = 0; i < MA * 8; ++i)
            acc[i / (4 * MA)][i / (2 * MA) & 1][i / 2 % MA][i & 1] =
                f32x4{0.f, 0.f, 0.f, 0.f};
    };
    clear();
    bf16x8 fa[MA][2], fb[2][2][2];
    const int p0 = (lg ^ (li >> 1)) * 16;      // of K 0-31; 32-63: ^ 64
    const char* af = smem + (wm * MB * 16 + li) * 128;
    const char* bf = smem + (wn * 32 + li) * 128;
    const char* af0 = smem + (wm * MA * 16 + li) * 128;
    auto read_x = [&](int buf, int g) {
#pragma unroll
        for (int k = 0; k < 2; ++k)
#pragma unroll
            for (int i = 0; i < MA; ++i)
                if (i < MT(g))
                    fa[i][k] = *reinterpret_cast<const bf16x8*>(
                        (MA == MB || g ? af : af0) + (p0 ^ k * 64) +
                        (buf * 4 + g) * LW_REGION + i * 2048);
    };
    auto read_w = [&](int buf, int g) {
#pragma unroll
        for (int k = 0; k < 2; ++k)
#pragma unroll
            for (int i = 0; i < 2; ++i)
                fb[g][i][k] = *reinterpret_cast<const bf16x8*>(
                    bf + (p0 ^ k * 64) + (buf * 4 + 2 + g) * LW_REGION +
                    i * 2048);
    };
    auto products = [&](int gx, int gw) {
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int k = 0; k < 2; ++k)
#pragma unroll
            for (int i = 0; i < MT(gx); ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    acc[gx][gw][i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                        fb[gw][j][k], fa[i][k], acc[gx][gw][i][j], 0, 0, 0);
        __builtin_amdgcn_s_setprio(0);
    };
    // (the builtin: the compiler has to know that nothing is under way)
    auto here = [&]() {
        __builtin_amdgcn_s_waitcnt(0xc07f);
        lw_barrier();
    };
    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;
    using I2 = std::integral_constant<int, 2>;
    using I3 = std::integral_constant<int, 3>;
    using I4 = std::integral_constant<int, 4>;
    using I5 = std::integral_constant<int, 5>;
    using I6 = std::integral_constant<int, 6>;
    using No = std::false_type;
    using Yes = std::true_type;

    // Step s of parity P lies in buffer P. Its regions are read in the order w P,
    // x 0, w !P, x 1, the first in the step before; each is loaded again, for step
    // s + 2 (`nx`), where all waves have read it, seven reads ahead. half: after two of the four `stores` have to be done
    auto step = [&](auto par, auto ahead, int nx, bool half) {
        constexpr int P = decltype(par)::value, L = decltype(ahead)::value;
        // L: steps after this one, 2 standing for more
        read_x(P, 0);
        if (L == 2) load_w(P, P, nx);
        if (L == 2) wait(I6(), No());
        else if (L == 1) wait(I5(), Yes());
        else wait(I1(), Yes());
        here();
        products(0, P);
        lw_barrier();
        read_w(P, !P);
        if (L == 2) load_x(P, 0, nx);
        if (L == 2) wait(I6(), No());
        else if (L == 1) wait(I4(), Yes());
        else wait(I0(), Yes());
        here();
        products(0, !P);
        lw_barrier();
        if (half) stores = false;
        read_x(P, 1);
        if (L == 2) load_w(P, !P, nx);
        if (L == 2) wait(I6(), No());
        else if (L == 1) wait(I3(), Yes());
        here();
        products(1, !P);
        lw_barrier();
        if (L) read_w(!P, !P);
        if (L == 2) load_x(P, 1, nx);
        if (L == 2) wait(I6(), No());
        else if (L == 1) wait(I2(), Yes());
        here();
        products(1, P);
        lw_barrier();
    };
    // ---- C layout: column li = row of x, rows lg * 4 + r = columns. Two tiles of
    // 16 columns side by side: lane rows swapped so that a lane has 8 columns of
    // one of them
    auto finish = [&](int fm, int fn, int fp) {
        const bool whole = fm + BM <= M && fn + BN <= N;
        const int l = lw_lane(), lg = l >> 4;
        const int r0 = fm + (l & 15);
        const int c0 = fn + wn * 32 +
                       (FORM == LW_PARTS ? lg * 4
                                         : (lg & 1) * 16 + (lg >> 1) * 8);
        auto put = [&](int row, int col, f32x4 v) {
            const long at = (long)row * N + col;
            if (FORM == LW_PARTS)
                *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(out) +
                                          (long)fp * M * N + at) = v;
            else
                *reinterpret_cast<f32x4*>(
                    reinterpret_cast<unsigned short*>(out) + at) = v;
        };
        auto rows = [&](int gx, int i, int gw, auto all) {
            const int row = r0 + gx * HM + (wm * MT(gx) + i) * 16;
            const int col = c0 + gw * 128;
            if constexpr (FORM == LW_PARTS) {
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    if (decltype(all)::value ||
                        (row < M && col + j * 16 < N))
                        put(row, col + j * 16, acc[gx][gw][i][j]);
            } else {
                uint2v u[2];
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    f32x4 z = acc[gx][gw][i][j];
                    if (FORM == LW_GATED) {
#pragma unroll
                        for (int r = 0; r < 4; ++r)
                            z[r] = z[r] *
                                   __builtin_amdgcn_rcpf(1.f + __expf(-z[r])) *
                                   acc[gx][1][i][j][r];
                    }
                    typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
                    u[j] = __builtin_bit_cast(
                        uint2v, bf16x4{(__bf16)z[0], (__bf16)z[1], (__bf16)z[2],
                                       (__bf16)z[3]});
                }
                const uint2v a =
                    __builtin_amdgcn_permlane16_swap(u[0][0], u[1][0], false,
                                                     false);
                const uint2v b =
                    __builtin_amdgcn_permlane16_swap(u[0][1], u[1][1], false,
                                                     false);
                typedef __attribute__((ext_vector_type(4))) unsigned uint4v;
                if (decltype(all)::value || (row < M && col < N))
                    put(row, col, __builtin_bit_cast(
                                      f32x4, uint4v{a[0], b[0], a[1], b[1]}));
            }
        };
        auto tiles = [&](auto all) {
#pragma unroll
            for (int gx = 0; gx < 2; ++gx)
#pragma unroll
                for (int i = 0; i < MT(gx); ++i)
#pragma unroll
                    for (int gw = 0; gw < (FORM == LW_GATED ? 1 : 2); ++gw)
                        rows(gx, i, gw, all);
        };
        if (whole) tiles(Yes());
        else tiles(No());
        stores = whole;
    };
    for (int i = 0; i < 2; ++i) {
        load_w(i, i, i);
        load_x(i, 0, i);
        load_w(i, !i, i);
        load_x(i, 1, i);
    }
    wait(I6(), No());
    lw_barrier();
    read_w(0, 0);
    here();
    // waves 4-7 read while 0-3 multiply, and the other way round
    if (wid >= 4) lw_barrier();
    int nx = 2;
    for (;;) {
        const int fm = m0, fn = n0, fp = part;
        const bool more = idx + stride < mine;
        for (int s = 0; s + 2 < n + 2 * more; s += 2) {
            if (nx == n) {
                idx += stride;
                tile(idx);
                aim();
                nx = 0;
            }
            step(I0(), I2(), nx, false);
            step(I1(), I2(), nx + 1, true);
            nx += 2;
        }
        if (!more) {
            step(I0(), I1(), 0, false);
            step(I1(), I0(), 0, false);
        }
        finish(fm, fn, fp);
        if (!more) break;
        clear();
    }
    if (wid < 4) lw_barrier();
}

// Microseconds of a launch as the planner sees it: rounds of 256 workgroups, a
// last one that leaves CUs idle faster a step, each with a start and an end.
// Steps of 128-row tiles take less than those of 256 rows: they draw 48 KB from
// L2, not 64, for half the products. Gated ones and output heads, which outweigh
// the caches: fitted to 50 sizes of 300 to 9216 rows, the choice the fastest of
// its own in all but one (4% behind).
static double lw_time(int M, int N, int K, int form, int tall) {
    static const double step[] = {0.82, 1.0, 1.26}, idle[] = {0.48, 0.45, 0.56},
                        busy[] = {0.45, 0.58, 0.46};
    const int BN = form == LW_GATED ? 128 : 256, i = tall - 2;
    const long tiles = ((M + tall * 64L - 1) / (tall * 64)) *
                       ((N + BN - 1) / BN);
    const double steps = K / 64 * step[i], full = tiles / 256,
                 left = (tiles % 256) / 256.0;
    double t = full * (steps + tall + 3);
    if (left > 0) {
        const double f = idle[i] + busy[i] * left;
        t += steps * (f < 1 ? f : 1) + tall + 3;
    }
    return t;
}

// The same of the narrow projections (S parts; 1: rows), fitted to 437 products
// of 4M weights and more, 257 to 6000 rows, every launch with weights that no
// cache holds, as in a model's step: a round starts slower and few workgroups
// gain less than above. Parts are written, and read in place of bf16 rows.
static double lw_time_parts(int M, int N, int K, int tall, int S) {
    static const double step[] = {0.84, 1.05, 1.36}, idle[] = {0.75, 0.71, 0.63},
                        busy[] = {0.42, 0.23, 0.28}, start[] = {3.6, 5.1, 4.4},
                        round[] = {0, 2.1, 6.0}, store[] = {0.22, 0.14, 0.08};
    const int i = tall - 2;
    const long tiles = ((M + tall * 64L - 1) / (tall * 64)) *
                       ((N + 255) / 256) * S;
    const double steps = K / 64 / S * step[i], full = tiles / 256,
                 left = (tiles % 256) / 256.0;
    double t = start[i] + full * (steps + round[i]);
    if (left > 0) {
        const double f = idle[i] + busy[i] * left;
        t += steps * (f < 1 ? f : 1) + round[i];
    }
    if (S > 1)
        t += (double)M * N / 1e6 * (4 * S * store[i] + 0.2 * (4 * S - 2));
    return t;
}

// Heights between those of 64 rows: a third fit, of all five in one run (174
// products of 4M weights and more and 86 gated ones, 257 to 12000 rows, weights
// that no cache holds), that only compares heights.
static double lw_time_rows(int M, int N, int K, int S, bool gated, int rows) {
    struct Fit { double step, idle, busy, start, round, store; };
    static const Fit fits[2][5] = {
        {{0.754, 0.722, 0.989, 5.7, 0, 0.244}, {0.88, 0.807, 0.148, 8.3, 0, 0.183},
         {0.998, 0.709, 0.231, 9.3, 0.6, 0.144},
         {1.137, 0.68, 0.214, 9.6, 1.9, 0.124},
         {1.285, 0.684, 0.184, 13.4, 0.2, 0.139}},
        {{0.821, 0.595, 0.746, 6.8, 0, 0}, {0.935, 0.707, 0.313, 6.6, 0, 0},
         {1.031, 0.748, 0.672, 3.2, 0.9, 0}, {1.181, 0.717, 0.239, 6.1, 0.8, 0},
         {1.345, 0.632, 0.315, 8.2, 0, 0}}};
    const Fit& f = fits[gated][rows / 32 - 4];
    const int BN = gated ? 128 : 256;
    const long tiles = ((M + rows - 1L) / rows) * ((N + BN - 1) / BN) * S;
    const double steps = K / 64 / S * f.step, full = tiles / 256,
                 left = (tiles % 256) / 256.0;
    double t = f.start + full * (steps + f.round);
    if (left > 0) {
        const double part = f.idle + f.busy * left;
        t += steps * (part < 1 ? part : 1) + f.round;
    }
    return S > 1 ? t + (double)M * N / 1e6 * 4 * S * f.store : t;
}

// Rows of a tile of a plan's 64 * tall: 160 for 192 and 224 for 256 where fewer
// of them stand over in the last round, and 3% of the time (4559x3072x8192: 18 by
// 12 tiles of 256 rows leave 40 CUs idle, 170 us; 21 by 12 of 224 154). A product
// that would take the height tall - 1 takes these, too, if they beat it by as
// much. Of the 260 products, 77 are 7% faster for it and one is 2% slower; all
// heights' results are the same.
static bool lw_between(int M, int N, int K, int S, bool gated, int tall) {
    return tall > 2 && lw_time_rows(M, N, K, S, gated, tall * 64 - 32) <
                           0.97 * lw_time_rows(M, N, K, S, gated, tall * 64);
}
extern "C" int linear_wide_rows(int M, int N, int K, int S, int form, int tall) {
    return tall * 64 -
           (lw_between(M, N, K, S, form == LW_GATED, tall) ? 32 : 0);
}

// The tile's height and number of parts (1: rows) that are fastest: tall + 8 *
// parts, or 0: left to the library. Parts only where LW_PARTS is asked for. +
// 128: the rows past the last whole tile are linear_mid.hip's, which reads the
// weights once more for them: where they would begin a round of their own
// (9217x3584x18944: 37 rows of tiles by 14 are 518 workgroups).
//
// The library's time is fitted to the same products: its rounds of 256 x 256
// tiles, operations and weights. Of 208 other products (330 to 12000 rows) the
// choice is more than 3% behind the library in one and 0.7% from the best on
// average; the times that were fitted to cached weights left it behind in 18,
// with the norm that follows, us, those in brackets: 512x3072x2048 20.6 (26.0),
// 512x2048x2048 16.3 (21.0), 1200x3072x3072 40.4 (47.2), 1400x2560x2560 36.3
// (46.4). Products of fewer weights stay here, up to 5 us behind the library:
// steps of such a stack that are not captured are bound by the host, which takes
// 6 us to launch one and 20 for the library's (six layers of 768, prompts of 300
// to 1023 tokens: 580 us against 770).
extern "C" int linear_wide_plan(int M, int N, int K, int form) {
    if (M < 1 || N < 8 || N % 8 || K < 256 || K % 128 || K > 1 << 22) return 0;
    int best = 0;
    double least = 1e30;
    for (int tall = 2; tall <= 4; ++tall)
        for (int S = 1; S <= (form == LW_PARTS ? 8 : 1); S *= 2) {
            if (S > 1 && (K / 64 / S < 8 || K % (128 * S))) break;
            auto time = [&](int rows) {
                return form == LW_PARTS ? lw_time_parts(rows, N, K, tall, S)
                                        : lw_time(rows, N, K, form, tall);
            };
            const double t = time(M);
            if (t < least) {
                least = t;
                best = tall + 8 * S;
            }
            const int tail = M % (tall * 64);
            const double bytes = (form == LW_GATED ? 4.0 : 2.0) * N * K;
            if (S > 1 || tail == 0 || tail == M || bytes >= 1LL << 32) continue;
            const double t2 = time(M - tail) + (form == LW_PARTS ? 12 : 8) +
                              bytes / 5.2e6 * (1 + 0.0035 * tail);
            if (t2 < 0.97 * least) {
                least = t2;
                best = tall + 8 + 128;
            }
        }
    if (best < 128) {
        const bool gated = form == LW_GATED;
        const int S = best / 8;
        const int rows = linear_wide_rows(M, N, K, S, form, best % 8);
        const double own = lw_time_rows(M, N, K, S, gated, best % 8 * 64);
        double now = lw_time_rows(M, N, K, S, gated, rows);
        for (int tall = 3; tall <= 4; ++tall) {
            if (!lw_between(M, N, K, S, gated, tall)) continue;
            const double t = lw_time_rows(M, N, K, S, gated, tall * 64 - 32);
            if (t >= 0.97 * own || t >= now) continue;
            now = t;
            best = tall + 8 * S;
        }
    }
    const double flops = 2.0 * M * N * K, bytes = 2.0 * N * K;
    if (form == LW_GATED) return best;
    if (form == LW_PARTS) {
        if ((long)N * K < 4 << 20) return best;
        const long tiles = ((M + 255L) / 256) * ((N + 255) / 256);
        const double library = 5.3 + (tiles + 255) / 256 * (K * 2.29e-3) +
                               flops * 0.73e-9 + bytes * 0.173e-6;
        return least <= library ? best : 0;
    }
    // output heads of a few hundred rows are bound by their weights (200 rows,
    // us, the library's in brackets: 32000x4096 76 (71), 128256x4096 232 (293))
    double library = flops / 1.45e9 * 1.25 + 14;
    if (least < bytes / 5.05e6 + 24) least = bytes / 5.05e6 + 24;
    if (library < bytes / 3.7e6) library = bytes / 3.7e6;
    return least <= library ? best : 0;
}

// x [M, K], w [N, K] (LW_GATED [2N, K]) and out [M, N] (LW_PARTS [S, M, N] fp32)
// contiguous, 16-byte aligned; K % (128 S) == 0, N % 8 == 0; S 1 but for LW_PARTS;
// rows of a tile: 128, 160 .. 256. Nonzero for anything else.
extern "C" int launch_linear_wide(const unsigned short* x,
                                  const unsigned short* w, void* out, int M,
                                  int N, int K, int S, int form, int rows,
                                  hipStream_t stream) {
    if (M < 1 || N < 8 || N % 8 || S < 1 || K < 1 || K % (128L * S)) return 1;
    if (form != LW_PARTS && S != 1) return 1;
    if (rows < 128 || rows > 256 || rows % 32) return 1;
    if (K > 1 << 22) return 1;                 // offsets in a tile: 32 bits
    const int BN = form == LW_GATED ? 128 : 256;
    const int TM = (M + rows - 1) / rows, TN = (N + BN - 1) / BN;
    if ((long)TM * TN * S > 1 << 30) return 1;
    const int strips = (TM + 7) / 8, strip = (TM + strips - 1) / strips;
    const bool stay = TM * TN * S > 256;       // a workgroup a CU
    const dim3 grid(stay ? 256 : TM * TN * S);
    const int stride = stay ? 32 : 1 << 30;
#define LW_ONE(F, A, B)                                                       \
    if (rows == (A + B) * 32) {                                               \
        hipLaunchKernelGGL((linear_wide_kernel<F, A, B>), grid, dim3(512),    \
                           LW_LDS, stream, x, w, out, M, N, K, S, TM, TN,     \
                           strip, stride);                                    \
        return 0;                                                             \
    }
#define LW_GO(F)                                                              \
    if (form == F) {                                                          \
        LW_ONE(F, 2, 2)                                                       \
        LW_ONE(F, 3, 2)                                                       \
        LW_ONE(F, 3, 3)                                                       \
        LW_ONE(F, 4, 3)                                                       \
        LW_ONE(F, 4, 4)                                                       \
    }
    LW_GO(LW_ROWS)
    LW_GO(LW_GATED)
    LW_GO(LW_PARTS)
#undef LW_ONE
#undef LW_GO
    return 1;
}
