// A decode step of a few sequences through the layers of a dense stack, in one
// launch: q|k|v, attention against the pages, output, gate and up (or the GPT-2
// family's up projection) and down, with norms, rotation, page store, activation
// and residual.
//
// Bound by the weights, and by what lies between two products: a launch after a
// launch costs 2.2 us here, and then a product waits 2 us more for its first
// weights; a layer was six launches. Here a workgroup a CU stays for the whole
// stack; weights depend on nothing, so the next product's are asked for under
// the last steps of this one, and what crosses the chip between products are a
// few KB of rows. A step with its logits, us, launch by launch / in one: 6 layers
// of 768 columns, 300 keys 213 / 172; 8 of 2048, 1000 keys 412 / 360; 8 of 4096,
// 3000 keys 924 / 810; 8 of 3584, two rows of 24000 keys 1058 / 979.
//  * Rows pass from workgroup to workgroup as words that say themselves whether
//    they are there: buffers are filled with DS_EMPTY (a NaN) before, a word is
//    stored once, and readers load it until it is something else. Every such
//    word is an agent-scope atomic, so no fence is needed, and a hop costs one
//    store and one load: 1.9 us from product to product with 256 workgroups,
//    where counters beside the data took 2.5 and a launch 2.2.
//  * A wave streams its eighth of K of 8 rows of W at a time (an octet: 8 rows
//    at two places along K, 128 bytes of a row together, as one left operand of
//    a 16x16x32 product; the input rows at both places as the other) through a
//    ring of DS_RING KB in LDS, over the ends of octets and products. It polls
//    its own eighth of the input rows; no wave waits for rows that it does not
//    read. Loads of a wave come back in order, so the words wait behind what of
//    the ring is still under way.
//  * A ninth wave adds up the eight and does all that follows a product.
//  * Attention is attn_stream.hip's tile of 32 keys a wave, eight waves a
//    workgroup, with keys straight into the operand's registers. Contexts of up
//    to DS_ALONE keys take one workgroup a key head; longer ones are split, and
//    waves of their own add the splits up. The step's own keys and values, of
//    all rows whose pages a context has, are taken from the words, not from
//    the pages that they are stored to meanwhile.
//  * Number c's octets of a product are c, c + DS_WGS and so on. Nothing has to
//    be resident together for that: a workgroup claims its number when it
//    starts, and after the first product each one sees that all numbers are
//    claimed, by running workgroups then; where they are not for a while
//    (another kernel holds CUs) it claims free ones itself and does their work
//    too. One that starts late and finds its number taken leaves. So a workgroup
//    only ever waits for others that run.
//  * A wait ends all the same: after DS_PATIENCE polls in which no workgroup with
//    several numbers, which take their time, got on (the share of one is done in
//    a millisecond). The host is told then (status), and from there on nothing is
//    stored that depends on a word that did not come, to pages in particular: the
//    others' waits end with it, and rows that no one is left to compute are NaN
//    or as they were.
#include "common.h"
#include "decode_stack.h"

typedef __attribute__((ext_vector_type(4))) short short4v;
typedef __attribute__((address_space(3))) short4v lds_short4v;
typedef __attribute__((ext_vector_type(4))) unsigned int ds_raw;

constexpr int DS_WAVES = 8;                    // that stream
constexpr int DS_RING = 8;                     // weight loads under way in each
// Steps that are read at once (1 / 2 / 3 / 4: us a layer of 768 columns 25.0 /
// 24.6 / 24.2 / 24.2, of 2048 35.3 / 35.2 / 34.7 / 35.0, of 4096 83.6 / 82.2 / 81.7 /
// 81.9)
constexpr int DS_BATCH = 3;
constexpr unsigned DS_EMPTY = 0xffffffffu;
constexpr int DS_KEYS = 32;                    // of a wave's tile
constexpr int DS_STEP = DS_WAVES * DS_KEYS;
// Keys that are not split, a tile of each wave (of 300 keys, a layer of 768 columns
// 24.7 us split and 25.2 not, 400 of 4096 columns 81.7 and 84.0), and least keys of
// a split (64: the same; 256: 1000 keys of 2048 columns 35.7 us, not 34.9).
constexpr int DS_ALONE = 256;
constexpr int DS_LEAST = 128;
constexpr int DS_PART = 18;                    // words: 16 columns of a split's
                                               // result, its maximum and sum
constexpr int DS_KEPT = 4;                     // octets of which much is in LDS
constexpr float DS_LOG2E = 1.44269504088896340736f;
enum { DS_LEAVE = -3, DS_OPEN = -2, DS_GO_ON = -1 };

DEV_INLINE unsigned long ds_load(const void* p) {
    return __hip_atomic_load(reinterpret_cast<const unsigned long*>(p),
                             __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
DEV_INLINE bool ds_there(unsigned long v) {
    return (unsigned)v != DS_EMPTY && (unsigned)(v >> 32) != DS_EMPTY;
}
// a word that is there (a result that looks like DS_EMPTY is another NaN)
DEV_INLINE unsigned ds_word(unsigned v) {
    return v == DS_EMPTY ? 0x7fff7fffu : v;
}
DEV_INLINE unsigned ds_word(float v) {
    return ds_word(__builtin_bit_cast(unsigned, v));
}
template <typename T> DEV_INLINE void ds_store(unsigned* p, T v) {
    __hip_atomic_store(p, ds_word(v), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T> DEV_INLINE void ds_store(unsigned* p, T v, T w) {
    __hip_atomic_store(reinterpret_cast<unsigned long*>(p),
                       ds_word(v) | (unsigned long)ds_word(w) << 32,
                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
DEV_INLINE float ds_low(unsigned long v) {
    return __builtin_bit_cast(float, (unsigned)v);
}
DEV_INLINE float ds_high(unsigned long v) {
    return __builtin_bit_cast(float, (unsigned)(v >> 32));
}
DEV_INLINE unsigned ds_load4(const unsigned* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Steps of a wave's input up to which all words are asked for at once (see until)
constexpr int DS_FEW = 6;
DEV_INLINE int ds_same(int v) { return __builtin_amdgcn_readfirstlane(v); }
DEV_INLINE unsigned ds_pack(float a, float b) {
    return f2bf(a) | (unsigned)f2bf(b) << 16;
}
// the same of another lane of the eight, without LDS
template <int CTRL> DEV_INLINE float ds_dpp(float v) {
    return __builtin_bit_cast(
        float, __builtin_amdgcn_update_dpp(
                   0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}
DEV_INLINE float ds_xor1(float v) { return ds_dpp<0xB1>(v); }
DEV_INLINE float ds_xor2(float v) { return ds_dpp<0x4E>(v); }
DEV_INLINE float ds_xor4(float v) { return ds_dpp<0x1B>(ds_dpp<0x141>(v)); }
DEV_INLINE float ds_wave_sum(float v) {
    v += ds_dpp<0x128>(v);                     // rotations of a row of 16
    v += ds_dpp<0x124>(v);
    v += ds_dpp<0x122>(v);
    v += ds_dpp<0x121>(v);
    return rows_sum(v);
}
// workgroup barrier that leaves loads from memory under way
DEV_INLINE void ds_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}
// 16 bytes a lane from base + off to LDS at `to` + lane * 16. The compiler does
// not see these loads: ds_wait counts them. (M0 is set where it is used.)
DEV_INLINE void ds_ask(const char* base, unsigned off, unsigned to,
                       bool streamed) {
    if (streamed)
        asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\t"
                     "global_load_lds_dwordx4 %0, %1 nt"
                     ::"v"(off), "s"(base), "s"(to) : "memory", "m0");
    else
        asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\t"
                     "global_load_lds_dwordx4 %0, %1"
                     ::"v"(off), "s"(base), "s"(to) : "memory", "m0");
}
// 4 bytes a lane
DEV_INLINE void ds_ask4(const char* base, unsigned off, unsigned to) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\t"
                 "global_load_lds_dword %0, %1"
                 ::"v"(off), "s"(base), "s"(to) : "memory", "m0");
}
// The same, unknown to the compiler: what is made of it is made where it is
// used, not before the loop over layers (that takes more registers than there
// are, and the ones put aside are loaded behind the weights: two rows of 24000
// keys 118 us a layer, not 113).
DEV_INLINE int ds_own(int v) {
    asm volatile("" : "+v"(v));
    return v;
}
// until at most `left` of this wave's loads are under way
template <int LEFT> DEV_INLINE void ds_wait() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LEFT) : "memory");
}

// the same pointer in all lanes, of memory
template <typename T> DEV_INLINE T* ds_uniform(T* p) {
    typedef __attribute__((address_space(1))) T* global;
    const unsigned long v = reinterpret_cast<unsigned long>(p);
    return (T*)(global)((unsigned long)(unsigned)ds_same((int)v) |
                        (unsigned long)(unsigned)ds_same((int)(v >> 32)) << 32);
}

// 8 elements of a page's row as an operand
DEV_INLINE bf16x8 ds_widen(uint2v x) {
    typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
    bf16x8 r;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const unsigned w = x[i];
        const bf16x2 a =
            __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, 1.f, false);
        const bf16x2 b =
            __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, 1.f, true);
        r[i * 4] = a[0];
        r[i * 4 + 1] = a[1];
        r[i * 4 + 2] = b[0];
        r[i * 4 + 3] = b[1];
    }
    return r;
}
// from memory, which the compiler is told: a choice between this and LDS is made
// one of addresses otherwise
template <bool NT = false, typename T> DEV_INLINE T ds_global(const T* p) {
    const auto from = (const __attribute__((address_space(1))) T*)p;
    if constexpr (NT) return __builtin_nontemporal_load(from);
    else return *from;
}

// A context's split: keys `from` up to `to` of number z's, of `len` keys, `per`
// keys each.
struct Span {
    int len, per, from, to;
    DEV_INLINE int splits() const { return (len + per - 1) / per; }
    DEV_INLINE bool none(int z) const { return z > 0 && from >= len; }
};
DEV_INLINE Span ds_span(int len, int Z, int z) {
    Span s;
    s.len = len;
    const int even = (len + Z - 1) / Z;
    s.per = max((even + DS_KEYS - 1) / DS_KEYS * DS_KEYS, DS_LEAST);
    if (len <= DS_ALONE || Z == 1) s.per = max(len, 1);
    s.from = z * s.per;
    s.to = min(len, s.from + s.per);
    return s;
}

template <bool LAYER, int HD, typename KVT>
__global__ __launch_bounds__((DS_WAVES + 1) * 64) void decode_stack_kernel(
    StackArgs args) {
    const int tid = threadIdx.x, lane = tid & 63;
    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int number = blockIdx.x % DS_WGS;
    // the rings; then input rows, or the attention waves' tiles
    extern __shared__ __attribute__((aligned(16))) char smem[];
    char* const area = smem + DS_WAVES * DS_RING * 1024;
    // the waves' sums of an octet, twice: [wave][place][row][8 columns]
    __shared__ float part[2][DS_WAVES][2][DS_ROWS][8];
    __shared__ float ml[16][DS_WAVES][2];      // attention: maxima and sums
    __shared__ short cols[DS_WGS];             // this workgroup's numbers
    // of the ninth wave's octets: biases, norm weights; the residual
    __shared__ unsigned operands[DS_KEPT][2][64];
    __shared__ float residual[DS_KEPT][64];
    __shared__ int slot_s[DS_ROWS], len_s[DS_ROWS];
    __shared__ int own_s[DS_ROWS];             // attention: keys of this step
    __shared__ int ncols, begin, gate;
    __shared__ int gone;                       // a wait has been given up
    __shared__ unsigned seen[DS_WAVES + 1];    // progress, when a wave last looked
    constexpr int LW = sizeof(StackLayer) / 4;
    __shared__ __attribute__((aligned(16))) int layers[(DS_LAYERS + 1) * LW];

    // ---- What the launch is told is kept in LDS, and read where it is needed:
    // scalar loads would cost 0.2 us each there (a line's first 1 us), and the
    // compiler takes all of them before the loop, into more registers than
    // there are.
    __shared__ StackHead told_s;
    const char* const told =
        (const char*)__builtin_amdgcn_kernarg_segment_ptr();
    int kw = reinterpret_cast<const int*>(told)[min(lane, 11)];
    for (int i = tid; i < (int)sizeof(StackHead) / 4;
         i += (DS_WAVES + 1) * 64)
        reinterpret_cast<int*>(&told_s)[i] =
            reinterpret_cast<const int*>(told)[i];
    for (int i = tid; i < (DS_LAYERS + 1) * LW; i += (DS_WAVES + 1) * 64)
        layers[i] = reinterpret_cast<const int*>(
            told + offsetof(StackArgs, layer))[i];
    int lo = args.lo, hi = args.hi, M = args.M;
    float* const turns = reinterpret_cast<float*>(area + args.turns);
    // the step's own keys and values: [row][2][HD / 2]
    auto fresh_at = [&](int n, int of) __attribute__((always_inline)) {
        return reinterpret_cast<unsigned*>(turns) + M * HD +
               (n * 2 + of) * (HD / 2);
    };
    const bool rope = args.cos_t != nullptr;
    int* const pages = reinterpret_cast<int*>(area + args.pages);
    const bool paged = args.area;
    asm volatile("s_waitcnt vmcnt(0)" : "+v"(kw), "+s"(lo), "+s"(hi), "+s"(M)
                 ::"memory");
    auto depth = [&](int k) __attribute__((always_inline)) {
        return __builtin_amdgcn_readlane(kw, k);
    };
    auto octets = [&](int k) __attribute__((always_inline)) {
        return __builtin_amdgcn_readlane(kw, 4 + k);
    };
    // pointer i of layer l
    auto pointer = [&](int l, int i) __attribute__((always_inline)) {
        return ds_uniform(reinterpret_cast<const char* const*>(
            layers + (l - lo) * LW)[i]);
    };
    const bool gelu = args.gelu, streamed = args.streamed;
    constexpr int hd_log2 = HD == 64 ? 6 : 7;
    static_assert(HD == 64 || HD == 128, "");
    // octets of product k that number c has
    auto count = [&](int k, int c) __attribute__((always_inline)) {
        const int n = octets(k) - c;
        return n > 0 ? (unsigned)(n + DS_WGS - 1) / DS_WGS : 0;
    };
#define DS_INT(name) ds_same(told_s.name)
#define DS_PTR(name) ds_uniform(told_s.name)
    // words of layer l
    auto at = [&](int l, int off) __attribute__((always_inline)) {
        return DS_PTR(words) + (long)l * DS_INT(stride) + off;
    };
    if (tid == 0) gone = 0;
    if (lane == 0) seen[wid] = DS_EMPTY;
    ds_barrier();                              // (0) all of it is there

    // Has this wait lasted long enough, or has another one? (Lane by lane: scalar
    // registers are what the kernel has too few of. With scalar values a step of six
    // layers takes 2 us more, for code that does not run.)
    auto enough = [&](int polls) __attribute__((always_inline)) {
        typedef __attribute__((address_space(1))) unsigned* global;
        unsigned* const state = (unsigned*)(global)told_s.state;
        bool end = __hip_atomic_load(&gone, __ATOMIC_RELAXED,
                                     __HIP_MEMORY_SCOPE_WORKGROUP) ||
                   ds_load4(state + 32) != DS_EMPTY;
        if ((polls & told_s.patience) == 0) {
            const unsigned now = ds_load4(state);
            end = end || now == seen[wid];
            seen[wid] = now;
        }
        if (end) {
            gone = 1;
            __hip_atomic_store(state + 32, 0u, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
        }
        return (bool)__any(end);
    };
    // Are all lanes' words there? If not, some clocks are left to the others
    // before they are asked for again: eight waves that ask without a pause keep
    // the ninth from issuing loads and stores at all.
    auto again = [&](bool there, int& polls) __attribute__((always_inline)) {
        if (__all(there)) return false;
        if (__builtin_expect((++polls & 31) == 0, 0) && enough(polls)) return false;
        __builtin_amdgcn_s_sleep(1);
        return true;
    };
    // Until the word at p is there: one request a wave, where all the words that
    // it will read would be asked for in vain. Where those are few, asking for
    // them all saves the second request: up to 768 bytes of a wave's input
    // (DS_FEW steps) a layer of 768 columns takes 25.0 us and not 25.9, of 2048
    // 34.9 and 35.4, but of 4096, at up to 1 KB, 83.5 and 82.7.
    auto until = [&](const unsigned* p) __attribute__((always_inline)) {
        int polls = 0;
        while (again(ds_load4(p) != DS_EMPTY, polls)) {}
    };

    if (wid == DS_WAVES) {
        // ------------------------------------------------ the ninth wave
        __builtin_amdgcn_s_setprio(3);         // the others wait for this one
        const int j = lane & 7, m = lane >> 3;
        const bool on = m < M;
        const int H = depth(DS_QKV);
        int buf = 0;
        unsigned* counters = DS_PTR(claims) + DS_WGS;
        // is it this workgroup's now?
        auto claim = [&](int c) __attribute__((always_inline)) {
            unsigned old = 0;
            if (lane == 0) {
                old = __hip_atomic_exchange(DS_PTR(claims) + c, 0u,
                                            __ATOMIC_RELAXED,
                                            __HIP_MEMORY_SCOPE_AGENT);
                if (old == DS_EMPTY)
                    __hip_atomic_fetch_add(counters + c % 8 * 32, 1u,
                                           __ATOMIC_RELAXED,
                                           __HIP_MEMORY_SCOPE_AGENT);
            }
            return __builtin_amdgcn_readfirstlane(old) == DS_EMPTY;
        };
        auto all_claimed = [&]() __attribute__((always_inline)) {
            bool full = true;                  // (counters start at -1)
            if (lane < 8)
                full = __hip_atomic_load(counters + lane * 32,
                                         __ATOMIC_RELAXED,
                                         __HIP_MEMORY_SCOPE_AGENT) ==
                       DS_WGS / 8 - 1;
            return (bool)__all(full);
        };
        const int mine = number;
        // What the step's rows are: slots, lengths, pages, rotation. The others
        // have them with their next barrier.
        int slot = 0, len = 0, position = 0;
        if (lane < M) {
            const int *slots = DS_PTR(slots), *pos = DS_PTR(pos);
            const int W = DS_INT(W), bs = DS_INT(bs);
            if (pos) position = pos[lane];
            len = DS_PTR(seq_lens)[lane];
            if (slots)
                slot = slots[lane];
            else
                slot = position < 0 || position / bs >= W
                           ? -1             // (no such position)
                           : DS_PTR(table)[lane * W + position / bs] * bs +
                                 position % bs;
        }
        const bool own = claim(mine);
        if (lane < M) {
            slot_s[lane] = slot;
            len_s[lane] = max(min(len, DS_INT(W) * DS_INT(bs)), 0);
        }
        if (paged)
            for (int i = lane; i < M * DS_INT(W); i += 64)
                pages[i] = DS_PTR(table)[i];
        if (rope)
            for (int i = lane; i < M * (HD / 2); i += 64) {
                const int row = i / (HD / 2), d = i % (HD / 2);
                const long from = turn_row(__shfl(position, row),
                                           DS_INT(turn_rows)) * (HD / 2) + d;
                turns[row * HD + d] = DS_PTR(cos_t)[from];
                turns[row * HD + HD / 2 + d] = DS_PTR(sin_t)[from];
            }
        if (lane == 0) {
            cols[0] = mine;
            ncols = 1;
        }

        float inv = 1.f;
        // 1 / rms of this lane's row: of rows that a product left, from their
        // sums of squares of 8 columns; of the first layer's, from the rows
        auto scales = [&](int l, int k) __attribute__((always_inline)) {
            const int Q = H / 8;               // (even)
            const float* squares = reinterpret_cast<const float*>(
                (k == DS_QKV ? at(l - 1, DS_INT(down)) : at(l, DS_INT(o))) +
                M * H / 2);
            float scale = 1.f;
            auto keep = [&](int row, float sum) __attribute__((always_inline)) {
                sum = ds_wave_sum(sum);
                if (m == row) scale = rsqrtf(sum / (float)H + told_s.eps);
            };
            if (l == 0 && k == DS_QKV) {
                for (int row = 0; row < M; ++row) {
                    float sum = 0.f;
                    for (int i = lane * 8; i < H; i += 512) {
                        float v[8];
                        load_bf16x8(DS_PTR(x) + row * H + i, v);
#pragma unroll
                        for (int e = 0; e < 8; ++e) sum = fmaf(v[e], v[e], sum);
                    }
                    keep(row, sum);
                }
                return scale;
            }
            // 16 loads at a time: of U for 128 sums each, rows beside each other
            // (one after the other, 4 rows of 768 columns take 2 us more a layer)
            auto rows = [&](auto u) __attribute__((always_inline)) {
                constexpr int U = decltype(u)::value, R = 16 / U;
                for (int r0 = 0; r0 < M; r0 += R) {
                    float sum[R] = {};
                    for (int i0 = 0; i0 < Q; i0 += U * 128) {
                        unsigned long v[R][U];
                        bool ok;
                        int polls = 0;
                        do {
                            ok = true;
#pragma unroll
                            for (int i = 0; i < R * U; ++i)
                                if (r0 + i / U < M && i0 + i % U * 128 < Q)
                                    v[i / U][i % U] = ds_load(
                                        squares + (r0 + i / U) * Q +
                                        min(i0 + i % U * 128 + lane * 2,
                                            Q - 2));
#pragma unroll
                            for (int i = 0; i < R * U; ++i)
                                if (r0 + i / U < M && i0 + i % U * 128 < Q)
                                    ok = ok && ds_there(v[i / U][i % U]);
                        } while (again(ok, polls));
#pragma unroll
                        for (int i = 0; i < R * U; ++i)
                            if (r0 + i / U < M &&
                                i0 + i % U * 128 + lane * 2 < Q)
                                sum[i / U] += ds_low(v[i / U][i % U]) +
                                              ds_high(v[i / U][i % U]);
                    }
#pragma unroll
                    for (int r = 0; r < R; ++r)
                        if (r0 + r < M) keep(r0 + r, sum[r]);
                }
            };
            if (M * Q > 256)
                until(reinterpret_cast<const unsigned*>(squares) + M * Q - 1);
            if (M > 2 && Q <= 256) rows(std::integral_constant<int, 2>());
            else rows(std::integral_constant<int, 8>());
            return scale;
        };
        bool passed = false;
        int nc = 1, parts = -1;
        // whether to go on: known to all with the first product's last barrier
        auto decide = [&]() __attribute__((always_inline)) {
#pragma unroll 1
            for (int k = 0; k < 32 && own && !passed; ++k)
                passed = all_claimed();
            if (lane == 0)
                begin = !own ? DS_LEAVE : passed ? DS_GO_ON : DS_OPEN;
        };
        // Biases and norm weights of a product's first octets are asked for when
        // the last product is done, into LDS: such loads wait behind the weights
        // that are under way. The residual stays in LDS.
        const unsigned kept = (unsigned)(unsigned long)(
            __attribute__((address_space(3))) char*)&operands[0][0][0];
        // of the octet's columns; the norm's next weights
        auto bias_at = [&](int k, int o) __attribute__((always_inline)) {
            if (k != DS_QKV) return o * 8 + j;
            constexpr int per = hd_log2 - 3;
            return (o >> per << hd_log2) + (o & ((1 << per) - 1)) * 4 + (j & 3) +
                   (j >> 2) * (HD / 2);
        };
        auto next_norm = [&](int l, int k) __attribute__((always_inline)) {
            if (LAYER || k == DS_QKV || k == DS_UP ||
                (k == DS_DOWN && l + 1 == DS_INT(all)))
                return (const char*)nullptr;
            return k == DS_O ? pointer(l, 9) : pointer(l + 1, 8);
        };
        auto fetch = [&](int l, int k) __attribute__((always_inline)) {
            const char* const bias = pointer(l, 4 + k);
            const char* const norm = next_norm(l, k);
            unsigned to = kept;
#pragma unroll 1
            for (int o = mine; o < min(octets(k), mine + DS_KEPT * DS_WGS);
                 o += DS_WGS, to += 512) {
                if (bias) ds_ask4(bias, (bias_at(k, o) & ~1) * 2, to);
                if (norm) ds_ask4(norm, ((o * 8 + j) & ~1) * 2, to + 256);
            }
        };
        auto pick = [&](unsigned v) __attribute__((always_inline)) {
            return __builtin_bit_cast(float, j & 1 ? v & 0xffff0000u : v << 16);
        };
        // Octet o of product k, the q-th of number cols[i]; dst: the words that
        // the product leaves. What can be done before the sums are there is.
        auto octet = [&](int l, int k, int o, int i, int q, const char* bias,
                         const char* norm, unsigned* dst)
                         __attribute__((always_inline)) {
            const int N = octets(k) * 8;       // (not of q|k|v, gate and up)
            const int col = o * 8 + j, where = m * N + col;
            const bool adds = k == DS_O || k == DS_DOWN;
            const bool in_lds = i == 0 && q < DS_KEPT;
            float add = 0.f, times = 1.f;
            if (bias)
                add = pick(in_lds ? operands[q][0][lane]
                                  : *reinterpret_cast<const unsigned*>(
                                        bias + (bias_at(k, o) & ~1) * 2));
            if (norm)
                times = pick(in_lds ? operands[q][1][lane]
                                    : *reinterpret_cast<const unsigned*>(
                                          norm + (col & ~1) * 2));
            if (adds) {
                const int at = min(m, M - 1) * N + col;
                if (in_lds && !(l == lo && k == DS_O))
                    add += residual[q][lane];
                else if (l == 0 && k == DS_O)
                    add += bf2f(DS_PTR(x)[at]);
                else
                    add += DS_PTR(x32)[at];
            }
            // of q|k|v: the head, the column, the rotation
            constexpr int per = hd_log2 - 3;
            const int head = o >> per, d0 = (o & ((1 << per) - 1)) * 4 + (j & 3);
            float cosine = 1.f, sine = 0.f;    // (a c - b s, b c + a s)
            if (k == DS_QKV && rope && head < DS_INT(nq) + DS_INT(nkv)) {
                const float* t = turns + min(m, M - 1) * HD + d0;
                cosine = t[0];
                sine = j < 4 ? -t[HD / 2] : t[HD / 2];
            }
            ds_barrier();                      // the waves' sums are there
            // (one order of three whose errors against 64 bits are the same)
            float p[DS_WAVES];
#pragma unroll
            for (int w = 0; w < DS_WAVES; ++w)
                p[w] = part[buf][w][0][m][j] + part[buf][w][1][m][j];
#pragma unroll
            for (int n = DS_WAVES / 2; n > 0; n /= 2)
#pragma unroll
                for (int w = 0; w < n; ++w) p[w] += p[w + n];
            buf ^= 1;
            const bool sound = !gone, put = on && sound;
            float z = p[0] * inv;
            if (k == DS_UP && !gelu) {
                const float u = ds_xor4(z);
                const float v = z / (1.f + __expf(-z)) * u;
                const float v1 = ds_xor1(v);
                if (put && j < 4 && j % 2 == 0)
                    ds_store(dst + (m * N / 2 + o * 4 + j) / 2, ds_pack(v, v1));
                return;
            }
            if (k != DS_QKV) z += add;
            if (adds) {
                const bool ends = k == DS_DOWN && l + 1 == DS_INT(all);
                if (in_lds) residual[q][lane] = z;
                if (ends) {
                    const float y = ds_xor1(z);
                    if (on && j % 2 == 0)
                        DS_PTR(out)[where / 2] = sound ? ds_pack(z, y)
                                                       : 0x7fff7fffu;
                    return;
                }
                if (LAYER) {
                    if (put) ds_store(dst + where, z);
                } else {
                    const float v = z * times, v1 = ds_xor1(v);
                    if (put && j % 2 == 0)
                        ds_store(dst + where / 2, ds_pack(v, v1));
                    float sq = z * z;
                    sq += ds_xor1(sq);
                    sq += ds_xor2(sq);
                    sq += ds_xor4(sq);
                    if (put && j == 0)
                        ds_store(dst + M * H / 2 + where / 8, sq);
                }
                // (also for the next launch)
                if (on && (!in_lds || (k == DS_DOWN && l + 1 == hi)))
                    DS_PTR(x32)[where] = z;
            } else if (k == DS_UP) {
                const float e = 0.7978845608028654f *
                                (z + 0.044715f * z * z * z);
                z = 0.5f * z * (1.f + tanhf(e));
                const float y = ds_xor1(z);
                if (put && j % 2 == 0) ds_store(dst + where / 2, ds_pack(z, y));
            } else {
                const int nq = DS_INT(nq), nkv = DS_INT(nkv);
                z += add;
                z = z * cosine + ds_xor4(z) * sine;
                const float y = ds_xor1(z);
                if (!put || j % 2) return;
                const int d = d0 + (j >> 2) * (HD / 2);
                if (head < nq) {
                    ds_store(dst + (((m * nq + head) << hd_log2) + d) / 2,
                             ds_pack(z, y));
                    return;
                }
                const bool is_k = head < nq + nkv;
                const int kvh = head - nq - (is_k ? 0 : nkv);
                unsigned word = ds_pack(z, y);
                unsigned short pair = 0;
                if (sizeof(KVT) == 1) {        // as the page has it
                    pair = f2fp8x2(bf2f(f2bf(z)), bf2f(f2bf(y)));
                    const float2v f = fp8x2_2f(pair);
                    word = ds_pack(f.x, f.y);
                }
                const int row = (m * 2 + !is_k) * nkv + kvh;
                ds_store(dst + DS_INT(new_kv) + ((row << hd_log2) + d) / 2,
                         word);
                const int slot = slot_s[m], bs = DS_INT(bs);
                if (slot < 0) return;          // no such position
                const long to =
                    ((((long)(slot / bs) * nkv + kvh) * bs + slot % bs)
                     << hd_log2) + d;
                char* cache = const_cast<char*>(pointer(l, is_k ? 12 : 13));
                if (sizeof(KVT) == 1)
                    reinterpret_cast<unsigned short*>(cache)[to / 2] = pair;
                else
                    reinterpret_cast<unsigned*>(cache)[to / 2] = word;
            }
        };

        fetch(lo, DS_QKV);
        for (int l = lo, k = 0, other = -1; l < hi;) {
            int some = 0;
            inv = 1.f;
            const char* const bias = pointer(l, 4 + k);
            const char* const norm = next_norm(l, k);
            unsigned* const dst =
                at(l, k == DS_QKV  ? 0
                      : k == DS_O  ? DS_INT(o)
                      : k == DS_UP ? DS_INT(up)
                                   : DS_INT(down));
            const bool start = l == lo && k == DS_QKV;
            for (int i = other >= 0 ? nc - 1 : 0; i < nc; ++i) {
                const int c = i ? ds_same(cols[i]) : mine, n = count(k, c);
                for (int q = 0; q < n; ++q) {
                    if (some++ == 0) {
                        ds_wait<0>();          // what fetch asked for
                        if (LAYER && (k == DS_QKV || k == DS_UP))
                            ds_barrier();      // (N) sums of the rows
                        if (!LAYER && (k == DS_QKV || k == DS_UP))
                            inv = scales(l, k);
                    }
                    if (start && i == 0 && q == n - 1) decide();
                    if (own) octet(l, k, c + q * DS_WGS, i, q, bias, norm, dst);
                    else ds_barrier();
                }
            }
            if (k < 3) fetch(l, k + 1);
            else if (l + 1 < hi) fetch(l + 1, DS_QKV);
            if (l == lo && k == DS_QKV) {
                if (other >= 0) {
                    ds_barrier();              // (3): gate has been read
                } else {
                    if (!some) {
                        decide();
                        ds_barrier();          // (1)
                    }
                    if (!own) return;
                }
                if (!passed || other >= 0) {
                    const long since = wall_clock64();
                    other = -1;
                    while (!passed && other < 0) {
                        passed = all_claimed();
                        if (passed || wall_clock64() - since < 2000) continue;
                        // 20 us
                        for (int i = 1; i < DS_WGS && other < 0; ++i) {
                            const int c = (mine + i) % DS_WGS;
                            if (claim(c)) other = c;
                        }
                    }
                    if (lane == 0) {
                        gate = other;          // (DS_GO_ON)
                        if (other >= 0) cols[nc] = other, ncols = nc + 1;
                    }
                    ds_barrier();              // (2)
                    if (other >= 0) {
                        ++nc;
                        continue;
                    }
                }
            }
            if (k == DS_QKV) {
                // items of attention (of one number the same in every layer)
                if (parts < 0 || nc > 1) {
                    parts = 0;
                    const int Z = DS_INT(Z);
                    for (int i = 0; i < nc; ++i) {
                        const int c = i ? ds_same(cols[i]) : mine;
                        for (int it = c; it < DS_INT(items); it += DS_WGS) {
                            const int len = len_s[it / Z / DS_INT(nkv)];
                            if (!ds_span(ds_same(len), Z, it % Z).none(it % Z))
                                ++parts;
                        }
                    }
                }
                for (int i = 0; i < parts; ++i) {
                    ds_barrier();              // (A)
                    ds_barrier();              // (B)
                }
            }
            if (++k == 4) k = 0, ++l;
        }
        return;
    }

    // ---------------------------------------------------- the waves of weights
    const int li = lane & 15, lg = lane >> 4;
    const int lj = li & 7, lk = (li >> 3) * 32 + lg * 8;
    const int xrow = min(lj, M - 1);
    // Of the products of a number, in lanes k * 8 + ..: its octets; this wave's
    // steps of an octet, and the first (<< 16); bytes from w to the first, and
    // from an octet's last step to the next octet's first; 2 K; 2 K half
    int plan = 0;
    auto prepare = [&](int c) __attribute__((always_inline)) {
        const int k = lane >> 3 & 3, f = lane & 7;
        const int K = told_s.K[k], o = told_s.octets[k];
        const int s0 = (unsigned)K / 64 * wid / DS_WAVES;
        const int n = (int)((unsigned)K / 64 * (wid + 1) / DS_WAVES) - s0;
        constexpr int per = hd_log2 - 3;       // log2 of a head's octets
        const bool fours = k == DS_UP && !gelu;
        const int row = k == DS_QKV
                            ? (c >> per << hd_log2) + (c & ((1 << per) - 1)) * 4
                            : c * (fours ? 4 : 8);
        const long off = ((long)row * K + s0 * 64) * 2;
        // (of q|k|v: whole heads further)
        const long jump = (long)DS_WGS * (fours ? 4 : 8) * K * 2 - (n - 1) * 128;
        plan = f == 0   ? (n && o > c ? (unsigned)(o - c + DS_WGS - 1) / DS_WGS
                                      : 0)
               : f == 1 ? n | s0 << 16
               : f == 2 ? (int)off
               : f == 3 ? (int)(off >> 32)
               : f == 4 ? (int)jump
               : f == 5 ? (int)(jump >> 32)
               : f == 6 ? K * 2
                        : (int)((unsigned)told_s.half[k] * K * 2);
    };
    prepare(number);
    auto planned = [&](int k, int f) __attribute__((always_inline)) {
        return __builtin_amdgcn_readlane(plan, k * 8 + f);
    };

    // ---- the stream of weights, a KB a step of 64 of K, into this wave's ring:
    // octet after octet of the numbers of this workgroup, product after product
    int gl = lo, gk = 0, gi = -1, gnc = 1;     // layer, product, index in cols
    int gleft = 0, goct = 0, gn = 0;           // steps, octets left; of an octet
    long gjump = 0;                            // to the next octet
    const char* gp = pointer(lo, 0);
    unsigned goff = 0;
    int told_l = layers[lane & 7];             // the layer's weights
    const unsigned ring = (unsigned)(unsigned long)(
        __attribute__((address_space(3))) char*)smem + wid * DS_RING * 1024;
    unsigned gslot = 0;                        // in bytes
    // on to the next number, or product, that has any
    auto seek = [&]() __attribute__((always_inline)) {
        goct = gleft = 0;                      // (none: the last address again)
        while (gl < hi) {
            if (++gi >= gnc) {
                gi = -1;
                if (++gk == 4) {
                    gk = 0;
                    ++gl;
                    told_l = layers[(gl - lo) * LW + (lane & 7)];
                }
                continue;
            }
            if (gnc > 1) prepare(gi ? ds_same(cols[gi]) : number);
            goct = planned(gk, 0);
            if (!goct) continue;
            gleft = gn = planned(gk, 1) & 0xffff;
            goff = (lj & 3) * (unsigned)planned(gk, 6) + lk * 2u +
                   (lj >> 2 ? (unsigned)planned(gk, 7) : 0u);
            const unsigned long from =
                (unsigned)__builtin_amdgcn_readlane(told_l, gk * 2) |
                (unsigned long)(unsigned)__builtin_amdgcn_readlane(
                    told_l, gk * 2 + 1) << 32;
            gp = (const char*)(const __attribute__((address_space(1))) char*)
                     from +
                 ((unsigned)planned(gk, 2) | (long)planned(gk, 3) << 32);
            gjump = (unsigned)planned(gk, 4) | (long)planned(gk, 5) << 32;
            return;
        }
    };
    auto ask = [&]() __attribute__((always_inline)) {
        ds_ask(gp, goff, ring + gslot, streamed);
        gslot += 1024;
        if (gslot == DS_RING * 1024) gslot = 0;
        if (goct == 0) return;
        if (--gleft) {
            gp += 128;
        } else if (--goct) {
            gp += gjump;
            gleft = gn;
        } else {
            seek();
        }
    };

    // ---- this wave's part of the rows that product k reads, in LDS
    char* xw = area;
    int xstride = 0;
    auto input = [&](int l, int k) __attribute__((always_inline)) {
        const int lane = ds_own(tid & 63);
        const int K = depth(k);
        const int s0 = planned(k, 1) >> 16, n = planned(k, 1) & 0xffff;
        xstride = n * 128 + 16;                // (rows in different banks)
        xw = area + M * (s0 * 128 + wid * 16);
        const bool raw = l == 0 && k == DS_QKV;
        if (LAYER && (k == DS_QKV || k == DS_UP)) {
            // Mean and deviation are of the whole row, to which each wave gives
            // the sums of its part (two columns a lane).
            const int H = K, e = lane * 2;
            const bool has = e < n * 64;
            const int col = s0 * 64 + (has ? e : 0);
            const unsigned nw = *reinterpret_cast<const unsigned*>(
                pointer(l, k == DS_QKV ? 8 : 9) + col * 2);
            const unsigned nb = *reinterpret_cast<const unsigned*>(
                pointer(l, k == DS_QKV ? 10 : 11) + col * 2);
            const unsigned* from =
                (k == DS_QKV ? at(l - 1, DS_INT(down)) : at(l, DS_INT(o))) +
                col;
            unsigned long v[DS_ROWS];
            bool ok;
            int polls = 0;
            if (!raw && n > 0 && M > 2)
                until(from - col + (M - 1) * H + s0 * 64 + n * 64 - 1);
            do {
                ok = true;
#pragma unroll
                for (int row = 0; row < DS_ROWS; ++row)
                    if (row < M) {
                        if (raw) {             // two of bf16
                            const unsigned x =
                                reinterpret_cast<const unsigned*>(
                                    DS_PTR(x))[(row * H + col) / 2];
                            v[row] = (unsigned long)(x & 0xffff0000u) << 32 |
                                     x << 16;
                        } else {
                            v[row] = ds_load(from + row * H);
                        }
                    }
#pragma unroll
                for (int row = 0; row < DS_ROWS; ++row)
                    if (row < M) ok = ok && ds_there(v[row]);
            } while (!raw && again(ok, polls));
#pragma unroll
            for (int row = 0; row < DS_ROWS; ++row)
                if (row < M) {
                    const float a0 = ds_low(v[row]), a1 = ds_high(v[row]);
                    const float sum = ds_wave_sum(has ? a0 + a1 : 0.f);
                    const float sq =
                        ds_wave_sum(has ? a0 * a0 + a1 * a1 : 0.f);
                    if (lane == 0) {
                        ml[row][wid][0] = sum;
                        ml[row][wid][1] = sq;
                    }
                }
            ds_barrier();                      // (N)
#pragma unroll
            for (int row = 0; row < DS_ROWS; ++row)
                if (row < M) {
                    float sum = 0.f, sq = 0.f;
#pragma unroll
                    for (int w = 0; w < DS_WAVES; ++w) {
                        sum += ml[row][w][0];
                        sq += ml[row][w][1];
                    }
                    const float mean = sum / (float)H;
                    const float dev =
                        rsqrtf(sq / (float)H - mean * mean + told_s.eps);
                    const float y0 = (ds_low(v[row]) - mean) * dev *
                                         bf2f((unsigned short)nw) +
                                     bf2f((unsigned short)nb);
                    const float y1 = (ds_high(v[row]) - mean) * dev *
                                         bf2f((unsigned short)(nw >> 16)) +
                                     bf2f((unsigned short)(nb >> 16));
                    if (has)
                        *reinterpret_cast<unsigned*>(xw + row * xstride +
                                                     e * 2) = ds_pack(y0, y1);
                }
        } else if (n > 0) {
            // 8 bytes a lane, `per` loads a row; a row's last lanes may read
            // its end twice
            const int per = (n + 3) / 4, loads = M * per;
            const char* x =
                (raw ? reinterpret_cast<const char*>(DS_PTR(x))
                     : reinterpret_cast<const char*>(
                           k == DS_QKV  ? at(l - 1, DS_INT(down))
                           : k == DS_O  ? at(l, DS_INT(att))
                           : k == DS_UP ? at(l, DS_INT(o))
                                        : at(l, DS_INT(up)))) + s0 * 128;
            const char* nwp = raw ? pointer(l, 8) + s0 * 128 : nullptr;
            const int last = n * 128 - 8;
            int i = 0;
            unsigned out = 0, in = 0;          // of a load's part of a row
            if (!raw && M * n > DS_FEW)
                until(reinterpret_cast<const unsigned*>(
                    x + (long)(M - 1) * K * 2 + n * 128 - 4));
            constexpr int B = 10;
            for (int l0 = 0; l0 < loads; l0 += B) {
                unsigned long v[B], w[B];
                unsigned off[B], to[B];
#pragma unroll
                for (int u = 0; u < B; ++u) {
                    const unsigned lane8 = min(lane * 8, last - i * 512);
                    off[u] = out + lane8;
                    to[u] = in + lane8;
                    if (raw && l0 + u < loads)
                        w[u] = *reinterpret_cast<const unsigned long*>(
                            nwp + i * 512 + lane8);
                    const bool over = ++i == per;
                    out += over ? K * 2 - (per - 1) * 512 : 512;
                    in += over ? xstride - (per - 1) * 512 : 512;
                    i = over ? 0 : i;
                }
                bool ok;
                int polls = 0;
                do {
                    ok = true;
#pragma unroll
                    for (int u = 0; u < B; ++u)
                        if (l0 + u < loads) v[u] = ds_load(x + off[u]);
#pragma unroll
                    for (int u = 0; u < B; ++u)
                        if (l0 + u < loads) ok = ok && ds_there(v[u]);
                } while (!raw && again(ok, polls));
#pragma unroll
                for (int u = 0; u < B; ++u) {
                    if (l0 + u >= loads) continue;
                    if (raw) {                 // times the norm's weight
                        unsigned long y = 0;
#pragma unroll
                        for (int e = 0; e < 64; e += 16)
                            y |= (unsigned long)f2bf(
                                     bf2f((unsigned short)(v[u] >> e)) *
                                     bf2f((unsigned short)(w[u] >> e)))
                                 << e;
                        v[u] = y;
                    }
                    *reinterpret_cast<unsigned long*>(xw + to[u]) = v[u];
                }
            }
        }
        WAVE_LDS_SYNC();
        if (k == DS_O) ds_wait<0>();           // (see combine)
    };

    // ---- products
    f32x4 acc{0.f, 0.f, 0.f, 0.f};
    int buf = 0;
    unsigned slot = wid * DS_RING * 1024 + lane * 16;    // to be read
    const unsigned slot_end = (wid + 1) * DS_RING * 1024;
    // rows of w 4 (lg & 1) .. + 3, input row lj; places of K apart
    const bool keeps = lj < M && (li >> 3) == (lg >> 1);
    // (told by a wave that the others do not wait for)
    auto got_on = [&]() __attribute__((always_inline)) {
        if (tid == 0)
            __hip_atomic_fetch_add(told_s.state, 1u, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
    };
    // number c's octets of product k, whose first steps are on their way
    auto product = [&](int k, int c) __attribute__((always_inline)) {
        const int n = planned(k, 1) & 0xffff;
        const char* x0 = xw + xrow * xstride + lk * 2;
        const int some = count(k, c);
        // Nothing is under way but the ring, which came before the rows did: the
        // compiler is told, or waits at every step for loads of its own.
        if (some) __builtin_amdgcn_s_waitcnt(0x0f70);        // vmcnt(0)
        for (int o = some; o > 0; --o) {
            const char* xp = x0;
            int i = 0;
            for (; i + DS_BATCH <= n; i += DS_BATCH, xp += 128 * DS_BATCH) {
                ds_wait<DS_RING - DS_BATCH>();
                bf16x8 w[DS_BATCH], x[DS_BATCH];
#pragma unroll
                for (int u = 0; u < DS_BATCH; ++u) {
                    w[u] = *reinterpret_cast<const bf16x8*>(smem + slot);
                    x[u] = *reinterpret_cast<const bf16x8*>(xp + u * 128);
                    slot += 1024;
                    if (slot >= slot_end) slot -= DS_RING * 1024;
                }
                // (read before the slots are asked for again)
                __builtin_amdgcn_s_waitcnt(0xc07f);
                if (gleft > DS_BATCH) {        // within an octet
#pragma unroll
                    for (int u = 0; u < DS_BATCH; ++u) {
                        ds_ask(gp, goff, ring + gslot, streamed);
                        gp += 128;
                        gslot += 1024;
                        if (gslot == DS_RING * 1024) gslot = 0;
                    }
                    gleft -= DS_BATCH;
                } else {
#pragma unroll 1
                    for (int u = 0; u < DS_BATCH; ++u) ask();
                }
#pragma unroll
                for (int u = 0; u < DS_BATCH; ++u)
                    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                        w[u], x[u], acc, 0, 0, 0);
            }
#pragma unroll 1
            for (; i < n; ++i, xp += 128) {
                ds_wait<DS_RING - 1>();
                const bf16x8 w = *reinterpret_cast<const bf16x8*>(smem + slot);
                const bf16x8 x = *reinterpret_cast<const bf16x8*>(xp);
                // (read before the slot is asked for again)
                __builtin_amdgcn_s_waitcnt(0xc07f);
                ask();
                acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w, x, acc, 0, 0,
                                                              0);
                slot += 1024;
                if (slot >= slot_end) slot -= DS_RING * 1024;
            }
            if (keeps)
                *reinterpret_cast<f32x4*>(
                    &part[buf][wid][li >> 3][lj][(lg & 1) * 4]) = acc;
            ds_barrier();
            if (__builtin_expect(gnc > 1, 0)) got_on();
            buf ^= 1;
            acc = f32x4{0.f, 0.f, 0.f, 0.f};
        }
    };

    // ---- attention of sequence and key head, one split: a wave takes tiles of
    // 32 keys on its own. Scores are S^T = K Q^T on 16x16x32 tiles (a column is
    // a query head), so that the weights are, as they stand, the right operand
    // of O^T = V^T P^T, whose keys follow the score tile's order through the
    // transposing LDS read.
    constexpr int KS = HD / 32, DT = HD / 16;
    constexpr int PC = 2 / sizeof(KVT);        // pieces of 8 of a load of V
    constexpr int CPR = HD / 8 / PC, RPI = 64 / CPR, NL = DS_KEYS / RPI;
    constexpr int RB = HD * 2, TILE = DS_KEYS * RB;
    const bool whole = DS_INT(bs) % DS_KEYS == 0;    // a tile is in one page
    auto page_of = [&](int m, int i) __attribute__((always_inline)) {
        if (paged) return pages[m * DS_INT(W) + i];
        return ds_global(DS_PTR(table) + (long)m * DS_INT(W) + i);
    };
    // (of the first item, the only one where there are no more than workgroups:
    // the same in every layer)
    int i_at = -1, i_m = 0, i_kvh = 0, i_z = 0;
    unsigned i_mine = 0;
    long i_base = 0;
    auto attention = [&](int l, int it) __attribute__((always_inline)) {
        const int bs = DS_INT(bs);
        if (__builtin_expect(it != i_at, 0)) {
            i_at = it;
            i_z = it % DS_INT(Z);
            i_m = it / DS_INT(Z) / DS_INT(nkv);
            i_kvh = it / DS_INT(Z) % DS_INT(nkv);
            const Span s = ds_span(ds_same(len_s[i_m]), DS_INT(Z), i_z);
            const int kb = s.from + wid * DS_KEYS;
            if (!s.none(i_z)) {
                // Which of its keys the step's rows store, -1: none; all waves
                // find the same. (Slots that several rows store to are this
                // row's, if it is one of them.)
                int own = -1;
                for (int p0 = s.from / bs; p0 * bs < s.to; p0 += 64) {
                    const int p = p0 + lane;
                    const int page = p * bs < s.to ? page_of(i_m, p) : -1;
                    for (int n = 0; n < M; ++n) {
                        const int slot = ds_same(slot_s[n]);
                        const int key = p * bs + slot % bs;
                        const unsigned long hit = __ballot(
                            slot >= 0 && page == slot / bs && key >= s.from &&
                            key < s.to);
                        if (hit && lane == n)
                            own = (p0 + __builtin_ctzl(hit)) * bs + slot % bs;
                    }
                }
                if (lane != i_m && own == __builtin_amdgcn_readlane(own, i_m))
                    own = -1;
                if (lane < M) own_s[lane] = own;
                // (of these, the ones in this wave's tiles)
                i_mine = __ballot(own >= kb &&
                                  (unsigned)(own - kb) % DS_STEP < DS_KEYS);
                if (whole && kb < s.to)        // the first tile's
                    i_base = (((long)ds_same(page_of(i_m, kb / bs)) *
                                   DS_INT(nkv) + i_kvh) * bs + kb % bs) * HD;
            }
        }
        const int m = i_m, kvh = i_kvh;
        const Span s = ds_span(ds_same(len_s[m]), DS_INT(Z), i_z);
        if (s.none(i_z)) return;
        const int G = DS_INT(G), nq = DS_INT(nq), nkv = DS_INT(nkv);
        const char* kc = pointer(l, 12);
        const char* vc = pointer(l, 13);
        auto v_swz = [](int row) {
            return 2 * (HD == 128 ? row & 7 : (row >> 1) & 3);
        };
        const bool round_q = sizeof(KVT) == 1;
        const float scale_log2 = round_q ? DS_LOG2E : told_s.scale * DS_LOG2E;
        char* const vt = area + wid * TILE;
        const int ld_row = lane / CPR, ld_c = lane % CPR * PC;

        typedef std::conditional_t<sizeof(KVT) == 2, ds_raw, uint2v> kraw;
        kraw rk[2][KS];
        ds_raw rv[NL];
        auto page_row = [&](int kb) __attribute__((always_inline)) {
            const int page = ds_same(page_of(m, kb / bs));
            return (((long)page * nkv + kvh) * bs + kb % bs) * HD;
        };
        auto row_of = [&](int key) __attribute__((always_inline)) {
            const int page = page_of(m, key / bs);
            return (((long)page * nkv + kvh) * bs + key % bs) * HD;
        };
        // NT: past L2; IN: the tile is in one page, at base (keys behind the last
        // one are not asked for: their scores are)
        auto keys_of = [&](int kb, long base, auto NT, auto IN)
                           __attribute__((always_inline)) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const char* from = kc + base * (long)sizeof(KVT);
                int at = (h * 16 + li) * HD;
                if constexpr (!IN()) {
                    from = kc + row_of(min(kb + h * 16 + li, s.to - 1)) *
                                    (long)sizeof(KVT);
                    at = 0;
                }
#pragma unroll
                for (int ks = 0; ks < KS; ++ks)
                    rk[h][ks] = ds_global<NT()>(reinterpret_cast<const kraw*>(
                        from + (unsigned)((at + ks * 32 + lg * 8) *
                                          (int)sizeof(KVT))));
            }
        };
        auto values_of = [&](int kb, long base, auto NT, auto IN)
                             __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < NL; ++i) {
                const char* from = vc + base * (long)sizeof(KVT);
                int at = min(ld_row + i * RPI, s.to - 1 - kb) * HD;
                if constexpr (!IN()) {
                    from = vc + row_of(min(kb + ld_row + i * RPI, s.to - 1)) *
                                    (long)sizeof(KVT);
                    at = 0;
                }
                rv[i] = ds_global<NT()>(reinterpret_cast<const ds_raw*>(
                    from + (unsigned)((at + ld_c * 8) * (int)sizeof(KVT))));
            }
        };
        const std::true_type yes;
        const std::false_type no;
        auto keys = [&](int kb, long base) __attribute__((always_inline)) {
            if (!whole) keys_of(kb, base, no, no);
            else if (streamed) keys_of(kb, base, yes, yes);
            else keys_of(kb, base, no, yes);
        };
        auto values = [&](int kb, long base) __attribute__((always_inline)) {
            if (!whole) values_of(kb, base, no, no);
            else if (streamed) values_of(kb, base, yes, yes);
            else values_of(kb, base, no, yes);
        };
        int kb = s.from + wid * DS_KEYS;
        if (kb < s.to) {
            keys(kb, i_base);
            values(kb, i_base);
        }

        // queries
        bf16x8 bq[KS];
        const unsigned mine = i_mine;          // rows
        int own = -1;                          // their keys
        if (kb < s.to) {                       // (others have nothing to ask)
            const unsigned* qw =
                at(l, 0) + (((m * nq + kvh * G + min(li, G - 1)) << hd_log2) +
                            lg * 8) / 2;
            // (the step's own key and value beside them, for the wave that has
            // their tile; of more rows than one after that)
            const int of = lane / (HD / 4) % 2, e2 = lane % (HD / 4) * 2;
            auto fresh_of = [&](int n) __attribute__((always_inline)) {
                return at(l, DS_INT(new_kv)) +
                       ((((n * 2 + of) * nkv + kvh) << hd_log2) / 2 + e2);
            };
            const int first = mine ? __builtin_ctz(mine) : 0;
            const unsigned* from = fresh_of(first);
            unsigned long q[KS][2], fresh_word = 0;
            bool ok;
            int polls = 0;
            do {
                ok = true;
                if (mine) {
                    fresh_word = ds_load(from);
                    ok = ds_there(fresh_word);
                }
#pragma unroll
                for (int ks = 0; ks < KS; ++ks)
#pragma unroll
                    for (int e = 0; e < 2; ++e) {
                        q[ks][e] = ds_load(qw + ks * 16 + e * 2);
                        ok = ok && ds_there(q[ks][e]);
                    }
            } while (again(ok, polls));
            if (mine) {
                if (lane < M) own = own_s[lane];
                *reinterpret_cast<unsigned long*>(fresh_at(first, of) + e2) =
                    fresh_word;
#pragma unroll 1
                for (unsigned b = mine & (mine - 1); __builtin_expect(b, 0);
                     b &= b - 1) {
                    const int n = __builtin_ctz(b);
                    polls = 0;
                    do fresh_word = ds_load(fresh_of(n));
                    while (again(ds_there(fresh_word), polls));
                    *reinterpret_cast<unsigned long*>(fresh_at(n, of) + e2) =
                        fresh_word;
                }
                WAVE_LDS_SYNC();
            }
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
                bq[ks] = __builtin_bit_cast(
                    bf16x8, ds_raw{(unsigned)q[ks][0],
                                   (unsigned)(q[ks][0] >> 32),
                                   (unsigned)q[ks][1],
                                   (unsigned)(q[ks][1] >> 32)});
                if (round_q) {                 // scaled, rounded like the pages
                    float f[8];
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        f[e] = (float)(__bf16)((float)bq[ks][e] * told_s.scale);
                    uint2v w;
#pragma unroll
                    for (int i = 0; i < 2; ++i)
                        w[i] = f2fp8x2(f[i * 4], f[i * 4 + 1]) |
                               (unsigned)f2fp8x2(f[i * 4 + 2], f[i * 4 + 3])
                                   << 16;
                    bq[ks] = ds_widen(w);
                }
            }
        }

        const int v_key = lg * 4 + (li >> 2);
        const int v_from = v_key * RB + (lane & 1) * 8 +
                           (((lane & 3) >> 1 ^ v_swz(v_key)) << 4);
        const int v_to = ld_row * RB + ((ld_c ^ v_swz(ld_row)) << 4);
        f32x4 o[DT];
        float mx = -1e30f, sum = 0.f;
#pragma unroll
        for (int d = 0; d < DT; ++d) o[d] = f32x4{0.f, 0.f, 0.f, 0.f};
        for (; kb < s.to; kb += DS_STEP) {
            const bool more = kb + DS_STEP < s.to;
            const long base = more && whole ? page_row(kb + DS_STEP) : 0;
            // rows whose keys are in this tile
            unsigned patch = 0;
            if (mine) patch = __ballot(own >= kb && own < kb + DS_KEYS);
            // values to LDS, 16-byte pieces xor-ed by the key
            const int to = ds_own(v_to), from = ds_own(v_from);
#pragma unroll
            for (int i = 0; i < NL; ++i) {
#pragma unroll
                for (int p = 0; p < PC; ++p) {
                    ds_raw x = rv[i];
                    if constexpr (sizeof(KVT) == 1)
                        x = __builtin_bit_cast(
                            ds_raw, ds_widen(uint2v{rv[i][p * 2],
                                                    rv[i][p * 2 + 1]}));
                    // (of keys RPI apart the same, or every other one's)
                    const int other = HD == 128 && RPI == 4 ? i % 2 * 128 : 0;
                    *reinterpret_cast<ds_raw*>(vt + (to ^ other) +
                                               i * RPI * RB + p * 16) = x;
                }
            }
            if (more) values(kb + DS_STEP, base);
            // (the last key's value stands in the tile's rows behind it, too)
            const unsigned* fresh_k[2] = {nullptr, nullptr};
#pragma unroll 1
            for (unsigned b = patch; b; b &= b - 1) {
                const int n = __builtin_ctz(b);
                const int key = __builtin_amdgcn_readlane(own, n);
                const int row = key - kb, c = lane % (HD / 8);
                const int end = key == s.to - 1 ? DS_KEYS : row + 1;
                const ds_raw x = *reinterpret_cast<const ds_raw*>(
                    fresh_at(n, 1) + c * 4);
                for (int r = row + lane / (HD / 8); r < end; r += 512 / HD)
                    *reinterpret_cast<ds_raw*>(
                        vt + r * RB + ((c ^ v_swz(r)) << 4)) = x;
#pragma unroll
                for (int h = 0; h < 2; ++h)
                    if (row == h * 16 + li) fresh_k[h] = fresh_at(n, 0);
            }
            f32x4 sc[2];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                sc[h] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int ks = 0; ks < KS; ++ks) {
                    bf16x8 ak;
                    if constexpr (sizeof(KVT) == 1) ak = ds_widen(rk[h][ks]);
                    else ak = __builtin_bit_cast(bf16x8, rk[h][ks]);
                    if (patch && fresh_k[h])
                        ak = *reinterpret_cast<const bf16x8*>(
                            fresh_k[h] + ks * 16 + lg * 4);
                    sc[h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                        ak, bq[ks], sc[h], 0, 0, 0);
                }
            }
            if (more) keys(kb + DS_STEP, base);
            if (kb + DS_KEYS > s.to) {
#pragma unroll
                for (int h = 0; h < 2; ++h)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        if (kb + h * 16 + lg * 4 + r >= s.to)
                            sc[h][r] = -INFINITY;
            }
            // online softmax, in powers of two
            float top = sc[0][0];
#pragma unroll
            for (int r = 0; r < 4; ++r)
                top = fmaxf(fmaxf(top, sc[0][r]), sc[1][r]);
            top = rows_max(top) * scale_log2;
            const float next = fmaxf(mx, top);
            if (__any(next > mx)) {
                const float alpha = __builtin_amdgcn_exp2f(mx - next);
                mx = next;
                sum *= alpha;
#pragma unroll
                for (int d = 0; d < DT; ++d)
#pragma unroll
                    for (int r = 0; r < 4; ++r) o[d][r] *= alpha;
            }
            bf16x8 p;
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    p[h * 4 + r] = (__bf16)__builtin_amdgcn_exp2f(
                        fmaf(sc[h][r], scale_log2, -mx));
            // the sum that divides is of the weights as they are multiplied:
            // what rounding does to both cancels
            sum = add_bf16x8(p, sum);
            WAVE_LDS_SYNC();
#pragma unroll
            for (int d = 0; d < DT; ++d) {
                const char* va = vt + (from ^ d * 32);
                const short4v a0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                    (lds_short4v*)va);
                const short4v a1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                    (lds_short4v*)(va + 16 * RB));
                o[d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                    __builtin_bit_cast(
                        bf16x8, __builtin_shufflevector(a0, a1, 0, 1, 2, 3, 4,
                                                        5, 6, 7)),
                    p, o[d], 0, 0, 0);
            }
            WAVE_LDS_SYNC();
        }
        // ---- the waves' sums meet in LDS, of those that had keys
        const int had = min((s.to - s.from + DS_KEYS - 1) / DS_KEYS, DS_WAVES);
        sum = rows_sum(sum);
        if (wid < had)
#pragma unroll
            for (int d = 0; d < DT; ++d)
                *reinterpret_cast<f32x4*>(vt + (d * 64 + lane) * 16) = o[d];
        if (lg == 0) {
            ml[li][wid][0] = mx;
            ml[li][wid][1] = sum;
        }
        // where this wave's columns of the result go
        const bool split = s.splits() > 1;
        unsigned* const to =
            split ? DS_PTR(parts) + (((long)it * G + li) * DT + wid) * DS_PART +
                        lg * 4
                  : at(l, DS_INT(att)) + (((m * nq + kvh * G + li) << hd_log2) +
                                          wid * 16 + lg * 4) / 2;
        ds_barrier();                          // (A)
        if (wid < DT) {
            const bool put = li < G && !gone;
            float wm[DS_WAVES], ws[DS_WAVES], top = -1e30f, all = 0.f;
            f32x4 x[DS_WAVES], y{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int w = 0; w < DS_WAVES; ++w) {
                wm[w] = ml[li][w][0];
                ws[w] = ml[li][w][1];
                x[w] = y;
                if (w < had)
                    x[w] = *reinterpret_cast<const f32x4*>(
                        area + w * TILE + (wid * 64 + lane) * 16);
            }
#pragma unroll
            for (int w = 0; w < DS_WAVES; ++w) top = fmaxf(top, wm[w]);
#pragma unroll
            for (int w = 0; w < DS_WAVES; ++w) {
                wm[w] = __builtin_amdgcn_exp2f(wm[w] - top);
                all = fmaf(wm[w], ws[w], all);
#pragma unroll
                for (int r = 0; r < 4; ++r) y[r] = fmaf(x[w][r], wm[w], y[r]);
            }
            if (put) {
                if (split) {
                    ds_store(to, y[0], y[1]);
                    ds_store(to + 2, y[2], y[3]);
                    if (lg == 0) ds_store(to + 16, top, all);
                } else {
                    // (no keys: zeros; a NaN stays one)
                    const float by = all == 0.f ? 0.f : 1.f / all;
                    ds_store(to, ds_pack(y[0] * by, y[1] * by),
                             ds_pack(y[2] * by, y[3] * by));
                }
            }
        }
        ds_barrier();                          // (B): the area is free again
        if (__builtin_expect(gnc > 1, 0)) got_on();
    };
    // A query head's splits, added up by a wave for 16 of its columns: two a lane,
    // eight lanes a split. Their words are left as they were found, for the next
    // layer, whose splits come after this sum.
    auto combine = [&](int l, int it) __attribute__((always_inline)) {
        const int nq = DS_INT(nq), G = DS_INT(G);
        const int m = it / nq, head = it % nq;
        const int nz = ds_span(ds_same(len_s[m]), DS_INT(Z), 0).splits();
        if (nz <= 1 || wid >= DT) return;      // (0: no keys, attention's zeros)
        constexpr int U = DS_SPLITS / 8;
        const int lane = ds_own(tid & 63);
        const int z0 = lane >> 3, c = lane & 7;
        const int step = G * DT * DS_PART;     // from a split to the next
        unsigned* const from =
            DS_PTR(parts) +
            (((long)(m * DS_INT(nkv) + head / G) * DS_INT(Z) * G + head % G) *
                 DT + wid) * DS_PART;
        unsigned* const to =
            at(l, DS_INT(att)) + ((it << hd_log2) + wid * 16 + c * 2) / 2;
        unsigned long v[U], e[U];
        bool ok;
        int polls = 0;
        until(from + (long)(nz - 1) * step + 17);
        do {
            ok = true;
#pragma unroll
            for (int u = 0; u < U; ++u) {
                v[u] = e[u] = 0;
                if (z0 + u * 8 >= nz) continue;
                const unsigned* at = from + (long)(z0 + u * 8) * step;
                v[u] = ds_load(at + c * 2);
                e[u] = ds_load(at + 16);
            }
#pragma unroll
            for (int u = 0; u < U; ++u)
                ok = ok && ds_there(v[u]) && ds_there(e[u]);
        } while (again(ok, polls));
        if (__builtin_expect(!__all(ok), 0)) return;
        auto empty = [&]() __attribute__((always_inline)) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                if (z0 + u * 8 >= nz) continue;
                unsigned long* at = reinterpret_cast<unsigned long*>(
                    from + (long)(z0 + u * 8) * step);
                __hip_atomic_store(at + c, ~0ul, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
                if (c == 0)
                    __hip_atomic_store(at + 8, ~0ul, __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
            }
        };
        float top = -1e30f, all = 0.f, y0 = 0.f, y1 = 0.f;
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (z0 + u * 8 < nz) top = fmaxf(top, ds_low(e[u]));
        top = rows_max(fmaxf(top, ds_dpp<0x128>(top)));      // (other 8 of 16)
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (z0 + u * 8 < nz) {
                const float f = __builtin_amdgcn_exp2f(ds_low(e[u]) - top);
                all = fmaf(f, ds_high(e[u]), all);
                y0 = fmaf(f, ds_low(v[u]), y0);
                y1 = fmaf(f, ds_high(v[u]), y1);
            }
        all = rows_sum(all + ds_dpp<0x128>(all));
        y0 = rows_sum(y0 + ds_dpp<0x128>(y0));
        y1 = rows_sum(y1 + ds_dpp<0x128>(y1));
        const float by = all == 0.f ? 0.f : 1.f / all;
        // The words are empty before any word that this workgroup leaves after,
        // on which the next layer's splits depend: input() waits for that, and
        // where no octet of the output follows, the result itself does.
        const bool last = it % DS_WGS >= octets(DS_O);
        if (last) {
            empty();
            ds_wait<0>();
        }
        if (z0 == 0) ds_store(to, ds_pack(y0 * by, y1 * by));
        if (!last) empty();
    };

    bool primed = false;
    for (int l = lo, k = 0, other = -1; l < hi;) {
        if (!primed) {
            seek();
#pragma unroll 1
            for (int u = 0; u < DS_RING; ++u) ask();
            primed = true;
        }
        int some = 0;
        if (other >= 0) some = count(k, other);
        else if (gnc == 1) some = count(k, number);
        else
            for (int i = 0; i < gnc; ++i) some += count(k, ds_same(cols[i]));
        if (some) input(l, k);
        for (int i = other >= 0 ? gnc - 1 : 0; i < gnc; ++i)
            product(k, i ? ds_same(cols[i]) : number);
        if (l == lo && k == DS_QKV) {
            bool on = false;
            if (other < 0) {
                if (!some) ds_barrier();       // (1)
                const int b = ds_same(begin);
                if (b == DS_LEAVE) break;
                on = b == DS_GO_ON;
            } else {
                ds_barrier();                  // (3)
            }
            if (!on) {
                ds_barrier();                  // (2)
                other = ds_same(gate);
                gnc = ds_same(ncols);
                // what is under way is of the next product: asked for again
                ds_wait<0>();
                gslot = 0;
                slot = wid * DS_RING * 1024 + lane * 16;
                gl = lo;
                told_l = layers[lane & 7];
                gk = other >= 0 ? DS_QKV : DS_O;
                gi = other >= 0 ? gnc - 2 : -1;
                primed = false;
                if (other >= 0) continue;
            }
        }
        if (k == DS_QKV) {
            for (int i = 0; i < gnc; ++i)
                for (int it = i ? ds_same(cols[i]) : number;
                     it < DS_INT(items); it += DS_WGS)
                    attention(l, it);
            if (DS_INT(Z) > 1)
                for (int i = 0; i < gnc; ++i)
                    for (int it = i ? ds_same(cols[i]) : number;
                         it < M * DS_INT(nq); it += DS_WGS)
                        combine(l, it);
        }
        if (++k == 4) k = 0, ++l;
    }
    ds_wait<0>();                              // nothing lands in LDS later
    if (gone && lane == 0 && told_s.status)
        __hip_atomic_store(told_s.status, 1, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_SYSTEM);
}

// LDS of the rings; of the rows of `K` columns or the attention's tiles; of the
// rows' rotation, new keys and values and, where there are few, their pages (up
// to 2 KB)
static long ds_area(int M, int K, int hd) {
    const long rows = (long)M * (K * 2 + DS_WAVES * 16);
    const long tiles = (long)DS_WAVES * DS_KEYS * hd * 2;
    return rows > tiles ? rows : tiles;
}
static long ds_lds(int M, int K, int hd) {
    return DS_WAVES * DS_RING * 1024 + ds_area(M, K, hd) + M * hd * 8 + 2048;
}
// ... beside what the kernel has without being asked
constexpr long DS_LDS = 160 * 1024 - 17 * 1024;

// Most rows of a step of a stack whose deepest product is K deep.
extern "C" int decode_stack_rows(int K, int hd) {
    int M = 0;
    while (M < DS_ROWS && ds_lds(M + 1, K, hd) <= DS_LDS) ++M;
    return M;
}

// Splits of the longest contexts: up to a workgroup a CU (a second item for some
// costs all a round: 6 rows of 12 heads 40 us a layer in 288 items, 35 in 216).
extern "C" int decode_stack_splits(long pairs, long keys) {
    if (keys <= DS_ALONE) return 1;
    long Z = DS_WGS / pairs;
    return Z > DS_SPLITS ? DS_SPLITS : Z < 1 ? 1 : (int)Z;
}

// The fields of `args` as decode_stack.h says, every word that passes, the
// claims and the state DS_EMPTY, all rows 16-byte aligned. Nonzero for sizes that
// the kernel does not take.
extern "C" int launch_decode_stack(const StackArgs* args, int hd, int fp8,
                                   int layer_norm, int wgs,
                                   hipStream_t stream) {
    StackArgs a = *args;
    const int layers = a.hi - a.lo;
    if (layers < 1 || layers > DS_LAYERS || a.M < 1) return 1;
    if (wgs < 1 || wgs > 2 * DS_WGS || (hd != 64 && hd != 128)) return 1;
    if (a.nkv < 1 || a.nq != a.G * a.nkv || a.G > 16 || a.Z < 1) return 1;
    if (a.items != a.M * a.nkv * a.Z) return 1;
    if (a.Z > DS_SPLITS || !(a.scale > 0.f) || a.patience < 31) return 1;
    int deepest = 0;
    for (int k = 0; k < 4; ++k) {
        const long K = a.K[k];
        if (K < 64 || K % 64 || a.octets[k] < 1) return 1;
        if (((long)a.half[k] + 4) * K * 2 >= 1L << 32) return 1;
        if (K > deepest) deepest = (int)K;
    }
    if (layer_norm && a.K[DS_QKV] > DS_LAYER_NORM) return 1;
    if (a.M > decode_stack_rows(deepest, hd)) return 1;
    const dim3 grid(wgs), block((DS_WAVES + 1) * 64);
    const int lds = (int)ds_lds(a.M, deepest, hd);
    a.turns = (int)ds_area(a.M, deepest, hd);
    a.pages = a.turns + a.M * hd * 8;
    a.area = a.pages + ((long)a.M * a.W * 4 <= 2048 ? 1 : 0);
#define DS_ONE(L, HD, T)                                                      \
    hipLaunchKernelGGL((decode_stack_kernel<L, HD, T>), grid, block, lds,     \
                       stream, a)
#define DS_GO(HD)                                                             \
    do {                                                                      \
        if (layer_norm && fp8) DS_ONE(true, HD, unsigned char);               \
        else if (layer_norm) DS_ONE(true, HD, unsigned short);                \
        else if (fp8) DS_ONE(false, HD, unsigned char);                       \
        else DS_ONE(false, HD, unsigned short);                               \
    } while (0)
    if (hd == 64) DS_GO(64);
    else DS_GO(128);
#undef DS_GO
#undef DS_ONE
    return 0;
}
