// Memory-bound fused kernels: RMSNorm, fused add+RMSNorm, RoPE, SwiGLU,
// paged-KV store. All bf16 I/O vectorized as short8 (16 B/lane — guide G13:
// hipcc does not auto-vectorize bf16 loads; scalar bf16 is ~2x slower).
//
// These replace what the reference ran inside transformers.generate()
// (bee2bee/hf.py:84-108) — each is one HBM round-trip, fused.
#include "common.h"

// ---------------------------------------------------------------- rmsnorm
// One workgroup per row. Row cached in LDS as fp32 between the two passes
// so the input is read from HBM exactly once.
template <bool FUSED_ADD>
__global__ void rmsnorm_kernel(
    const unsigned short* __restrict__ x,      // [T, H]
    const unsigned short* __restrict__ resid,  // [T, H] or null
    const unsigned short* __restrict__ w,      // [H]
    unsigned short* __restrict__ y,            // [T, H]
    unsigned short* __restrict__ resid_out,    // [T, H] or null
    int H, float eps) {
    extern __shared__ __attribute__((aligned(16))) char smem_raw[];
    float* row = reinterpret_cast<float*>(smem_raw);       // [H]
    __shared__ float red[8];

    const long t = blockIdx.x;
    const unsigned short* xr = x + t * (long)H;
    const unsigned short* rr = FUSED_ADD ? resid + t * (long)H : nullptr;
    unsigned short* ro = FUSED_ADD ? resid_out + t * (long)H : nullptr;

    float sumsq = 0.f;
    for (int i = threadIdx.x * 8; i < H; i += blockDim.x * 8) {
        float v[8];
        load_bf16x8(xr + i, v);
        if (FUSED_ADD) {
            float r[8];
            load_bf16x8(rr + i, r);
#pragma unroll
            for (int j = 0; j < 8; ++j) v[j] += r[j];
            store_bf16x8(ro + i, v);
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            row[i + j] = v[j];
            sumsq += v[j] * v[j];
        }
    }
    // block reduction: wave-level then cross-wave through LDS
    sumsq = wave_sum(sumsq);
    const int wid = threadIdx.x / WAVE;
    const int lane = threadIdx.x % WAVE;
    if (lane == 0) red[wid] = sumsq;
    __syncthreads();
    const int nw = blockDim.x / WAVE;
    float total = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) total += (i < nw) ? red[i] : 0.f;
    const float inv = rsqrtf(total / (float)H + eps);

    unsigned short* yr = y + t * (long)H;
    for (int i = threadIdx.x * 8; i < H; i += blockDim.x * 8) {
        float wv[8], o[8];
        load_bf16x8(w + i, wv);
#pragma unroll
        for (int j = 0; j < 8; ++j) o[j] = row[i + j] * inv * wv[j];
        store_bf16x8(yr + i, o);
    }
}

// -------------------------------------------------------------- layernorm
// GPT-2-family LayerNorm (mean/variance, weight + bias), same one-HBM-read
// structure as rmsnorm_kernel: row cached fp32 in LDS between passes.
template <bool FUSED_ADD>
__global__ void layernorm_kernel(
    const unsigned short* __restrict__ x,      // [T, H]
    const unsigned short* __restrict__ resid,  // [T, H] or null
    const unsigned short* __restrict__ w,      // [H]
    const unsigned short* __restrict__ b,      // [H]
    unsigned short* __restrict__ y,            // [T, H]
    unsigned short* __restrict__ resid_out,    // [T, H] or null
    int H, float eps) {
    extern __shared__ __attribute__((aligned(16))) char smem_raw[];
    float* row = reinterpret_cast<float*>(smem_raw);  // [H]
    __shared__ float red[8], red2[8];

    const long t = blockIdx.x;
    const unsigned short* xr = x + t * (long)H;
    const unsigned short* rr = FUSED_ADD ? resid + t * (long)H : nullptr;
    unsigned short* ro = FUSED_ADD ? resid_out + t * (long)H : nullptr;

    float lsum = 0.f, lsumsq = 0.f;
    for (int i = threadIdx.x * 8; i < H; i += blockDim.x * 8) {
        float v[8];
        load_bf16x8(xr + i, v);
        if (FUSED_ADD) {
            float r[8];
            load_bf16x8(rr + i, r);
#pragma unroll
            for (int j = 0; j < 8; ++j) v[j] += r[j];
            store_bf16x8(ro + i, v);
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            row[i + j] = v[j];
            lsum += v[j];
            lsumsq += v[j] * v[j];
        }
    }
    lsum = wave_sum(lsum);
    lsumsq = wave_sum(lsumsq);
    const int wid = threadIdx.x / WAVE;
    const int lane = threadIdx.x % WAVE;
    if (lane == 0) { red[wid] = lsum; red2[wid] = lsumsq; }
    __syncthreads();
    const int nw = blockDim.x / WAVE;
    float tot = 0.f, totsq = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        tot += (i < nw) ? red[i] : 0.f;
        totsq += (i < nw) ? red2[i] : 0.f;
    }
    const float mean = tot / (float)H;
    const float var = totsq / (float)H - mean * mean;
    const float inv = rsqrtf(var + eps);

    unsigned short* yr = y + t * (long)H;
    for (int i = threadIdx.x * 8; i < H; i += blockDim.x * 8) {
        float wv[8], bv[8], o[8];
        load_bf16x8(w + i, wv);
        load_bf16x8(b + i, bv);
#pragma unroll
        for (int j = 0; j < 8; ++j)
            o[j] = (row[i + j] - mean) * inv * wv[j] + bv[j];
        store_bf16x8(yr + i, o);
    }
}

// ------------------------------------------------------------------ gelu
// HF gelu_new (tanh approximation) — matches transformers GPT-2 exactly.
__global__ void gelu_kernel(
    const unsigned short* __restrict__ x,  // [N] (flattened, 8-aligned)
    unsigned short* __restrict__ y,
    long n8) {
    for (long idx = blockIdx.x * (long)blockDim.x + threadIdx.x; idx < n8;
         idx += (long)gridDim.x * blockDim.x) {
        float v[8], o[8];
        load_bf16x8(x + idx * 8, v);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const float u = v[j];
            const float c = 0.7978845608028654f * (u + 0.044715f * u * u * u);
            o[j] = 0.5f * u * (1.f + tanhf(c));
        }
        store_bf16x8(y + idx * 8, o);
    }
}

// ------------------------------------------------------------------- rope
// Llama rotate-half RoPE, in place on strided q/k views of the fused qkv
// projection. One wave per (token, head); lane owns pair (d, d+hd/2).
// cos/sin tables are host-precomputed fp32 (guide App. B: no device trig).
__global__ void rope_kernel(
    unsigned short* __restrict__ q,  // [T, nq, hd], token stride sq
    unsigned short* __restrict__ k,  // [T, nkv, hd], token stride sk
    const int* __restrict__ pos,     // [T]
    const float* __restrict__ cos_t, // [table, hd/2]
    const float* __restrict__ sin_t, int table,
    int T, int nq, int nkv, int hd, long sq, long sk) {
    const int glob_wave = (blockIdx.x * blockDim.x + threadIdx.x) / WAVE;
    const int lane = threadIdx.x % WAVE;
    const int heads = nq + nkv;
    if (glob_wave >= T * heads) return;
    const int t = glob_wave / heads;
    const int h = glob_wave % heads;
    unsigned short* base = (h < nq) ? q + (long)t * sq + (long)h * hd
                                    : k + (long)t * sk + (long)(h - nq) * hd;
    const int half = hd / 2;
    const long tab = turn_row(pos[t], table) * half;
    for (int d = lane; d < half; d += WAVE) {
        float c = cos_t[tab + d];
        float s = sin_t[tab + d];
        float x1 = bf2f(base[d]);
        float x2 = bf2f(base[d + half]);
        base[d] = f2bf(x1 * c - x2 * s);
        base[d + half] = f2bf(x2 * c + x1 * s);
    }
}

// ---------------------------------------------------------- kv_cache_store
// Scatter new K/V rows into the paged pool. One wave per (token, kv head).
__global__ void kv_store_kernel(
    const unsigned short* __restrict__ k,  // [T, nkv, hd], token stride sk
    const unsigned short* __restrict__ v,
    unsigned short* __restrict__ k_cache,  // [nb, nkv, bs, hd]
    unsigned short* __restrict__ v_cache,
    const int* __restrict__ slots,         // [T]
    int T, int nkv, int hd, int bs, long sk, long sv) {
    const int glob_wave = (blockIdx.x * blockDim.x + threadIdx.x) / WAVE;
    const int lane = threadIdx.x % WAVE;
    if (glob_wave >= T * nkv) return;
    const int t = glob_wave / nkv;
    const int h = glob_wave % nkv;
    const int slot = slots[t];
    if (slot < 0) return;            // no such position
    const int blk = slot / bs, off = slot % bs;
    const long dst = (((long)blk * nkv + h) * bs + off) * hd;
    const unsigned short* ks = k + (long)t * sk + (long)h * hd;
    const unsigned short* vs = v + (long)t * sv + (long)h * hd;
    for (int d = lane * 2; d + 1 < hd; d += WAVE * 2) {
        *reinterpret_cast<short2v*>(k_cache + dst + d) =
            *reinterpret_cast<const short2v*>(ks + d);
        *reinterpret_cast<short2v*>(v_cache + dst + d) =
            *reinterpret_cast<const short2v*>(vs + d);
    }
    if (hd % 2) { /* head dims are even for all supported models */ }
}

// fp8 (OCP e4m3) KV cache variant: quantize at store time (RNE pack), so
// the decode kernels read HALF the bytes. Scale is 1.0 (e4m3 covers +-448;
// post-RMSNorm K/V magnitudes sit well inside — opt-in, documented).
__global__ void kv_store_fp8_kernel(
    const unsigned short* __restrict__ k,  // [T, nkv, hd] bf16
    const unsigned short* __restrict__ v,
    unsigned char* __restrict__ k_cache,   // [nb, nkv, bs, hd] fp8
    unsigned char* __restrict__ v_cache,
    const int* __restrict__ slots,
    int T, int nkv, int hd, int bs, long sk, long sv) {
    const int glob_wave = (blockIdx.x * blockDim.x + threadIdx.x) / WAVE;
    const int lane = threadIdx.x % WAVE;
    if (glob_wave >= T * nkv) return;
    const int t = glob_wave / nkv;
    const int h = glob_wave % nkv;
    const int slot = slots[t];
    if (slot < 0) return;            // no such position
    const int blk = slot / bs, off = slot % bs;
    const long dst = (((long)blk * nkv + h) * bs + off) * hd;
    const unsigned short* ks = k + (long)t * sk + (long)h * hd;
    const unsigned short* vs = v + (long)t * sv + (long)h * hd;
    for (int d = lane * 2; d + 1 < hd; d += WAVE * 2) {
        const short2v kk = *reinterpret_cast<const short2v*>(ks + d);
        const short2v vv = *reinterpret_cast<const short2v*>(vs + d);
        *reinterpret_cast<unsigned short*>(k_cache + dst + d) =
            f2fp8x2(bf2f((unsigned short)kk[0]), bf2f((unsigned short)kk[1]));
        *reinterpret_cast<unsigned short*>(v_cache + dst + d) =
            f2fp8x2(bf2f((unsigned short)vv[0]), bf2f((unsigned short)vv[1]));
    }
}

// ------------------------------------------------------------- rope_store
// What stands between the q|k|v projection and attention, in one pass: the
// projection's parts summed (S > 0: fp32 [S, T, N]) or its bf16 rows taken
// (S == 0, in qkv itself), bias added, q and k rotated (pos null: not), the
// result left in qkv [T, N] and k and v scattered into the paged pool (bf16,
// or OCP fp8 bytes). A thread takes 8 coordinates of a head's first half and
// their partners in the second. Bound by its bytes at thousands of tokens (8512
// tokens of 28 + 2x4 heads of 128: 38 us with the bias; as an add, a rotation
// of 2-byte accesses and a copy it was 44 + 64 + 12), by the latency of its parts
// at tens: all of them (PARTS; 0: rows, -1: a number that is not known) are asked
// for before the first is added, by a wave a workgroup.
template <typename CT, int PARTS>
__global__ __launch_bounds__(256) void qkv_rope_store_kernel(
    const float* __restrict__ part, int S, unsigned short* __restrict__ qkv,
    const unsigned short* __restrict__ bias, const int* __restrict__ pos,
    const float* __restrict__ cos_t, const float* __restrict__ sin_t, int table,
    CT* __restrict__ k_cache, CT* __restrict__ v_cache,
    const int* __restrict__ slots, long T, int nq, int nkv, int hd, int bs) {
    const int heads = nq + 2 * nkv, half = hd / 2, per = hd / 16;
    const long idx = blockIdx.x * (long)blockDim.x + threadIdx.x;
    const int c = idx % per;
    const int h = idx / per % heads;
    const long t = idx / per / heads;
    if (t >= T) return;
    const int N = heads * hd, d = c * 8, n = h * hd + d;
    unsigned short* row = qkv + t * N + n;
    float a[8], b[8];
    if constexpr (PARTS > 0) {
        f32x4 u[PARTS][2], w[PARTS][2];
#pragma unroll
        for (int s = 0; s < PARTS; ++s)
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const float* p = part + ((long)s * T + t) * N + n;
                u[s][q] = reinterpret_cast<const f32x4*>(p)[q];
                w[s][q] = reinterpret_cast<const f32x4*>(p + half)[q];
            }
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            a[e] = b[e] = 0.f;
#pragma unroll
            for (int s = 0; s < PARTS; ++s) {
                a[e] += u[s][e / 4][e % 4];
                b[e] += w[s][e / 4][e % 4];
            }
        }
    } else if (PARTS < 0) {
#pragma unroll
        for (int e = 0; e < 8; ++e) a[e] = b[e] = 0.f;
        for (int s = 0; s < S; ++s) {
            const float* p = part + ((long)s * T + t) * N + n;
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const f32x4 u = reinterpret_cast<const f32x4*>(p)[q];
                const f32x4 w = reinterpret_cast<const f32x4*>(p + half)[q];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    a[q * 4 + e] += u[e];
                    b[q * 4 + e] += w[e];
                }
            }
        }
    } else {
        load_bf16x8(row, a);
        load_bf16x8(row + half, b);
    }
    if (bias) {
        float u[8], w[8];
        load_bf16x8(bias + n, u);
        load_bf16x8(bias + n + half, w);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            a[e] += u[e];
            b[e] += w[e];
        }
    }
    const bool turns = pos && h < nq + nkv;
    if (turns) {
        const long tab = turn_row(pos[t], table) * half + d;
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const f32x4 cs = reinterpret_cast<const f32x4*>(cos_t + tab)[q];
            const f32x4 sn = reinterpret_cast<const f32x4*>(sin_t + tab)[q];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float x = a[q * 4 + e], y = b[q * 4 + e];
                a[q * 4 + e] = x * cs[e] - y * sn[e];
                b[q * 4 + e] = y * cs[e] + x * sn[e];
            }
        }
    }
    if (S > 0 || bias || turns) {
        store_bf16x8(row, a);
        store_bf16x8(row + half, b);
    }
    if (h < nq) return;
    const int kvh = (h - nq) % nkv, slot = slots[t];
    if (slot < 0) return;            // no such position
    const long dst =
        (((long)(slot / bs) * nkv + kvh) * bs + slot % bs) * hd + d;
    CT* cache = (h < nq + nkv ? k_cache : v_cache) + dst;
    if (sizeof(CT) == 2) {
        unsigned short* o = reinterpret_cast<unsigned short*>(cache);
        store_bf16x8(o, a);
        store_bf16x8(o + half, b);
    } else {
        unsigned int w[4];
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const float* x = q ? b : a;
            float r[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) r[e] = bf2f(f2bf(x[e]));
#pragma unroll
            for (int e = 0; e < 2; ++e)
                w[q * 2 + e] =
                    f2fp8x2(r[e * 4], r[e * 4 + 1]) |
                    (unsigned int)f2fp8x2(r[e * 4 + 2], r[e * 4 + 3]) << 16;
        }
        *reinterpret_cast<uint2v*>(cache) = uint2v{w[0], w[1]};
        *reinterpret_cast<uint2v*>(cache + half) = uint2v{w[2], w[3]};
    }
}

// ----------------------------------------------- what a step starts with
// Bound by their launches: each is one for what were five and four. A captured
// decode step of one row, 8 layers: 248 -> 231 us at distilgpt2's sizes (both
// kernels), 501 -> 490 us at llama3.2-1b's (the slots alone).

// table[pos / bs] * bs + pos % bs of a row's table: where its new key and value
// go; -1, which the kernels that store leave out, for a position that the table
// does not have.
DEV_INLINE int decode_slot(const int* table, int pos, int W, int bs) {
    const int page = pos / bs;
    return pos < 0 || page >= W ? -1 : table[page] * bs + pos % bs;
}

__global__ void decode_slots_kernel(const int* __restrict__ table,
                                    const int* __restrict__ pos,
                                    int* __restrict__ slots, int B, int W,
                                    long row_stride, int bs) {
    const int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= B) return;
    slots[b] = decode_slot(table + b * row_stride, pos[b], W, bs);
}

// The same, and order: the B <= ORDER_MAX rows by their lengths, longest first (of
// the same length: as they stand). A row's place is the number of rows before it:
// four waves count a quarter of the others each, for 64 rows. 2.1 us at 24 rows, 3.0
// at 100, 4.0 at 200, 7.3 at 512, 23 at 2048.
constexpr int ORDER_MAX = 2048;
__global__ __launch_bounds__(256) void decode_plan_kernel(
    const int* __restrict__ table, const int* __restrict__ pos,
    int* __restrict__ slots, const int* __restrict__ lens,
    int* __restrict__ order, int B, int W, long row_stride, int bs) {
    __shared__ __attribute__((aligned(16))) int len_s[ORDER_MAX];
    __shared__ int places[4][64];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const int quads = (B + 3) / 4;
    for (int i = threadIdx.x; i < quads * 4; i += 256)
        len_s[i] = i < B ? lens[i] : INT_MIN;  // (behind all others)
    const int b = blockIdx.x * 64 + lane;
    if (wid == 0 && b < B)
        slots[b] = decode_slot(table + b * row_stride, pos[b], W, bs);
    __syncthreads();
    const int mine = b < B ? len_s[b] : 0;
    int n = 0;
    for (int i = wid; i < quads; i += 4) {
        const int4 l = reinterpret_cast<const int4*>(len_s)[i];
        const int v[4] = {l.x, l.y, l.z, l.w};
#pragma unroll
        for (int e = 0; e < 4; ++e)
            n += v[e] > mine || (v[e] == mine && i * 4 + e < b);
    }
    places[wid][lane] = n;
    __syncthreads();
    if (wid == 0 && b < B)
        order[places[0][lane] + places[1][lane] + places[2][lane] +
              places[3][lane]] = b;
}

// out[t] = embed[ids[t]] + pos_embed[pos[t]], one workgroup a token; a row of
// NaN for an id or a position that the tables do not have
__global__ void embed_positions_kernel(
    const long* __restrict__ ids, const unsigned short* __restrict__ embed,
    const int* __restrict__ pos, const unsigned short* __restrict__ pos_embed,
    unsigned short* __restrict__ out, int H, long vocab, int positions) {
    const long t = blockIdx.x, id = ids[t];
    const int p = pos[t];
    const bool known = id >= 0 && id < vocab && p >= 0 && p < positions;
    for (int i = threadIdx.x * 8; i < H; i += blockDim.x * 8) {
        float a[8], b[8];
        if (known) {
            load_bf16x8(embed + id * H + i, a);
            load_bf16x8(pos_embed + (long)p * H + i, b);
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) a[e] = known ? a[e] + b[e] : NAN;
        store_bf16x8(out + t * H + i, a);
    }
}

// ----------------------------------------------------------------- swiglu
// out[t, i] = silu(gu[t, i]) * gu[t, I + i]; grid-stride, short8 loads.
__global__ void swiglu_kernel(
    const unsigned short* __restrict__ gu,  // [T, 2I]
    unsigned short* __restrict__ out,       // [T, I]
    long T, long I) {
    const long total = T * I / 8;
    for (long idx = blockIdx.x * blockDim.x + threadIdx.x; idx < total;
         idx += (long)gridDim.x * blockDim.x) {
        const long t = idx / (I / 8);
        const long i = (idx % (I / 8)) * 8;
        float g[8], u[8], o[8];
        load_bf16x8(gu + t * 2 * I + i, g);
        load_bf16x8(gu + t * 2 * I + I + i, u);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            float sig = 1.f / (1.f + __expf(-g[j]));
            o[j] = g[j] * sig * u[j];
        }
        store_bf16x8(out + t * I + i, o);
    }
}

// ------------------------------------------------------------- launchers
extern "C" {

void launch_rmsnorm(const unsigned short* x, const unsigned short* w,
                    unsigned short* y, long T, int H, float eps,
                    hipStream_t stream) {
    const int smem = H * 4;
    hipLaunchKernelGGL((rmsnorm_kernel<false>), dim3(T), dim3(256), smem,
                       stream, x, nullptr, w, y, nullptr, H, eps);
}

void launch_layernorm(const unsigned short* x, const unsigned short* w,
                      const unsigned short* b, unsigned short* y, long T,
                      int H, float eps, hipStream_t stream) {
    const int smem = H * 4;
    hipLaunchKernelGGL((layernorm_kernel<false>), dim3(T), dim3(256), smem,
                       stream, x, nullptr, w, b, y, nullptr, H, eps);
}

void launch_fused_add_layernorm(const unsigned short* x,
                                const unsigned short* resid,
                                const unsigned short* w,
                                const unsigned short* b, unsigned short* y,
                                unsigned short* resid_out, long T, int H,
                                float eps, hipStream_t stream) {
    const int smem = H * 4;
    hipLaunchKernelGGL((layernorm_kernel<true>), dim3(T), dim3(256), smem,
                       stream, x, resid, w, b, y, resid_out, H, eps);
}

void launch_gelu(const unsigned short* x, unsigned short* y, long n,
                 hipStream_t stream) {
    const long n8 = n / 8;
    long blocks = (n8 + 255) / 256;
    if (blocks > 2048) blocks = 2048;  // grid-stride
    if (blocks < 1) blocks = 1;
    hipLaunchKernelGGL(gelu_kernel, dim3(blocks), dim3(256), 0, stream, x, y,
                       n8);
}

void launch_fused_add_rmsnorm(const unsigned short* x,
                              const unsigned short* resid,
                              const unsigned short* w, unsigned short* y,
                              unsigned short* resid_out, long T, int H,
                              float eps, hipStream_t stream) {
    const int smem = H * 4;
    hipLaunchKernelGGL((rmsnorm_kernel<true>), dim3(T), dim3(256), smem,
                       stream, x, resid, w, y, resid_out, H, eps);
}

void launch_rope(unsigned short* q, unsigned short* k, const int* pos,
                 const float* cos_t, const float* sin_t, int table, int T, int nq,
                 int nkv, int hd, long sq, long sk, hipStream_t stream) {
    const long waves = (long)T * (nq + nkv);
    const long blocks = (waves + 3) / 4;
    hipLaunchKernelGGL(rope_kernel, dim3(blocks), dim3(256), 0, stream, q, k,
                       pos, cos_t, sin_t, table, T, nq, nkv, hd, sq, sk);
}

void launch_kv_store(const unsigned short* k, const unsigned short* v,
                     unsigned short* k_cache, unsigned short* v_cache,
                     const int* slots, int T, int nkv, int hd, int bs,
                     long sk, long sv, hipStream_t stream) {
    const long waves = (long)T * nkv;
    const long blocks = (waves + 3) / 4;
    hipLaunchKernelGGL(kv_store_kernel, dim3(blocks), dim3(256), 0, stream, k,
                       v, k_cache, v_cache, slots, T, nkv, hd, bs, sk, sv);
}

void launch_kv_store_fp8(const unsigned short* k, const unsigned short* v,
                         unsigned char* k_cache, unsigned char* v_cache,
                         const int* slots, int T, int nkv, int hd, int bs,
                         long sk, long sv, hipStream_t stream) {
    const long waves = (long)T * nkv;
    const long blocks = (waves + 3) / 4;
    hipLaunchKernelGGL(kv_store_fp8_kernel, dim3(blocks), dim3(256), 0,
                       stream, k, v, k_cache, v_cache, slots, T, nkv, hd, bs,
                       sk, sv);
}

void launch_decode_slots(const int* table, const int* pos, int* slots, int B,
                         int W, long row_stride, int bs, hipStream_t stream) {
    if (B == 0) return;
    hipLaunchKernelGGL(decode_slots_kernel, dim3((B + 255) / 256), dim3(256),
                       0, stream, table, pos, slots, B, W, row_stride, bs);
}

// nonzero for more rows than it takes
int launch_decode_plan(const int* table, const int* pos, int* slots,
                       const int* lens, int* order, int B, int W,
                       long row_stride, int bs, hipStream_t stream) {
    if (B < 1 || B > ORDER_MAX) return 1;
    hipLaunchKernelGGL(decode_plan_kernel, dim3((B + 63) / 64), dim3(256), 0,
                       stream, table, pos, slots, lens, order, B, W, row_stride,
                       bs);
    return 0;
}

void launch_embed_positions(const long* ids, const unsigned short* embed,
                            const int* pos, const unsigned short* pos_embed,
                            unsigned short* out, long T, int H, long vocab,
                            int positions, hipStream_t stream) {
    if (T == 0) return;
    hipLaunchKernelGGL(embed_positions_kernel, dim3(T), dim3(128), 0, stream,
                       ids, embed, pos, pos_embed, out, H, vocab, positions);
}

// hd % 16 == 0; qkv, bias, tables and pools 16-byte aligned; nonzero otherwise
int launch_qkv_rope_store(const float* part, int S, unsigned short* qkv,
                      const unsigned short* bias, const int* pos,
                      const float* cos_t, const float* sin_t, int table,
                      void* k_cache, void* v_cache, const int* slots, long T, int nq, int nkv,
                      int hd, int bs, int fp8, hipStream_t stream) {
    if (hd % 16) return 1;
    const long n = T * (nq + 2 * nkv) * (hd / 16);
    if (n == 0) return 0;
    const int threads = n < 256 * 256 ? 64 : 256;
#define RS_ONE(CT, P)                                                         \
    hipLaunchKernelGGL((qkv_rope_store_kernel<CT, P>),                        \
                       dim3((n + threads - 1) / threads), dim3(threads), 0,   \
                       stream, part, S, qkv, bias, pos, cos_t, sin_t, table,  \
                       (CT*)k_cache, (CT*)v_cache, slots, T, nq, nkv, hd, bs)
#define RS_GO(CT)                                                             \
    do {                                                                      \
        if (S == 0) RS_ONE(CT, 0);                                            \
        else if (S == 1) RS_ONE(CT, 1);                                       \
        else if (S == 2) RS_ONE(CT, 2);                                       \
        else if (S == 4) RS_ONE(CT, 4);                                       \
        else RS_ONE(CT, -1);                                                  \
    } while (0)
    if (fp8) RS_GO(unsigned char);
    else RS_GO(unsigned short);
#undef RS_ONE
#undef RS_GO
    return 0;
}

void launch_swiglu(const unsigned short* gu, unsigned short* out, long T,
                   long I, hipStream_t stream) {
    const long total = T * I / 8;
    long blocks = (total + 255) / 256;
    if (blocks > 2048) blocks = 2048;  // grid-stride (guide G11)
    if (blocks < 1) blocks = 1;
    hipLaunchKernelGGL(swiglu_kernel, dim3(blocks), dim3(256), 0, stream, gu,
                       out, T, I);
}

}  // extern "C"
