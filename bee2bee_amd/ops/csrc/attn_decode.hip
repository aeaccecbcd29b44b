// Paged GQA decode attention for head sizes other than 64 and 128 (those are
// attn_stream.hip's, at a positive scale) — three-stage flash-decoding:
//   1. attn_scores:  S = q.K^T + chunk-level softmax -> p, (m,l) scratch
//   2. attn_pv:      partial_o = p.V per chunk (p from scratch, LDS-staged)
//   3. attn_combine: merge chunk partials, normalize, write bf16 out
//
// Replaces: the reference's decode path inside transformers.generate()
// (bee2bee/hf.py:84-108). Numerics reference: ops/reference.py attn_decode.
#include "common.h"

#define DEC_BLOCK 256
#define DEC_WAVES 4
#define DEC_CHUNK 256  // keys per workgroup (DEC_WAVES x 64)

// KV element loaders, templated on the cache storage type:
//   unsigned short = bf16 (2 B/elem), unsigned char = OCP fp8 e4m3 (1 B).
template <typename KVT>
__device__ __forceinline__ bf16x8 load_kv_bf16x8(const KVT* p);
template <>
__device__ __forceinline__ bf16x8 load_kv_bf16x8(const unsigned short* p) {
    return *reinterpret_cast<const bf16x8*>(p);
}
template <>
__device__ __forceinline__ bf16x8 load_kv_bf16x8(const unsigned char* p) {
    float f[8];
    load_fp8x8(p, f);
    bf16x8 r;
#pragma unroll
    for (int e = 0; e < 8; ++e) r[e] = (__bf16)f[e];
    return r;
}
// raw 2-element cache pair (batched loads keep the raw bytes in flight,
// converting only when consumed)
template <typename KVT> struct kv_pair_t;
template <> struct kv_pair_t<unsigned short> { short2v v; };
template <> struct kv_pair_t<unsigned char> { u8x2 v; };
__device__ __forceinline__ float2v kv_pair_f32(kv_pair_t<unsigned short> p) {
    return float2v{bf2f((unsigned short)p.v[0]), bf2f((unsigned short)p.v[1])};
}
__device__ __forceinline__ float2v kv_pair_f32(kv_pair_t<unsigned char> p) {
    unsigned short w = (unsigned short)p.v[0] |
                       ((unsigned short)p.v[1] << 8);
    return fp8x2_2f(w);
}

// ------------------------------------------------------------ stage 1: S
template <int G, typename KVT>
__global__ __launch_bounds__(DEC_BLOCK) void attn_scores_kernel(
    const unsigned short* __restrict__ q,        // [B, nq, hd] (strided)
    const KVT* __restrict__ k_cache,             // [nb, nkv, bs, hd]
    const int* __restrict__ block_table,         // [B, W]
    const int* __restrict__ seq_lens,            // [B]
    unsigned short* __restrict__ p_out,          // [B, nkv, C, CHUNK, G] bf16
    float* __restrict__ part_ml,                 // [B, nkv, C, G, 2]
    int nkv, int W, int bs, int hd, int C, long q_stride, float scale) {
    const int b = blockIdx.x;
    const int kvh = blockIdx.y;
    const int L = min(seq_lens[b], W * bs);    // (what its pages hold)
    if ((int)blockIdx.z * DEC_CHUNK >= L) return;
    const int lane = threadIdx.x % WAVE;
    const int wid = threadIdx.x / WAVE;

    extern __shared__ __attribute__((aligned(16))) char smem_raw[];
    unsigned short* q_s = reinterpret_cast<unsigned short*>(smem_raw);  // [G*hd]
    float* red = reinterpret_cast<float*>(smem_raw + ((G * hd * 2 + 15) & ~15));
    // red: [DEC_WAVES][G][2] wave-level m / sum

    for (int i = threadIdx.x; i < G * hd; i += DEC_BLOCK) {
        const int g = i / hd, d = i % hd;
        q_s[i] = f2bf(
            bf2f(q[(long)b * q_stride + (kvh * G + g) * (long)hd + d]) * scale);
    }
    __syncthreads();

    const int* bt = block_table + (long)b * W;
    // loop chunks with stride gridDim.z — the PV and combine stages walk
    // ALL chunks of (b, kvh), so every chunk's p/(m,l) must be produced even
    // when the launcher picks Z < ceil(L/DEC_CHUNK) (a single-
    // chunk kernel left chunks >= Z uninitialized for hd not in {64,128})
    for (int chunk = blockIdx.z; chunk * DEC_CHUNK < L; chunk += gridDim.z) {
    const int start = chunk * DEC_CHUNK;
    const int key = start + threadIdx.x;  // one key per thread
    const bool valid = key < L;

    float s[G];
#pragma unroll
    for (int g = 0; g < G; ++g) s[g] = -1e30f;
    if (valid) {
        const int page = bt[key / bs];
        BB_KASSERT(page >= 0);  // block table row must be fully mapped
        const KVT* kr =
            k_cache + (((long)page * nkv + kvh) * bs + key % bs) * hd;
#pragma unroll
        for (int g = 0; g < G; ++g) s[g] = 0.f;
        for (int d = 0; d < hd; d += 8) {
            const bf16x8 kraw = load_kv_bf16x8<KVT>(kr + d);
#pragma unroll
            for (int g = 0; g < G; ++g) {
                const short8 qraw =
                    *reinterpret_cast<const short8*>(q_s + g * hd + d);
#pragma unroll
                for (int j = 0; j < 8; ++j)
                    s[g] = fmaf((float)kraw[j],
                                bf2f((unsigned short)qraw[j]), s[g]);
            }
        }
    }

    // chunk-level softmax: wave max -> LDS -> chunk max; then exp + sums
    float wmax[G];
#pragma unroll
    for (int g = 0; g < G; ++g) wmax[g] = wave_max(s[g]);
    if (lane == 0) {
#pragma unroll
        for (int g = 0; g < G; ++g) red[(wid * G + g) * 2] = wmax[g];
    }
    __syncthreads();
    float M[G];
#pragma unroll
    for (int g = 0; g < G; ++g) {
        float m = red[g * 2];
        for (int w2 = 1; w2 < DEC_WAVES; ++w2)
            m = fmaxf(m, red[(w2 * G + g) * 2]);
        M[g] = m;
    }
    float p[G], wsum[G];
#pragma unroll
    for (int g = 0; g < G; ++g) {
        // round to bf16 BEFORE summing so l matches the p that PV consumes
        p[g] = valid ? bf2f(f2bf(__expf(s[g] - M[g]))) : 0.f;
        wsum[g] = wave_sum(p[g]);
    }
    __syncthreads();  // red reuse (second slot written below)
    if (lane == 0) {
#pragma unroll
        for (int g = 0; g < G; ++g) red[(wid * G + g) * 2 + 1] = wsum[g];
    }
    // coalesced p write: [key][G] bf16 (p in [0,1]; bf16 halves the
    // G-proportional scratch traffic)
    {
        unsigned short* prow =
            p_out + ((((long)b * nkv + kvh) * C + chunk) * DEC_CHUNK +
                     threadIdx.x) * G;
#pragma unroll
        for (int g = 0; g < G; ++g) prow[g] = f2bf(p[g]);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        float* pml = part_ml + ((((long)b * nkv + kvh) * C + chunk) * G) * 2;
#pragma unroll
        for (int g = 0; g < G; ++g) {
            float lsum = 0.f;
            for (int w2 = 0; w2 < DEC_WAVES; ++w2)
                lsum += red[(w2 * G + g) * 2 + 1];
            pml[g * 2] = M[g];
            pml[g * 2 + 1] = lsum;
        }
    }
    __syncthreads();  // red reused by the next chunk iteration
    }  // chunk loop
}


// ----------------------------------------------------------- stage 2: PV
// When FOLD (launcher sets it iff gridDim.z == 1, i.e. every chunk of this
// (b, kvh) runs serially in THIS workgroup: B*nkv >= 4096), the kernel carries the running flash-decoding
// merge (M, l, acc) across chunks in registers and writes the normalized
// bf16 output directly: no part_o round-trip, no combine kernel.
template <int G, bool FOLD, typename KVT>
__global__ __launch_bounds__(DEC_BLOCK) void attn_pv_kernel(
    const KVT* __restrict__ v_cache,             // [nb, nkv, bs, hd]
    const int* __restrict__ block_table,
    const int* __restrict__ seq_lens,
    const unsigned short* __restrict__ p_in,     // [B,nkv,C,CHUNK,G] bf16
    float* __restrict__ part_o,                  // [B, nkv, C, G, hd]
    const float* __restrict__ part_ml,           // [B, nkv, C, G, 2]
    unsigned short* __restrict__ out,            // [B, nq, hd] (FOLD only)
    float* __restrict__ out_ml,                  // optional [B, nq, 2]:
                                                 // final (m, l) per q head —
                                                 // the cross-rank merge
                                                 // state for context
                                                 // parallelism (parallel/cp)
    int nkv, int W, int bs, int hd, int C) {
    const int b = blockIdx.x;
    const int kvh = blockIdx.y;
    const int L = min(seq_lens[b], W * bs);    // (what its pages hold)
    if ((int)blockIdx.z * DEC_CHUNK >= L) return;
    const int lane = threadIdx.x % WAVE;
    const int wid = threadIdx.x / WAVE;

    extern __shared__ __attribute__((aligned(16))) char smem_raw[];
    float* p_s = reinterpret_cast<float*>(smem_raw);  // [CHUNK][G]
    long* voff_s = reinterpret_cast<long*>(p_s + DEC_CHUNK * G);  // [CHUNK]
    float* merge = reinterpret_cast<float*>(voff_s + DEC_CHUNK);  // [Wv][G][hd]
    // FOLD running state lives in LDS so the hot loop stays at ~64 VGPRs
    // (a register version measured 101 VGPRs -> 5 waves/SIMD). Each head
    // group g is OWNED by wave g%DEC_WAVES: the per-chunk merge + fold and
    // the final normalize run G-way parallel across waves instead of
    // serializing on wave 0 (the r1 kernel's measured latency tail), and
    // per-g slices stay single-writer so no extra barriers appear.
    float* run = merge + DEC_WAVES * G * hd;   // [G][hd] running acc
    float* runml = run + G * hd;               // [G][2] running (m, l)
    if (FOLD) {
        for (int g = wid; g < G; g += DEC_WAVES) {
            for (int i = lane; i < hd; i += WAVE) run[g * hd + i] = 0.f;
            if (lane == 0) {
                runml[g * 2] = -1e30f;
                runml[g * 2 + 1] = 0.f;
            }
        }
    }

    for (int chunk = blockIdx.z; chunk * DEC_CHUNK < L; chunk += gridDim.z) {
    const int start = chunk * DEC_CHUNK;
    // stage p for the whole chunk into LDS, widening bf16 -> fp32 so the
    // inner fma loop reads full-rate f32x4
    {
        const unsigned short* psrc =
            p_in + (((long)b * nkv + kvh) * C + chunk) * DEC_CHUNK * G;
        for (int i = threadIdx.x; i < DEC_CHUNK * G / 8; i += DEC_BLOCK) {
            float v[8];
            load_bf16x8(psrc + i * 8, v);
#pragma unroll
            for (int j = 0; j < 8; ++j) p_s[i * 8 + j] = v[j];
        }
    }
    // per-thread V row offset (one chained block-table load per key)
    {
        const int* bt = block_table + (long)b * W;
        const int key = start + threadIdx.x;
        long voff = 0;
        if (key < L) {
            const int page = bt[key / bs];
            voff = (((long)page * nkv + kvh) * bs + key % bs) * hd;
        }
        voff_s[threadIdx.x] = voff;
    }
    __syncthreads();

    // wave wid accumulates keys [wid*64, wid*64+64) of the chunk;
    // lane owns output dims (d0, d0+1)
    const int d0 = lane * 2;
    const int wave_start = wid * WAVE;
    const int nkeys = min(WAVE, L - (start + wave_start));
    float o0[G], o1[G];
#pragma unroll
    for (int g = 0; g < G; ++g) o0[g] = o1[g] = 0.f;
    if (d0 < hd && nkeys > 0) {
        const long* voffs = voff_s + wave_start;
        const float* pw = p_s + wave_start * G;
        int t = 0;
        for (; t + 32 <= nkeys; t += 32) {  // 32 V loads in flight
            kv_pair_t<KVT> vv[32];
#pragma unroll
            for (int j = 0; j < 32; ++j)
                vv[j] = *reinterpret_cast<const kv_pair_t<KVT>*>(
                    v_cache + voffs[t + j] + d0);
#pragma unroll
            for (int j = 0; j < 32; ++j) {
                const float2v vf = kv_pair_f32(vv[j]);
                const float* pt = pw + (t + j) * G;
#pragma unroll
                for (int g = 0; g < G; ++g) {
                    o0[g] = fmaf(pt[g], vf.x, o0[g]);
                    o1[g] = fmaf(pt[g], vf.y, o1[g]);
                }
            }
        }
        for (; t < nkeys; ++t) {
            const kv_pair_t<KVT> vv =
                *reinterpret_cast<const kv_pair_t<KVT>*>(
                    v_cache + voffs[t] + d0);
            const float2v vf = kv_pair_f32(vv);
            const float* pt = pw + t * G;
#pragma unroll
            for (int g = 0; g < G; ++g) {
                o0[g] = fmaf(pt[g], vf.x, o0[g]);
                o1[g] = fmaf(pt[g], vf.y, o1[g]);
            }
        }
    }

    // all waves used the same chunk max, so cross-wave merge is a plain sum
    float* mw = merge + wid * G * hd;
    if (d0 < hd) {
#pragma unroll
        for (int g = 0; g < G; ++g) {
            mw[g * hd + d0] = o0[g];
            mw[g * hd + d0 + 1] = o1[g];
        }
    }
    __syncthreads();
    if (d0 < hd) {
        const long base = (((long)b * nkv + kvh) * C + chunk) * G;
        for (int g = wid; g < G; g += DEC_WAVES) {
            float a0 = 0.f, a1 = 0.f;
            for (int w2 = 0; w2 < DEC_WAVES; ++w2) {
                a0 += merge[(w2 * G + g) * hd + d0];
                a1 += merge[(w2 * G + g) * hd + d0 + 1];
            }
            if (FOLD) {
                // online merge with this chunk's (m, l) from the scores pass
                const float mc = part_ml[(base + g) * 2];
                const float lc = part_ml[(base + g) * 2 + 1];
                const float mold = runml[g * 2];
                const float mn = fmaxf(mold, mc);
                const float alpha = __expf(mold - mn);
                const float beta = __expf(mc - mn);
                run[g * hd + d0] = run[g * hd + d0] * alpha + a0 * beta;
                run[g * hd + d0 + 1] =
                    run[g * hd + d0 + 1] * alpha + a1 * beta;
                if (lane == 0) {
                    runml[g * 2] = mn;
                    runml[g * 2 + 1] = runml[g * 2 + 1] * alpha + lc * beta;
                }
            } else {
                float* po = part_o + (base + g) * hd;
                po[d0] = a0;
                po[d0 + 1] = a1;
            }
        }
    }
    __syncthreads();  // LDS buffers reused by the next chunk iteration
    }  // chunk loop

    if (FOLD) {
        const int d0f = lane * 2;
        const int nq = nkv * G;
        if (d0f < hd) {
            for (int g = wid; g < G; g += DEC_WAVES) {
                const float lr = runml[g * 2 + 1];
                const float inv = (lr > 0.f) ? 1.f / lr : 0.f;
                unsigned short* orow =
                    out + ((long)b * nq + kvh * G + g) * hd;
                orow[d0f] = f2bf(run[g * hd + d0f] * inv);
                orow[d0f + 1] = f2bf(run[g * hd + d0f + 1] * inv);
            }
        }
        if (out_ml != nullptr && lane == 0) {
            for (int g = wid; g < G; g += DEC_WAVES) {
                float* mlrow = out_ml + ((long)b * nq + kvh * G + g) * 2;
                mlrow[0] = runml[g * 2];
                mlrow[1] = runml[g * 2 + 1];
            }
        }
    }
}

// ------------------------------------------------------ stage 3: combine
template <int G>
__global__ __launch_bounds__(DEC_BLOCK) void attn_decode_combine_kernel(
    const float* __restrict__ part_o,   // [B, nkv, C, G, hd]
    const float* __restrict__ part_ml,  // [B, nkv, C, G, 2]
    const int* __restrict__ seq_lens,
    unsigned short* __restrict__ out,   // [B, nq, hd]
    float* __restrict__ out_ml,         // optional [B, nq, 2] (see PV)
    int nkv, int hd, int C) {
    const int b = blockIdx.x;
    const int kvh = blockIdx.y;
    const int g = blockIdx.z;  // one block per (seq, kv head, q head)
    const int nq = nkv * G;
    const int L = seq_lens[b];
    const int nc = min((L + DEC_CHUNK - 1) / DEC_CHUNK, C);
    const long base = ((long)b * nkv + kvh) * C;

    // stage this head's (m, l) pairs once
    __shared__ float ml_s[128][2];  // C <= 128 (32768-token contexts)
    for (int c = threadIdx.x; c < nc; c += DEC_BLOCK) {
        ml_s[c][0] = part_ml[((base + c) * G + g) * 2];
        ml_s[c][1] = part_ml[((base + c) * G + g) * 2 + 1];
    }
    __syncthreads();
    float M = -1e30f;
    for (int c = 0; c < nc; ++c) M = fmaxf(M, ml_s[c][0]);
    float Ltot = 0.f;
    for (int c = 0; c < nc; ++c) Ltot += __expf(ml_s[c][0] - M) * ml_s[c][1];
    const float inv = (Ltot > 0.f) ? 1.f / Ltot : 0.f;
    if (out_ml != nullptr && threadIdx.x == 0) {
        float* mlrow = out_ml + ((long)b * nq + kvh * G + g) * 2;
        mlrow[0] = M;
        mlrow[1] = Ltot;
    }

    for (int d = threadIdx.x; d < hd; d += DEC_BLOCK) {
        float acc = 0.f;
        for (int c = 0; c < nc; ++c)
            acc += __expf(ml_s[c][0] - M) *
                   part_o[((base + c) * G + g) * hd + d];
        out[((long)b * nq + kvh * G + g) * hd + d] = f2bf(acc * inv);
    }
}

extern "C" void launch_attn_decode(
    const unsigned short* q, const void* k_cache, const void* v_cache,
    const int* block_table, const int* seq_lens, unsigned short* p_buf,
    float* part_o, float* part_ml, unsigned short* out, float* out_ml,
    int B, int nkv,
    int G, int W, int bs, int hd, int C, long q_stride, float scale,
    int fp8, hipStream_t stream) {
    // enough blocks to fill the chip, but chunks loop within a block so the
    // cold-start/tail phases amortize over multiple 64 KB K/V bursts
    int Z = (4096 + B * nkv - 1) / (B * nkv);
    if (Z > C) Z = C;
    if (Z < 1) Z = 1;
    dim3 grid(B, nkv, Z);
    dim3 cgrid(B, nkv, G);
    const int smem_s = ((G * hd * 2 + 15) & ~15) + DEC_WAVES * G * 2 * 4;
    const int smem_pv = DEC_CHUNK * G * 4 + DEC_CHUNK * 8 +
                        DEC_WAVES * G * hd * 4 +
                        G * hd * 4 + G * 8;  // + FOLD running state
#define LAUNCH_T(GG, KVT)                                                      \
    do {                                                                       \
        const KVT* kc = reinterpret_cast<const KVT*>(k_cache);                 \
        const KVT* vc = reinterpret_cast<const KVT*>(v_cache);                 \
        hipLaunchKernelGGL((attn_scores_kernel<GG, KVT>), grid,                \
                           dim3(DEC_BLOCK), smem_s, stream, q, kc,             \
                           block_table, seq_lens, p_buf, part_ml, nkv, W, bs,  \
                           hd, C, q_stride, scale);                            \
        if (Z == 1) {                                                          \
            hipLaunchKernelGGL((attn_pv_kernel<GG, true, KVT>), grid,          \
                               dim3(DEC_BLOCK), smem_pv, stream, vc,           \
                               block_table, seq_lens, p_buf, part_o, part_ml,  \
                               out, out_ml, nkv, W, bs, hd, C);                \
        } else {                                                               \
            hipLaunchKernelGGL((attn_pv_kernel<GG, false, KVT>), grid,         \
                               dim3(DEC_BLOCK), smem_pv, stream, vc,           \
                               block_table, seq_lens, p_buf, part_o,           \
                               part_ml, out, nullptr, nkv, W, bs, hd, C);      \
            hipLaunchKernelGGL(attn_decode_combine_kernel<GG>, cgrid,          \
                               dim3(DEC_BLOCK), 0, stream, part_o, part_ml,    \
                               seq_lens, out, out_ml, nkv, hd, C);             \
        }                                                                      \
    } while (0)
#define LAUNCH(GG)                                                             \
    do {                                                                       \
        if (fp8) LAUNCH_T(GG, unsigned char);                                  \
        else LAUNCH_T(GG, unsigned short);                                     \
    } while (0)
    switch (G) {
        case 1: LAUNCH(1); break;
        case 2: LAUNCH(2); break;
        case 3: LAUNCH(3); break;
        case 4: LAUNCH(4); break;
        case 5: LAUNCH(5); break;
        case 6: LAUNCH(6); break;
        case 7: LAUNCH(7); break;  // Qwen2.5-7B: 28 q / 4 kv heads
        case 8: LAUNCH(8); break;
        default: LAUNCH(16); break;
    }
#undef LAUNCH
#undef LAUNCH_T
}
