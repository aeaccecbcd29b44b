// Torch bindings of the projections of a few rows (linear_rows.hip), of some tens
// (linear_mid.hip) and more (linear_wide.hip), of the pass between q|k|v and
// attention, and of a decode step's layers in one launch (decode_stack.hip).
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>
#include <hip/hip_runtime.h>
#include <algorithm>
#include <limits>
#include "decode_stack.h"

using torch::Tensor;
using c10::optional;

extern "C" int launch_linear_rows(
    const void*, int, const unsigned short*, const unsigned short*,
    const unsigned short*, const unsigned short*, const float*, const void*,
    int, void*, int, const unsigned short*, unsigned short*, float*, int, int,
    int, float, int, int, const int*, const float*, const float*, int,
    const int*, void*, void*, int, int, int, int, int, hipStream_t);
extern "C" int decode_stack_rows(int, int);
extern "C" int decode_stack_splits(long, long);
extern "C" int launch_decode_stack(const StackArgs*, int, int, int, int,
                                   hipStream_t);
extern "C" int linear_mid_splits(int, int);
extern "C" int launch_linear_mid(const unsigned short*, const unsigned short*,
                                 const unsigned short*, void*, int, int, int,
                                 int, int, int, const float*, float,
                                 hipStream_t);
extern "C" int linear_wide_plan(int, int, int, int);
extern "C" int linear_wide_rows(int, int, int, int, int, int);
extern "C" int launch_linear_wide(const unsigned short*, const unsigned short*,
                                  void*, int, int, int, int, int, int,
                                  hipStream_t);
extern "C" int launch_add_norm_parts(
    const float*, const unsigned short*, const void*, int,
    const unsigned short*, const unsigned short*, void*, int, unsigned short*,
    int, int, int, float, hipStream_t);
extern "C" int launch_qkv_rope_store(
    const float*, int, unsigned short*, const unsigned short*, const int*,
    const float*, const float*, int, void*, void*, const int*, long, int, int,
    int, int, int, hipStream_t);

extern "C" int launch_decode_plan(const int*, const int*, int*, const int*,
                                  int*, int, int, long, int, hipStream_t);
extern "C" void launch_decode_slots(const int*, const int*, int*, int, int,
                                    long, int, hipStream_t);
extern "C" void launch_embed_positions(const long*, const unsigned short*,
                                       const int*, const unsigned short*,
                                       unsigned short*, long, int, long, int,
                                       hipStream_t);

namespace {

enum { EPI_PLAIN = 0, EPI_GLU = 1, EPI_GELU = 2, EPI_QKV = 3 };

hipStream_t stream() {
    return at::hip::getCurrentHIPStreamMasqueradingAsCUDA().stream();
}

bool is_f32(const Tensor& t) { return t.scalar_type() == torch::kFloat32; }

// t as the kernel reads it: contiguous, 16-byte aligned (copied if it is not)
Tensor dense(const Tensor& t, const char* name, bool f32_too = false) {
    TORCH_CHECK(t.is_cuda() && (t.scalar_type() == torch::kBFloat16 ||
                                (f32_too && is_f32(t))),
                name, f32_too ? " must be bf16 or fp32 on the GPU"
                              : " must be bf16 on the GPU");
    if (t.is_contiguous() &&
        reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0)
        return t;
    return t.clone(at::MemoryFormat::Contiguous);
}

// one value a column; undefined without the tensor
Tensor column(const optional<Tensor>& t, long n, const char* name) {
    if (!t.has_value()) return Tensor();
    TORCH_CHECK(t->numel() == n, name, " must have ", n, " values");
    return dense(*t, name);
}

const unsigned short* ptr(const Tensor& t) {
    return t.defined()
               ? reinterpret_cast<const unsigned short*>(t.data_ptr())
               : nullptr;
}

unsigned short* mut(Tensor& t) {
    return reinterpret_cast<unsigned short*>(t.data_ptr());
}

// The rotation's tables as kernels read them, [rows, hd / 2] each.
struct Turns {
    const float *cos_t = nullptr, *sin_t = nullptr;
    int rows = 0;
};
Turns turns(const optional<Tensor>& cos_t, const optional<Tensor>& sin_t,
            long hd) {
    const Tensor &c = cos_t.value(), &s = sin_t.value();
    for (const Tensor* t : {&c, &s})
        TORCH_CHECK(t->is_cuda() && t->scalar_type() == torch::kFloat32 &&
                    t->is_contiguous() && t->dim() == 2 && t->size(0) >= 1 &&
                    t->size(1) == hd / 2,
                    "rotation tables [rows, head size / 2] fp32");
    return {c.data_ptr<float>(), s.data_ptr<float>(),
            (int)std::min(c.size(0), s.size(0))};
}

struct Rows {
    Tensor x, w, norm_w, norm_b, squares;
    int M, N, K, norm;
    const float* sq() const {
        return squares.defined() ? squares.data_ptr<float>() : nullptr;
    }
};

// norm_b given: layer norm; norm_w alone: RMS norm; squares: RMS norm of rows
// that are multiplied by its weight already
Rows rows_of(const Tensor& x, const Tensor& w, const optional<Tensor>& norm_w,
             const optional<Tensor>& norm_b,
             const optional<Tensor>& squares) {
    TORCH_CHECK(x.dim() == 2 && w.dim() == 2 && x.size(1) == w.size(1),
                "x [M, K] and w [N, K]");
    Rows r;
    r.M = x.size(0);
    r.K = x.size(1);
    r.N = w.size(0);
    TORCH_CHECK(r.M >= 1 && r.M <= 16, "1 to 16 rows");
    TORCH_CHECK(r.K % 32 == 0, "K must be a multiple of 32");
    TORCH_CHECK(norm_w.has_value() || !norm_b.has_value());
    r.x = dense(x, "x", norm_b.has_value());
    r.w = dense(w, "w");
    r.norm_w = column(norm_w, r.K, "norm weight");
    r.norm_b = column(norm_b, r.K, "norm bias");
    r.norm = !norm_w.has_value() ? 0 : norm_b.has_value() ? 2 : 1;
    if (squares.has_value()) {
        TORCH_CHECK(r.norm == 0 && squares->is_cuda() && is_f32(*squares) &&
                    squares->dim() == 2 && squares->size(0) == r.M &&
                    squares->size(1) == r.K / 8 && squares->is_contiguous(),
                    "squares [M, K / 8] fp32, in the norm's place");
        r.squares = *squares;
        r.norm = 3;
    }
    return r;
}

// Gated projections of a few rows that linear_mid.hip's rings take: where they
// are long enough for a ring to pay, which starts later than waves that load for
// themselves. The rule does not look at the number of rows, on which a row's
// result does not depend. Measured (us, 1 / 8 / 16 rows, linear_rows.hip in
// brackets): 2x14336x4096 37.1 (36.5) / 37.9 (42.4) / 39 (51.7), 2x18944x3584
// 44 (43.7) / 44.2 (52.2) / 45.6 (57.9), but 2x8192x3072 19.6 (18.9) / 19.9
// (21.1) / 21.0 (23.2), 2x8192x2048 14.0 (13.7) / 13.8 (14.9) / 13.8 (15.6).
bool streams_gated(const Rows& r, int64_t act) {
    return act == EPI_GLU && (r.norm == 0 || r.norm == 3) && r.K % 64 == 0 &&
           (long)r.N * r.K >= 100000000 && (long)r.N * r.K < 1L << 31;
}

// x of a layer norm, and resid, may be fp32; keep32: so is the result. then_w,
// the weight of the RMS norm that reads the result: also the result times it, and
// the sums of squares of 8 columns each, in scaled and squares_out
Tensor rows_product(const Tensor& x, const Tensor& w,
                    const optional<Tensor>& bias,
                    const optional<Tensor>& resid,
                    const optional<Tensor>& norm_w,
                    const optional<Tensor>& norm_b,
                    const optional<Tensor>& squares, double eps, int64_t act,
                    bool keep32, const optional<Tensor>& then_w,
                    Tensor& scaled, Tensor& squares_out) {
    const Rows r = rows_of(x, w, norm_w, norm_b, squares);
    TORCH_CHECK(act == EPI_PLAIN || act == EPI_GLU || act == EPI_GELU);
    TORCH_CHECK(act != EPI_GLU || (r.N % 32 == 0 && !bias.has_value()));
    TORCH_CHECK(act == EPI_PLAIN || !(resid.has_value() || keep32));
    const int N = act == EPI_GLU ? r.N / 2 : r.N;
    if (resid.has_value())
        TORCH_CHECK(resid->dim() == 2 && resid->size(0) == r.M &&
                    resid->size(1) == N, "resid [M, N]");
    const Tensor b = column(bias, N, "bias");
    const Tensor add =
        resid.has_value() ? dense(*resid, "resid", true) : Tensor();
    const auto bf16 = r.w.options();
    const auto f32 = bf16.dtype(torch::kFloat32);
    Tensor y = torch::empty({r.M, N}, keep32 ? f32 : bf16);
    const Tensor tw = column(then_w, N, "the next norm's weight");
    if (tw.defined()) {
        TORCH_CHECK(N % 8 == 0);
        scaled = torch::empty({r.M, N}, bf16);
        squares_out = torch::empty({r.M, N / 8}, f32);
    }
    if (streams_gated(r, act)) {
        TORCH_CHECK(launch_linear_mid(ptr(r.x), ptr(r.w), nullptr,
                                      y.data_ptr(), r.M, N, r.K, 1, 1, 0,
                                      r.sq(), (float)eps, stream()) == 0);
        return y;
    }
    TORCH_CHECK(launch_linear_rows(
                    r.x.data_ptr(), is_f32(r.x), ptr(r.norm_w),
                    ptr(r.norm_b), ptr(r.w), ptr(b), r.sq(),
                    add.defined() ? add.data_ptr() : nullptr,
                    add.defined() && is_f32(add), y.data_ptr(), keep32,
                    ptr(tw), tw.defined() ? mut(scaled) : nullptr,
                    tw.defined() ? squares_out.data_ptr<float>() : nullptr,
                    r.M, N, r.K, (float)eps, r.norm, (int)act, nullptr,
                    nullptr, nullptr, 0, nullptr, nullptr, nullptr, 0, 0, 0,
                    0, 0, stream()) == 0);
    return y;
}

Tensor rows_linear(const Tensor& x, const Tensor& w,
                   const optional<Tensor>& bias,
                   const optional<Tensor>& resid,
                   const optional<Tensor>& norm_w,
                   const optional<Tensor>& norm_b,
                   const optional<Tensor>& squares, double eps, int64_t act,
                   bool keep32) {
    Tensor none;
    return rows_product(x, w, bias, resid, norm_w, norm_b, squares, eps, act,
                        keep32, optional<Tensor>(), none, none);
}

// -> the result, its rows times then_w, the sums of squares
std::tuple<Tensor, Tensor, Tensor> rows_sum(
    const Tensor& x, const Tensor& w, const optional<Tensor>& bias,
    const optional<Tensor>& resid, const optional<Tensor>& norm_w,
    const optional<Tensor>& norm_b, const optional<Tensor>& squares,
    double eps, bool keep32, const Tensor& then_w) {
    Tensor scaled, sums;
    Tensor y = rows_product(x, w, bias, resid, norm_w, norm_b, squares, eps,
                            EPI_PLAIN, keep32, then_w, scaled, sums);
    return {y, scaled, sums};
}

// -> rotated queries [M, nq, hd]; rotated keys and the values go to the pages
Tensor rows_qkv(const Tensor& x, const Tensor& w, const optional<Tensor>& bias,
                const optional<Tensor>& norm_w, const optional<Tensor>& norm_b,
                const optional<Tensor>& squares, double eps, int64_t nq,
                const optional<Tensor>& pos,
                const optional<Tensor>& cos_t, const optional<Tensor>& sin_t,
                Tensor& k_cache, Tensor& v_cache, const Tensor& slots) {
    const Rows r = rows_of(x, w, norm_w, norm_b, squares);
    const bool fp8 = k_cache.scalar_type() == torch::kUInt8;
    TORCH_CHECK(k_cache.dim() == 4 && k_cache.sizes() == v_cache.sizes() &&
                k_cache.scalar_type() == v_cache.scalar_type() &&
                k_cache.is_contiguous() && v_cache.is_contiguous());
    TORCH_CHECK(fp8 || k_cache.scalar_type() == torch::kBFloat16);
    const int nkv = k_cache.size(1), bs = k_cache.size(2),
              hd = k_cache.size(3);
    TORCH_CHECK(hd % 32 == 0 && r.N == (nq + 2 * nkv) * hd);
    TORCH_CHECK(slots.scalar_type() == torch::kInt32 &&
                slots.is_contiguous() && slots.numel() == r.M);
    Turns by;
    if (pos.has_value()) {
        TORCH_CHECK(pos->scalar_type() == torch::kInt32 &&
                    pos->is_contiguous() && pos->numel() == r.M);
        by = turns(cos_t, sin_t, hd);
    }
    const Tensor b = column(bias, r.N, "bias");
    Tensor q = torch::empty({r.M, nq, hd}, r.w.options());
    TORCH_CHECK(launch_linear_rows(
                    r.x.data_ptr(), is_f32(r.x), ptr(r.norm_w),
                    ptr(r.norm_b), ptr(r.w), ptr(b), r.sq(), nullptr, 0,
                    q.data_ptr(), 0, nullptr, nullptr, nullptr, r.M, r.N, r.K,
                    (float)eps, r.norm, EPI_QKV,
                    pos.has_value() ? pos->data_ptr<int>() : nullptr,
                    by.cos_t, by.sin_t, by.rows,
                    slots.data_ptr<int>(), k_cache.data_ptr(),
                    v_cache.data_ptr(), nq, nkv, hd, bs, fp8, stream()) == 0);
    return q;
}

// Most rows of a decode step whose layers decode_stack takes, 0 for a stack that
// it does not take (among them the group sizes that attn_decode refuses).
int64_t stack_rows(int64_t hidden, int64_t nq, int64_t nkv, int64_t hd,
                   int64_t inner, bool layer_norm) {
    const int64_t deepest = std::max(std::max(hidden, nq * hd), inner);
    const int64_t G = nkv < 1 || nq % nkv ? 0 : nq / nkv;
    if ((hd != 64 && hd != 128) || !((G >= 1 && G <= 8) || G == 16) ||
        hidden % 64 || inner % 64 || deepest > 1 << 16 ||
        (layer_norm && hidden > DS_LAYER_NORM))
        return 0;
    return decode_stack_rows((int)deepest, (int)hd);
}

// The layers of a decode step, x [M, H] to the last one's result. A layer is 14
// tensors: w_qkv, w_o, w_up, w_down, their biases, the two norms' weights, their
// biases (layer norm: all given), pages of keys and of values. wgs: workgroups
// (DS_WGS; fewer do the work of the others, more find it taken). status: see decode_stack.h, pinned.
// absent: so many of the last numbers are marked as taken, by nobody.
Tensor decode_stack(const Tensor& x,
                    const std::vector<std::vector<optional<Tensor>>>& layers,
                    int64_t nq, bool gelu, double eps, double scale,
                    const optional<Tensor>& pos, const optional<Tensor>& cos_t,
                    const optional<Tensor>& sin_t,
                    const optional<Tensor>& slots, const Tensor& table,
                    const Tensor& seq_lens, int64_t wgs,
                    const optional<Tensor>& status, int64_t patience,
                    int64_t absent) {
    const int L = layers.size();
    TORCH_CHECK(L >= 1 && layers[0].size() == 14);
    const Tensor xd = dense(x, "x");
    TORCH_CHECK(xd.dim() == 2);
    const Tensor& k0 = layers[0][12].value();
    TORCH_CHECK(k0.dim() == 4);
    const int M = xd.size(0), H = xd.size(1), nkv = k0.size(1),
              bs = k0.size(2), hd = k0.size(3);
    const bool fp8 = k0.scalar_type() == torch::kUInt8;
    TORCH_CHECK(fp8 || k0.scalar_type() == torch::kBFloat16);
    const bool norm_b = layers[0][10].has_value();
    const int Q = nq * hd, N = (nq + 2 * nkv) * hd;
    const int I = layers[0][3].value().size(1);
    TORCH_CHECK(M >= 1 && M <= stack_rows(H, nq, nkv, hd, I, norm_b), "rows");
    auto ints = [&](const Tensor& t, long n, const char* name) {
        TORCH_CHECK(t.is_cuda() && t.scalar_type() == torch::kInt32 &&
                    t.is_contiguous() && t.numel() >= n, name);
        return t.data_ptr<int>();
    };
    // tables and lengths may be of more rows, contexts as long as attn_decode's
    TORCH_CHECK(table.dim() == 2 && table.size(1) > 0);
    TORCH_CHECK(table.size(1) * bs <= 32768,
                "decode supports up to 32768-token contexts for now");

    StackArgs a{};
    a.M = M;
    a.gelu = gelu;
    a.nq = nq;
    a.nkv = nkv;
    a.G = nq / nkv;
    a.bs = bs;
    a.W = table.size(1);
    a.eps = (float)eps;
    a.scale = (float)scale;
    a.all = L;
    TORCH_CHECK(slots.has_value() || pos.has_value(), "slots or positions");
    if (slots.has_value()) {
        a.slots = ints(*slots, M, "slots");
        TORCH_CHECK(slots->numel() == M, "slots");
    }
    a.table = ints(table, (long)M * a.W, "table");
    a.seq_lens = ints(seq_lens, M, "seq_lens");
    if (pos.has_value()) {
        a.pos = ints(*pos, M, "positions");
        TORCH_CHECK(pos->numel() == M, "positions");
    }
    if (pos.has_value() && cos_t.has_value()) {
        const Turns by = turns(cos_t, sin_t, hd);
        a.cos_t = by.cos_t;
        a.sin_t = by.sin_t;
        a.turn_rows = by.rows;
    }
    const int up = gelu ? I : 2 * I;
    const int K[4] = {H, Q, H, I}, rows[4] = {N, H, up, H};
    for (int k = 0; k < 4; ++k) {
        a.K[k] = K[k];
        a.octets[k] = rows[k] / 8;
        a.half[k] = k == DS_QKV ? hd / 2 : k == DS_UP && !gelu ? I : 4;
    }
    // (as linear_rows.hip: stacks of more than 768)
    a.streamed = std::min(H, I) > 768 || std::max(up, I) > 4096;
    a.Z = decode_stack_splits((long)M * nkv, (long)a.W * bs);

    // words that pass, a layer's after the other's: queries, the step's own keys
    // and values, attention's result, the rows after attention, activations, the
    // rows after the layer
    const long after = norm_b ? (long)M * H : (long)M * H / 2 + M * H / 8;
    a.new_kv = M * Q / 2;
    a.att = a.new_kv + M * nkv * hd;
    a.o = a.att + M * Q / 2;
    a.up = a.o + after;
    a.down = a.up + M * I / 2;
    a.stride = (a.down + after + 31) / 32 * 32;
    const int launches = (L + DS_LAYERS - 1) / DS_LAYERS;
    a.items = M * nkv * a.Z;
    const long parts = a.Z > 1 ? (long)a.items * a.G * (hd / 16 * 18) : 0;
    const long claims = (long)launches * DS_CLAIMS;
    Tensor work = torch::full({claims + DS_STATE + (long)L * a.stride + parts},
                              -1,
                              xd.options().dtype(torch::kInt32));
    unsigned* words = reinterpret_cast<unsigned*>(work.data_ptr());
    a.state = words + claims;
    a.words = a.state + DS_STATE;
    a.parts = a.words + (long)L * a.stride;
    TORCH_CHECK(absent >= 0 && absent < DS_WGS && patience >= 1 &&
                patience <= DS_PATIENCE);
    for (int i = 0; i < launches; ++i)
        for (int c = DS_WGS - absent; c < DS_WGS; ++c) {
            work[(long)i * DS_CLAIMS + c].zero_();
            work[(long)i * DS_CLAIMS + DS_WGS + c % 8 * 32].add_(1);
        }
    a.patience = 31;                           // (see decode_stack.h)
    while (a.patience < patience - 1) a.patience = a.patience * 2 + 1;
    if (status.has_value()) {
        TORCH_CHECK(status->device().is_cpu() && status->numel() == 1 &&
                    status->scalar_type() == torch::kInt32 &&
                    status->is_pinned(), "status: one pinned int32");
        a.status = status->data_ptr<int>();
    }
    Tensor x32 = torch::empty({M, H}, xd.options().dtype(torch::kFloat32));
    Tensor out = torch::empty({M, H}, xd.options());
    a.x = ptr(xd);
    a.x32 = x32.data_ptr<float>();
    a.out = reinterpret_cast<unsigned*>(out.data_ptr());

    std::vector<StackLayer> told(L + 1);
    std::vector<Tensor> kept;                  // copies of what is not dense
    auto keep = [&](const Tensor& t) {
        kept.push_back(t);
        return ptr(t);
    };
    for (int l = 0; l < L; ++l) {
        const auto& t = layers[l];
        TORCH_CHECK(t.size() == 14);
        StackLayer& s = told[l];
        for (int k = 0; k < 4; ++k) {
            const Tensor w = dense(t[k].value(), "weights");
            TORCH_CHECK(w.dim() == 2 && w.size(0) == rows[k] &&
                        w.size(1) == K[k], "sizes of the layer's products");
            s.w[k] = keep(w);
            TORCH_CHECK(k != DS_UP || gelu || !t[4 + k].has_value());
            s.bias[k] = keep(column(t[4 + k], rows[k], "bias"));
        }
        for (int i = 0; i < 2; ++i) {
            TORCH_CHECK(t[8 + i].has_value() &&
                        t[10 + i].has_value() == norm_b, "norms");
            s.norm[i] = keep(column(t[8 + i], H, "norm weight"));
            s.norm_bias[i] = keep(column(t[10 + i], H, "norm bias"));
        }
        for (int i = 12; i < 14; ++i) {
            const Tensor& c = t[i].value();
            TORCH_CHECK(c.is_cuda() && c.sizes() == k0.sizes() &&
                        c.scalar_type() == k0.scalar_type() &&
                        c.is_contiguous() &&
                        reinterpret_cast<uintptr_t>(c.data_ptr()) % 16 == 0,
                        "pages");
            (i == 12 ? s.k_cache : s.v_cache) = c.data_ptr();
        }
    }
    for (int i = 0; i < launches; ++i) {
        a.lo = i * DS_LAYERS;
        a.hi = std::min(L, a.lo + DS_LAYERS);
        a.claims = words + (long)i * DS_CLAIMS;
        std::copy(told.begin() + a.lo, told.begin() + a.hi + 1, a.layer);
        TORCH_CHECK(launch_decode_stack(&a, hd, fp8, norm_b, (int)wgs,
                                        stream()) == 0);
    }
    return out;
}

// parts [S, M, N] fp32, whose sum over S is x w^T
Tensor mid_linear(const Tensor& x, const Tensor& w) {
    TORCH_CHECK(x.dim() == 2 && w.dim() == 2 && x.size(1) == w.size(1),
                "x [M, K] and w [N, K]");
    const int M = x.size(0), K = x.size(1), N = w.size(0);
    TORCH_CHECK(M >= 1 && M <= 256, "1 to 256 rows");
    TORCH_CHECK(K % 64 == 0 && N % 4 == 0);
    const Tensor xd = dense(x, "x"), wd = dense(w, "w");
    const int S = linear_mid_splits(N, K);
    Tensor part = torch::empty({S, M, N},
                               x.options().dtype(torch::kFloat32));
    TORCH_CHECK(launch_linear_mid(ptr(xd), ptr(wd), nullptr, part.data_ptr(),
                                  M, N, K, S, 0, 0, nullptr, 0.f, stream()) == 0);
    return part;
}

// act(x w^T + bias) in bf16; act swiglu: w holds the gate's rows, then the
// values'
Tensor mid_rows_linear(const Tensor& x, const Tensor& w,
                       const optional<Tensor>& bias, int64_t act) {
    TORCH_CHECK(x.dim() == 2 && w.dim() == 2 && x.size(1) == w.size(1),
                "x [M, K] and w [N, K]");
    TORCH_CHECK(act == EPI_PLAIN || act == EPI_GLU || act == EPI_GELU);
    const bool glu = act == EPI_GLU;
    TORCH_CHECK(!glu || (w.size(0) % 16 == 0 && !bias.has_value()));
    const int M = x.size(0), K = x.size(1), N = w.size(0) / (glu ? 2 : 1);
    TORCH_CHECK(M >= 1 && M <= 256, "1 to 256 rows");
    TORCH_CHECK(K % 64 == 0 && N % 4 == 0);
    const Tensor xd = dense(x, "x"), wd = dense(w, "w"),
                 b = column(bias, N, "bias");
    Tensor y = torch::empty({M, N}, xd.options());
    TORCH_CHECK(launch_linear_mid(ptr(xd), ptr(wd), ptr(b), y.data_ptr(), M,
                                  N, K, 1, glu ? 1 : 2, act == EPI_GELU,
                                  nullptr, 0.f, stream()) == 0);
    return y;
}

// Wide products: forms of linear_wide.hip
enum { WIDE_ROWS = 0, WIDE_GATED = 1, WIDE_PARTS = 2 };

int64_t wide_plan(int64_t M, int64_t N, int64_t K, int64_t form) {
    TORCH_CHECK(form >= WIDE_ROWS && form <= WIDE_PARTS);
    const int64_t most = std::numeric_limits<int>::max();
    if (M > most || N > most || K > most) return 0;
    return linear_wide_plan(M, N, K, form);
}

// rows of a tile of that plan
int64_t wide_height(int64_t M, int64_t N, int64_t K, int64_t plan, bool gated) {
    TORCH_CHECK(M >= 1 && plan % 8 >= 2 && plan % 8 <= 4 && plan >= 8);
    return linear_wide_rows(M, N, K, plan / 8 % 16,
                            gated ? WIDE_GATED : WIDE_ROWS, plan % 8);
}

// x w^T in bf16; silu(gate) * value of w's two halves (gated); or, where the
// plan has several parts, [S, M, N] fp32
Tensor wide_linear(const Tensor& x, const Tensor& w, int64_t plan,
                   bool gated) {
    TORCH_CHECK(x.dim() == 2 && w.dim() == 2 && x.size(1) == w.size(1),
                "x [M, K] and w [N, K]");
    const int64_t tall = plan % 8, S = plan / 8 % 16;
    TORCH_CHECK(tall >= 2 && tall <= 4 && S >= 1 && S <= 8, "a plan");
    TORCH_CHECK(!gated || (S == 1 && w.size(0) % 16 == 0));
    TORCH_CHECK(x.size(0) >= 1 && x.size(1) % 64 == 0 &&
                x.size(1) >= 128 * S && w.size(0) % 8 == 0);
    const Tensor xd = dense(x, "x"), wd = dense(w, "w");
    const int M = x.size(0), K = x.size(1), N = w.size(0) / (gated ? 2 : 1);
    const int form = gated ? WIDE_GATED : S > 1 ? WIDE_PARTS : WIDE_ROWS;
    Tensor y = S > 1 ? torch::empty({S, M, N},
                                    x.options().dtype(torch::kFloat32))
                     : torch::empty({M, N}, xd.options());
    // rows past the last whole tile, if the plan has them apart
    const int tail = plan >= 128 ? M % (tall * 64) : 0;
    TORCH_CHECK(plan < 256 && (tail == 0 || (S == 1 && tail < M)), "a plan");
    TORCH_CHECK(launch_linear_wide(ptr(xd), ptr(wd), y.data_ptr(), M - tail,
                                   N, K, S, form,
                                   linear_wide_rows(M - tail, N, K, S, form,
                                                    tall),
                                   stream()) == 0);
    if (tail)
        TORCH_CHECK(launch_linear_mid(
                        ptr(xd) + (long)(M - tail) * K, ptr(wd), nullptr,
                        mut(y) + (long)(M - tail) * N, tail, N, K, 1,
                        gated ? 1 : 2, 0, nullptr, 0.f, stream()) == 0);
    return y;
}

const float* parts(const Tensor& t, long M, long N) {
    TORCH_CHECK(t.is_cuda() && t.scalar_type() == torch::kFloat32 &&
                t.is_contiguous() && t.dim() == 3 && t.size(1) == M &&
                t.size(2) == N, "parts [S, M, N] fp32");
    return t.data_ptr<float>();
}

// -> norm(resid + sum of the parts + bias) (undefined without a norm), and
// that sum in bf16 or fp32; resid is either
std::vector<optional<Tensor>> add_norm_parts(
    const Tensor& part, const optional<Tensor>& bias, const Tensor& resid,
    const optional<Tensor>& norm_w, const optional<Tensor>& norm_b,
    double eps, bool sum32) {
    TORCH_CHECK(resid.dim() == 2);
    TORCH_CHECK(norm_w.has_value() || !norm_b.has_value());
    const int M = resid.size(0), H = resid.size(1);
    TORCH_CHECK(M >= 1 && H % 8 == 0 && H <= 8192);
    const Tensor r = dense(resid, "resid", true), b = column(bias, H, "bias"),
                 nw = column(norm_w, H, "norm weight"),
                 nb = column(norm_b, H, "norm bias");
    const auto bf16 = r.options().dtype(torch::kBFloat16);
    Tensor sum = torch::empty({M, H}, sum32 ? r.options().dtype(torch::kFloat32)
                                            : bf16), y;
    if (norm_w.has_value()) y = torch::empty({M, H}, bf16);
    TORCH_CHECK(launch_add_norm_parts(
                    parts(part, M, H), ptr(b), r.data_ptr(), is_f32(r), ptr(nw),
                    ptr(nb), sum.data_ptr(), sum32,
                    y.defined() ? mut(y) : nullptr, M, H,
                    part.size(0), (float)eps, stream()) == 0);
    return {y.defined() ? optional<Tensor>(y) : optional<Tensor>(), sum};
}

// qkv: the projection's bf16 rows [T, N], changed in place, or its fp32 parts
// [S, T, N]; -> [T, N] with bias added and q, k rotated; k, v also stored
Tensor rope_store_qkv(const Tensor& qkv, const optional<Tensor>& bias,
                      int64_t nq, const optional<Tensor>& pos,
                      const optional<Tensor>& cos_t,
                      const optional<Tensor>& sin_t, Tensor& k_cache,
                      Tensor& v_cache, const Tensor& slots) {
    const bool split = qkv.dim() == 3;
    const long T = qkv.size(-2), N = qkv.size(-1);
    const bool fp8 = k_cache.scalar_type() == torch::kUInt8;
    TORCH_CHECK(k_cache.dim() == 4 && k_cache.sizes() == v_cache.sizes() &&
                k_cache.scalar_type() == v_cache.scalar_type() &&
                k_cache.is_contiguous() && v_cache.is_contiguous());
    TORCH_CHECK(fp8 || k_cache.scalar_type() == torch::kBFloat16);
    const int nkv = k_cache.size(1), bs = k_cache.size(2),
              hd = k_cache.size(3);
    TORCH_CHECK(hd % 16 == 0 && N == (nq + 2 * nkv) * hd);
    TORCH_CHECK(slots.scalar_type() == torch::kInt32 &&
                slots.is_contiguous() && slots.numel() == T);
    Turns by;
    if (pos.has_value()) {
        TORCH_CHECK(pos->scalar_type() == torch::kInt32 &&
                    pos->is_contiguous() && pos->numel() == T);
        by = turns(cos_t, sin_t, hd);
    }
    const Tensor b = column(bias, N, "bias");
    const float* p = split ? parts(qkv, T, N) : nullptr;
    Tensor out = split ? torch::empty({T, N}, qkv.options().dtype(
                                                  torch::kBFloat16))
                       : dense(qkv, "qkv");
    TORCH_CHECK(launch_qkv_rope_store(
                    p, split ? qkv.size(0) : 0, mut(out), ptr(b),
                    pos.has_value() ? pos->data_ptr<int>() : nullptr,
                    by.cos_t, by.sin_t, by.rows,
                    k_cache.data_ptr(), v_cache.data_ptr(),
                    slots.data_ptr<int>(), T, nq, nkv, hd, bs, fp8,
                    stream()) == 0);
    return out;
}

void check_decode(const Tensor& table, const Tensor& pos, int64_t bs) {
    TORCH_CHECK(table.is_cuda() && table.scalar_type() == torch::kInt32 &&
                table.dim() == 2 && table.stride(1) == 1);
    TORCH_CHECK(pos.is_cuda() && pos.scalar_type() == torch::kInt32 &&
                pos.is_contiguous() && pos.dim() == 1 &&
                pos.size(0) <= table.size(0) && bs > 0);
}

Tensor decode_slots(const Tensor& table, const Tensor& pos, int64_t bs) {
    check_decode(table, pos, bs);
    Tensor slots = torch::empty_like(pos);
    launch_decode_slots(table.data_ptr<int>(), pos.data_ptr<int>(),
                        slots.data_ptr<int>(), pos.size(0), table.size(1),
                        table.stride(0), bs, stream());
    return slots;
}

// the same, and the rows by length, longest first
std::vector<Tensor> decode_plan(const Tensor& table, const Tensor& pos,
                                int64_t bs, const Tensor& lens) {
    check_decode(table, pos, bs);
    TORCH_CHECK(lens.is_cuda() && lens.scalar_type() == torch::kInt32 &&
                lens.is_contiguous() && lens.dim() == 1 &&
                lens.size(0) >= pos.size(0), "lengths of the rows");
    Tensor slots = torch::empty_like(pos), order = torch::empty_like(pos);
    TORCH_CHECK(launch_decode_plan(table.data_ptr<int>(), pos.data_ptr<int>(),
                                   slots.data_ptr<int>(), lens.data_ptr<int>(),
                                   order.data_ptr<int>(), pos.size(0),
                                   table.size(1), table.stride(0), bs,
                                   stream()) == 0, "1 to 2048 rows");
    return {slots, order};
}

// [T, H] bf16 = embed[ids] + pos_embed[pos]
Tensor embed_positions(const Tensor& ids, const Tensor& embed,
                       const Tensor& pos, const Tensor& pos_embed) {
    TORCH_CHECK(ids.is_cuda() && ids.scalar_type() == torch::kInt64 &&
                ids.is_contiguous() && ids.dim() == 1);
    TORCH_CHECK(pos.is_cuda() && pos.scalar_type() == torch::kInt32 &&
                pos.is_contiguous() && pos.sizes() == ids.sizes());
    const Tensor e = dense(embed, "embed"), p = dense(pos_embed, "pos_embed");
    TORCH_CHECK(e.dim() == 2 && p.dim() == 2 && e.size(1) == p.size(1) &&
                e.size(1) % 8 == 0);
    Tensor out = torch::empty({ids.size(0), e.size(1)}, e.options());
    launch_embed_positions(reinterpret_cast<const long*>(ids.data_ptr()),
                           ptr(e), pos.data_ptr<int>(), ptr(p), mut(out),
                           ids.size(0), e.size(1), e.size(0), p.size(0),
                           stream());
    return out;
}

}  // namespace

void register_rows_ops(pybind11::module_& m) {
    m.def("rows_linear", &rows_linear,
          "projection of a few rows: norm, product, bias, activation, residual");
    m.def("rows_sum", &rows_sum,
          "the same without activation, and what the next RMS norm takes");
    m.def("rows_qkv", &rows_qkv,
          "norm, q|k|v projection, rotation and page store of a few rows");
    m.def("stack_rows", &stack_rows,
          "most rows of a decode step whose layers are one launch");
    m.def("decode_stack", &decode_stack, "the layers of a decode step");
    m.def("mid_linear", &mid_linear,
          "projection of some tens of rows as fp32 parts over K");
    m.def("mid_rows_linear", &mid_rows_linear,
          "projection of some tens of rows, with bias and activation");
    m.def("wide_plan", &wide_plan,
          "tile and parts of a projection of many rows, 0 for the library");
    m.def("wide_height", &wide_height, "rows of a tile of a plan");
    m.def("wide_linear", &wide_linear,
          "projection of many rows, gated or as parts where wanted");
    m.def("add_norm_parts", &add_norm_parts,
          "residual add of a projection's parts, and the next norm");
    m.def("decode_slots", &decode_slots, "page slots of a decode step's rows");
    m.def("decode_plan", &decode_plan,
          "page slots of a decode step's rows, and the rows by length");
    m.def("embed_positions", &embed_positions,
          "token and learned position embeddings, added");
    m.def("rope_store_qkv", &rope_store_qkv,
          "bias, rotation and page store of q|k|v rows or parts");
}
