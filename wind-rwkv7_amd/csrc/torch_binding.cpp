// The eager path of the Python operators in native code: checks, allocation, autograd nodes and launches.
//
// A pass through the Python autograd Functions costs some 200 us of host time per forward + backward (seven views and
// their nodes, a dozen Python allocations, argument conversion for three library calls with up to 35 pointers), more
// than the kernels of the headline shape need; here the same work is one call of a few microseconds each way.  The
// kernels stay behind the C ABI (include/wind_rwkv7.h): this file only calls it, through the library the Python side has
// loaded.  Every function returns None when its arguments are not the plain case (contiguous tensors of the expected
// types on one GPU, supported sizes); the caller then takes the Python path, which names what is wrong, pads a LoRA rank,
// and so on, and which is also what torch.compile traces.
#include <dlfcn.h>

#include <ATen/ATen.h>
#include <ATen/TensorSubclassLikeUtils.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/utils/pybind.h>

#include "../../include/wind_rwkv7.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::Variable;
using torch::autograd::variable_list;
namespace py = pybind11;

#define WIND_SYMBOLS(X)                                                                                              \
    X(strerror) X(checkpoint_interval) X(head_size_supported) X(attn_head_size_supported)                            \
    X(attn_saved_bytes) X(attn_fwd_workspace_bytes) X(attn_bwd_workspace_bytes)                                      \
    X(attn_forward) X(attn_prefill) X(attn_backward)                                                                 \
    X(attn_ln_saved_bytes) X(attn_ln_fwd_workspace_bytes) X(attn_ln_bwd_workspace_bytes)                             \
    X(attn_ln_forward) X(attn_ln_prefill) X(attn_ln_backward)                                                        \
    X(attn_f32_saved_bytes) X(attn_f32_forward) X(attn_f32_prefill) X(attn_f32_backward)                             \
    X(ddlerp_bwd_workspace_bytes) X(ddlerp_forward) X(ddlerp_backward)                                               \
    X(expand_loras_bwd_workspace_bytes) X(expand_loras_forward) X(expand_loras_backward) X(cast_to_bf16)

struct Lib {
#define X(name) decltype(&wind_rwkv7_##name) name = nullptr;
    WIND_SYMBOLS(X)
#undef X
} L;

void load(const std::string& path) {
    void* handle = dlopen(path.c_str(), RTLD_NOW | RTLD_LOCAL);
    TORCH_CHECK(handle, "cannot load ", path, ": ", dlerror());
#define X(name)                                                                                       \
    L.name = reinterpret_cast<decltype(L.name)>(dlsym(handle, "wind_rwkv7_" #name));                  \
    TORCH_CHECK(L.name, path, " has no wind_rwkv7_" #name);
    WIND_SYMBOLS(X)
#undef X
}

void check(int code) { TORCH_CHECK(code == 0, "wind_rwkv7 error ", code, ": ", L.strerror(code)); }

void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

// A tensor the kernels can take as it is: dense, contiguous, on a GPU, no subclass and no transform around it.
bool plain(const Tensor& t, at::ScalarType dtype) {
    return t.defined() && t.is_cuda() && t.scalar_type() == dtype && t.layout() == at::kStrided && !at::isTensorSubclassLike(t) &&
           t.is_contiguous();
}
bool plain_like(const Tensor& t, const Tensor& like) {
    return plain(t, like.scalar_type()) && t.device() == like.device() && t.sizes() == like.sizes();
}
bool plain_param(const Tensor& t, const Tensor& like) {   // a float32 or bf16 parameter beside the sequence `like`
    return t.defined() && (plain(t, at::kFloat) || plain(t, at::kBFloat16)) && t.device() == like.device();
}

bool differentiating(std::initializer_list<const Tensor*> ts) {
    if (!at::GradMode::is_enabled()) return false;
    for (const Tensor* t : ts)
        if (t->defined() && t->requires_grad()) return true;
    return false;
}

Tensor scratch_bytes(size_t n, const Tensor& like) {
    return at::empty({(int64_t)std::max<size_t>(n, 256)}, like.options().dtype(at::kByte));
}
void* ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
int state_code(const Tensor& t) { return t.defined() && t.scalar_type() == at::kFloat ? WIND_RWKV7_F32 : WIND_RWKV7_BF16; }
Tensor contiguous_or_zeros(const Tensor& g, const Tensor& like) { return g.defined() ? g.contiguous() : at::zeros_like(like); }

struct Shape {
    int B, T, H, C;
};
// [B,T,H*C] -> sizes, or B = 0 where the index ranges of the C ABI (int) do not hold
Shape shape_of(const Tensor& t, int64_t C) {
    const auto s = t.sizes();
    constexpr int64_t most = std::numeric_limits<int>::max();
    if (t.dim() != 3 || C <= 0 || C > most || s[2] % C || s[0] > most || s[1] > most || s[2] > most) return {0, 0, 0, 0};
    return {(int)s[0], (int)s[1], (int)(s[2] / C), (int)C};
}

// (In the autograd nodes the sequences stand in the C ABI's order w, q, k, v, a, b; needs_input_grad counts tensors only.)
// ------------------------------------------------------------------------------------------------
// WKV7 on bf16 sequences
// ------------------------------------------------------------------------------------------------
struct Kept {   // what an autograd node keeps besides tensors
    Shape s;
    int interval;
    at::ScalarType state_type;
    bool has_s0;
};
void keep(AutogradContext* ctx, const Kept& k) {
    ctx->saved_data["k"] = std::vector<int64_t>{k.s.B, k.s.T, k.s.H, k.s.C, k.interval, (int64_t)k.state_type, k.has_s0};
}
Kept kept(AutogradContext* ctx) {
    const auto v = ctx->saved_data["k"].toIntVector();
    return {{(int)v[0], (int)v[1], (int)v[2], (int)v[3]}, (int)v[4], (at::ScalarType)v[5], v[6] != 0};
}
void same_interval(const Kept& k) {
    const int now = L.checkpoint_interval();
    TORCH_CHECK(now == k.interval, "checkpoint interval changed between forward (", k.interval, ") and backward (", now,
                "): set it between whole forward + backward passes only");
}

struct Wkv7 : torch::autograd::Function<Wkv7> {
    static variable_list run(const Shape& s, const Tensor& w, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& a,
                             const Tensor& b, const Tensor& s0, Tensor* saved) {
        Tensor y = at::empty_like(v);
        Tensor sT = at::empty({s.B, s.H, s.C, s.C}, s0.defined() ? s0.options() : v.options());
        // one allocation for the saved tensor and the forward's scratch behind it (both are multiples of 256 bytes)
        const size_t ws = std::max<size_t>(L.attn_fwd_workspace_bytes(s.B, s.T, s.H, s.C), 256);
        const size_t keep_bytes = saved ? (L.attn_saved_bytes(s.B, s.T, s.H, s.C) + 255) / 256 * 256 : 0;
        Tensor mem = scratch_bytes(keep_bytes + ws, v);
        char* base = static_cast<char*>(mem.data_ptr());
        check((saved ? L.attn_forward : L.attn_prefill)(
            s.B, s.T, s.H, s.C, WIND_RWKV7_BF16, state_code(s0), ptr(w), ptr(q), ptr(k), ptr(v), ptr(a), ptr(b), ptr(s0), ptr(y),
            base, ptr(sT), base + keep_bytes, ws, stream_of(v)));
        if (saved) *saved = mem;
        return {y, sT};
    }
    // (a node takes no undefined tensor: without an initial state `state` is any tensor)
    static variable_list forward(AutogradContext* ctx, Shape s, bool has_s0, const Tensor& w, const Tensor& q, const Tensor& k,
                                 const Tensor& v, const Tensor& a, const Tensor& b, const Tensor& state) {
        Tensor saved;
        variable_list out = run(s, w, q, k, v, a, b, has_s0 ? state : Tensor(), &saved);
        ctx->set_materialize_grads(false);
        ctx->save_for_backward({w, q, k, v, a, b, saved});
        keep(ctx, {s, L.checkpoint_interval(), out[1].scalar_type(), has_s0});
        return out;
    }
    static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
        const auto t = ctx->get_saved_variables();
        const Kept kp = kept(ctx);
        const Shape& s = kp.s;
        same_interval(kp);
        c10::DeviceGuard guard(t[0].device());
        const Tensor dy = contiguous_or_zeros(grads[0], t[3]);
        const Tensor dsT = grads[1].defined() ? grads[1].contiguous() : Tensor();
        variable_list d(6);
        for (auto& g : d) g = at::empty_like(t[3]);
        Tensor ds0;
        if (kp.has_s0 && ctx->needs_input_grad(6)) ds0 = at::empty({s.B, s.H, s.C, s.C}, t[3].options().dtype(kp.state_type));
        const size_t ws = L.attn_bwd_workspace_bytes(s.B, s.T, s.H, s.C);
        const Tensor mem = scratch_bytes(ws, dy);
        check(L.attn_backward(s.B, s.T, s.H, s.C, WIND_RWKV7_BF16, kp.state_type == at::kFloat ? WIND_RWKV7_F32 : WIND_RWKV7_BF16,
                              ptr(t[0]), ptr(t[1]), ptr(t[2]), ptr(t[3]), ptr(t[4]), ptr(t[5]), ptr(dy), ptr(t[6]), ptr(dsT), ptr(d[0]),
                              ptr(d[1]), ptr(d[2]), ptr(d[3]), ptr(d[4]), ptr(d[5]), ptr(ds0), ptr(mem), mem.numel(), stream_of(dy)));
        return {Tensor(), Tensor(), d[0], d[1], d[2], d[3], d[4], d[5], ds0};
    }
};

// ------------------------------------------------------------------------------------------------
// WKV7 on float32 sequences
// ------------------------------------------------------------------------------------------------
struct Wkv7F32 : torch::autograd::Function<Wkv7F32> {
    static variable_list run(const Shape& s, const Tensor& w, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& a,
                             const Tensor& b, const Tensor& s0, Tensor* saved) {
        Tensor y = at::empty_like(v), sT = at::empty_like(s0);
        if (saved) {
            *saved = scratch_bytes(L.attn_f32_saved_bytes(s.B, s.T, s.H, s.C), v);
            check(L.attn_f32_forward(s.B, s.T, s.H, s.C, ptr(w), ptr(q), ptr(k), ptr(v), ptr(a), ptr(b), ptr(s0), ptr(y), ptr(*saved),
                                     ptr(sT), stream_of(v)));
        } else {
            check(L.attn_f32_prefill(s.B, s.T, s.H, s.C, ptr(w), ptr(q), ptr(k), ptr(v), ptr(a), ptr(b), ptr(s0), ptr(y), ptr(sT),
                                     stream_of(v)));
        }
        return {y, sT};
    }
    static variable_list forward(AutogradContext* ctx, Shape s, const Tensor& w, const Tensor& q, const Tensor& k, const Tensor& v,
                                 const Tensor& a, const Tensor& b, const Tensor& s0) {
        Tensor saved;
        variable_list out = run(s, w, q, k, v, a, b, s0, &saved);
        ctx->set_materialize_grads(false);
        ctx->save_for_backward({w, q, k, v, a, b, saved});
        keep(ctx, {s, 0, at::kFloat, true});
        return out;
    }
    static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
        const auto t = ctx->get_saved_variables();
        const Shape s = kept(ctx).s;
        c10::DeviceGuard guard(t[0].device());
        const Tensor dy = contiguous_or_zeros(grads[0], t[3]);
        const Tensor dsT = grads[1].defined() ? grads[1].contiguous() : at::zeros({s.B, s.H, s.C, s.C}, t[3].options());
        variable_list d(6);
        for (auto& g : d) g = at::empty_like(t[3]);
        Tensor ds0 = at::empty_like(dsT);
        check(L.attn_f32_backward(s.B, s.T, s.H, s.C, ptr(t[0]), ptr(t[1]), ptr(t[2]), ptr(t[3]), ptr(t[4]), ptr(t[5]), ptr(dy), ptr(t[6]),
                                  ptr(dsT), ptr(d[0]), ptr(d[1]), ptr(d[2]), ptr(d[3]), ptr(d[4]), ptr(d[5]), ptr(ds0), stream_of(dy)));
        return {Tensor(), d[0], d[1], d[2], d[3], d[4], d[5], ds0};
    }
};

py::object attn(const Tensor& r, const Tensor& w, const Tensor& k, const Tensor& v, const Tensor& a, const Tensor& b,
                int64_t head_size, const std::optional<Tensor>& s0_, bool return_state) {
    if (!w.defined() || (w.scalar_type() != at::kBFloat16 && w.scalar_type() != at::kFloat)) return py::none();
    const bool f32 = w.scalar_type() == at::kFloat;
    if (!plain(w, w.scalar_type())) return py::none();
    for (const Tensor* t : {&r, &k, &v, &a, &b})
        if (!plain_like(*t, w)) return py::none();
    const Shape s = shape_of(w, head_size);
    if (s.B <= 0 || !(f32 ? L.attn_f32_saved_bytes : L.attn_saved_bytes)(s.B, s.T, s.H, s.C)) return py::none();
    Tensor s0 = s0_.value_or(Tensor());
    if (s0.defined()) {
        if (!(plain(s0, at::kFloat) || (!f32 && plain(s0, at::kBFloat16))) || s0.device() != w.device() ||
            s0.sizes() != at::IntArrayRef({s.B, s.H, s.C, s.C}))
            return py::none();
    }
    c10::DeviceGuard guard(w.device());
    if (f32 && !s0.defined()) s0 = at::zeros({s.B, s.H, s.C, s.C}, w.options());
    variable_list out;
    if (differentiating({&r, &w, &k, &v, &a, &b, &s0}))
        out = f32 ? Wkv7F32::apply(s, w, r, k, v, a, b, s0) : Wkv7::apply(s, s0.defined(), w, r, k, v, a, b, s0.defined() ? s0 : w);
    else
        out = f32 ? Wkv7F32::run(s, w, r, k, v, a, b, s0, nullptr) : Wkv7::run(s, w, r, k, v, a, b, s0, nullptr);
    if (return_state) return py::make_tuple(out[0], out[1]);
    return py::cast(out[0]);
}

// ------------------------------------------------------------------------------------------------
// WKV7 with the GroupNorm + bonus + gate epilogue
// ------------------------------------------------------------------------------------------------
struct Wkv7Ln : torch::autograd::Function<Wkv7Ln> {
    static variable_list run(const Shape& s, const Tensor& w, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& a,
                             const Tensor& b, const Tensor& g, const Tensor& params, const Tensor& s0, Tensor* saved) {
        Tensor y = at::empty_like(v);
        Tensor sT = at::empty({s.B, s.H, s.C, s.C}, s0.defined() ? s0.options() : v.options());
        const size_t ws = std::max<size_t>(L.attn_ln_fwd_workspace_bytes(s.B, s.T, s.H, s.C), 256);
        const size_t keep_bytes = (L.attn_ln_saved_bytes(s.B, s.T, s.H, s.C) + 255) / 256 * 256;
        Tensor mem = scratch_bytes(keep_bytes + ws, v);
        char* base = static_cast<char*>(mem.data_ptr());
        check((saved ? L.attn_ln_forward : L.attn_ln_prefill)(
            s.B, s.T, s.H, s.C, WIND_RWKV7_BF16, state_code(s0), ptr(w), ptr(q), ptr(k), ptr(v), ptr(a), ptr(b), ptr(g), ptr(params),
            ptr(s0), ptr(y), base, ptr(sT), base + keep_bytes, ws, stream_of(v)));
        if (saved) *saved = mem;
        return {y, sT};
    }
    static variable_list forward(AutogradContext* ctx, Shape s, bool has_s0, const Tensor& w, const Tensor& q, const Tensor& k,
                                 const Tensor& v, const Tensor& a, const Tensor& b, const Tensor& g, const Tensor& params,
                                 const Tensor& state) {
        Tensor saved;
        variable_list out = run(s, w, q, k, v, a, b, g, params, has_s0 ? state : Tensor(), &saved);
        ctx->set_materialize_grads(false);
        ctx->save_for_backward({w, q, k, v, a, b, g, params, saved});
        keep(ctx, {s, L.checkpoint_interval(), out[1].scalar_type(), has_s0});
        return out;
    }
    static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
        const auto t = ctx->get_saved_variables();
        const Kept kp = kept(ctx);
        const Shape& s = kp.s;
        same_interval(kp);
        c10::DeviceGuard guard(t[0].device());
        const Tensor dy = contiguous_or_zeros(grads[0], t[3]);
        const Tensor dsT = grads[1].defined() ? grads[1].contiguous() : Tensor();
        variable_list d(7);
        for (auto& x : d) x = at::empty_like(t[3]);
        Tensor dparams = at::empty_like(t[7]), ds0;
        if (kp.has_s0 && ctx->needs_input_grad(8)) ds0 = at::empty({s.B, s.H, s.C, s.C}, t[3].options().dtype(kp.state_type));
        const Tensor mem = scratch_bytes(L.attn_ln_bwd_workspace_bytes(s.B, s.T, s.H, s.C), dy);
        check(L.attn_ln_backward(s.B, s.T, s.H, s.C, WIND_RWKV7_BF16, kp.state_type == at::kFloat ? WIND_RWKV7_F32 : WIND_RWKV7_BF16,
                                 ptr(t[0]), ptr(t[1]), ptr(t[2]), ptr(t[3]), ptr(t[4]), ptr(t[5]), ptr(t[6]), ptr(t[7]), ptr(dy), ptr(t[8]),
                                 ptr(dsT), ptr(d[0]), ptr(d[1]), ptr(d[2]), ptr(d[3]), ptr(d[4]), ptr(d[5]), ptr(d[6]), ptr(dparams), ptr(ds0),
                                 ptr(mem), mem.numel(), stream_of(dy)));
        return {Tensor(), Tensor(), d[0], d[1], d[2], d[3], d[4], d[5], d[6], dparams, ds0};
    }
};

py::object attn_ln(const Tensor& r, const Tensor& w, const Tensor& k, const Tensor& v, const Tensor& a, const Tensor& b,
                   const Tensor& g, const Tensor& params, int64_t head_size, const std::optional<Tensor>& s0_, bool return_state) {
    if (!w.defined() || !plain(w, at::kBFloat16)) return py::none();
    for (const Tensor* t : {&r, &k, &v, &a, &b, &g})
        if (!plain_like(*t, w)) return py::none();
    const Shape s = shape_of(w, head_size);
    if (s.B <= 0 || !L.attn_ln_saved_bytes(s.B, s.T, s.H, s.C)) return py::none();
    if (!plain(params, at::kFloat) || params.device() != w.device() || params.sizes() != at::IntArrayRef({3, (int64_t)s.H * s.C}))
        return py::none();
    const Tensor s0 = s0_.value_or(Tensor());
    if (s0.defined() && (!(plain(s0, at::kFloat) || plain(s0, at::kBFloat16)) || s0.device() != w.device() ||
                         s0.sizes() != at::IntArrayRef({s.B, s.H, s.C, s.C})))
        return py::none();
    c10::DeviceGuard guard(w.device());
    variable_list out;
    if (differentiating({&r, &w, &k, &v, &a, &b, &g, &params, &s0}))
        out = Wkv7Ln::apply(s, s0.defined(), w, r, k, v, a, b, g, params, s0.defined() ? s0 : w);
    else
        out = Wkv7Ln::run(s, w, r, k, v, a, b, g, params, s0, nullptr);
    if (return_state) return py::make_tuple(out[0], out[1]);
    return py::cast(out[0]);
}

// ------------------------------------------------------------------------------------------------
// parameters as bf16, and their gradients
// ------------------------------------------------------------------------------------------------
constexpr int64_t ALIGN_ELEMS_BF16 = 128, ALIGN_ELEMS_F32 = 64;   // 256 bytes
int64_t round_up(int64_t n, int64_t m) { return (n + m - 1) / m * m; }

// bf16 device pointers of the parameters: their own where they are bf16, otherwise into `flat`, which one launch fills
// (in `flat` each starts on a 256-byte boundary).  `flat` given: it was filled by the forward, only the pointers are wanted.
std::vector<void*> bf16_pointers(const std::vector<Tensor>& params, Tensor& flat) {
    std::vector<void*> out;
    bool all_bf16 = true;
    for (const auto& p : params) all_bf16 = all_bf16 && p.scalar_type() == at::kBFloat16;
    if (all_bf16) {
        for (const auto& p : params) out.push_back(p.data_ptr());
        return out;
    }
    std::vector<long long> offset, numel;
    std::vector<const void*> src;
    std::vector<int> dtype;
    long long total = 0;
    for (const auto& p : params) {
        offset.push_back(total);
        numel.push_back(p.numel());
        src.push_back(p.data_ptr());
        dtype.push_back(p.scalar_type() == at::kFloat ? WIND_RWKV7_F32 : WIND_RWKV7_BF16);
        total += round_up(p.numel(), ALIGN_ELEMS_BF16);
    }
    if (!flat.defined()) {
        flat = at::empty({total}, params[0].options().dtype(at::kBFloat16));
        check(L.cast_to_bf16((int)params.size(), src.data(), dtype.data(), numel.data(), offset.data(), flat.data_ptr(), stream_of(flat)));
    }
    for (long long o : offset) out.push_back(static_cast<char*>(flat.data_ptr()) + 2 * o);
    return out;
}

// float32 gradients of tensors of the given shapes in one buffer, and the tensors to hand back: views of it, or of one
// bf16 copy of it where the parameters are bf16.
struct FlatGrads {
    std::vector<std::vector<int64_t>> shapes;
    std::vector<int64_t> offset;
    Tensor flat;
    FlatGrads(std::vector<std::vector<int64_t>> sh, const Tensor& like) : shapes(std::move(sh)) {
        int64_t total = 0;
        for (const auto& s : shapes) {
            offset.push_back(total);
            total += round_up(c10::multiply_integers(s), ALIGN_ELEMS_F32);
        }
        flat = at::empty({total}, like.options().dtype(at::kFloat));
    }
    void* p(size_t i) const { return static_cast<float*>(flat.data_ptr()) + offset[i]; }
    variable_list tensors(at::ScalarType dtype) const {
        const Tensor all = flat.to(dtype);
        variable_list out;
        for (size_t i = 0; i < shapes.size(); i++) {
            std::vector<int64_t> stride(shapes[i].size());
            int64_t n = 1;
            for (size_t d = stride.size(); d-- > 0; n *= shapes[i][d]) stride[d] = n;
            out.push_back(all.as_strided(shapes[i], stride, offset[i]));
        }
        return out;
    }
};

// ------------------------------------------------------------------------------------------------
// ddlerp
// ------------------------------------------------------------------------------------------------
struct DDLerp : torch::autograd::Function<DDLerp> {
    static variable_list forward(AutogradContext* ctx, const Tensor& x, const Tensor& alpha, const Tensor& Lw, const Tensor& R,
                                 const Tensor& beta) {
        at::AutoDispatchBelowADInplaceOrView below;   // (the four outputs are slices of one buffer, not views to autograd)
        const int B = x.size(0), T = x.size(1), C = x.size(2), D = R.size(2);
        Tensor flat;
        const auto p = bf16_pointers({alpha, Lw, R, beta}, flat);
        Tensor y = at::empty({4, B, T, C}, x.options()), mid = at::empty({2, B, T, 4 * D}, x.options());
        void* bder = static_cast<char*>(mid.data_ptr()) + mid.numel();   // the second half (2 bytes an element)
        check(L.ddlerp_forward(B, T, C, D, ptr(x), p[0], p[1], p[2], p[3], ptr(mid), bder, ptr(y), stream_of(x)));
        ctx->save_for_backward({x, alpha, Lw, R, beta, flat, mid});
        return {y.select(0, 0), y.select(0, 1), y.select(0, 2), y.select(0, 3)};
    }
    static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
        const auto t = ctx->get_saved_variables();
        const Tensor& x = t[0];
        const int B = x.size(0), T = x.size(1), C = x.size(2), D = t[3].size(2);
        c10::DeviceGuard guard(x.device());
        Tensor flat = t[5], dy[4];
        const auto p = bf16_pointers({t[1], t[2], t[3], t[4]}, flat);
        for (int i = 0; i < 4; i++) dy[i] = contiguous_or_zeros(grads[i], x);
        Tensor dx = at::empty_like(x);
        const FlatGrads g({{C}, {4 * D, C}, {4, C, D}, {4, 1, 1, C}}, x);
        const Tensor ws = scratch_bytes(L.ddlerp_bwd_workspace_bytes(B, T, C, D), x);
        const Tensor& mid = t[6];
        check(L.ddlerp_backward(B, T, C, D, ptr(x), p[0], p[1], p[2], p[3], ptr(mid), static_cast<char*>(mid.data_ptr()) + mid.numel(),
                                ptr(dy[0]), ptr(dy[1]), ptr(dy[2]), ptr(dy[3]), ptr(dx), g.p(0), g.p(1), g.p(2), g.p(3), ptr(ws),
                                ws.numel(), stream_of(x)));
        variable_list out = g.tensors(t[1].scalar_type());
        out.insert(out.begin(), dx);
        return out;
    }
};

py::object ddlerp(const Tensor& x, const Tensor& alpha, const Tensor& Lw, const Tensor& R, const Tensor& beta) {
    if (!x.defined() || !plain(x, at::kBFloat16) || x.dim() != 3 || R.dim() != 3) return py::none();
    const Shape s = shape_of(x, x.size(2));
    const int64_t C = s.C, D = R.size(2);
    if (s.B <= 0 || (D != 32 && D != 64) || !L.ddlerp_bwd_workspace_bytes(s.B, s.T, s.C, (int)D)) return py::none();
    for (const Tensor* t : {&alpha, &Lw, &R, &beta})
        if (!plain_param(*t, x) || t->scalar_type() != alpha.scalar_type()) return py::none();
    if (alpha.sizes() != at::IntArrayRef({C}) || Lw.sizes() != at::IntArrayRef({4 * D, C}) || R.sizes() != at::IntArrayRef({4, C, D}) ||
        beta.sizes() != at::IntArrayRef({4, 1, 1, C}))
        return py::none();
    c10::DeviceGuard guard(x.device());
    const variable_list y = DDLerp::apply(x, alpha, Lw, R, beta);
    return py::make_tuple(y[0], y[1], y[2], y[3]);
}

// ------------------------------------------------------------------------------------------------
// expand_loras: 0 w_in, 1 k_in, 2-5 the activations z, a, ma, mk, 6-9 their weights, 10-13 the biases w, a, ma, mk
// ------------------------------------------------------------------------------------------------
struct ExpandLoras : torch::autograd::Function<ExpandLoras> {
    template <class... Ts>
    static variable_list forward(AutogradContext* ctx, int64_t head_size, const Ts&... tensors) {
        at::AutoDispatchBelowADInplaceOrView below;
        const variable_list in{tensors...};
        const int B = in[0].size(0), T = in[0].size(1), C = in[0].size(2), D = in[2].size(2);
        variable_list save(in);
        for (int i = 2; i < 6; i++) save[i] = in[i].contiguous();
        Tensor flat;
        const auto p = bf16_pointers(std::vector<Tensor>(in.begin() + 6, in.end()), flat);
        variable_list out(4);
        for (auto& o : out) o = at::empty_like(in[0]);
        check(L.expand_loras_forward(B, T, C, D, (int)head_size, ptr(in[0]), ptr(in[1]), ptr(save[2]), ptr(save[3]), ptr(save[4]),
                                     ptr(save[5]), p[0], p[1], p[2], p[3], p[4], p[5], p[6], p[7], ptr(out[0]), ptr(out[1]), ptr(out[2]),
                                     ptr(out[3]), stream_of(in[0])));
        save.push_back(flat);
        ctx->save_for_backward(save);
        ctx->saved_data["head_size"] = head_size;
        return out;
    }
    static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
        const auto in = ctx->get_saved_variables();
        const int B = in[0].size(0), T = in[0].size(1), C = in[0].size(2), D = in[2].size(2);
        c10::DeviceGuard guard(in[0].device());
        Tensor flat = in[14], dy[4];
        const auto p = bf16_pointers(std::vector<Tensor>(in.begin() + 6, in.begin() + 14), flat);
        for (int i = 0; i < 4; i++) dy[i] = contiguous_or_zeros(grads[i], in[0]);
        variable_list d(6);
        for (int i = 0; i < 6; i++) d[i] = at::empty_like(in[i]);
        const FlatGrads g({{C, D}, {C, D}, {C, D}, {C, D}, {C}, {C}, {C}, {C}}, in[0]);
        const Tensor ws = scratch_bytes(L.expand_loras_bwd_workspace_bytes(B, T, C, D), in[0]);
        check(L.expand_loras_backward(
            B, T, C, D, (int)ctx->saved_data["head_size"].toInt(), ptr(in[0]), ptr(in[1]), ptr(in[2]), ptr(in[3]), ptr(in[4]), ptr(in[5]),
            p[0], p[1], p[2], p[3], p[4], p[5], p[6], p[7], ptr(dy[0]), ptr(dy[1]), ptr(dy[2]), ptr(dy[3]), ptr(d[0]), ptr(d[1]), ptr(d[2]),
            ptr(d[3]), ptr(d[4]), ptr(d[5]), g.p(0), g.p(1), g.p(2), g.p(3), g.p(4), g.p(5), g.p(6), g.p(7), ptr(ws), ws.numel(),
            stream_of(in[0])));
        variable_list out{Tensor()};
        out.insert(out.end(), d.begin(), d.end());
        for (auto& t : g.tensors(in[6].scalar_type())) out.push_back(t);
        return out;
    }
};

template <size_t... I>
variable_list expand_loras_node(int64_t head_size, const variable_list& in, std::index_sequence<I...>) {
    return ExpandLoras::apply(head_size, in[I]...);
}

py::object expand_loras(const variable_list& in, int64_t head_size) {
    if (in.size() != 14) return py::none();
    const Tensor& w = in[0];
    if ( !w.defined() || !plain(w, at::kBFloat16) || !plain_like(in[1], w) || in[2].dim() != 3) return py::none();
    const Shape s = shape_of(w, head_size);
    const int64_t C = s.H * (int64_t)s.C, D = in[2].size(2);
    if (s.B <= 0 || C % 64 || head_size % 16 || (D != 16 && D != 32 && D != 64)) return py::none();
    if (!L.expand_loras_bwd_workspace_bytes(s.B, s.T, (int)C, (int)D)) return py::none();
    for (int i = 2; i < 6; i++) {   // (the activations may be strided: they are made contiguous)
        const Tensor& t = in[i];
        if (!t.defined() || !t.is_cuda() || t.scalar_type() != at::kBFloat16 || t.layout() != at::kStrided || at::isTensorSubclassLike(t) ||
            t.device() != w.device() || t.sizes() != at::IntArrayRef({s.B, s.T, D}))
            return py::none();
    }
    for (int i = 6; i < 14; i++)
        if (!plain_param(in[i], w) || in[i].scalar_type() != in[6].scalar_type() ||
            in[i].sizes() != (i < 10 ? at::IntArrayRef({C, D}) : at::IntArrayRef({C})))
            return py::none();
    c10::DeviceGuard guard(w.device());
    const variable_list y = expand_loras_node(head_size, in, std::make_index_sequence<14>());
    return py::make_tuple(y[0], y[1], y[2], y[3]);
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
    m.def("load", &load);
    m.def("attn", &attn);
    m.def("attn_ln", &attn_ln);
    m.def("ddlerp", &ddlerp);
    m.def("expand_loras", &expand_loras);
}
