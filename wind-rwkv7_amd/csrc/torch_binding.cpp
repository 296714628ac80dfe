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
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/pybind.h>
#include <torch/version.h>

#include "../../include/wind_rwkv7.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::Variable;
using torch::autograd::variable_list;
namespace py = pybind11;

#define WIND_SYMBOLS(X)                                                                                              \
    X(strerror) X(checkpoint_interval) X(head_size_supported) X(attn_head_size_supported)                            \
    X(attn_saved_bytes) X(attn_fwd_workspace_bytes) X(attn_train_workspace_bytes) X(attn_bwd_workspace_bytes)        \
    X(attn_forward) X(attn_prefill) X(attn_backward)                                                                 \
    X(attn_ln_saved_bytes) X(attn_ln_bwd_workspace_bytes)                                                            \
    X(attn_ln_forward) X(attn_ln_prefill) X(attn_ln_prefill_ragged) X(attn_ln_backward)                                                        \
    X(attn_f32_saved_bytes) X(attn_f32_forward) X(attn_f32_prefill) X(attn_f32_backward_split)                       \
    X(attn_f32_bwd_workspace_bytes)                                                                                  \
    X(ddlerp_bwd_workspace_bytes) X(ddlerp_forward) X(ddlerp_backward)                                               \
    X(expand_loras_bwd_workspace_bytes) X(expand_loras_forward) X(expand_loras_forward_padded) X(expand_loras_backward) X(cast_to_bf16)             \
    X(ddlerp_first_workspace_bytes) X(ddlerp_first) X(attn_ln_tokens) X(pad_rows) X(linear_wgrad_workspace_bytes) X(linear_wgrad)           \
    X(block_wgrads_workspace_bytes) X(block_wgrads) X(mixer_decode_workspace_bytes) X(mixer_decode) \
    X(mixer_prompt) X(linear_group) X(pack_weights) X(pack_weights_pad_rows) X(expand_loras_backward_to)

struct Lib {
#define X(name) decltype(&wind_rwkv7_##name) name = nullptr;
    WIND_SYMBOLS(X)
#undef X
} L;

PyObject* error_class = nullptr;   // WindRwkv7Error(code, message); kept for good

void load(const std::string& path, const py::object& error) {
    void* handle = dlopen(path.c_str(), RTLD_NOW | RTLD_LOCAL);
    TORCH_CHECK(handle, "cannot load ", path, ": ", dlerror());
#define X(name)                                                                                       \
    L.name = reinterpret_cast<decltype(L.name)>(dlsym(handle, "wind_rwkv7_" #name));                  \
    TORCH_CHECK(L.name, path, " has no wind_rwkv7_" #name);
    WIND_SYMBOLS(X)
#undef X
    error_class = py::object(error).release().ptr();
}

// An entry point's error as the Python class, out of a call as out of a backward pass (autograd's engine takes a python_error
// to the thread that waits for it).
void check(int code) {
    if (code == 0) return;
    py::gil_scoped_acquire gil;
    const py::object error = py::reinterpret_borrow<py::object>(error_class)(code, L.strerror(code));
    PyErr_SetObject(error_class, error.ptr());
    python_error e;
    e.persist();
    throw e;
}

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

bool aligned(const Tensor& t) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0; }
// x in bf16, dense and where 16-byte accesses may go (a view may start anywhere)
Tensor dense_bf16(const Tensor& x) {
    const Tensor t = x.to(at::kBFloat16).contiguous();
    return aligned(t) ? t : t.clone();
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

// The forward's saved tensor and its scratch: two allocations where the scratch is large, so that a node keeps what its backward pass
// reads and no more (1 x 1536 tokens x 64 heads 63 MB instead of 142), and the second as large as the backward's workspace where they are of a
// size, so that the pool hands it on.  Forward + backward in a captured pass, us, one allocation / two / two of a size: 1 x 2048 x 40 152 / 160 /
// 149 (the gradients get the scratch's memory where the sizes differ), 1 x 1536 x 64 173 / 176 / 150, 1 x 2560 x 20 146 / - / 135, attn_ln 4 x 1024 x 12
// 132 / 132 / 123; eager the same.
// One allocation below 32 MiB, what the L2s of the eight XCDs hold together: there memory that another XCD has just used costs more
// than it saves (1 x 1536 x 8 heads 76.5 / - / 82.7, 1 x 1536 x 16 83.5 / - / 86.5).  And at other head sizes, whose states are five times the
// records: 8 x 1024 x 6 of 128 226 / 240 / 226, 2 x 512 x 6 77 / 77 / 84.
struct ForwardMemory {
    Tensor kept, own;
    void* workspace;
    size_t bytes;
    ForwardMemory(const Shape& s, size_t saved_bytes, size_t backward_bytes, bool saves, const Tensor& like)
        : bytes(std::max<size_t>((saves ? L.attn_train_workspace_bytes : L.attn_fwd_workspace_bytes)(s.B, s.T, s.H, s.C), 256)) {
        const size_t first = (saved_bytes + 255) / 256 * 256;
        const bool apart = saves && bytes > 32 << 20 && L.head_size_supported(s.C);
        kept = scratch_bytes(first + (apart ? 0 : bytes), like);
        if (apart) own = scratch_bytes(backward_bytes <= 2 * bytes ? std::max(bytes, backward_bytes) : bytes, like);
        workspace = apart ? ptr(own) : static_cast<char*>(ptr(kept)) + first;
    }
};

struct Wkv7 : torch::autograd::Function<Wkv7> {
    static variable_list run(const Shape& s, const Tensor& w, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& a,
                             const Tensor& b, const Tensor& s0, Tensor* saved) {
        Tensor y = at::empty_like(v);
        Tensor sT = at::empty({s.B, s.H, s.C, s.C}, s0.defined() ? s0.options() : v.options());
        const ForwardMemory mem(s, saved ? L.attn_saved_bytes(s.B, s.T, s.H, s.C) : 0, L.attn_bwd_workspace_bytes(s.B, s.T, s.H, s.C), saved, v);
        check((saved ? L.attn_forward : L.attn_prefill)(
            s.B, s.T, s.H, s.C, WIND_RWKV7_BF16, state_code(s0), ptr(w), ptr(q), ptr(k), ptr(v), ptr(a), ptr(b), ptr(s0), ptr(y),
            ptr(mem.kept), ptr(sT), mem.workspace, mem.bytes, stream_of(v)));
        if (saved) *saved = mem.kept;
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
        const Tensor mem = scratch_bytes(L.attn_bwd_workspace_bytes(s.B, s.T, s.H, s.C), dy);   // (ahead of the gradients: see ForwardMemory)
        variable_list d(6);
        for (auto& g : d) g = at::empty_like(t[3]);
        Tensor ds0;
        if (kp.has_s0 && ctx->needs_input_grad(6)) ds0 = at::empty({s.B, s.H, s.C, s.C}, t[3].options().dtype(kp.state_type));
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
        const Tensor mem = scratch_bytes(L.attn_f32_bwd_workspace_bytes(s.B, s.T, s.H, s.C), t[3]);
        check(L.attn_f32_backward_split(s.B, s.T, s.H, s.C, ptr(t[0]), ptr(t[1]), ptr(t[2]), ptr(t[3]), ptr(t[4]), ptr(t[5]), ptr(dy), ptr(t[6]),
                                  ptr(dsT), ptr(d[0]), ptr(d[1]), ptr(d[2]), ptr(d[3]), ptr(d[4]), ptr(d[5]), ptr(ds0), ptr(mem), mem.numel(),
                                        stream_of(dy)));
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
        const ForwardMemory mem(s, L.attn_ln_saved_bytes(s.B, s.T, s.H, s.C), L.attn_ln_bwd_workspace_bytes(s.B, s.T, s.H, s.C), saved, v);
        check((saved ? L.attn_ln_forward : L.attn_ln_prefill)(
            s.B, s.T, s.H, s.C, WIND_RWKV7_BF16, state_code(s0), ptr(w), ptr(q), ptr(k), ptr(v), ptr(a), ptr(b), ptr(g), ptr(params),
            ptr(s0), ptr(y), ptr(mem.kept), ptr(sT), mem.workspace, mem.bytes, stream_of(v)));
        if (saved) *saved = mem.kept;
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
        const Tensor mem = scratch_bytes(L.attn_ln_bwd_workspace_bytes(s.B, s.T, s.H, s.C), dy);
        variable_list d(7);
        for (auto& x : d) x = at::empty_like(t[3]);
        Tensor dparams = at::empty_like(t[7]), ds0;
        if (kp.has_s0 && ctx->needs_input_grad(8)) ds0 = at::empty({s.B, s.H, s.C, s.C}, t[3].options().dtype(kp.state_type));
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

// The parameters as bf16: the tensors themselves where all of them are, and aligned, otherwise copies in one buffer that one
// launch fills (each on a 256-byte boundary).  A node saves what it multiplied - `saved` - and not a parameter it has a copy
// of, which may be written to before the backward pass.
struct Bf16Params {
    variable_list own;   // the parameters, or none
    Tensor flat;         // the copies, or undefined
    explicit Bf16Params(const variable_list& params) {
        bool direct = true;
        for (const auto& p : params) direct = direct && p.scalar_type() == at::kBFloat16 && aligned(p);
        if (direct) {
            own = params;
            return;
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
        flat = at::empty({total}, params[0].options().dtype(at::kBFloat16));
        check(L.cast_to_bf16((int)params.size(), src.data(), dtype.data(), numel.data(), offset.data(), flat.data_ptr(), stream_of(flat)));
    }
    // from the tail of a node's saved variables: one flat buffer, or the parameters
    Bf16Params(variable_list::const_iterator first, variable_list::const_iterator last) {
        if (last - first == 1) flat = *first;
        else own.assign(first, last);
    }
    variable_list saved() const { return flat.defined() ? variable_list{flat} : own; }
    std::vector<void*> pointers(std::initializer_list<int64_t> numel) const {
        std::vector<void*> out;
        if (!flat.defined())
            for (const auto& p : own) out.push_back(p.data_ptr());
        int64_t o = 0;
        for (int64_t n : numel) {
            if (flat.defined()) out.push_back(static_cast<char*>(flat.data_ptr()) + 2 * o);
            o += round_up(n, ALIGN_ELEMS_BF16);
        }
        return out;
    }
};

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
        const Bf16Params params({alpha, Lw, R, beta});
        const auto p = params.pointers({C, 4 * D * C, 4 * D * C, 4 * C});
        Tensor y = at::empty({4, B, T, C}, x.options()), mid = at::empty({2, B, T, 4 * D}, x.options());
        void* bder = static_cast<char*>(mid.data_ptr()) + mid.numel();   // the second half (2 bytes an element)
        check(L.ddlerp_forward(B, T, C, D, ptr(x), p[0], p[1], p[2], p[3], ptr(mid), bder, ptr(y), stream_of(x)));
        variable_list save{x, mid};
        for (const auto& t : params.saved()) save.push_back(t);
        ctx->save_for_backward(save);
        ctx->saved_data["type"] = alpha.scalar_type();
        return {y.select(0, 0), y.select(0, 1), y.select(0, 2), y.select(0, 3)};
    }
    static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
        const auto t = ctx->get_saved_variables();
        const Tensor& x = t[0];
        const Tensor& mid = t[1];
        const int B = x.size(0), T = x.size(1), C = x.size(2), D = mid.size(3) / 4;
        c10::DeviceGuard guard(x.device());
        Tensor dy[4];
        const auto p = Bf16Params(t.begin() + 2, t.end()).pointers({C, 4 * D * C, 4 * D * C, 4 * C});
        for (int i = 0; i < 4; i++) dy[i] = contiguous_or_zeros(grads[i], x);
        Tensor dx = at::empty_like(x);
        const FlatGrads g({{C}, {4 * D, C}, {4, C, D}, {4, 1, 1, C}}, x);
        const Tensor ws = scratch_bytes(L.ddlerp_bwd_workspace_bytes(B, T, C, D), x);
        check(L.ddlerp_backward(B, T, C, D, ptr(x), p[0], p[1], p[2], p[3], ptr(mid), static_cast<char*>(mid.data_ptr()) + mid.numel(),
                                ptr(dy[0]), ptr(dy[1]), ptr(dy[2]), ptr(dy[3]), ptr(dx), g.p(0), g.p(1), g.p(2), g.p(3), ptr(ws),
                                ws.numel(), stream_of(x)));
        variable_list out = g.tensors(ctx->saved_data["type"].toScalarType());
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
        variable_list save(in.begin(), in.begin() + 6);
        for (int i = 2; i < 6; i++) save[i] = in[i].contiguous();
        const Bf16Params params(variable_list(in.begin() + 6, in.end()));
        const auto p = params.pointers({C * D, C * D, C * D, C * D, C, C, C, C});
        variable_list out(4);
        for (auto& o : out) o = at::empty_like(in[0]);
        check(L.expand_loras_forward(B, T, C, D, (int)head_size, ptr(in[0]), ptr(in[1]), ptr(save[2]), ptr(save[3]), ptr(save[4]),
                                     ptr(save[5]), p[0], p[1], p[2], p[3], p[4], p[5], p[6], p[7], ptr(out[0]), ptr(out[1]), ptr(out[2]),
                                     ptr(out[3]), stream_of(in[0])));
        for (const auto& t : params.saved()) save.push_back(t);
        ctx->save_for_backward(save);
        ctx->saved_data["head_size"] = head_size;
        ctx->saved_data["type"] = in[6].scalar_type();
        return out;
    }
    static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
        const auto in = ctx->get_saved_variables();
        const int B = in[0].size(0), T = in[0].size(1), C = in[0].size(2), D = in[2].size(2);
        c10::DeviceGuard guard(in[0].device());
        Tensor dy[4];
        const auto p = Bf16Params(in.begin() + 6, in.end()).pointers({C * D, C * D, C * D, C * D, C, C, C, C});
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
        for (auto& t : g.tensors(ctx->saved_data["type"].toScalarType())) out.push_back(t);
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

// ------------------------------------------------------------------------------------------------
// TimeMixer: the whole block as one node (training), as one call (prompts) and one token at a time
// ------------------------------------------------------------------------------------------------
// The block's parameters: the weights in the order of wind_rwkv7_mixer_weights, then the GroupNorm's and the bonus.
enum Param {
    MAA_X, MAA, MAA_W1, MAA_W2, WR, WK, WV, WO, GATE_W1, DECAY_W1, KKK_W1, MK_W1, AAA_W1, MA_W1, GATE_W2, DECAY_W2, KKK_W2,
    MK_W2, AAA_W2, MA_W2, DECAY, AAAAA, MISC_A, MISC_K, LN_W, LN_B, FAAAA, PARAMS
};
constexpr int WEIGHTS = LN_W;   // the ones whose bf16 copies the kernels take
const char* const PARAM_NAMES[PARAMS] = {
    "time_maa_x", "time_maa", "time_maa_w1", "time_maa_w2", "Wr", "Wk", "Wv", "Wo", "gate_w1", "time_decay_w1", "time_kkk_w1",
    "mk_w1", "time_aaa_w1", "ma_w1", "gate_w2", "time_decay_w2", "time_kkk_w2", "mk_w2", "time_aaa_w2", "ma_w2", "time_decay",
    "time_aaaaa", "time_misc_a", "time_misc_k", "weight", "bias", "time_faaaa"};
constexpr int R_MIX = 32, R_DECAY = 64, R_GATE = 128, R_LORA = 16;   // LoRA ranks (time_mixer.py:69-94); R_LORA: aaa, kkk, ma, mk
constexpr int W_KKMK = 2 * R_LORA, W_DECAY_AAA_MA = R_DECAY + 2 * R_LORA;

std::vector<int64_t> param_shape(int i, int64_t C) {
    switch (i) {
        case MAA: return {4, 1, 1, C};
        case MAA_W1: return {4 * R_MIX, C};
        case MAA_W2: return {4, C, R_MIX};
        case WR: case WK: case WV: case WO: return {C, C};
        case GATE_W1: return {R_GATE, C};
        case DECAY_W1: return {R_DECAY, C};
        case KKK_W1: case MK_W1: case AAA_W1: case MA_W1: return {R_LORA, C};
        case GATE_W2: return {C, R_GATE};
        case DECAY_W2: return {C, R_DECAY};
        case KKK_W2: case MK_W2: case AAA_W2: case MA_W2: return {C, R_LORA};
        default: return {C};
    }
}
// Where each parameter lies in a buffer of all of them, in elements.  Every piece is a multiple of 64 elements, so the two
// concatenated first halves [kkk; mk] and [decay; aaa; ma] are one matrix each and the GroupNorm's weight, bias and the
// bonus are the [3, C] tensor of attn_ln.
struct ParamLayout {
    int64_t at[PARAMS + 1];
    explicit ParamLayout(int64_t C) {
        static const int order[PARAMS] = {WR, WK, WV, WO, GATE_W1, KKK_W1, MK_W1, DECAY_W1, AAA_W1, MA_W1, GATE_W2, DECAY_W2, MAA_W1,
                                          MAA_W2, KKK_W2, MK_W2, AAA_W2, MA_W2, MAA_X, MAA, DECAY, AAAAA, MISC_A, MISC_K, LN_W, LN_B, FAAAA};
        int64_t o = 0;
        for (int i : order) {
            at[i] = o;
            o += c10::multiply_integers(param_shape(i, C));
        }
        at[PARAMS] = o;
    }
};

// The weights as the kernels take them, in one buffer (bf16 elements): copies of all of them in ParamLayout's places, the
// [3, C] float32 parameters of attn_ln, and for a backward pass the transposed copies of the projections' weights.
struct WeightLayout {
    ParamLayout at_;
    int64_t C, ln, Tr, Tk, Tv, To, Tg1, Tkkmk, Tw1, Tg2, Tw2, total[2];   // total[whether the transposed copies are there]
    explicit WeightLayout(int64_t C_) : at_(C_), C(C_) {
        int64_t o = at_.at[LN_W];
        auto take = [&](int64_t n) { const int64_t r = o; o += n; return r; };
        ln = take(2 * 3 * C);
        total[0] = o;
        Tr = take(C * C), Tk = take(C * C), Tv = take(C * C), To = take(C * C);
        Tg1 = take(C * R_GATE), Tkkmk = take(C * W_KKMK), Tw1 = take(C * W_DECAY_AAA_MA), Tg2 = take(C * R_GATE), Tw2 = take(C * R_DECAY);
        total[1] = o;
    }
};
using B16 = c10::BFloat16;
B16* at_elem(const Tensor& t, int64_t o) { return static_cast<B16*>(t.data_ptr()) + o; }

// A prompt's rows on their way to whole chunks, in the launch that packs the weights: x [B,T,C] to out, [B,C] of it to last (may be undefined)
struct Padding {
    Tensor x, out, last;
};

void pack_weights(const WeightLayout& L_, const variable_list& p, const Tensor& buf, bool transposed, const Padding& pad = {}) {
    wind_rwkv7_pack t[PARAMS];
    for (int i = 0; i < PARAMS; i++) {
        const auto shape = param_shape(i, L_.C);
        const bool norm = i >= WEIGHTS;
        t[i].src = p[i].data_ptr();
        t[i].src_dtype = p[i].scalar_type() == at::kFloat ? WIND_RWKV7_F32 : WIND_RWKV7_BF16;
        t[i].dst_dtype = norm ? WIND_RWKV7_F32 : WIND_RWKV7_BF16;
        t[i].dst = at_elem(buf, norm ? L_.ln + 2 * (L_.at_.at[i] - L_.at_.at[LN_W]) : L_.at_.at[i]);
        t[i].cols = (int)shape.back();
        t[i].rows = (int)(p[i].numel() / shape.back());
        t[i].dstT = nullptr;
        t[i].ldT = 0;
    }
    if (transposed) {
        auto turn = [&](int i, int64_t at, int64_t ld) { t[i].dstT = at_elem(buf, at), t[i].ldT = ld; };
        turn(WR, L_.Tr, L_.C), turn(WK, L_.Tk, L_.C), turn(WV, L_.Tv, L_.C), turn(WO, L_.To, L_.C);
        turn(GATE_W1, L_.Tg1, R_GATE), turn(GATE_W2, L_.Tg2, L_.C), turn(DECAY_W2, L_.Tw2, L_.C);
        turn(KKK_W1, L_.Tkkmk, W_KKMK), turn(MK_W1, L_.Tkkmk + R_LORA, W_KKMK);
        turn(DECAY_W1, L_.Tw1, W_DECAY_AAA_MA), turn(AAA_W1, L_.Tw1 + R_DECAY, W_DECAY_AAA_MA);
        turn(MA_W1, L_.Tw1 + R_DECAY + R_LORA, W_DECAY_AAA_MA);
    }
    if (pad.x.defined())
        check(L.pack_weights_pad_rows(PARAMS, t, pad.x.size(0), pad.x.size(1), pad.out.size(1), pad.x.size(2), ptr(pad.x), ptr(pad.out), ptr(pad.last),
                                      stream_of(buf)));
    else
        check(L.pack_weights(PARAMS, t, stream_of(buf)));
}

struct Block {   // the sizes of a call
    int64_t B, T, C, H;
    int64_t rows() const { return B * T; }
    int64_t N() const { return C / H; }
    int64_t plane() const { return rows() * C; }
};

// Activations of a block in one buffer; offsets in elements (all multiples of 256: rows() is a multiple of 16).  Where no
// backward pass asks for them, what is made after the streams are multiplied takes their place: nine planes for thirteen.
struct Activations {
    int64_t streams, r, k, v, g, w2, w, k2, kk, b, mid, der, tg1, tw1, kk1, mk1, a1, ma1, total;
    Activations(const Block& s, bool save) {
        int64_t o = 0;
        auto take = [&](int64_t n) { const int64_t r = o; o += n; return r; };
        const int64_t M = s.rows(), P = s.plane();
        streams = take(4 * P);
        r = take(P), k = take(P), v = take(P), kk = take(P), b = take(P);
        g = save ? take(P) : streams, w2 = save ? take(P) : streams + P, w = save ? take(P) : streams + 2 * P;
        k2 = save ? take(P) : streams + 3 * P;
        mid = take(4 * R_MIX * M), der = take(4 * R_MIX * M);
        tg1 = take(R_GATE * M), tw1 = take(R_DECAY * M);
        kk1 = take(R_LORA * M), mk1 = take(R_LORA * M), a1 = take(R_LORA * M), ma1 = take(R_LORA * M);
        total = o;
    }
};

// Products out = in W^T on the same rows in one launch (wind_rwkv7_linear_group).  The library's kernel for a single large
// product is the better one by a quarter where each fills the chip several times over, so there a large product goes to it.
// Measured, us for three C x C products as one group / as three library calls, at 1.2e10, 2.5e10 and 1e11 rows x columns x
// contraction length each: C = 512 114/166, 237/204; 768 84/78, 189/143, 720/589; 1536 79/82, 156/124, 637/480; 2048 80/98,
// 175/133, 627/497; 4096 96/95, 178/146, 649/470.  A second segment is a second library call that reads the result back and
// adds to it in bf16; here it is more of the same sum (one product, 128 indices in the second segment, own / library): C =
// 768 71/83, 1024 76/88, 1536 64/63, 2048 78/58, 4096 88/62 at 2.5e10, so with one it takes a contraction of 2048 as well.
struct Products {
    static constexpr double LIBRARY_FROM = 2.5e10;   // rows x columns x contraction length
    static constexpr int LIBRARY_FROM_K = 2048;      // with a second segment
    std::vector<wind_rwkv7_linear> ps;
    void add(const void* in, const void* W, int64_t K, int64_t N) {
        wind_rwkv7_linear p{};
        p.A[0] = in, p.W[0] = W, p.lda[0] = p.ldw[0] = K, p.K[0] = (int)K;
        p.N = (int)N;
        ps.push_back(p);
    }
    void plus(const void* in, const void* W, int64_t K) {
        auto& p = ps.back();
        p.A[1] = in, p.W[1] = W, p.lda[1] = p.ldw[1] = K, p.K[1] = (int)K;
    }
    void to(void* out, int64_t width, int op = 0, const void* aux = nullptr, int64_t ld = 0) {
        auto& p = ps.back();
        const int t = p.npieces++;
        p.out[t] = out, p.width[t] = (int)width, p.ld_out[t] = ld ? ld : width, p.op[t] = op, p.aux[t] = aux;
    }
    void run(int64_t rows, const Tensor& like) {
        std::vector<wind_rwkv7_linear> group;
        for (const auto& p : ps) {
            if ((double)rows * p.N * p.K[0] < LIBRARY_FROM || (p.K[1] && p.K[0] < LIBRARY_FROM_K) || p.npieces > 1 || p.op[0]) {
                group.push_back(p);
                continue;
            }
            auto view = [&](const void* q, int64_t r, int64_t c) { return at::from_blob(const_cast<void*>(q), {r, c}, like.options()); };
            Tensor out = view(p.out[0], rows, p.N);
            at::mm_out(out, view(p.A[0], rows, p.K[0]), view(p.W[0], p.N, p.K[0]).t());
            if (p.K[1]) at::addmm_out(out, out, view(p.A[1], rows, p.K[1]), view(p.W[1], p.N, p.K[1]).t());
        }
        if (!group.empty()) check(L.linear_group((int)group.size(), rows, group.data(), stream_of(like)));
    }
};

// dW = dy^T x for several pairs on the same tokens, the output projection's first (a single pair goes through its own entry point).
// Whatever runs on its own leaves fp32 partial tiles from every compute unit, 147 KB each, which are written and read again: a 768 x 768 product
// of 8192 tokens is 22 us + 8 of sums for 12 us of products.  So all of a pass go together, unless the grid that makes falls badly on
// the compute units: that is decided behind the entry point (first_alone in linear_wgrad.hip).
struct WeightGrads {
    std::vector<int> O, I;
    std::vector<const void*> dy, x;
    std::vector<long long> ld_dy, ld_x;
    std::vector<void*> dW;
    void add(const void* d, int o, const void* a, int i, void* w) {
        dy.push_back(d), O.push_back(o), ld_dy.push_back(o), x.push_back(a), I.push_back(i), ld_x.push_back(i), dW.push_back(w);
    }
    void run(int64_t tokens, const Tensor& like, void* stream) {
        const int n = (int)O.size();
        if (n == 0) return;
        if (n == 1) {
            const Tensor ws = scratch_bytes(L.linear_wgrad_workspace_bytes(tokens, O[0], I[0]), like);
            check(L.linear_wgrad(tokens, O[0], I[0], dy[0], ld_dy[0], x[0], ld_x[0], dW[0], WIND_RWKV7_F32, ptr(ws), ws.numel(), stream));
            return;
        }
        const Tensor ws = scratch_bytes(L.block_wgrads_workspace_bytes(n, tokens, O.data(), I.data()), like);
        check(L.block_wgrads(n, tokens, O.data(), I.data(), dy.data(), ld_dy.data(), x.data(), ld_x.data(), dW.data(), WIND_RWKV7_F32,
                             ptr(ws), ws.numel(), stream));
    }
};

// What a forward pass leaves: the caller's results and what a backward pass needs.
struct BlockBuffers {
    Tensor weights, acts, saved, ya, y, sT;   // ya: what the output projection multiplies
    static int64_t saved_bytes(const Block& s) { return L.attn_ln_saved_bytes(s.B, s.T, s.H, s.N()); }
    BlockBuffers(const Block& s, const Tensor& xb, bool save, int64_t valid, at::ScalarType state_type) {
        weights = at::empty({WeightLayout(s.C).total[save]}, xb.options());
        acts = at::empty({Activations(s, save).total}, xb.options());
        saved = scratch_bytes(saved_bytes(s), xb);
        ya = at::empty({s.plane()}, xb.options());
        y = at::empty({s.B, valid, s.C}, xb.options());
        sT = at::empty({s.B, s.H, s.N(), s.N()}, xb.options().dtype(state_type));
    }
    BlockBuffers(Tensor w, Tensor a, Tensor s, Tensor ya_, Tensor y_, Tensor st)
        : weights(std::move(w)), acts(std::move(a)), saved(std::move(s)), ya(std::move(ya_)), y(std::move(y_)), sT(std::move(st)) {}
};

// A continued sequence's first token and the carried one before it, both float32 or both bf16 (no defined tensors: there is
// none).  Its streams are made in fp32 on the parameters themselves.
struct First {
    Tensor x, prev;   // [B,C], x's rows anywhere
    First() = default;
    First(const Tensor& x_first, const Tensor& x_prev) : x(x_first), prev(x_prev) {
        if (x.scalar_type() != at::kBFloat16 || prev.scalar_type() != at::kBFloat16) x = x.to(at::kFloat), prev = prev.to(at::kFloat);
        if (x.stride(1) != 1) x = x.contiguous();
        prev = prev.contiguous();
    }
    // y[k * y_stream + b * y_seq ..]: stream k of sequence b
    void streams(const variable_list& p, void* y, int64_t y_stream, int64_t y_seq) const {
        const int B = x.size(0), C = x.size(1);
        Tensor w[4] = {p[MAA_X], p[MAA_W1], p[MAA_W2], p[MAA]};
        bool f32 = false;
        for (const auto& t : w) f32 = f32 || t.scalar_type() == at::kFloat;
        if (f32)
            for (auto& t : w) t = t.to(at::kFloat);
        const wind_rwkv7_first_tokens t{ptr(x),      ptr(prev), ptr(w[0]), ptr(w[1]),       ptr(w[2]), ptr(w[3]),
                                        x.stride(0), y_stream,  y_seq,     state_code(x), state_code(w[0])};
        const Tensor ws = scratch_bytes(L.ddlerp_first_workspace_bytes(B, R_MIX), x);
        check(L.ddlerp_first(B, C, R_MIX, &t, y, ptr(ws), ws.numel(), stream_of(x)));
    }
};

// x [B,T,C] bf16 contiguous, T a multiple of 16.  `save`: keep what the backward needs.  `first` / s0: a carried state
// (undefined: zero).  `valid` < T (head size 64, not with `save`): the tokens from there on are padding, y has none of
// them.  The sequence kernels then take the whole chunks and leave the tokens after them to attn_ln_prefill_ragged's second half, which keeps the
// state in fp32 from token to token (a chunk's products would round those tokens' share of it to bf16 operands).
void block_forward(const Block& s, const Tensor& xb, const variable_list& p, bool save, int64_t valid, const First& first,
                   const Tensor& s0, const BlockBuffers& f, const Padding& pad = {}) {
    const int B = s.B, T = s.T, C = s.C, H = s.H, N = s.N();
    const int64_t M = s.rows(), P = s.plane();
    void* stream = stream_of(xb);
    const WeightLayout W(C);
    const Activations A(s, save);
    pack_weights(W, p, f.weights, save, pad);
    auto a = [&](int64_t o) -> void* { return at_elem(f.acts, o); };
    auto w = [&](int i) -> void* { return at_elem(f.weights, W.at_.at[i]); };
    check(L.ddlerp_forward(B, T, C, R_MIX, ptr(xb), w(MAA_X), w(MAA_W1), w(MAA_W2), w(MAA), a(A.mid), a(A.der), a(A.streams), stream));
    if (first.x.defined()) first.streams(p, a(A.streams), P, (int64_t)T * C);
    const void *xrg = a(A.streams), *xwa = a(A.streams + P), *xk = a(A.streams + 2 * P), *xv = a(A.streams + 3 * P);
    {
        Products halves;
        halves.add(xrg, w(WR), C, C), halves.to(a(A.r), C);
        halves.add(xk, w(WK), C, C), halves.to(a(A.k), C);
        halves.add(xv, w(WV), C, C), halves.to(a(A.v), C);
        halves.add(xrg, w(GATE_W1), C, R_GATE), halves.to(a(A.tg1), R_GATE, 1);
        halves.add(xwa, w(DECAY_W1), C, W_DECAY_AAA_MA);
        halves.to(a(A.tw1), R_DECAY, 1), halves.to(a(A.a1), R_LORA), halves.to(a(A.ma1), R_LORA);
        halves.add(xk, w(KKK_W1), C, W_KKMK), halves.to(a(A.kk1), R_LORA), halves.to(a(A.mk1), R_LORA);
        halves.run(M, xb);
        Products second;
        second.add(a(A.tg1), w(GATE_W2), R_GATE, C), second.to(a(A.g), C);
        second.add(a(A.tw1), w(DECAY_W2), R_DECAY, C), second.to(a(A.w2), C);
        second.run(M, xb);
    }
    const int whole = (int)(valid / 16 * 16), rest = (int)(valid - whole);
    Tensor kept;
    if (rest && whole) kept = at::empty({3, B, T - whole, C}, xb.options());   // (T is valid rounded up: the last chunk)
    check(L.expand_loras_forward_padded(B, T, C, R_LORA, N, a(A.w2), a(A.k), a(A.kk1), a(A.a1), a(A.ma1), a(A.mk1), w(KKK_W2), w(AAA_W2),
                                        w(MA_W2), w(MK_W2), w(DECAY), w(AAAAA), w(MISC_A), w(MISC_K), a(A.w), a(A.k2), a(A.kk), a(A.b),
                                        kept.defined() ? ptr(kept) : nullptr, stream));
    if (whole && rest) {
        const Tensor ws = scratch_bytes(L.attn_fwd_workspace_bytes(B, T, H, N), xb);
        check(L.attn_ln_prefill_ragged(B, T, H, N, rest, state_code(f.sT), a(A.w), a(A.r), a(A.k2), a(A.v), a(A.kk), a(A.b), a(A.g),
                                       at_elem(f.weights, W.ln), ptr(kept), ptr(s0), ptr(f.ya), ptr(f.saved), ptr(f.sT), ptr(ws), ws.numel(), stream));
    } else if (whole) {
        const Tensor ws = scratch_bytes((save ? L.attn_train_workspace_bytes : L.attn_fwd_workspace_bytes)(B, T, H, N), xb);
        check((save ? L.attn_ln_forward : L.attn_ln_prefill)(
            B, T, H, N, WIND_RWKV7_BF16, state_code(f.sT), a(A.w), a(A.r), a(A.k2), a(A.v), a(A.kk), a(A.b), a(A.g), at_elem(f.weights, W.ln),
            ptr(s0), ptr(f.ya), ptr(f.saved), ptr(f.sT), ptr(ws), ws.numel(), stream));
    } else {   // (fewer tokens than a chunk)
        check(L.attn_ln_tokens(B, T, H, N, 0, rest, state_code(f.sT), a(A.w), a(A.r), a(A.k2), a(A.v), a(A.kk), a(A.b), a(A.g),
                               at_elem(f.weights, W.ln), T, 0, ptr(s0), ptr(f.ya), ptr(f.sT), stream));
    }
    Products out;
    if (!rest) {
        out.add(ptr(f.ya), w(WO), C, C), out.to(ptr(f.y), C);
        out.run(M, xb);
    } else if (B <= WIND_RWKV7_LINEAR_GROUP_MAX) {   // a product per sequence: one launch, each straight to its place
        for (int64_t b = 0; b < B; b++) out.add(at_elem(f.ya, b * T * C), w(WO), C, C), out.to(at_elem(f.y, b * valid * C), C);
        out.run(valid, xb);
    } else {
        out.add(ptr(f.ya), w(WO), C, C), out.to(a(A.w), C);   // (w is done with)
        out.run(M, xb);
        check(L.pad_rows(B, T, (int)valid, C, a(A.w), ptr(f.y), nullptr, stream));
    }
}

// The stages of a backward pass that the wanted gradients ask for; need(i): parameter i's is wanted, x: the input's.
struct Stages {
    bool streams, gate, decay, expand, attn;   // down to: the four streams, the first halves of gate and decay, the LoRA expansion, WKV7
    template <class Need>
    Stages(bool x, const Need& need) {
        auto any = [&](std::initializer_list<int> is) {
            for (int i : is)
                if (need(i)) return true;
            return false;
        };
        streams = x || any({MAA_X, MAA, MAA_W1, MAA_W2});
        gate = streams || need(GATE_W1);
        decay = streams || any({DECAY_W1, AAA_W1, MA_W1});
        expand = decay || any({WK, KKK_W1, MK_W1, DECAY_W2, KKK_W2, AAA_W2, MA_W2, MK_W2, DECAY, AAAAA, MISC_A, MISC_K});
        attn = gate || expand || any({WR, WV, GATE_W2, LN_W, LN_B, FAAAA});
    }
};

// Where the gradients lie, float32: the wanted ones in one buffer, in `at` from its start (the matrices that one product
// computes together are neighbours, wanted or not); the others that a stage writes all the same behind them, in a scratch
// buffer (offsets from `kept` on).
struct GradLayout {
    int64_t at[PARAMS], kept = 0, total = 0;
    template <class Need>
    GradLayout(int64_t C, const Need& need) {
        static const std::vector<int> groups[] = {{WR}, {WK}, {WV}, {WO}, {GATE_W1}, {KKK_W1, MK_W1}, {DECAY_W1, AAA_W1, MA_W1}, {GATE_W2}, {DECAY_W2},
                                                  {MAA_W1}, {MAA_W2}, {KKK_W2}, {MK_W2}, {AAA_W2}, {MA_W2}, {MAA_X}, {MAA}, {DECAY}, {AAAAA}, {MISC_A},
                                                  {MISC_K}, {LN_W, LN_B, FAAAA}};
        for (bool wanted : {true, false}) {
            for (const auto& g : groups) {
                bool any = false;
                for (int i : g) any = any || need(i);
                if (any != wanted) continue;
                // (a weight gradient of the products that nobody wants is not computed)
                if (!wanted && (g[0] == WR || g[0] == WK || g[0] == WV || g[0] == WO || g[0] == GATE_W1 || g[0] == KKK_W1 || g[0] == DECAY_W1 ||
                                g[0] == GATE_W2 || g[0] == DECAY_W2))
                    continue;
                for (int i : g) at[i] = total, total += c10::multiply_integers(param_shape(i, C));
            }
            if (wanted) kept = total;
        }
    }
    // the gradient of parameter i as its caller takes it: a view of the buffer of the wanted ones in that type
    static Tensor view(const Tensor& flat, int i, int64_t C, int64_t offset) {
        const auto shape = param_shape(i, C);
        std::vector<int64_t> stride(shape.size());
        int64_t n = 1;
        for (size_t k = stride.size(); k-- > 0; n *= shape[k]) stride[k] = n;
        return flat.as_strided(shape, stride, offset);
    }
};

// dx and the wanted gradients of the parameters (in `flat`, GradLayout's first `kept` floats); need(i): whether parameter i's
// is wanted.  A stage that nothing wanted lies behind does not run; without Stages::attn only ya is there to go back through.
template <class Need>
void block_backward(const Block& s, const Tensor& xb, const Tensor& weights, const Tensor& acts, const Tensor& saved, const Tensor& ya,
                    const Tensor& dout, const Stages& st, const Tensor& dx, const Tensor& flat, const Need& need) {
    const int B = s.B, T = s.T, C = s.C, H = s.H, N = s.N();
    const int64_t M = s.rows(), P = s.plane();
    void* stream = stream_of(dout);
    const GradLayout G(C, need);
    Tensor unwanted;
    auto g = [&](int i) -> void* {
        const bool kept = G.at[i] < G.kept;
        return static_cast<float*>((kept ? flat : unwanted).data_ptr()) + G.at[i] - (kept ? 0 : G.kept);
    };
    WeightGrads wg;   // (run at the end: everything that they multiply is kept until then)
    if (need(WO)) wg.add(ptr(dout), C, ptr(ya), C, g(WO));
    if (!st.attn) {
        wg.run(M, dout, stream);
        return;
    }
    if (G.total > G.kept) unwanted = at::empty({G.total - G.kept}, flat.options());
    const WeightLayout W(C);
    const Activations A(s, true);
    // gradients of activations: nine planes, reused as they are consumed, and the gradients of the three first halves
    const int64_t o_g1 = 9 * P, o_kkmk = o_g1 + R_GATE * M, o_w1 = o_kkmk + W_KKMK * M, total = o_w1 + W_DECAY_AAA_MA * M;
    const Tensor buf = at::empty({total}, xb.options());
    auto a = [&](int64_t o) -> void* { return at_elem(acts, o); };
    auto d = [&](int64_t o) -> void* { return at_elem(buf, o); };
    auto w = [&](int i) -> void* { return at_elem(weights, W.at_.at[i]); };
    auto t = [&](int64_t o) -> void* { return at_elem(weights, o); };
    size_t ws_bytes = L.attn_ln_bwd_workspace_bytes(B, T, H, N);
    if (st.expand) ws_bytes = std::max(ws_bytes, L.expand_loras_bwd_workspace_bytes(B, T, C, R_LORA));
    if (st.streams) ws_bytes = std::max(ws_bytes, L.ddlerp_bwd_workspace_bytes(B, T, C, R_MIX));
    const Tensor ws = scratch_bytes(ws_bytes, xb);

    // planes: 0 dya then dw2, 1 dr, 2 dw, 3 dk', 4 dv, 5 dkk, 6 db, 7 dg, 8 dk
    {
        Products p;
        p.add(ptr(dout), t(W.To), C, C), p.to(d(0), C);
        p.run(M, xb);
    }
    check(L.attn_ln_backward(B, T, H, N, WIND_RWKV7_BF16, WIND_RWKV7_BF16, a(A.w), a(A.r), a(A.k2), a(A.v), a(A.kk), a(A.b), a(A.g), t(W.ln), d(0),
                             ptr(saved), nullptr, d(2 * P), d(P), d(3 * P), d(4 * P), d(5 * P), d(6 * P), d(7 * P), g(LN_W), nullptr, ptr(ws),
                             ws.numel(), stream));
    B16 *dkkmk = at_elem(buf, o_kkmk), *dw1 = at_elem(buf, o_w1);
    const long long ld_din[4] = {W_KKMK, W_DECAY_AAA_MA, W_DECAY_AAA_MA, W_KKMK};
    if (st.expand)
        check(L.expand_loras_backward_to(B, T, C, R_LORA, N, a(A.w2), a(A.k), a(A.kk1), a(A.a1), a(A.ma1), a(A.mk1), w(KKK_W2), w(AAA_W2), w(MA_W2),
                                         w(MK_W2), w(DECAY), w(AAAAA), w(MISC_A), w(MISC_K), d(2 * P), d(3 * P), d(5 * P), d(6 * P), d(0),
                                         d(8 * P), dkkmk, dw1 + R_DECAY, dw1 + R_DECAY + R_LORA, dkkmk + R_LORA, ld_din, g(KKK_W2), g(AAA_W2),
                                         g(MA_W2), g(MK_W2), g(DECAY), g(AAAAA), g(MISC_A), g(MISC_K), ptr(ws), ws.numel(), stream));
    {
        Products p;   // through the derivative of the tanh between the halves
        if (st.gate) p.add(d(7 * P), t(W.Tg2), C, R_GATE), p.to(d(o_g1), R_GATE, 2, a(A.tg1));
        if (st.decay) p.add(d(0), t(W.Tw2), C, R_DECAY), p.to(dw1, R_DECAY, 2, a(A.tw1), W_DECAY_AAA_MA);
        p.run(M, xb);
    }
    // the streams' gradients go to the planes that are free now: 2, 5, 3, 6
    void *dxrg = d(2 * P), *dxwa = d(5 * P), *dxk = d(3 * P), *dxv = d(6 * P);
    {
        Products p;
        if (st.streams) {
            p.add(d(P), t(W.Tr), C, C), p.plus(d(o_g1), t(W.Tg1), R_GATE), p.to(dxrg, C);
            p.add(d(8 * P), t(W.Tk), C, C), p.plus(dkkmk, t(W.Tkkmk), W_KKMK), p.to(dxk, C);
            p.add(d(4 * P), t(W.Tv), C, C), p.to(dxv, C);
            p.add(dw1, t(W.Tw1), W_DECAY_AAA_MA, C), p.to(dxwa, C);
        }
        p.run(M, xb);
    }
    if (need(WR)) wg.add(d(P), C, a(A.streams), C, g(WR));
    if (need(GATE_W1)) wg.add(d(o_g1), R_GATE, a(A.streams), C, g(GATE_W1));
    if (need(WK)) wg.add(d(8 * P), C, a(A.streams + 2 * P), C, g(WK));
    if (need(KKK_W1) || need(MK_W1)) wg.add(dkkmk, W_KKMK, a(A.streams + 2 * P), C, g(KKK_W1));
    if (need(WV)) wg.add(d(4 * P), C, a(A.streams + 3 * P), C, g(WV));
    if (need(DECAY_W1) || need(AAA_W1) || need(MA_W1)) wg.add(dw1, W_DECAY_AAA_MA, a(A.streams + P), C, g(DECAY_W1));
    if (need(GATE_W2)) wg.add(d(7 * P), C, a(A.tg1), R_GATE, g(GATE_W2));
    if (need(DECAY_W2)) wg.add(d(0), C, a(A.tw1), R_DECAY, g(DECAY_W2));
    wg.run(M, xb, stream);
    if (st.streams)
        check(L.ddlerp_backward(B, T, C, R_MIX, ptr(xb), w(MAA_X), w(MAA_W1), w(MAA_W2), w(MAA), a(A.mid), a(A.der), dxrg, dxwa, dxk, dxv, ptr(dx),
                                g(MAA_X), g(MAA_W1), g(MAA_W2), g(MAA), ptr(ws), ws.numel(), stream));
}

struct MixerBlock : torch::autograd::Function<MixerBlock> {
    template <class... Ts>
    static variable_list forward(AutogradContext* ctx, int64_t H, const Tensor& x, const Ts&... params) {
        at::AutoDispatchBelowADInplaceOrView below;
        const Block s{x.size(0), x.size(1), x.size(2), H};
        const variable_list p{params...};
        const Tensor xb = dense_bf16(x);
        const bool attn = Stages(x.requires_grad(), [&](int i) { return p[i].requires_grad(); }).attn;
        const BlockBuffers f(s, xb, attn, s.T, at::kBFloat16);
        block_forward(s, xb, p, attn, s.T, First(), Tensor(), f);
        if (attn) ctx->save_for_backward({f.ya, xb, f.weights, f.acts, f.saved});
        else ctx->save_for_backward({f.ya});
        std::vector<int64_t> kept{s.B, s.T, s.C, H, L.checkpoint_interval(), (int64_t)x.scalar_type()};
        for (const auto& t : p) kept.push_back((int64_t)t.scalar_type());
        ctx->saved_data["k"] = kept;
        return {f.y};
    }
    static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
        auto t = ctx->get_saved_variables();
        t.resize(5);
        const auto kept = ctx->saved_data["k"].toIntVector();
        const int64_t* types = kept.data() + 6;
        const Block s{kept[0], kept[1], kept[2], kept[3]};
        same_interval({{}, (int)kept[4], at::kBFloat16, false});
        c10::DeviceGuard guard(t[0].device());
        at::AutoDispatchBelowADInplaceOrView below;
        auto need = [&](int i) { return ctx->needs_input_grad(1 + i); };
        const bool need_x = ctx->needs_input_grad(0);
        const Stages st(need_x, need);
        const GradLayout G(s.C, need);
        const Tensor dx = st.streams ? at::empty_like(t[1]) : Tensor(), flat = at::empty({G.kept}, t[0].options().dtype(at::kFloat));
        block_backward(s, t[1], t[2], t[3], t[4], t[0], dense_bf16(grads[0]), st, dx, flat, need);
        variable_list out{Tensor(), need_x ? dx.to((at::ScalarType)kept[5]) : Tensor()};
        Tensor flat16;   // bf16 parameters: one conversion of the whole buffer
        for (int i = 0; i < PARAMS; i++) {
            if (!need(i)) {
                out.emplace_back();
                continue;
            }
            const bool f32 = types[i] == (int64_t)at::kFloat;
            if (!f32 && !flat16.defined()) flat16 = flat.to(at::kBFloat16);
            out.push_back(GradLayout::view(f32 ? flat : flat16, i, s.C, G.at[i]));
        }
        return out;
    }
};

// The same two passes as the registered operators that torch.compile records: every buffer comes from the caller, an empty
// tensor stands for one that is not there.  need[0]: x's gradient is wanted, need[1 + i]: parameter i's.  block_sizes: the
// elements of `weights` without and with the transposed copies and of `acts` per token without and with a backward; whether the backward goes further than
// the output projection; the elements of `flat`, and each wanted gradient's place in it.
std::vector<int64_t> block_sizes(int64_t C, const std::vector<bool>& need) {
    TORCH_CHECK(need.size() == PARAMS + 1, "one flag for x and one per parameter");
    auto of = [&](int i) { return (bool)need[1 + i]; };
    const WeightLayout W(C);
    const GradLayout G(C, of);
    std::vector<int64_t> r{W.total[0], W.total[1], Activations({1, 16, C, 1}, false).total / 16, Activations({1, 16, C, 1}, true).total / 16, Stages(need[0], of).attn, G.kept};
    for (int i = 0; i < PARAMS; i++) r.push_back(of(i) ? G.at[i] : -1);
    return r;
}
void traced_block_forward(const Tensor& xb, const variable_list& p, int64_t H, const Tensor& x_first, const Tensor& x_prev, const Tensor& s0,
                          const Tensor& weights, const Tensor& acts, const Tensor& saved, const Tensor& ya, const Tensor& y, const Tensor& sT,
                          bool save) {
    c10::DeviceGuard guard(xb.device());
    at::AutoDispatchBelowADInplaceOrView below;
    const Block s{xb.size(0), xb.size(1), xb.size(2), H};
    block_forward(s, dense_bf16(xb), p, save, s.T, x_prev.numel() ? First(x_first, x_prev) : First(), s0.numel() ? s0 : Tensor(),
                  BlockBuffers(weights, acts, saved, ya, y, sT));
}
void traced_block_backward(const Tensor& xb, const Tensor& weights, const Tensor& acts, const Tensor& saved, const Tensor& ya, const Tensor& dout,
                           int64_t H, const std::vector<bool>& need, const Tensor& dx, const Tensor& flat) {
    TORCH_CHECK(need.size() == PARAMS + 1, "one flag for x and one per parameter");
    c10::DeviceGuard guard(xb.device());
    at::AutoDispatchBelowADInplaceOrView below;
    auto of = [&](int i) { return (bool)need[1 + i]; };
    block_backward({xb.size(0), xb.size(1), xb.size(2), H}, dense_bf16(xb), weights, acts, saved, ya, dense_bf16(dout), Stages(need[0], of), dx,
                   flat, of);
}

template <size_t... I>
Tensor mixer_node(int64_t H, const Tensor& x, const variable_list& p, std::index_sequence<I...>) {
    return MixerBlock::apply(H, x, p[I]...)[0];
}

// The parameters by name out of the module's (and its GroupNorm's) `_parameters`; false where one is missing or not a
// plain float32 / bf16 tensor of the expected shape on x's device.
bool mixer_params(const py::dict& own, const py::dict& norm, const Tensor& x, variable_list& out) {
    static PyObject* names[PARAMS] = {};
    if (!names[0])
        for (int i = 0; i < PARAMS; i++) names[i] = PyUnicode_InternFromString(PARAM_NAMES[i]);
    const int64_t C = x.size(-1);
    out.clear();
    out.reserve(PARAMS);
    for (int i = 0; i < PARAMS; i++) {
        PyObject* o = PyDict_GetItem((i == LN_W || i == LN_B ? norm : own).ptr(), names[i]);   // (borrowed)
        if (!o || !THPVariable_Check(o)) return false;
        const Tensor& t = THPVariable_Unpack(o);
        if (!plain_param(t, x) || t.sizes() != at::IntArrayRef(param_shape(i, C))) return false;
        out.push_back(t);
    }
    return true;
}
bool floating(const Tensor& t) {
    return t.scalar_type() == at::kBFloat16 || t.scalar_type() == at::kFloat || t.scalar_type() == at::kHalf || t.scalar_type() == at::kDouble;
}

// A ragged prompt this short runs token by token on a state in registers, in the four launches of a step; the sequence kernels take some twenty launches whatever the length.  (Whole chunks stay with them: the same bits as the
// same tokens inside a longer call.)
constexpr int64_t SHORT_PROMPT = 64, SHORT_PROMPT_ROWS = 512;

py::object short_prompt(int64_t B, int64_t T, int64_t C, int64_t H, const Tensor& x, const variable_list& p, const Tensor& x_prev,
                        const Tensor& s0, at::ScalarType state_type, bool return_state) {
    at::AutoDispatchBelowADInplaceOrView below;
    const Tensor xb = dense_bf16(x);
    const WeightLayout W(C);
    const Tensor packed = at::empty({W.total[0]}, xb.options());
    pack_weights(W, p, packed, false);
    const void* w[WEIGHTS + 1];
    for (int i = 0; i < WEIGHTS; i++) w[i] = at_elem(packed, W.at_.at[i]);
    w[WEIGHTS] = at_elem(packed, W.ln);
    wind_rwkv7_mixer_weights weights;
    static_assert(sizeof(w) == sizeof(weights), "the enumeration above is the header's order");
    memcpy(&weights, w, sizeof(w));
    const Tensor y = at::empty({B, T, C}, xb.options()), sT = at::empty({B, H, 64, 64}, xb.options().dtype(state_type));
    const bool carry_here = return_state && x.scalar_type() == at::kBFloat16;   // (the carried token keeps x's own type)
    const Tensor carry = carry_here ? at::empty({B, C}, xb.options()) : return_state ? x.select(1, T - 1).clone() : Tensor();
    const Tensor ws = scratch_bytes(L.mixer_decode_workspace_bytes((int)(B * T), (int)C), xb);
    const Tensor prev = x_prev.defined() ? dense_bf16(x_prev) : Tensor();   // (as `step` takes it)
    check(L.mixer_prompt((int)B, (int)T, (int)C, (int)H, state_type == at::kFloat ? WIND_RWKV7_F32 : WIND_RWKV7_BF16, &weights, ptr(xb), ptr(prev),
                         ptr(s0), ptr(sT), ptr(y), carry_here ? ptr(carry) : nullptr, ptr(ws), ws.numel(), stream_of(xb)));
    if (!return_state) return py::cast(y);
    return py::make_tuple(y, py::make_tuple(carry, sT));
}

py::object mixer(const Tensor& x, const py::dict& own, const py::dict& norm, int64_t H, const std::optional<Tensor>& x_prev_,
                 const std::optional<Tensor>& s0_, bool return_state) {
    if (!x.defined() || !x.is_cuda() || !floating(x) || x.layout() != at::kStrided || at::isTensorSubclassLike(x) || x.dim() != 3 || H <= 0 ||
        x.size(2) % H || x.numel() == 0)
        return py::none();
    const bool stateful = return_state || x_prev_ || s0_;
    const int64_t T = x.size(1);
    const Block s{x.size(0), (T + 15) / 16 * 16, x.size(2), H};
    if (T % 16 && (!stateful || s.N() != 64)) return py::none();
    if (s.rows() > std::numeric_limits<int>::max() || s.C % 64 || !L.attn_ln_saved_bytes(s.B, s.T, s.H, s.N()) ||
        !L.expand_loras_bwd_workspace_bytes(s.B, s.T, s.C, R_LORA) || !L.ddlerp_bwd_workspace_bytes(s.B, s.T, s.C, R_MIX))
        return py::none();
    variable_list p;
    if (!mixer_params(own, norm, x, p)) return py::none();
    bool grad = x.requires_grad();
    for (const auto& t : p) grad = grad || t.requires_grad();
    grad = grad && at::GradMode::is_enabled();
    c10::DeviceGuard guard(x.device());
    if (grad) return stateful ? py::object(py::none()) : py::cast(mixer_node(H, x, p, std::make_index_sequence<PARAMS>()));
    Tensor x_prev, s0;
    if (x_prev_) {
        if (!x_prev_->is_cuda() || !floating(*x_prev_) || x_prev_->device() != x.device() || x_prev_->sizes() != at::IntArrayRef({s.B, s.C})) return py::none();
        x_prev = *x_prev_;
    }
    if (s0_) {
        s0 = *s0_;
        if (!(plain(s0, at::kFloat) || plain(s0, at::kBFloat16)) || s0.device() != x.device() ||
            s0.sizes() != at::IntArrayRef({s.B, s.H, s.N(), s.N()}))
            return py::none();
    }
    const at::ScalarType state_type = s0.defined() ? s0.scalar_type() : stateful ? at::kFloat : at::kBFloat16;
    if (T % 16 && s.N() == 64 && T <= SHORT_PROMPT && s.B * T <= SHORT_PROMPT_ROWS) return short_prompt(s.B, T, s.C, H, x, p, x_prev, s0, state_type, return_state);
    Tensor xb = dense_bf16(x), carry;
    Padding pad;
    if (s.T != T) {
        pad.x = xb, pad.out = xb = at::empty({s.B, s.T, s.C}, xb.options());
        if (return_state && x.scalar_type() == at::kBFloat16) pad.last = carry = at::empty({s.B, s.C}, xb.options());   // (the carried token keeps x's own type)
    }
    const BlockBuffers f(s, xb, false, T, state_type);
    block_forward(s, xb, p, false, T, x_prev.defined() ? First(x.select(1, 0), x_prev) : First(), s0, f, pad);
    if (!return_state) return py::cast(f.y);
    return py::make_tuple(f.y, py::make_tuple(carry.defined() ? carry : x.select(1, T - 1).clone(), f.sT));
}

// One token per sequence.  `cache` = (key, 24 bf16 copies, [3,C] float32, workspaces by batch) as the module keeps it;
// None where it is not there or a parameter has changed since (the caller then remakes it and calls again).
py::object mixer_step(const Tensor& x, const Tensor& x_prev, const Tensor& S, const py::dict& own, const py::dict& norm, const py::object& cache,
                      int64_t H) {
    if (!x.defined() || x.dim() != 2 || !x.is_cuda() || !floating(x) || at::isTensorSubclassLike(x) || !floating(x_prev) ||
        x_prev.device() != x.device() || x_prev.sizes() != x.sizes() || H <= 0)
        return py::none();
    const int64_t B = x.size(0), C = x.size(1);
    if (!(plain(S, at::kFloat) || plain(S, at::kBFloat16)) || S.device() != x.device() || C != 64 * H ||
        S.sizes() != at::IntArrayRef({B, H, 64, 64}) || !PyTuple_Check(cache.ptr()) || PyTuple_GET_SIZE(cache.ptr()) != 4)
        return py::none();
    variable_list p;
    if (!mixer_params(own, norm, x, p)) return py::none();
    PyObject *key = PyTuple_GET_ITEM(cache.ptr(), 0), *copies = PyTuple_GET_ITEM(cache.ptr(), 1);
    if (!PyTuple_Check(key) || PyTuple_GET_SIZE(key) != PARAMS || !PyList_Check(copies) || PyList_GET_SIZE(copies) != WEIGHTS) return py::none();
    for (int i = 0; i < PARAMS; i++) {
        PyObject* pair = PyTuple_GET_ITEM(key, i);
        if (PyLong_AsVoidPtr(PyTuple_GET_ITEM(pair, 0)) != p[i].data_ptr() || PyLong_AsLongLong(PyTuple_GET_ITEM(pair, 1)) != (long long)p[i]._version())
            return py::none();
    }
    const void* w[WEIGHTS + 1];
    static_assert(sizeof(w) == sizeof(wind_rwkv7_mixer_weights), "the enumeration above is the header's order");
    for (int i = 0; i < WEIGHTS; i++) {
        PyObject* o = PyList_GET_ITEM(copies, i);
        if (!THPVariable_Check(o) || THPVariable_Unpack(o).device() != x.device()) return py::none();
        w[i] = THPVariable_Unpack(o).data_ptr();
    }
    w[WEIGHTS] = THPVariable_Unpack(PyTuple_GET_ITEM(cache.ptr(), 2)).data_ptr();
    wind_rwkv7_mixer_weights weights;
    memcpy(&weights, w, sizeof(w));
    c10::DeviceGuard guard(x.device());
    at::AutoDispatchBelowADInplaceOrView below;
    // the workspace belongs to the call (the allocator hands the same memory out again on this stream): two threads or
    // streams stepping one module do not share it
    const Tensor ws = scratch_bytes(L.mixer_decode_workspace_bytes((int)B, (int)C), x);
    const Tensor xb = dense_bf16(x), xp = dense_bf16(x_prev);
    const Tensor y = at::empty({B, C}, xb.options()), carry = at::empty({B, C}, xb.options());
    check(L.mixer_decode((int)B, (int)C, (int)H, state_code(S), &weights, ptr(xb), ptr(xp), ptr(S), ptr(y), ptr(carry), ptr(ws), ws.numel(), stream_of(x)));
    return py::make_tuple(y, py::make_tuple(carry, S));
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
    py::register_local_exception_translator([](std::exception_ptr p) {
        try {
            if (p) std::rethrow_exception(p);
        } catch (python_error& e) {
            e.restore();
        }
    });
    m.attr("torch_version") = TORCH_VERSION;   // (without the build's suffix)
    m.def("load", &load);
    m.def("attn", &attn);
    m.def("attn_ln", &attn_ln);
    m.def("ddlerp", &ddlerp);
    m.def("expand_loras", &expand_loras);
    m.def("mixer", &mixer);
    m.def("mixer_step", &mixer_step);
    m.def("block_sizes", &block_sizes);
    m.def("block_forward", &traced_block_forward);
    m.def("block_backward", &traced_block_backward);
}
