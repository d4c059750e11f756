// The host side of the calls that a program makes most, as a Python extension module: checks, allocation, launch and the
// autograd node, for operands that need nothing else.
//
// With small operands a call waits for the host. Through a Python autograd function with ctypes launches a forward and a
// backward take 105 to 160 us whatever their size (the interpreter's part of the function alone 48); here 52 to 80, of which the
// engine's own handing over to its thread and back is 25. One pass, us, before and here: softmax [4, 8, 512, 512] 124 / 53,
// rotary of 34 MB 144 / 88 (its kernels' time), LayerNorm of 67 MB 118 / 73 (its kernels), attention [1024, 4, 12, 64] 158 / 84
// (kernels 76), a decoding step of a layer of 768 features 213 / 107.
//
// A function returns NotImplemented where anything is unusual: the caller then goes on in Python, which takes, refuses and
// explains as it always did. So a check here may be stricter than the one there, never looser. Unusual is
//  - a tensor that is not a torch.Tensor or Parameter itself, or that torch follows beyond autograd (vmap and the other function
//    transforms, forward mode, tracing, modes, views by conjugation or negation),
//  - an operand on the CPU, of another type or size than the kernels take, of no elements, on another device than the rest.
// The nodes are torch's own C++ ones (torch::autograd::Function): saved tensors go through SavedVariable (version check,
// hooks), nothing else is kept, and a backward runs on whatever thread and stream the engine gives it.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/autocast_mode.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/forward_grad.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include "../../include/neox_hotpath.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::Function;
using torch::autograd::Variable;
using torch::autograd::variable_list;
using MaybeTensor = std::optional<Tensor>;

// ---------------------------------------------------------------------------------------------------------------- operands
const c10::DispatchKeySet kFollowedKeys(
    {c10::DispatchKey::Python, c10::DispatchKey::PythonTLSSnapshot, c10::DispatchKey::FuncTorchBatched,
     c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Functionalize, c10::DispatchKey::Conjugate,
     c10::DispatchKey::Negative, c10::DispatchKey::ZeroTensor, c10::DispatchKey::Batched, c10::DispatchKey::Fake});

// Whether torch follows operations beyond autograd right now, whatever they are on.
bool followed()
{
    return torch::jit::tracer::isTracing() || c10::impl::dispatch_mode_enabled() || at::impl::torch_function_mode_enabled() ||
           c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode) ||
           c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::Functionalize) ||
           torch::autograd::ForwardADLevel::try_get_by_idx(0) != nullptr;
}

bool take(PyObject* o, Tensor& t)
{
    if (!THPVariable_CheckExact(o)) return false;
    t = THPVariable_Unpack(o);
    return t.is_cuda() && t.layout() == at::kStrided && !t.key_set().has_any(kFollowedKeys) && t.numel() > 0;
}

bool take(PyObject* o, MaybeTensor& t)
{
    if (o == Py_None) {
        t.reset();
        return true;
    }
    Tensor inner;
    if (!take(o, inner)) return false;
    t = std::move(inner);
    return true;
}

bool take(PyObject* o, double& v)
{
    if (PyLong_CheckExact(o)) {
        v = PyLong_AsDouble(o);
        if (!PyErr_Occurred()) return true;
        PyErr_Clear();
        return false;
    }
    if (!PyFloat_CheckExact(o)) return false;
    v = PyFloat_AS_DOUBLE(o);
    return true;
}

bool take(PyObject* o, int64_t& v)
{
    if (!PyLong_CheckExact(o)) return false;
    int overflow = 0;
    v = PyLong_AsLongLongAndOverflow(o, &overflow);
    return overflow == 0;
}

bool take(PyObject* o, bool& v)
{
    v = o == Py_True;
    return v || o == Py_False;
}

template <size_t... I, typename... T>
bool take_all(PyObject* const* args, std::index_sequence<I...>, T&... to)
{
    return (take(args[I], to) && ...);
}
template <typename... T>
bool take_all(PyObject* const* args, Py_ssize_t count, T&... to)
{
    return count == (Py_ssize_t)sizeof...(T) && take_all(args, std::index_sequence_for<T...>{}, to...);
}

int type_code(at::ScalarType t)
{
    return t == at::kHalf ? NHP_F16 : t == at::kBFloat16 ? NHP_BF16 : t == at::kFloat ? NHP_F32 : -1;
}
bool is_half(const Tensor& t) { return t.scalar_type() == at::kHalf || t.scalar_type() == at::kBFloat16; }
bool alike(const Tensor& a, const Tensor& b) { return a.scalar_type() == b.scalar_type() && a.device() == b.device(); }

void* ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
void* ptr(const MaybeTensor& t) { return t ? t->data_ptr() : nullptr; }
void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }
Tensor bytes(int64_t n, const Tensor& like) { return n > 0 ? at::empty({n}, like.options().dtype(at::kByte)) : Tensor(); }
Tensor defined_or_none(const MaybeTensor& t) { return t ? *t : Tensor(); }
MaybeTensor contiguous(const MaybeTensor& t) { return t ? MaybeTensor(t->contiguous()) : t; }
Tensor contiguous_or_none(const Tensor& t) { return t.defined() ? t.contiguous() : t; }

void check(int status, const char* who)
{
    TORCH_CHECK(status == NHP_OK, who, ": ", nhp_status_string(status), " (status ", status, ")");
}

// A vector of `cols` values for a norm: its own type or fp32, the same for all of them.
bool parameters_fit(const Tensor& x, std::initializer_list<const MaybeTensor*> parameters, int64_t cols, int& code)
{
    code = type_code(x.scalar_type());
    bool first = true;
    for (const MaybeTensor* p : parameters) {
        if (!*p) continue;
        const Tensor& t = **p;
        const int own = type_code(t.scalar_type());
        if (t.numel() != cols || t.device() != x.device() || (own != type_code(x.scalar_type()) && own != NHP_F32)) return false;
        if (!first && own != code) return false;
        code = own;
        first = false;
    }
    return true;
}

at::ScalarType parameter_type(int code, const Tensor& x) { return code == NHP_F32 ? at::kFloat : x.scalar_type(); }

Tensor new_parameter(bool wanted, int64_t cols, int code, const Tensor& like)
{
    return wanted ? at::empty({cols}, like.options().dtype(parameter_type(code, like))) : Tensor();
}

// Which of the inputs that the graph has edges for want a gradient; inputs that were not given have none.
struct Wanted {
    const AutogradContext* ctx;
    size_t edge = 0;
    bool next(bool given) { return given && ctx->needs_input_grad(edge++); }
};

// ------------------------------------------------------------------------------------------------------------------- norms
struct LayerNormNode : Function<LayerNormNode> {
    static Tensor forward(AutogradContext* ctx, const Tensor& x, const MaybeTensor& weight, const MaybeTensor& bias, double eps,
                          int64_t pcode)
    {
        const Tensor src = x.contiguous();
        const MaybeTensor w = contiguous(weight), b = contiguous(bias);
        const int64_t cols = src.size(-1), rows = src.numel() / cols;
        const int code = type_code(src.scalar_type());
        const c10::DeviceGuard guard(src.device());
        Tensor y = at::empty_like(src);
        const Tensor mean = at::empty({rows}, src.options().dtype(at::kFloat)), rstd = at::empty({rows}, mean.options());
        check(nhp_layernorm_fwd(y.data_ptr(), mean.data_ptr<float>(), rstd.data_ptr<float>(), src.data_ptr(), ptr(w), ptr(b),
                                (float)eps, rows, cols, code, (int)pcode, stream_of(src)), "LayerNorm");
        ctx->save_for_backward({src, defined_or_none(w), mean, rstd});
        ctx->saved_data["conf"] = std::vector<int64_t>{code, pcode, bias.has_value()};
        return y;
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads)
    {
        const variable_list saved = ctx->get_saved_variables();
        const auto conf = ctx->saved_data["conf"].toIntVector();
        const Tensor src = saved[0].contiguous(), w = contiguous_or_none(saved[1]), mean = saved[2].contiguous(), rstd = saved[3].contiguous();
        const Tensor g = grads[0].contiguous();
        const int64_t cols = src.size(-1), rows = src.numel() / cols;
        const c10::DeviceGuard guard(src.device());
        Wanted wanted{ctx, 1};
        Tensor dx = at::empty_like(src);
        Tensor dw = new_parameter(wanted.next(w.defined()), cols, (int)conf[1], src);
        Tensor db = new_parameter(wanted.next(conf[2]), cols, (int)conf[1], src);
        Tensor ws;
        if (dw.defined() || db.defined()) ws = bytes(nhp_norm_bwd_workspace_bytes(rows, cols, (int)conf[0]), src);
        check(nhp_layernorm_bwd(dx.data_ptr(), ptr(dw), ptr(db), g.data_ptr(), src.data_ptr(), mean.data_ptr<float>(),
                                rstd.data_ptr<float>(), ptr(w), ptr(ws), rows, cols, (int)conf[0], (int)conf[1], stream_of(src)),
              "LayerNorm backward");
        return {dx, dw, db, Tensor(), Tensor()};
    }
};

struct LayerNormPairNode : Function<LayerNormPairNode> {
    static variable_list forward(AutogradContext* ctx, const Tensor& x, const MaybeTensor& weight1, const MaybeTensor& bias1,
                                 const MaybeTensor& weight2, const MaybeTensor& bias2, double eps, int64_t pcode)
    {
        const Tensor src = x.contiguous();
        const MaybeTensor w1 = contiguous(weight1), b1 = contiguous(bias1), w2 = contiguous(weight2), b2 = contiguous(bias2);
        const int64_t cols = src.size(-1), rows = src.numel() / cols;
        const int code = type_code(src.scalar_type());
        const c10::DeviceGuard guard(src.device());
        Tensor y1 = at::empty_like(src), y2 = at::empty_like(src);
        const Tensor mean = at::empty({rows}, src.options().dtype(at::kFloat)), rstd = at::empty({rows}, mean.options());
        check(nhp_layernorm_pair_fwd(y1.data_ptr(), y2.data_ptr(), mean.data_ptr<float>(), rstd.data_ptr<float>(), src.data_ptr(),
                                     ptr(w1), ptr(b1), ptr(w2), ptr(b2), (float)eps, rows, cols, code, (int)pcode, stream_of(src)),
              "LayerNorm pair");
        ctx->save_for_backward({src, defined_or_none(w1), defined_or_none(w2), mean, rstd});
        ctx->saved_data["conf"] = std::vector<int64_t>{code, pcode, b1.has_value(), b2.has_value()};
        return {y1, y2};
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads)
    {
        const variable_list saved = ctx->get_saved_variables();
        const auto conf = ctx->saved_data["conf"].toIntVector();
        const Tensor src = saved[0].contiguous(), w1 = contiguous_or_none(saved[1]), w2 = contiguous_or_none(saved[2]);
        const Tensor mean = saved[3].contiguous(), rstd = saved[4].contiguous();
        const Tensor g1 = grads[0].contiguous(), g2 = grads[1].contiguous();
        const int64_t cols = src.size(-1), rows = src.numel() / cols;
        const c10::DeviceGuard guard(src.device());
        Wanted wanted{ctx, 1};
        const int pcode = (int)conf[1];
        Tensor dx = at::empty_like(src);
        Tensor dw1 = new_parameter(wanted.next(w1.defined()), cols, pcode, src), db1 = new_parameter(wanted.next(conf[2]), cols, pcode, src);
        Tensor dw2 = new_parameter(wanted.next(w2.defined()), cols, pcode, src), db2 = new_parameter(wanted.next(conf[3]), cols, pcode, src);
        Tensor ws;
        if (dw1.defined() || db1.defined() || dw2.defined() || db2.defined())
            ws = bytes(nhp_layernorm_pair_bwd_workspace_bytes(rows, cols, (int)conf[0]), src);
        check(nhp_layernorm_pair_bwd(dx.data_ptr(), ptr(dw1), ptr(db1), ptr(dw2), ptr(db2), g1.data_ptr(), g2.data_ptr(), src.data_ptr(),
                                     mean.data_ptr<float>(), rstd.data_ptr<float>(), ptr(w1), ptr(w2), ptr(ws), rows, cols,
                                     (int)conf[0], pcode, stream_of(src)), "LayerNorm pair backward");
        return {dx, dw1, db1, dw2, db2, Tensor(), Tensor()};
    }
};

struct RMSNormNode : Function<RMSNormNode> {
    static Tensor forward(AutogradContext* ctx, const Tensor& x, const MaybeTensor& scale, const MaybeTensor& offset, double eps,
                          int64_t eps_mode, int64_t stat, int64_t pcode)
    {
        const Tensor src = x.contiguous();
        const MaybeTensor s = contiguous(scale), o = contiguous(offset);
        const int64_t cols = src.size(-1), rows = src.numel() / cols;
        const int code = type_code(src.scalar_type());
        const c10::DeviceGuard guard(src.device());
        Tensor y = at::empty_like(src);
        const Tensor inv = at::empty({rows}, src.options().dtype(at::kFloat));
        check(nhp_rmsnorm_partial_fwd(y.data_ptr(), inv.data_ptr<float>(), src.data_ptr(), ptr(s), ptr(o), (float)eps, (int)eps_mode,
                                      rows, cols, stat, code, (int)pcode, stream_of(src)), "RMSNorm");
        ctx->save_for_backward({src, defined_or_none(s), inv});
        ctx->saved_data["conf"] = std::vector<int64_t>{code, pcode, offset.has_value(), eps_mode, stat};
        ctx->saved_data["eps"] = eps;
        return y;
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads)
    {
        const variable_list saved = ctx->get_saved_variables();
        const auto conf = ctx->saved_data["conf"].toIntVector();
        const Tensor src = saved[0].contiguous(), s = contiguous_or_none(saved[1]), inv = saved[2].contiguous(), g = grads[0].contiguous();
        const int64_t cols = src.size(-1), rows = src.numel() / cols;
        const c10::DeviceGuard guard(src.device());
        Wanted wanted{ctx, 1};
        Tensor dx = at::empty_like(src);
        Tensor ds = new_parameter(wanted.next(s.defined()), cols, (int)conf[1], src);
        Tensor dof = new_parameter(wanted.next(conf[2]), cols, (int)conf[1], src);
        Tensor ws;
        if (ds.defined() || dof.defined()) ws = bytes(nhp_norm_bwd_workspace_bytes(rows, cols, (int)conf[0]), src);
        check(nhp_rmsnorm_partial_bwd(dx.data_ptr(), ptr(ds), ptr(dof), g.data_ptr(), src.data_ptr(), inv.data_ptr<float>(), ptr(s),
                                      ptr(ws), (float)ctx->saved_data["eps"].toDouble(), (int)conf[3], rows, cols, conf[4], (int)conf[0],
                                      (int)conf[1], stream_of(src)), "RMSNorm backward");
        return {dx, ds, dof, Tensor(), Tensor(), Tensor(), Tensor()};
    }
};

// ------------------------------------------------------------------------------------------------------------- activations
struct BiasGeluNode : Function<BiasGeluNode> {
    static Tensor forward(AutogradContext* ctx, const Tensor& x, const MaybeTensor& bias)
    {
        const Tensor src = x.contiguous();
        const MaybeTensor b = contiguous(bias);
        const int64_t cols = src.size(-1), rows = src.numel() / cols;
        const c10::DeviceGuard guard(src.device());
        Tensor out = at::empty_like(src);
        check(nhp_bias_gelu_fwd(out.data_ptr(), src.data_ptr(), ptr(b), rows, cols, type_code(src.scalar_type()), stream_of(src)), "bias_gelu");
        ctx->save_for_backward({x, defined_or_none(bias)});
        return out;
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads)
    {
        const variable_list saved = ctx->get_saved_variables();
        const Tensor src = saved[0].contiguous(), b = contiguous_or_none(saved[1]), g = grads[0].contiguous();
        const int64_t cols = src.size(-1), rows = src.numel() / cols;
        const int code = type_code(src.scalar_type());
        const c10::DeviceGuard guard(src.device());
        Tensor dx = at::empty_like(src), db, ws;
        if (b.defined() && ctx->needs_input_grad(1)) {
            db = at::empty_like(b);
            ws = bytes(nhp_bias_gelu_bwd_workspace_bytes(rows, cols, code), src);
        }
        check(nhp_bias_gelu_bwd(dx.data_ptr(), g.data_ptr(), src.data_ptr(), ptr(b), ptr(db), ptr(ws), rows, cols, code, stream_of(src)),
              "bias_gelu_back");
        return {dx, db};
    }
};

struct GatedNode : Function<GatedNode> {
    static Tensor forward(AutogradContext* ctx, const Tensor& x, int64_t act)
    {
        const Tensor src = x.contiguous();
        const int64_t features = src.size(-1) / 2, rows = src.numel() / (2 * features);
        const c10::DeviceGuard guard(src.device());
        auto shape = src.sizes().vec();
        shape.back() = features;
        Tensor out = at::empty(shape, src.options());
        check(nhp_gated_act_fwd(out.data_ptr(), src.data_ptr(), nullptr, rows, features, (int)act, type_code(src.scalar_type()), stream_of(src)),
              "Gated_Activation");
        ctx->save_for_backward({src});
        ctx->saved_data["act"] = act;
        return out;
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads)
    {
        const Tensor src = ctx->get_saved_variables()[0].contiguous(), g = grads[0].contiguous();
        const int64_t features = src.size(-1) / 2, rows = src.numel() / (2 * features);
        const c10::DeviceGuard guard(src.device());
        Tensor dx = at::empty_like(src);
        check(nhp_gated_act_bwd(dx.data_ptr(), g.data_ptr(), src.data_ptr(), nullptr, rows, features, (int)ctx->saved_data["act"].toInt(),
                                type_code(src.scalar_type()), stream_of(src)), "Gated_Activation backward");
        return {dx, Tensor()};
    }
};

// ----------------------------------------------------------------------------------------------------------------- softmax
struct CausalSoftmaxNode : Function<CausalSoftmaxNode> {
    static Tensor forward(AutogradContext* ctx, const Tensor& x, double scale, int64_t window)
    {
        const int64_t s = x.size(-1), matrices = x.numel() / (s * s);
        const c10::DeviceGuard guard(x.device());
        Tensor y = at::empty_like(x);
        check(nhp_causal_softmax_blocks_fwd(y.data_ptr(), x.data_ptr(), (float)scale, matrices, s, window, 0, nullptr, nullptr, nullptr, 1,
                                            type_code(x.scalar_type()), stream_of(x)),
              "scaled_upper_triang_masked_softmax_cuda.forward");
        ctx->save_for_backward({y});
        ctx->saved_data["scale"] = scale;
        ctx->saved_data["window"] = window;
        return y;
    }
    // in place on the gradient, as the reference's kernel
    static variable_list backward(AutogradContext* ctx, variable_list grads)
    {
        const Tensor y = ctx->get_saved_variables()[0].contiguous();
        Tensor g = grads[0].detach().contiguous();
        const int64_t s = y.size(-1), matrices = y.numel() / (s * s);
        const c10::DeviceGuard guard(y.device());
        check(nhp_causal_softmax_blocks_bwd(g.data_ptr(), g.data_ptr(), y.data_ptr(), (float)ctx->saved_data["scale"].toDouble(), matrices, s,
                                            ctx->saved_data["window"].toInt(), 0, nullptr, 1, type_code(y.scalar_type()), stream_of(y)),
              "scaled_upper_triang_masked_softmax_cuda.backward");
        return {g, Tensor(), Tensor()};
    }
};

struct MaskedSoftmaxNode : Function<MaskedSoftmaxNode> {
    static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& mask, double scale)
    {
        const Tensor src = x.contiguous(), m = mask.contiguous();
        const c10::DeviceGuard guard(src.device());
        Tensor y = at::empty_like(src);
        check(nhp_masked_softmax_ex_fwd(y.data_ptr(), src.data_ptr(), static_cast<const uint8_t*>(m.data_ptr()), (float)scale, src.size(0),
                                        src.size(1), src.size(2), src.size(3), m.size(0), nullptr, nullptr, nullptr,
                                        type_code(src.scalar_type()), stream_of(src)), "scaled_masked_softmax_cuda.forward");
        ctx->save_for_backward({y});
        ctx->saved_data["scale"] = scale;
        return y;
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads)
    {
        const Tensor y = ctx->get_saved_variables()[0].contiguous();
        Tensor g = grads[0].detach().contiguous();
        const int64_t sk = y.size(3);
        const c10::DeviceGuard guard(y.device());
        check(nhp_masked_softmax_bwd(g.data_ptr(), g.data_ptr(), y.data_ptr(), (float)ctx->saved_data["scale"].toDouble(), y.numel() / sk, sk,
                                     type_code(y.scalar_type()), stream_of(y)), "scaled_masked_softmax_cuda.backward");
        return {g, Tensor(), Tensor()};
    }
};

// ------------------------------------------------------------------------------------------------------------------ rotary
using RopeKernel = decltype(&nhp_rope_cached_qk_fwd);

void rotate(RopeKernel kernel, const Tensor& q_out, const Tensor& k_out, const Tensor& q, const Tensor& k, const Tensor& cos,
            const Tensor& sin, const char* who)
{
    check(kernel(q_out.data_ptr(), k_out.data_ptr(), q.data_ptr(), k.data_ptr(), cos.data_ptr(), sin.data_ptr(), q.size(0), q.size(1),
                 q.size(2), k.size(2), q.size(3), cos.size(3), q.strides().data(), k.strides().data(), q_out.strides().data(),
                 k_out.strides().data(), type_code(q.scalar_type()), type_code(cos.scalar_type()), stream_of(q)), who);
}

// Tables [S, 1, 1, d2] whose rows from `offset` on hold `rows` positions of tensors like `t`
bool tables_fit(const Tensor& cos, const Tensor& sin, const Tensor& t, int64_t head, int64_t rows, int64_t offset)
{
    return cos.dim() == 4 && cos.sizes() == sin.sizes() && alike(cos, sin) && cos.device() == t.device() && cos.size(1) == 1 &&
           cos.size(2) == 1 && cos.size(3) <= head && (cos.scalar_type() == at::kFloat || cos.scalar_type() == t.scalar_type()) &&
           offset >= 0 && rows > 0 && offset + rows <= cos.size(0);
}
Tensor table_rows(const Tensor& table, int64_t offset, int64_t rows)
{
    return offset == 0 && table.size(0) == rows ? table : table.narrow(0, offset, rows);
}

struct RotaryNode : Function<RotaryNode> {
    static variable_list forward(AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& cos, const Tensor& sin)
    {
        const c10::DeviceGuard guard(q.device());
        Tensor q_out = at::empty(q.sizes(), q.options()), k_out = at::empty(k.sizes(), k.options());
        rotate(nhp_rope_cached_qk_fwd, q_out, k_out, q, k, cos.contiguous(), sin.contiguous(),
               "fused_rotary_positional_embedding.forward_cached_qk");
        ctx->save_for_backward({cos, sin});
        return {q_out, k_out};
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads)
    {
        const variable_list saved = ctx->get_saved_variables();
        const Tensor &gq = grads[0], &gk = grads[1];
        const c10::DeviceGuard guard(gq.device());
        Tensor dq = at::empty(gq.sizes(), gq.options()), dk = at::empty(gk.sizes(), gk.options());
        rotate(nhp_rope_cached_qk_bwd, dq, dk, gq, gk, saved[0].contiguous(), saved[1].contiguous(),
               "fused_rotary_positional_embedding.backward_cached_qk");
        return {dq, dk, Tensor(), Tensor()};
    }
};

// The three parts of a projection's output: [sq, b, np, 3 * hn] (`heads` == 0), or [sq, b, (np + 2 * nkv) * hn]
struct Parts {
    Tensor q, k, v;
};
Parts parts_of(const Tensor& mixed, int64_t heads, int64_t kv_heads)
{
    if (heads == 0) {
        const int64_t hn = mixed.size(-1) / 3;
        return {mixed.narrow(-1, 0, hn), mixed.narrow(-1, hn, hn), mixed.narrow(-1, 2 * hn, hn)};
    }
    const int64_t sq = mixed.size(0), b = mixed.size(1), hn = mixed.size(2) / (heads + 2 * kv_heads);
    return {mixed.narrow(-1, 0, heads * hn).view({sq, b, heads, hn}), mixed.narrow(-1, heads * hn, kv_heads * hn).view({sq, b, kv_heads, hn}),
            mixed.narrow(-1, (heads + kv_heads) * hn, kv_heads * hn).view({sq, b, kv_heads, hn})};
}

struct SplitRotaryNode : Function<SplitRotaryNode> {
    static variable_list forward(AutogradContext* ctx, const Tensor& mixed, const Tensor& cos, const Tensor& sin, int64_t heads,
                                 int64_t kv_heads)
    {
        const c10::DeviceGuard guard(mixed.device());
        const Parts in = parts_of(mixed, heads, kv_heads);
        Tensor q, k;
        if (heads == 0) {
            q = at::empty(in.q.sizes(), in.q.options());
            k = at::empty(in.k.sizes(), in.k.options());
        } else {   // head-major, as the grouped products take them without a copy
            q = at::empty({in.q.size(1), in.q.size(2), in.q.size(0), in.q.size(3)}, in.q.options()).permute({2, 0, 1, 3});
            k = at::empty({in.k.size(1), in.k.size(2), in.k.size(0), in.k.size(3)}, in.k.options()).permute({2, 0, 1, 3});
        }
        rotate(nhp_rope_cached_qk_fwd, q, k, in.q, in.k, cos.contiguous(), sin.contiguous(),
               "fused_rotary_positional_embedding.forward_cached_qk");
        ctx->save_for_backward({cos, sin});
        ctx->saved_data["heads"] = std::vector<int64_t>{heads, kv_heads};
        return {q, k, in.v};
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads)
    {
        const variable_list saved = ctx->get_saved_variables();
        const auto heads = ctx->saved_data["heads"].toIntVector();
        const Tensor &gq = grads[0], &gk = grads[1], &gv = grads[2];
        const int64_t sq = gq.size(0), b = gq.size(1), np = gq.size(2), hn = gq.size(3);
        const c10::DeviceGuard guard(gq.device());
        Tensor grad = heads[0] == 0 ? at::empty({sq, b, np, 3 * hn}, gq.options())
                                    : at::empty({sq, b, (heads[0] + 2 * heads[1]) * hn}, gq.options());
        Parts to = parts_of(grad, heads[0], heads[1]);
        rotate(nhp_rope_cached_qk_bwd, to.q, to.k, gq, gk, saved[0].contiguous(), saved[1].contiguous(),
               "fused_rotary_positional_embedding.backward_cached_qk");
        to.v.copy_(gv);
        return {grad, Tensor(), Tensor(), Tensor(), Tensor()};
    }
};

// ------------------------------------------------------------------------------------------------------------ residual adds
// Sum over all but the last dimension, fp32 sums in a fixed order, one rounding.
Tensor column_sum(const Tensor& t)
{
    const Tensor src = t.contiguous();
    const int64_t cols = src.size(-1), rows = src.numel() / cols;
    const int code = type_code(src.scalar_type());
    Tensor out = at::empty({cols}, src.options());
    const Tensor ws = bytes(nhp_column_sum_workspace_bytes(rows, cols, code), src);
    check(nhp_column_sum(out.data_ptr(), src.data_ptr(), ptr(ws), rows, cols, code, stream_of(src)), "bias_dropout_add backward");
    return out;
}

struct AddResidualNode : Function<AddResidualNode> {
    static Tensor forward(AutogradContext* ctx, const Tensor& x, const MaybeTensor& bias, const MaybeTensor& residual)
    {
        const Tensor src = x.contiguous();
        const MaybeTensor b = contiguous(bias), res = contiguous(residual);
        const int64_t cols = src.size(-1), rows = src.numel() / cols;
        const c10::DeviceGuard guard(src.device());
        Tensor out = at::empty_like(src);
        check(nhp_bias_add_residual(out.data_ptr(), src.data_ptr(), ptr(b), ptr(res), rows, cols, type_code(src.scalar_type()), stream_of(src)),
              "bias_dropout_add");
        ctx->saved_data["bias"] = bias ? bias->sizes().vec() : std::vector<int64_t>{};
        ctx->saved_data["given"] = std::vector<int64_t>{bias.has_value(), residual.has_value()};
        return out;
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads)
    {
        const auto given = ctx->saved_data["given"].toIntVector();
        const Tensor& grad = grads[0];
        const c10::DeviceGuard guard(grad.device());
        Wanted wanted{ctx, 1};
        Tensor gb, gr;
        if (wanted.next(given[0])) gb = column_sum(grad).view(ctx->saved_data["bias"].toIntVector());
        if (wanted.next(given[1])) gr = grad;
        return {grad, gb, gr};
    }
};

struct AddResidualPairNode : Function<AddResidualPairNode> {
    static Tensor forward(AutogradContext* ctx, const Tensor& x1, const MaybeTensor& bias1, const Tensor& x2, const MaybeTensor& bias2,
                          const Tensor& residual)
    {
        const Tensor a = x1.contiguous(), c = x2.contiguous(), res = residual.contiguous();
        const MaybeTensor b1 = contiguous(bias1), b2 = contiguous(bias2);
        const int64_t cols = a.size(-1), rows = a.numel() / cols;
        const c10::DeviceGuard guard(a.device());
        Tensor out = at::empty_like(a);
        check(nhp_bias_add_residual_pair(out.data_ptr(), a.data_ptr(), ptr(b1), c.data_ptr(), ptr(b2), res.data_ptr(), rows, cols,
                                         type_code(a.scalar_type()), stream_of(a)), "bias_add_residual_pair");
        ctx->saved_data["bias1"] = bias1 ? bias1->sizes().vec() : std::vector<int64_t>{};
        ctx->saved_data["bias2"] = bias2 ? bias2->sizes().vec() : std::vector<int64_t>{};
        ctx->saved_data["given"] = std::vector<int64_t>{bias1.has_value(), bias2.has_value()};
        return out;
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads)
    {
        const auto given = ctx->saved_data["given"].toIntVector();
        const Tensor& grad = grads[0];
        const c10::DeviceGuard guard(grad.device());
        Wanted wanted{ctx, 1};
        const bool need1 = wanted.next(given[0]);
        wanted.next(true);
        const bool need2 = wanted.next(given[1]);
        const bool need_residual = wanted.next(true);
        Tensor sum, g1, g2;
        if (need1 || need2) sum = column_sum(grad);
        if (need1) g1 = sum.view(ctx->saved_data["bias1"].toIntVector());
        if (need2) g2 = sum.view(ctx->saved_data["bias2"].toIntVector());
        return {grad, g1, grad, g2, need_residual ? grad : Tensor()};
    }
};

// --------------------------------------------------------------------------------------------------------------- attention
// Element strides over position, batch entry and head; that of a dimension of one entry means nothing and is 0.
struct Strides3 {
    int64_t s[3];
    explicit Strides3(const Tensor& t)
    {
        for (int i = 0; i < 3; ++i) s[i] = t.size(i) > 1 ? t.stride(i) : 0;
    }
    Strides3(int64_t a, int64_t b, int64_t c) : s{a, b, c} {}
};

// `t`, or a copy where the kernels cannot read it: they want contiguous features and 16-byte aligned rows
Tensor readable(const Tensor& t)
{
    const Strides3 st(t);
    if (t.stride(3) == 1 && ((st.s[0] | st.s[1] | st.s[2]) & 7) == 0 && reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0 && st.s[0] < (1 << 24))
        return t;
    return t.clone(at::MemoryFormat::Contiguous);
}

// The context in the layout that the caller gets and its strides: [sq, b, np * hn] with `merged`, [b, np, sq, hn] without
std::pair<Tensor, Strides3> new_context(const Tensor& q, bool merged)
{
    const int64_t sq = q.size(0), b = q.size(1), np = q.size(2), hn = q.size(3);
    if (merged) return {at::empty({sq, b, np * hn}, q.options()), Strides3(sq > 1 ? b * np * hn : 0, np * hn, hn)};
    return {at::empty({b, np, sq, hn}, q.options()), Strides3(hn, np * sq * hn, sq * hn)};
}

// What makes q, k and v belong together, and sizes that the kernels can address
bool attention_fits(const Tensor& q, const Tensor& k, const Tensor& v)
{
    if (!is_half(q) || !alike(q, k) || !alike(q, v) || q.dim() != 4 || k.dim() != 4 || v.sizes() != k.sizes()) return false;
    const int64_t sq = q.size(0), b = q.size(1), np = q.size(2), hn = q.size(3), sk = k.size(0), nkv = k.size(2);
    return (hn == 64 || hn == 80 || hn == 96 || hn == 128) && k.size(3) == hn && k.size(1) == b && np % nkv == 0 && sq <= sk && sk < (1 << 24) &&
           (sq == 1 || b * np * hn < (1 << 24)) && (sk == 1 || b * nkv * hn < (1 << 24)) && (b * np + 7) / 8 * 8 * ((sk + 127) / 128) < (1 << 24) &&
           sk * b * nkv * hn < ((int64_t)1 << 35);
}

struct CausalAttentionNode : Function<CausalAttentionNode> {
    static Tensor forward(AutogradContext* ctx, const Tensor& q_in, const Tensor& k_in, const Tensor& v_in, double scale, int64_t window,
                          bool merged, bool differentiated)
    {
        const c10::DeviceGuard guard(q_in.device());
        const Tensor q = readable(q_in), k = readable(k_in), v = readable(v_in);
        const int64_t sq = q.size(0), b = q.size(1), np = q.size(2), hn = q.size(3), sk = k.size(0), nkv = k.size(2);
        auto [out, out_strides] = new_context(q, merged);
        Tensor kept, lse;
        if (differentiated) {   // the caller may change the context in place: the backward has one of its own
            kept = at::empty_like(out);
            lse = at::empty({b * np, sq}, q.options().dtype(at::kFloat));
        }
        check(nhp_attention_fwd_keep(out.data_ptr(), ptr(kept), static_cast<float*>(ptr(lse)), q.data_ptr(), k.data_ptr(), v.data_ptr(), nullptr,
                                     1, 0.0f, (float)scale, window, b, np, nkv, sq, sk, hn, Strides3(q).s, Strides3(k).s, Strides3(v).s,
                                     out_strides.s, type_code(q.scalar_type()), stream_of(q)), "CausalAttention");
        if (differentiated) {
            ctx->save_for_backward({q, k, v, kept, lse});
            ctx->saved_data["scale"] = scale;
            ctx->saved_data["conf"] = std::vector<int64_t>{window, merged, out_strides.s[0], out_strides.s[1], out_strides.s[2]};
        }
        return out;
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads)
    {
        const variable_list saved = ctx->get_saved_variables();
        const auto conf = ctx->saved_data["conf"].toIntVector();
        const c10::DeviceGuard guard(saved[0].device());
        // (a hook on saved tensors may hand them back laid out otherwise)
        const Tensor q = readable(saved[0]), k = readable(saved[1]), v = readable(saved[2]), out = saved[3].contiguous(), lse = saved[4].contiguous();
        const int64_t sq = q.size(0), b = q.size(1), np = q.size(2), hn = q.size(3), sk = k.size(0), nkv = k.size(2);
        const Tensor g = readable(conf[1] ? grads[0].reshape({sq, b, np, hn}) : grads[0].permute({2, 0, 1, 3}));
        Tensor dq = at::empty(q.sizes(), q.options()), dk = at::empty(k.sizes(), k.options()), dv = at::empty(v.sizes(), v.options());
        const Tensor ws = bytes(nhp_attention_bwd_workspace_bytes(b, np, nkv, sq, sk, hn), q);
        check(nhp_attention_bwd(dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), g.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(),
                                out.data_ptr(), lse.data_ptr<float>(), ptr(ws), (float)ctx->saved_data["scale"].toDouble(), conf[0], b, np, nkv, sq,
                                sk, hn, Strides3(dq).s, Strides3(dk).s, Strides3(dv).s, Strides3(g).s, Strides3(q).s, Strides3(k).s,
                                Strides3(v).s, conf.data() + 2, type_code(q.scalar_type()), stream_of(q)), "CausalAttention backward");
        return {ctx->needs_input_grad(0) ? dq : Tensor(), ctx->needs_input_grad(1) ? dk : Tensor(), ctx->needs_input_grad(2) ? dv : Tensor(),
                Tensor(), Tensor(), Tensor(), Tensor()};
    }
};

bool wants_grad(std::initializer_list<const Tensor*> tensors)
{
    if (!at::GradMode::is_enabled()) return false;
    for (const Tensor* t : tensors)
        if (t->requires_grad()) return true;
    return false;
}

// --------------------------------------------------------------------------------------------------------- entry points
PyObject* not_here() { Py_RETURN_NOTIMPLEMENTED; }

// What `work` returns, other Python threads running meanwhile: an allocation may wait for the driver and a launch for a queue
// that is full. What comes back into Python (hooks on saved tensors, anomaly mode) takes the lock by itself. (0.2 us a call.)
template <typename F>
auto unlocked(F work)
{
    struct Lock {
        PyThreadState* const state = PyEval_SaveThread();
        ~Lock() { PyEval_RestoreThread(state); }
    } lock;
    return work();
}

PyObject* pack(const variable_list& tensors)
{
    PyObject* tuple = PyTuple_New((Py_ssize_t)tensors.size());
    if (!tuple) throw python_error();
    for (size_t i = 0; i < tensors.size(); ++i) PyTuple_SET_ITEM(tuple, (Py_ssize_t)i, THPVariable_Wrap(tensors[i]));
    return tuple;
}

// layer_norm(x, weight, bias, eps)
PyObject* py_layer_norm(PyObject*, PyObject* const* args, Py_ssize_t count)
{
    HANDLE_TH_ERRORS
    Tensor x;
    MaybeTensor w, b;
    double eps;
    int pcode;
    if (followed() || !take_all(args, count, x, w, b, eps) || x.dim() < 1 || type_code(x.scalar_type()) < 0 ||
        !parameters_fit(x, {&w, &b}, x.size(-1), pcode))
        return not_here();
    return THPVariable_Wrap(unlocked([&] { return LayerNormNode::apply(x, w, b, eps, (int64_t)pcode); }));
    END_HANDLE_TH_ERRORS
}

// layer_norm_pair(x, weight1, bias1, weight2, bias2, eps)
PyObject* py_layer_norm_pair(PyObject*, PyObject* const* args, Py_ssize_t count)
{
    HANDLE_TH_ERRORS
    Tensor x;
    MaybeTensor w1, b1, w2, b2;
    double eps;
    int pcode;
    if (followed() || !take_all(args, count, x, w1, b1, w2, b2, eps) || x.dim() < 1 || type_code(x.scalar_type()) < 0 ||
        !parameters_fit(x, {&w1, &b1, &w2, &b2}, x.size(-1), pcode))
        return not_here();
    return pack(unlocked([&] { return LayerNormPairNode::apply(x, w1, b1, w2, b2, eps, (int64_t)pcode); }));
    END_HANDLE_TH_ERRORS
}

// rms_norm(x, scale, offset, eps, eps_mode, features of the statistics)
PyObject* py_rms_norm(PyObject*, PyObject* const* args, Py_ssize_t count)
{
    HANDLE_TH_ERRORS
    Tensor x;
    MaybeTensor s, o;
    double eps;
    int64_t mode, stat;
    int pcode;
    if (followed() || !take_all(args, count, x, s, o, eps, mode, stat) || x.dim() < 1 || type_code(x.scalar_type()) < 0 ||
        !parameters_fit(x, {&s, &o}, x.size(-1), pcode) || mode < 0 || mode > 2 || stat < 1 || stat > x.size(-1))
        return not_here();
    return THPVariable_Wrap(unlocked([&] { return RMSNormNode::apply(x, s, o, eps, mode, stat, (int64_t)pcode); }));
    END_HANDLE_TH_ERRORS
}

// bias_gelu(x, bias)
PyObject* py_bias_gelu(PyObject*, PyObject* const* args, Py_ssize_t count)
{
    HANDLE_TH_ERRORS
    Tensor x;
    MaybeTensor b;
    if (followed() || !take_all(args, count, x, b) || x.dim() < 1 || type_code(x.scalar_type()) < 0) return not_here();
    if (b && (b->dim() != 1 || b->size(0) != x.size(-1) || !alike(*b, x))) return not_here();
    return THPVariable_Wrap(unlocked([&] { return BiasGeluNode::apply(x, b); }));
    END_HANDLE_TH_ERRORS
}

// gated(x, activation code)
PyObject* py_gated(PyObject*, PyObject* const* args, Py_ssize_t count)
{
    HANDLE_TH_ERRORS
    Tensor x;
    int64_t act;
    if (followed() || !take_all(args, count, x, act) || x.dim() < 1 || x.size(-1) % 2 || type_code(x.scalar_type()) < 0) return not_here();
    return THPVariable_Wrap(unlocked([&] { return GatedNode::apply(x, act); }));
    END_HANDLE_TH_ERRORS
}

// causal_softmax(scores, scale, window)
PyObject* py_causal_softmax(PyObject*, PyObject* const* args, Py_ssize_t count)
{
    HANDLE_TH_ERRORS
    Tensor x;
    double scale;
    int64_t window;
    if (followed() || !take_all(args, count, x, scale, window) || x.dim() != 4 || x.size(2) != x.size(3) || !is_half(x) || !x.is_contiguous())
        return not_here();
    return THPVariable_Wrap(unlocked([&] { return CausalSoftmaxNode::apply(x, scale, window); }));
    END_HANDLE_TH_ERRORS
}

// masked_softmax(scores, mask, scale)
PyObject* py_masked_softmax(PyObject*, PyObject* const* args, Py_ssize_t count)
{
    HANDLE_TH_ERRORS
    Tensor x, mask;
    double scale;
    if (followed() || !take_all(args, count, x, mask, scale) || x.dim() != 4 || mask.dim() != 4 || !is_half(x) || mask.requires_grad() ||
        mask.element_size() != 1 || mask.device() != x.device() || x.size(2) < 2 || (mask.size(0) != 1 && mask.size(0) != x.size(0)) ||
        mask.size(1) != 1 || mask.size(2) != x.size(2) || mask.size(3) != x.size(3))
        return not_here();
    return THPVariable_Wrap(unlocked([&] { return MaskedSoftmaxNode::apply(x, mask, scale); }));
    END_HANDLE_TH_ERRORS
}

// rotary(q, k, cos, sin, offset)
PyObject* py_rotary(PyObject*, PyObject* const* args, Py_ssize_t count)
{
    HANDLE_TH_ERRORS
    Tensor q, k, cos, sin;
    int64_t offset;
    if (followed() || !take_all(args, count, q, k, cos, sin, offset) || q.dim() != 4 || k.dim() != 4 || type_code(q.scalar_type()) < 0 ||
        !alike(q, k) || q.size(0) != k.size(0) || q.size(1) != k.size(1) || q.size(3) != k.size(3) ||
        !tables_fit(cos, sin, q, q.size(3), q.size(0), offset))
        return not_here();
    return pack(unlocked([&] { return RotaryNode::apply(q, k, table_rows(cos, offset, q.size(0)), table_rows(sin, offset, q.size(0))); }));
    END_HANDLE_TH_ERRORS
}

// split_rotary(projection, cos, sin, offset, heads, key/value heads), both 0 for one that is [sq, b, np, 3 * hn]
PyObject* py_split_rotary(PyObject*, PyObject* const* args, Py_ssize_t count)
{
    HANDLE_TH_ERRORS
    Tensor mixed, cos, sin;
    int64_t offset, heads, kv_heads;
    if (followed() || !take_all(args, count, mixed, cos, sin, offset, heads, kv_heads) || type_code(mixed.scalar_type()) < 0 ||
        mixed.dim() != (heads == 0 ? 4 : 3) || heads < 0 || (heads > 0 && kv_heads < 1) || mixed.stride(-1) != 1)
        return not_here();
    const int64_t divided = heads == 0 ? 3 : heads + 2 * kv_heads, hn = mixed.size(-1) / divided;
    if (mixed.size(-1) % divided || !tables_fit(cos, sin, mixed, hn, mixed.size(0), offset)) return not_here();
    return pack(unlocked([&] { return SplitRotaryNode::apply(mixed, table_rows(cos, offset, mixed.size(0)), table_rows(sin, offset, mixed.size(0)), heads, kv_heads); }));
    END_HANDLE_TH_ERRORS
}

bool bias_fits(const MaybeTensor& b, const Tensor& x) { return !b || (b->dim() == 1 && b->size(0) == x.size(-1) && alike(*b, x)); }

// add_residual(x, bias, residual)
PyObject* py_add_residual(PyObject*, PyObject* const* args, Py_ssize_t count)
{
    HANDLE_TH_ERRORS
    Tensor x;
    MaybeTensor b, r;
    if (followed() || !take_all(args, count, x, b, r) || x.dim() < 1 || type_code(x.scalar_type()) < 0 || !bias_fits(b, x) ||
        (r && (r->sizes() != x.sizes() || !alike(*r, x))))
        return not_here();
    return THPVariable_Wrap(unlocked([&] { return AddResidualNode::apply(x, b, r); }));
    END_HANDLE_TH_ERRORS
}

// add_residual_pair(x1, bias1, x2, bias2, residual)
PyObject* py_add_residual_pair(PyObject*, PyObject* const* args, Py_ssize_t count)
{
    HANDLE_TH_ERRORS
    Tensor x1, x2, r;
    MaybeTensor b1, b2;
    if (followed() || !take_all(args, count, x1, b1, x2, b2, r) || x1.dim() < 1 || type_code(x1.scalar_type()) < 0 || !bias_fits(b1, x1) ||
        !bias_fits(b2, x1) || x2.sizes() != x1.sizes() || !alike(x2, x1) || r.sizes() != x1.sizes() || !alike(r, x1))
        return not_here();
    return THPVariable_Wrap(unlocked([&] { return AddResidualPairNode::apply(x1, b1, x2, b2, r); }));
    END_HANDLE_TH_ERRORS
}

// causal_attention(q, k, v, scale, window or -1, merged)
PyObject* py_causal_attention(PyObject*, PyObject* const* args, Py_ssize_t count)
{
    HANDLE_TH_ERRORS
    Tensor q, k, v;
    double scale;
    int64_t window;
    bool merged;
    if (followed() || !take_all(args, count, q, k, v, scale, window, merged) || !attention_fits(q, k, v)) return not_here();
    return THPVariable_Wrap(unlocked([&] { return CausalAttentionNode::apply(q, k, v, scale, window, merged, wants_grad({&q, &k, &v})); }));
    END_HANDLE_TH_ERRORS
}

// masked_attention(q, k, v, mask, scale, fill, merged); the caller has seen that mask and operands fit and nobody differentiates
PyObject* py_masked_attention(PyObject*, PyObject* const* args, Py_ssize_t count)
{
    HANDLE_TH_ERRORS
    Tensor q, k, v, mask;
    double scale, fill;
    bool merged;
    if (followed() || !take_all(args, count, q, k, v, mask, scale, fill, merged) || !attention_fits(q, k, v) || wants_grad({&q, &k, &v})) return not_here();
    const int64_t sq = q.size(0), b = q.size(1), sk = k.size(0);
    if (mask.scalar_type() != at::kBool || mask.device() != q.device() || mask.dim() != 4 || (mask.size(0) != 1 && mask.size(0) != b) ||
        mask.size(1) != 1 || mask.size(2) != sq || mask.size(3) != sk || sk > 65536 || mask.size(0) * sq >= (1 << 26))
        return not_here();
    return THPVariable_Wrap(unlocked([&] {
        const at::NoGradGuard no_grad;
        const c10::DeviceGuard guard(q.device());
        q = readable(q);
        k = readable(k);
        v = readable(v);
        mask = mask.contiguous();
        const Tensor bits = at::empty({mask.size(0), sq, (sk + 63) / 64}, q.options().dtype(at::kLong));
        auto [out, out_strides] = new_context(q, merged);
        check(nhp_attention_mask_bits(bits.data_ptr(), mask.data_ptr(), mask.size(0), sq, sk, stream_of(q)), "masked_attention");
        check(nhp_attention_fwd_keep(out.data_ptr(), nullptr, nullptr, q.data_ptr(), k.data_ptr(), v.data_ptr(), bits.data_ptr(), mask.size(0),
                                     (float)fill, (float)scale, -1, b, q.size(2), k.size(2), sq, sk, q.size(3), Strides3(q).s, Strides3(k).s,
                                     Strides3(v).s, out_strides.s, type_code(q.scalar_type()), stream_of(q)), "masked_attention");
        return out;
    }));
    END_HANDLE_TH_ERRORS
}

// Cached keys or values as the kernels read them
bool rows_readable(const Tensor& past)
{
    return past.stride(4) == 1 && ((past.stride(0) | past.stride(1) | past.stride(2) | past.stride(3)) & 7) == 0 && past.stride(1) < (1 << 24) &&
           reinterpret_cast<uintptr_t>(past.data_ptr()) % 16 == 0;
}

bool cache_fits(const Tensor& k, const Tensor& v, int64_t past)
{
    if (!is_half(k) || k.dim() != 4 || v.sizes() != k.sizes() || !alike(k, v)) return false;
    const int64_t sk = past + k.size(0), heads = k.size(1) * k.size(2), hn = k.size(3);
    return hn % 8 == 0 && heads * hn < (1 << 24) && sk < (1 << 24) && sk * heads < ((int64_t)1 << 31);
}

bool continues(const Tensor& past, const Tensor& k)
{
    return past.dim() == 5 && past.size(0) == 2 && past.size(2) == k.size(1) && past.size(3) == k.size(2) && past.size(4) == k.size(3) &&
           alike(past, k);
}

Strides3 past_strides(const Tensor& past)
{
    return {past.size(1) > 1 ? past.stride(1) : 0, past.size(2) > 1 ? past.stride(2) : 0, past.size(3) > 1 ? past.stride(3) : 0};
}

// decode_attention(q, k, v, layer_past, mask, scale, fill, merged) -> (context, present); the caller has seen that they fit
PyObject* py_decode_attention(PyObject*, PyObject* const* args, Py_ssize_t count)
{
    HANDLE_TH_ERRORS
    Tensor q, k, v, past, mask;
    double scale, fill;
    bool merged;
    if (followed() || !take_all(args, count, q, k, v, past, mask, scale, fill, merged) || !attention_fits(q, k, v) || !continues(past, k) ||
        !rows_readable(past) || !cache_fits(k, v, past.size(1)) || wants_grad({&q, &k, &v, &past}))
        return not_here();
    const int64_t sq = q.size(0), b = q.size(1), np = q.size(2), hn = q.size(3), nkv = k.size(2), n = past.size(1), sk = n + sq;
    if (k.size(0) != sq || sk < 4 || sq * (np / nkv) > 32 || mask.scalar_type() != at::kBool || mask.device() != q.device() || mask.dim() != 4 ||
        (mask.size(0) != 1 && mask.size(0) != b) || mask.size(1) != 1 || mask.size(2) != sq || mask.size(3) != sk)
        return not_here();
    return pack(unlocked([&] {
        const at::NoGradGuard no_grad;
        const c10::DeviceGuard guard(q.device());
        q = readable(q);
        k = readable(k);
        v = readable(v);
        if (mask.stride(3) != 1) mask = mask.contiguous();
        auto [out, out_strides] = new_context(q, merged);
        Tensor present = at::empty({2, sk, b, nkv, hn}, k.options());
        const Tensor ws = bytes(nhp_attention_decode_workspace_bytes(b, np, nkv, sq, n, hn), q);
        const char* keys = static_cast<const char*>(past.data_ptr());
        const Strides3 ps = past_strides(past);
        check(nhp_attention_decode(out.data_ptr(), present.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(), keys, keys + 2 * past.stride(0),
                                   mask.data_ptr(), mask.size(0) > 1 ? mask.stride(0) : 0, mask.stride(2), (float)fill, ptr(ws), (float)scale, b, np,
                                   nkv, sq, n, hn, out_strides.s, Strides3(q).s, Strides3(k).s, Strides3(v).s, ps.s, ps.s,
                                   type_code(q.scalar_type()), stream_of(q)), "decode_attention");
        return variable_list{out, present};
    }));
    END_HANDLE_TH_ERRORS
}

// append_to_cache(k, v, layer_past or None) -> present; the caller has seen that they fit
PyObject* py_append_to_cache(PyObject*, PyObject* const* args, Py_ssize_t count)
{
    HANDLE_TH_ERRORS
    Tensor k, v;
    MaybeTensor past;
    if (followed() || !take_all(args, count, k, v, past) || wants_grad({&k, &v}) || !cache_fits(k, v, past ? past->size(1) : 0)) return not_here();
    if (past && (!continues(*past, k) || !rows_readable(*past) || wants_grad({&*past}))) return not_here();
    return THPVariable_Wrap(unlocked([&] {
        const at::NoGradGuard no_grad;
        const c10::DeviceGuard guard(k.device());
        k = readable(k);
        v = readable(v);
        const int64_t n = past ? past->size(1) : 0, sq = k.size(0), b = k.size(1), nkv = k.size(2), hn = k.size(3);
        Tensor present = at::empty({2, n + sq, b, nkv, hn}, k.options());
        const char* keys = past ? static_cast<const char*>(past->data_ptr()) : nullptr;
        const Strides3 ps = past ? past_strides(*past) : Strides3(0, 0, 0);
        check(nhp_kv_cache_append(present.data_ptr(), k.data_ptr(), v.data_ptr(), keys, past ? keys + 2 * past->stride(0) : nullptr, b, nkv, sq, n, hn,
                                  Strides3(k).s, Strides3(v).s, past ? ps.s : nullptr, past ? ps.s : nullptr, type_code(k.scalar_type()), stream_of(k)),
              "append_to_cache");
        return present;
    }));
    END_HANDLE_TH_ERRORS
}

// Whether nobody differentiates x W^T, the operands as the kernels read them
bool rows_ready(const Tensor& x, const Tensor& w, const MaybeTensor& b)
{
    if (followed() || at::autocast::is_autocast_enabled(at::kCUDA) || x.dim() < 1 || w.dim() != 2 || !is_half(x) || !alike(x, w)) return false;
    const int64_t n = w.size(0), k = w.size(1);
    return x.size(-1) == k && k % 32 == 0 && k <= 16384 && n % 16 == 0 && n <= (1 << 24) && w.is_contiguous() && x.is_contiguous() &&
           reinterpret_cast<uintptr_t>(x.data_ptr()) % 16 == 0 && reinterpret_cast<uintptr_t>(w.data_ptr()) % 16 == 0 &&
           (!b || (b->dim() == 1 && b->size(0) == n && alike(*b, x) && b->is_contiguous() && !wants_grad({&*b}))) && !wants_grad({&x, &w});
}

bool are_few(const Tensor& x, const Tensor& w, int64_t most, int64_t most_split)
{
    const int64_t n = w.size(0), k = w.size(1);
    return x.numel() <= (std::min(n, k) <= 2048 || k > 4096 ? most_split : most) * k;
}

bool few_rows(const Tensor& x, const Tensor& w, const MaybeTensor& b, int64_t most, int64_t most_split)
{
    return rows_ready(x, w, b) && are_few(x, w, most, most_split);
}

Tensor new_rows(const Tensor& x, int64_t width)
{
    auto shape = x.sizes().vec();
    shape.back() = width;
    return at::empty(shape, x.options());
}

// linear(x, weight, bias, most rows, most rows of a layer that is narrow or split): x W^T (+ bias)
PyObject* py_linear(PyObject*, PyObject* const* args, Py_ssize_t count)
{
    HANDLE_TH_ERRORS
    Tensor x, w;
    MaybeTensor b;
    int64_t most, most_split;
    if (!take_all(args, count, x, w, b, most, most_split) || !rows_ready(x, w, b)) return not_here();
    const int64_t n = w.size(0), k = w.size(1), rows = x.numel() / k;
    const bool few = are_few(x, w, most, most_split);
    if (!few && (!nhp_linear_tiles_pay(rows, n, k) || (b && reinterpret_cast<uintptr_t>(b->data_ptr()) % 16))) return not_here();
    return THPVariable_Wrap(unlocked([&] {
        const at::NoGradGuard no_grad;
        const c10::DeviceGuard guard(x.device());
        Tensor y = new_rows(x, n);
        if (!few) {
            check(nhp_linear_tiles(y.data_ptr(), x.data_ptr(), w.data_ptr(), ptr(b), rows, n, k, type_code(x.scalar_type()), stream_of(x)), "linear");
            return y;
        }
        const Tensor ws = bytes(nhp_linear_decode_workspace_bytes(rows, n, k), x);
        check(nhp_linear_decode(y.data_ptr(), x.data_ptr(), w.data_ptr(), ptr(b), ptr(ws), rows, n, k, type_code(x.scalar_type()), stream_of(x)), "linear");
        return y;
    }));
    END_HANDLE_TH_ERRORS
}

// linear_act(x, weight, bias, act, most rows, most rows ..): the activation of x W^T
PyObject* py_linear_act(PyObject*, PyObject* const* args, Py_ssize_t count)
{
    HANDLE_TH_ERRORS
    Tensor x, w;
    MaybeTensor b;
    int64_t act, most, most_split;
    if (!take_all(args, count, x, w, b, act, most, most_split) || !few_rows(x, w, b, most, most_split)) return not_here();
    const bool gated = act != NHP_LINEAR_BIAS_GELU;
    if (gated && (b || w.size(0) % 32 || act < NHP_GATE_SWISH || act > NHP_GATE_IDENTITY)) return not_here();
    return THPVariable_Wrap(unlocked([&] {
        const at::NoGradGuard no_grad;
        const c10::DeviceGuard guard(x.device());
        const int64_t n = w.size(0), k = w.size(1), rows = x.numel() / k;
        Tensor y = new_rows(x, gated ? n / 2 : n);
        const Tensor ws = bytes(nhp_linear_decode_workspace_bytes(rows, n, k), x);
        check(nhp_linear_decode_act(y.data_ptr(), x.data_ptr(), w.data_ptr(), ptr(b), ptr(ws), rows, n, k, (int)act, type_code(x.scalar_type()),
                                    stream_of(x)), "linear and activation");
        return y;
    }));
    END_HANDLE_TH_ERRORS
}

// linear_add(x, weight, bias, x1, bias1, residual, most rows, most rows ..): residual + (x W^T + bias), or with x1
// residual + ((x1 + bias1) + (x W^T + bias))
PyObject* py_linear_add(PyObject*, PyObject* const* args, Py_ssize_t count)
{
    HANDLE_TH_ERRORS
    Tensor x, w, r;
    MaybeTensor b, x1, b1;
    int64_t most, most_split;
    if (!take_all(args, count, x, w, b, x1, b1, r, most, most_split) || !few_rows(x, w, b, most, most_split) || (b1 && !x1)) return not_here();
    const int64_t n = w.size(0), k = w.size(1), rows = x.numel() / k;
    if (r.dim() != x.dim() || r.size(-1) != n || r.numel() != rows * n || !alike(r, x) || !r.is_contiguous() || wants_grad({&r})) return not_here();
    for (int64_t i = 0; i + 1 < x.dim(); ++i)
        if (r.size(i) != x.size(i)) return not_here();
    if (x1 && (x1->sizes() != r.sizes() || !alike(*x1, x) || !x1->is_contiguous() || wants_grad({&*x1}))) return not_here();
    if (b1 && (b1->dim() != 1 || b1->size(0) != n || !alike(*b1, x) || !b1->is_contiguous() || wants_grad({&*b1}))) return not_here();
    return THPVariable_Wrap(unlocked([&] {
        const at::NoGradGuard no_grad;
        const c10::DeviceGuard guard(x.device());
        Tensor y = new_rows(x, n);
        const Tensor ws = bytes(nhp_linear_decode_workspace_bytes(rows, n, k), x);
        check(nhp_linear_decode_add(y.data_ptr(), x.data_ptr(), w.data_ptr(), ptr(b), ptr(x1), ptr(b1), r.data_ptr(), ptr(ws), rows, n, k,
                                    type_code(x.scalar_type()), stream_of(x)), "linear and residual");
        return y;
    }));
    END_HANDLE_TH_ERRORS
}

#define NATIVE(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_##name)), METH_FASTCALL, nullptr}
PyMethodDef kMethods[] = {NATIVE(layer_norm),       NATIVE(layer_norm_pair),  NATIVE(rms_norm),          NATIVE(bias_gelu),
                          NATIVE(gated),            NATIVE(causal_softmax),   NATIVE(masked_softmax),    NATIVE(rotary),
                          NATIVE(split_rotary),     NATIVE(add_residual),     NATIVE(add_residual_pair), NATIVE(causal_attention),
                          NATIVE(masked_attention), NATIVE(decode_attention), NATIVE(append_to_cache),   NATIVE(linear),
                          NATIVE(linear_act),       NATIVE(linear_add),
                          {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

// BUILT_FOR: the versions of torch, of Python and of the library's interface that this file was compiled against
PyMODINIT_FUNC PyInit__native()
{
    PyObject* module = PyModule_Create(&kModule);
    if (!module) return nullptr;
    PyObject* versions = Py_BuildValue("(ssi)", NHP_TORCH_VERSION, Py_STRINGIFY(PY_MAJOR_VERSION) "." Py_STRINGIFY(PY_MINOR_VERSION), NHP_ABI_VERSION);
    if (!versions || PyModule_AddObject(module, "BUILT_FOR", versions) < 0) {
        Py_XDECREF(versions);
        Py_DECREF(module);
        return nullptr;
    }
    return module;
}
