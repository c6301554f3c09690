// Native torch binding of libenatten.so: the operators enatten::na{1,2}d_{fwd,bwd}
// and the differentiable enatten::natten{1,2}d, registered from C++ so that neither
// the forward nor the backward runs any Python.  (The backward of a Python
// autograd.Function is called on the autograd engine's device thread; measured per
// forward+backward on small inputs, the host side costs about 180 us that way and
// about a third of it from here.)  Host code only: tensors and streams come from
// torch, all device work goes through the C ABI in enatten.h.
//
// Same contract as the reference Functions (e_natten/triton.py:425-483 for 1D,
// :487-548 for 2D): q, k, v of one shape, dtype and device in, one tensor out,
// gradients for q, k and v only.
#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/functions/basic_ops.h>
#include <torch/library.h>

#include <algorithm>
#include <tuple>

#include "enatten.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

int dtype_code(const Tensor &t) {
    switch (t.scalar_type()) {
        case at::kFloat: return ENATTEN_F32;
        case at::kBFloat16: return ENATTEN_BF16;
        case at::kHalf: return ENATTEN_F16;
        case at::kDouble: return ENATTEN_F64;
        default: return -1;
    }
}

// The checks of the Python host side, with the same error classes: ValueError for
// bad shapes, dtypes and kernel sizes, RuntimeError for tensors that are not on
// the GPU.
void validate(const char *what, const Tensor &q, const Tensor &k, const Tensor &v, int64_t ks,
              int64_t ndim, bool check_device = true) {
    TORCH_CHECK_VALUE(q.dim() == ndim, what, ": expected ",
                      ndim == 5 ? "[B, heads, H, W, head_dim]" : "[B, heads, T, head_dim]",
                      " tensors, got ", q.dim(), "-D q");
    TORCH_CHECK_VALUE(k.sizes() == q.sizes() && v.sizes() == q.sizes(), what,
                      ": q, k and v must have the same shape, got ", q.sizes(), ", ", k.sizes(),
                      ", ", v.sizes());
    TORCH_CHECK_VALUE(k.scalar_type() == q.scalar_type() && v.scalar_type() == q.scalar_type(),
                      what, ": q, k and v must share a dtype");
    TORCH_CHECK_VALUE(dtype_code(q) >= 0, what, ": dtype ", q.scalar_type(),
                      " is not supported (float32, bfloat16, float16, float64)");
    TORCH_CHECK_VALUE(k.device() == q.device() && v.device() == q.device(), what,
                      ": q, k and v must be on the same device");
    TORCH_CHECK_VALUE(ks >= 1 && ks % 2 == 1, what, ": kernel_size must be odd and >= 1, got ", ks);
    for (int64_t d = 2; d < ndim - 1; d++)
        TORCH_CHECK_VALUE(q.size(d) >= ks, what, ": input of extent ", q.sizes().slice(2, ndim - 3),
                          " is smaller than kernel_size ", ks);
    TORCH_CHECK_VALUE(q.numel() > 0, what, ": empty tensors are not supported");
    TORCH_CHECK_VALUE(q.size(-1) <= 1024, what, ": head_dim ", q.size(-1),
                      " exceeds the supported maximum of 1024");
    // meta tensors (shape inference under tracing) pass: every operator returns outputs of
    // the right shape for them without touching the library
    TORCH_CHECK(!check_device || q.is_cuda() || q.is_meta(), what,
                ": tensors must be on the GPU; this build has no CPU path");
}

// The kernels take any strides on the leading axes but need unit stride on the
// channel axis.
Tensor kernel_layout(const Tensor &t) {
    return (t.stride(-1) != 1 && t.size(-1) != 1) ? t.contiguous() : t;
}

void check_rc(int rc) {
    if (rc == ENATTEN_OK) return;
    const char *msg = enatten_last_error();
    TORCH_CHECK_VALUE(rc != ENATTEN_EINVAL, msg);
    TORCH_CHECK(false, msg);
}

void check_bwd_extras(const char *what, const Tensor &q, const Tensor &o, const Tensor &d_o) {
    TORCH_CHECK_VALUE(d_o.sizes() == q.sizes() && o.sizes() == q.sizes(), what,
                      ": o and d_o must have the shape of q");
    TORCH_CHECK_VALUE(d_o.scalar_type() == q.scalar_type() && o.scalar_type() == q.scalar_type(),
                      what, ": o and d_o must have the dtype of q");
}

std::tuple<Tensor, Tensor> na2d_fwd(const Tensor &q_, const Tensor &k_, const Tensor &v_,
                                    int64_t ks, double scale) {
    validate("enatten::na2d_fwd", q_, k_, v_, ks, 5);
    if (q_.is_meta())
        return {at::empty_like(kernel_layout(q_)),
                at::empty({q_.size(0), q_.size(1), q_.size(2), q_.size(3)}, q_.options().dtype(at::kFloat))};
    const c10::DeviceGuard guard(q_.device());
    const Tensor q = kernel_layout(q_), k = kernel_layout(k_), v = kernel_layout(v_);
    const int B = q.size(0), N = q.size(1), H = q.size(2), W = q.size(3), D = q.size(4);
    // like the reference's zeros_like(Q) (e_natten/triton.py:502) the output takes the
    // memory order of q
    Tensor o = kernel_layout(at::empty_like(q));
    Tensor lse = at::empty({B, N, H, W}, q.options().dtype(at::kFloat));
    check_rc(enatten2d_fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(),
                           lse.data_ptr<float>(), B, N, H, W, D, (int)ks, dtype_code(q),
                           q.strides().data(), k.strides().data(), v.strides().data(),
                           o.strides().data(), (float)scale,
                           c10::hip::getCurrentHIPStream().stream()));
    return {o, lse};
}

std::tuple<Tensor, Tensor, Tensor> na2d_bwd(const Tensor &q_, const Tensor &k_, const Tensor &v_,
                                            const Tensor &o_, const Tensor &lse_,
                                            const Tensor &d_o_, int64_t ks, double scale) {
    validate("enatten::na2d_bwd", q_, k_, v_, ks, 5);
    check_bwd_extras("enatten::na2d_bwd", q_, o_, d_o_);
    if (q_.is_meta()) {
        const Tensor g = at::empty(q_.sizes(), q_.options());
        return {g, at::empty_like(g), at::empty_like(g)};
    }
    const c10::DeviceGuard guard(q_.device());
    const Tensor q = kernel_layout(q_), k = kernel_layout(k_), v = kernel_layout(v_);
    const Tensor o = kernel_layout(o_), d_o = kernel_layout(d_o_), lse = lse_.contiguous();
    const int B = q.size(0), N = q.size(1), H = q.size(2), W = q.size(3), D = q.size(4);
    Tensor dq = at::empty({B, N, H, W, D}, q.options());
    Tensor dk = at::empty_like(dq), dv = at::empty_like(dq);
    Tensor ws = at::empty({(int64_t)enatten2d_bwd_workspace_bytes(B, N, H, W, D, (int)ks, dtype_code(q))},
                          q.options().dtype(at::kByte));
    check_rc(enatten2d_bwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), d_o.data_ptr(),
                           lse.data_ptr<float>(), dq.data_ptr(), dk.data_ptr(), dv.data_ptr(),
                           ws.data_ptr(), B, N, H, W, D, (int)ks, dtype_code(q),
                           q.strides().data(), k.strides().data(), v.strides().data(),
                           o.strides().data(), d_o.strides().data(), (float)scale,
                           c10::hip::getCurrentHIPStream().stream()));
    return {dq, dk, dv};
}

std::tuple<Tensor, Tensor> na1d_fwd(const Tensor &q_, const Tensor &k_, const Tensor &v_,
                                    int64_t ks, double scale) {
    validate("enatten::na1d_fwd", q_, k_, v_, ks, 4);
    if (q_.is_meta())
        return {at::empty_like(kernel_layout(q_)),
                at::empty({q_.size(0), q_.size(1), q_.size(2)}, q_.options().dtype(at::kFloat))};
    const c10::DeviceGuard guard(q_.device());
    const Tensor q = kernel_layout(q_), k = kernel_layout(k_), v = kernel_layout(v_);
    const int B = q.size(0), N = q.size(1), T = q.size(2), D = q.size(3);
    Tensor o = kernel_layout(at::empty_like(q));
    Tensor lse = at::empty({B, N, T}, q.options().dtype(at::kFloat));
    check_rc(enatten1d_fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(),
                           lse.data_ptr<float>(), B, N, T, D, (int)ks, dtype_code(q),
                           q.strides().data(), k.strides().data(), v.strides().data(),
                           o.strides().data(), (float)scale,
                           c10::hip::getCurrentHIPStream().stream()));
    return {o, lse};
}

std::tuple<Tensor, Tensor, Tensor> na1d_bwd(const Tensor &q_, const Tensor &k_, const Tensor &v_,
                                            const Tensor &o_, const Tensor &lse_,
                                            const Tensor &d_o_, int64_t ks, double scale) {
    validate("enatten::na1d_bwd", q_, k_, v_, ks, 4);
    check_bwd_extras("enatten::na1d_bwd", q_, o_, d_o_);
    if (q_.is_meta()) {
        const Tensor g = at::empty(q_.sizes(), q_.options());
        return {g, at::empty_like(g), at::empty_like(g)};
    }
    const c10::DeviceGuard guard(q_.device());
    const Tensor q = kernel_layout(q_), k = kernel_layout(k_), v = kernel_layout(v_);
    const Tensor o = kernel_layout(o_), d_o = kernel_layout(d_o_), lse = lse_.contiguous();
    const int B = q.size(0), N = q.size(1), T = q.size(2), D = q.size(3);
    Tensor dq = at::empty({B, N, T, D}, q.options());
    Tensor dk = at::empty_like(dq), dv = at::empty_like(dq);
    Tensor ws = at::empty({(int64_t)enatten1d_bwd_workspace_bytes(B, N, T)},
                          q.options().dtype(at::kByte));
    check_rc(enatten1d_bwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), d_o.data_ptr(),
                           lse.data_ptr<float>(), dq.data_ptr(), dk.data_ptr(), dv.data_ptr(),
                           ws.data_ptr(), B, N, T, D, (int)ks, dtype_code(q), q.strides().data(),
                           k.strides().data(), v.strides().data(), o.strides().data(),
                           d_o.strides().data(), (float)scale,
                           c10::hip::getCurrentHIPStream().stream()));
    return {dq, dk, dv};
}

// The composite operators reach the four kernels' operators through the dispatcher, not
// by a C++ call: tensor subclasses and modes above the backend keys (fake tensors under
// torch.compile, functorch wrappers) then see them as opaque operators with a meta kernel.
std::tuple<Tensor, Tensor> call_fwd(bool two_d, const Tensor &q, const Tensor &k, const Tensor &v,
                                    int64_t ks, double scale) {
    using Sig = std::tuple<Tensor, Tensor>(const Tensor &, const Tensor &, const Tensor &, int64_t,
                                           double);
    static const auto op2 =
        c10::Dispatcher::singleton().findSchemaOrThrow("enatten::na2d_fwd", "").typed<Sig>();
    static const auto op1 =
        c10::Dispatcher::singleton().findSchemaOrThrow("enatten::na1d_fwd", "").typed<Sig>();
    return (two_d ? op2 : op1).call(q, k, v, ks, scale);
}
std::tuple<Tensor, Tensor, Tensor> call_bwd(bool two_d, const Tensor &q, const Tensor &k,
                                            const Tensor &v, const Tensor &o, const Tensor &lse,
                                            const Tensor &d_o, int64_t ks, double scale) {
    using Sig = std::tuple<Tensor, Tensor, Tensor>(const Tensor &, const Tensor &, const Tensor &,
                                                   const Tensor &, const Tensor &, const Tensor &,
                                                   int64_t, double);
    static const auto op2 =
        c10::Dispatcher::singleton().findSchemaOrThrow("enatten::na2d_bwd", "").typed<Sig>();
    static const auto op1 =
        c10::Dispatcher::singleton().findSchemaOrThrow("enatten::na1d_bwd", "").typed<Sig>();
    return (two_d ? op2 : op1).call(q, k, v, o, lse, d_o, ks, scale);
}

// One autograd node for both operators: the forward keeps (q, k, v, o, lse), the
// backward returns (dQ, dK, dV) and no gradient for kernel_size and scale.
template <bool TWO_D>
struct NattenFn : public torch::autograd::Function<NattenFn<TWO_D>> {
    static Tensor forward(AutogradContext *ctx, const Tensor &q, const Tensor &k, const Tensor &v,
                          int64_t ks, double scale) {
        at::AutoDispatchBelowADInplaceOrView below;
        Tensor o, lse;
        std::tie(o, lse) = call_fwd(TWO_D, q, k, v, ks, scale);
        ctx->save_for_backward({q, k, v, o, lse});
        ctx->saved_data["kernel_size"] = ks;
        ctx->saved_data["scale"] = scale;
        return o;
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        const variable_list s = ctx->get_saved_variables();
        const int64_t ks = ctx->saved_data["kernel_size"].toInt();
        const double scale = ctx->saved_data["scale"].toDouble();
        at::AutoDispatchBelowADInplaceOrView below;
        Tensor dq, dk, dv;
        std::tie(dq, dk, dv) = call_bwd(TWO_D, s[0], s[1], s[2], s[3], s[4], grads[0], ks, scale);
        return {dq, dk, dv, Tensor(), Tensor()};
    }
};

// Gradients that carry no graph of their own.  Where the upstream gradient requires one
// (create_graph), they are handed on through a node that raises when it is differentiated, as a
// Python function marked once_differentiable does, instead of counting as constants.
variable_list once_differentiable(variable_list out, const variable_list &grads) {
    bool wanted = false;
    for (const Tensor &g : grads) wanted = wanted || (g.defined() && g.requires_grad());
    if (!wanted || !at::GradMode::is_enabled()) return out;
    for (Tensor &t : out)
        if (t.defined()) t = t.detach().set_requires_grad(true);
    return torch::autograd::DelayedError("the gradients of this operator cannot be differentiated again",
                                         (int64_t)out.size())(std::move(out));
}

// Dilated neighborhoods: the contract of enatten2d_fwd_dilated.  The output is contiguous.
void validate_dilation(const char *what, const Tensor &q, const Tensor &k, const Tensor &v, int64_t ks,
                       int64_t dil) {
    validate(what, q, k, v, ks, 5);
    TORCH_CHECK_VALUE(dil >= 1, what, ": dilation must be >= 1, got ", dil);
    TORCH_CHECK_VALUE(std::min(q.size(2), q.size(3)) / dil >= ks, what, ": input of extent ",
                      q.sizes().slice(2, 2), " is smaller than kernel_size * dilation = ", ks, " * ", dil);
}
std::tuple<Tensor, Tensor> na2d_dilated_fwd(const Tensor &q_, const Tensor &k_, const Tensor &v_,
                                            int64_t ks, double scale, int64_t dil) {
    validate_dilation("enatten::na2d_dilated_fwd", q_, k_, v_, ks, dil);
    if (q_.is_meta())
        return {at::empty(q_.sizes(), q_.options()),
                at::empty(q_.sizes().slice(0, 4), q_.options().dtype(at::kFloat))};
    const c10::DeviceGuard guard(q_.device());
    const Tensor q = kernel_layout(q_), k = kernel_layout(k_), v = kernel_layout(v_);
    const int B = q.size(0), N = q.size(1), H = q.size(2), W = q.size(3), D = q.size(4);
    Tensor o = at::empty(q.sizes(), q.options());
    Tensor lse = at::empty({B, N, H, W}, q.options().dtype(at::kFloat));
    check_rc(enatten2d_fwd_dilated(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(),
                                   lse.data_ptr<float>(), B, N, H, W, D, (int)ks, (int)dil, dtype_code(q),
                                   q.strides().data(), k.strides().data(), v.strides().data(),
                                   o.strides().data(), (float)scale,
                                   c10::hip::getCurrentHIPStream().stream()));
    return {o, lse};
}
std::tuple<Tensor, Tensor, Tensor> na2d_dilated_bwd(const Tensor &q_, const Tensor &k_, const Tensor &v_,
                                                    const Tensor &o_, const Tensor &lse_,
                                                    const Tensor &d_o_, int64_t ks, double scale,
                                                    int64_t dil) {
    validate_dilation("enatten::na2d_dilated_bwd", q_, k_, v_, ks, dil);
    check_bwd_extras("enatten::na2d_dilated_bwd", q_, o_, d_o_);
    if (q_.is_meta()) {
        const Tensor g = at::empty(q_.sizes(), q_.options());
        return {g, at::empty_like(g), at::empty_like(g)};
    }
    const c10::DeviceGuard guard(q_.device());
    const Tensor q = kernel_layout(q_), k = kernel_layout(k_), v = kernel_layout(v_);
    const Tensor o = kernel_layout(o_), d_o = kernel_layout(d_o_), lse = lse_.contiguous();
    const int B = q.size(0), N = q.size(1), H = q.size(2), W = q.size(3), D = q.size(4);
    Tensor dq = at::empty(q.sizes(), q.options());
    Tensor dk = at::empty_like(dq), dv = at::empty_like(dq);
    Tensor ws = at::empty({(int64_t)enatten2d_bwd_dilated_workspace_bytes(B, N, H, W, dtype_code(q))},
                          q.options().dtype(at::kByte));
    check_rc(enatten2d_bwd_dilated(
        q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), d_o.data_ptr(), lse.data_ptr<float>(),
        dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), ws.data_ptr(), B, N, H, W, D, (int)ks, (int)dil,
        dtype_code(q), q.strides().data(), k.strides().data(), v.strides().data(), o.strides().data(),
        d_o.strides().data(), (float)scale, c10::hip::getCurrentHIPStream().stream()));
    return {dq, dk, dv};
}
// (through the dispatcher, as call_fwd and call_bwd)
std::tuple<Tensor, Tensor> call_dilated_fwd(const Tensor &q, const Tensor &k, const Tensor &v, int64_t ks,
                                            double scale, int64_t dil) {
    static const auto op = c10::Dispatcher::singleton()
                               .findSchemaOrThrow("enatten::na2d_dilated_fwd", "")
                               .typed<decltype(na2d_dilated_fwd)>();
    return op.call(q, k, v, ks, scale, dil);
}
struct DilatedFn : public torch::autograd::Function<DilatedFn> {
    static Tensor forward(AutogradContext *ctx, const Tensor &q, const Tensor &k, const Tensor &v,
                          int64_t ks, double scale, int64_t dil) {
        at::AutoDispatchBelowADInplaceOrView below;
        Tensor o, lse;
        std::tie(o, lse) = call_dilated_fwd(q, k, v, ks, scale, dil);
        ctx->save_for_backward({q, k, v, o, lse});
        ctx->saved_data["kernel_size"] = ks;
        ctx->saved_data["scale"] = scale;
        ctx->saved_data["dilation"] = dil;
        return o;
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        const variable_list s = ctx->get_saved_variables();
        const int64_t ks = ctx->saved_data["kernel_size"].toInt(), dil = ctx->saved_data["dilation"].toInt();
        const double scale = ctx->saved_data["scale"].toDouble();
        static const auto op = c10::Dispatcher::singleton()
                                   .findSchemaOrThrow("enatten::na2d_dilated_bwd", "")
                                   .typed<decltype(na2d_dilated_bwd)>();
        Tensor dq, dk, dv;
        {
            at::AutoDispatchBelowADInplaceOrView below;
            std::tie(dq, dk, dv) = op.call(s[0], s[1], s[2], s[3], s[4], grads[0], ks, scale, dil);
        }
        return once_differentiable({dq, dk, dv, Tensor(), Tensor(), Tensor()}, grads);
    }
};
Tensor natten2d_dilated_autograd(const Tensor &q, const Tensor &k, const Tensor &v, int64_t ks,
                                 double scale, int64_t dil) {
    return DilatedFn::apply(q, k, v, ks, scale, dil);
}
Tensor natten2d_dilated_plain(const Tensor &q, const Tensor &k, const Tensor &v, int64_t ks,
                              double scale, int64_t dil) {
    return std::get<0>(call_dilated_fwd(q, k, v, ks, scale, dil));
}

// Rectangular and causal windows and the relative position bias (enatten2d_fwd_window): the
// rules of the Python host side, 2D ([B, heads, H, W, d], rpb [heads, 2 kh - 1, 2 kw - 1]) and 1D
// ([B, heads, T, d] as an image of one row, rpb [heads, 2 k - 1]).
struct Window {
    int64_t kh, kw;
    bool ch, cw;
    double scale;
};
void validate_window(const Tensor &q, const Tensor &k, const Tensor &v, const c10::optional<Tensor> &rpb,
                     const Window &w, bool two_d) {
    const char *what = two_d ? "natten2d" : "natten1d";
    validate(what, q, k, v, 1, two_d ? 5 : 4, false);
    auto axis = [&](const char *name, int64_t L, int64_t ks, bool causal) {
        TORCH_CHECK_VALUE(ks >= 1 && (causal || ks % 2 == 1), what, ": kernel_size along ", name,
                          " must be >= 1, and odd unless that axis is causal, got ", ks);
        TORCH_CHECK_VALUE(L >= ks, what, ": input has ", L, " ", name, ", fewer than kernel_size ", ks);
    };
    if (two_d) axis("rows", q.size(2), w.kh, w.ch);
    axis(two_d ? "columns" : "positions", q.size(-2), w.kw, w.cw);
    if (rpb.has_value()) {
        const Tensor &r = *rpb;
        const bool shape_ok = two_d ? r.dim() == 3 && r.size(0) == q.size(1) && r.size(1) == 2 * w.kh - 1 &&
                                          r.size(2) == 2 * w.kw - 1
                                    : r.dim() == 2 && r.size(0) == q.size(1) && r.size(1) == 2 * w.kw - 1;
        TORCH_CHECK_VALUE(shape_ok, what, ": rpb must have shape [heads, 2*kernel_size-1 along each axis], got ", r.sizes());
        TORCH_CHECK_VALUE(r.scalar_type() == q.scalar_type() && r.device() == q.device(), what,
                          ": rpb must have the dtype and device of q");
        TORCH_CHECK_VALUE(!w.ch && !w.cw, what, ": a relative position bias goes with centred axes only");
    }
    TORCH_CHECK(q.is_cuda() || q.is_meta(), what,
                ": tensors must be on the GPU; this build has no CPU path");
}
// (batch, head, row, column) extents and strides of a tensor; a sequence is an image of one row
struct Image {
    int B, N, H, W, D;
    explicit Image(const Tensor &t)
        : B(t.size(0)), N(t.size(1)), H(t.dim() == 5 ? t.size(2) : 1), W(t.size(-2)), D(t.size(-1)) {}
};
struct Strides {
    int64_t s[4];
    explicit Strides(const Tensor &t)
        : s{t.stride(0), t.stride(1), t.dim() == 5 ? t.stride(2) : 0, t.stride(-2)} {}
    operator const int64_t *() const { return s; }
};
// One pair of operators for both: [B, heads, H, W, d] or [B, heads, T, d] with kh = 1, ch = false.
std::tuple<Tensor, Tensor> na_window_fwd(const Tensor &q_, const Tensor &k_, const Tensor &v_,
                                         const c10::optional<Tensor> &rpb_, int64_t kh, int64_t kw, bool ch,
                                         bool cw, double scale) {
    const bool two_d = q_.dim() == 5;
    validate_window(q_, k_, v_, rpb_, Window{kh, kw, ch, cw, scale}, two_d);
    const Image im(q_);
    const auto lse_of = [&] { return at::empty({im.B, im.N, im.H, im.W}, q_.options().dtype(at::kFloat)); };
    if (q_.is_meta()) return {kernel_layout(at::empty_like(kernel_layout(q_))), lse_of()};
    const c10::DeviceGuard guard(q_.device());
    const Tensor q = kernel_layout(q_), k = kernel_layout(k_), v = kernel_layout(v_);
    const Tensor rpb = rpb_.has_value() ? rpb_->contiguous() : Tensor();
    Tensor o = kernel_layout(at::empty_like(q)), lse = lse_of();
    check_rc(enatten2d_fwd_window(q.data_ptr(), k.data_ptr(), v.data_ptr(),
                                  rpb.defined() ? rpb.data_ptr() : nullptr, o.data_ptr(), lse.data_ptr<float>(),
                                  im.B, im.N, im.H, im.W, im.D, (int)kh, (int)kw, ch, cw, dtype_code(q),
                                  Strides(q), Strides(k), Strides(v), Strides(o), (float)scale,
                                  c10::hip::getCurrentHIPStream().stream()));
    return {o, lse};
}
// (dQ, dK, dV, dRPB); without a bias the last one is empty
std::tuple<Tensor, Tensor, Tensor, Tensor> na_window_bwd(const Tensor &q_, const Tensor &k_, const Tensor &v_,
                                                         const c10::optional<Tensor> &rpb_, const Tensor &o_,
                                                         const Tensor &lse_, const Tensor &d_o_, int64_t kh,
                                                         int64_t kw, bool ch, bool cw, double scale) {
    validate_window(q_, k_, v_, rpb_, Window{kh, kw, ch, cw, scale}, q_.dim() == 5);
    check_bwd_extras("enatten::na_window_bwd", q_, o_, d_o_);
    const bool bias = rpb_.has_value();
    Tensor dq, dk, dv, d_rpb;
    const c10::DeviceGuard guard(q_.device());
    dq = at::empty(q_.sizes(), q_.options());
    dk = at::empty_like(dq), dv = at::empty_like(dq);
    d_rpb = at::empty(bias ? rpb_->sizes() : at::IntArrayRef({0}), bias ? q_.options() : q_.options().dtype(at::kFloat));
    if (!q_.is_meta()) {
        const Tensor q = kernel_layout(q_), k = kernel_layout(k_), v = kernel_layout(v_);
        const Tensor o = kernel_layout(o_), d_o = kernel_layout(d_o_), lse = lse_.contiguous();
        const Tensor rpb = bias ? rpb_->contiguous() : Tensor();
        const Image im(q);
        Tensor ws = at::empty({(int64_t)enatten2d_bwd_window_workspace_bytes(im.B, im.N, im.H, im.W, (int)kh,
                                                                             (int)kw, bias)},
                              q.options().dtype(at::kByte));
        check_rc(enatten2d_bwd_window_typed(
            q.data_ptr(), k.data_ptr(), v.data_ptr(), bias ? rpb.data_ptr() : nullptr, o.data_ptr(),
            d_o.data_ptr(), lse.data_ptr<float>(), dq.data_ptr(), dk.data_ptr(), dv.data_ptr(),
            bias ? d_rpb.data_ptr() : nullptr, ws.data_ptr(), im.B, im.N, im.H, im.W, im.D, (int)kh,
            (int)kw, ch, cw, dtype_code(q), Strides(q), Strides(k), Strides(v), Strides(o), Strides(d_o),
            (float)scale, c10::hip::getCurrentHIPStream().stream()));
    }
    return {dq, dk, dv, d_rpb};
}
// (through the dispatcher, as call_fwd and call_bwd)
std::tuple<Tensor, Tensor> call_window_fwd(const Tensor &q, const Tensor &k, const Tensor &v,
                                           const c10::optional<Tensor> &rpb, int64_t kh, int64_t kw, bool ch,
                                           bool cw, double scale) {
    static const auto op = c10::Dispatcher::singleton()
                               .findSchemaOrThrow("enatten::na_window_fwd", "")
                               .typed<decltype(na_window_fwd)>();
    return op.call(q, k, v, rpb, kh, kw, ch, cw, scale);
}
struct WindowFn : public torch::autograd::Function<WindowFn> {
    static Tensor forward(AutogradContext *ctx, const Tensor &q, const Tensor &k, const Tensor &v,
                          const c10::optional<Tensor> &rpb, int64_t kh, int64_t kw, bool ch, bool cw,
                          double scale) {
        at::AutoDispatchBelowADInplaceOrView below;
        Tensor o, lse;
        std::tie(o, lse) = call_window_fwd(q, k, v, rpb, kh, kw, ch, cw, scale);
        ctx->save_for_backward({q, k, v, o, lse, rpb.has_value() ? *rpb : Tensor()});
        ctx->saved_data["kh"] = kh;
        ctx->saved_data["kw"] = kw;
        ctx->saved_data["causal"] = (int64_t)ch | ((int64_t)cw << 1);
        ctx->saved_data["scale"] = scale;
        return o;
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        const variable_list s = ctx->get_saved_variables();
        const int64_t causal = ctx->saved_data["causal"].toInt();
        const c10::optional<Tensor> rpb = s[5].defined() ? c10::optional<Tensor>(s[5]) : c10::nullopt;
        static const auto op = c10::Dispatcher::singleton()
                                   .findSchemaOrThrow("enatten::na_window_bwd", "")
                                   .typed<decltype(na_window_bwd)>();
        Tensor dq, dk, dv, d_rpb;
        {
            at::AutoDispatchBelowADInplaceOrView below;
            std::tie(dq, dk, dv, d_rpb) =
                op.call(s[0], s[1], s[2], rpb, s[3], s[4], grads[0], ctx->saved_data["kh"].toInt(),
                        ctx->saved_data["kw"].toInt(), (causal & 1) != 0, (causal & 2) != 0,
                        ctx->saved_data["scale"].toDouble());
        }
        return once_differentiable({dq, dk, dv, rpb.has_value() ? d_rpb : Tensor(), Tensor(), Tensor(),
                                    Tensor(), Tensor(), Tensor()}, grads);
    }
};
Tensor natten2d_window_autograd(const Tensor &q, const Tensor &k, const Tensor &v,
                                const c10::optional<Tensor> &rpb, int64_t kh, int64_t kw, bool ch, bool cw,
                                double scale) {
    validate_window(q, k, v, rpb, Window{kh, kw, ch, cw, scale}, true);
    return WindowFn::apply(q, k, v, rpb, kh, kw, ch, cw, scale);
}
Tensor natten2d_window_plain(const Tensor &q, const Tensor &k, const Tensor &v,
                             const c10::optional<Tensor> &rpb, int64_t kh, int64_t kw, bool ch, bool cw,
                             double scale) {
    validate_window(q, k, v, rpb, Window{kh, kw, ch, cw, scale}, true);
    return std::get<0>(call_window_fwd(q, k, v, rpb, kh, kw, ch, cw, scale));
}
Tensor natten1d_window_autograd(const Tensor &q, const Tensor &k, const Tensor &v,
                                const c10::optional<Tensor> &rpb, int64_t ks, bool causal, double scale) {
    validate_window(q, k, v, rpb, Window{1, ks, false, causal, scale}, false);
    return WindowFn::apply(q, k, v, rpb, (int64_t)1, ks, false, causal, scale);
}
Tensor natten1d_window_plain(const Tensor &q, const Tensor &k, const Tensor &v,
                             const c10::optional<Tensor> &rpb, int64_t ks, bool causal, double scale) {
    validate_window(q, k, v, rpb, Window{1, ks, false, causal, scale}, false);
    return std::get<0>(call_window_fwd(q, k, v, rpb, 1, ks, false, causal, scale));
}

Tensor natten2d_autograd(const Tensor &q, const Tensor &k, const Tensor &v, int64_t ks,
                         double scale) {
    return NattenFn<true>::apply(q, k, v, ks, scale);
}
Tensor natten1d_autograd(const Tensor &q, const Tensor &k, const Tensor &v, int64_t ks,
                         double scale) {
    return NattenFn<false>::apply(q, k, v, ks, scale);
}
Tensor natten2d_plain(const Tensor &q, const Tensor &k, const Tensor &v, int64_t ks, double scale) {
    return std::get<0>(call_fwd(true, q, k, v, ks, scale));
}
Tensor natten1d_plain(const Tensor &q, const Tensor &k, const Tensor &v, int64_t ks, double scale) {
    return std::get<0>(call_fwd(false, q, k, v, ks, scale));
}

}  // namespace

TORCH_LIBRARY(enatten, m) {
    m.def("na2d_fwd(Tensor q, Tensor k, Tensor v, int kernel_size, float scale) -> (Tensor, Tensor)");
    m.def("na2d_bwd(Tensor q, Tensor k, Tensor v, Tensor o, Tensor lse, Tensor d_o, "
          "int kernel_size, float scale) -> (Tensor, Tensor, Tensor)");
    m.def("na1d_fwd(Tensor q, Tensor k, Tensor v, int kernel_size, float scale) -> (Tensor, Tensor)");
    m.def("na1d_bwd(Tensor q, Tensor k, Tensor v, Tensor o, Tensor lse, Tensor d_o, "
          "int kernel_size, float scale) -> (Tensor, Tensor, Tensor)");
    m.def("na2d_dilated_fwd(Tensor q, Tensor k, Tensor v, int kernel_size, float scale, int dilation) "
          "-> (Tensor, Tensor)");
    m.def("na2d_dilated_bwd(Tensor q, Tensor k, Tensor v, Tensor o, Tensor lse, Tensor d_o, "
          "int kernel_size, float scale, int dilation) -> (Tensor, Tensor, Tensor)");
    m.def("na_window_fwd(Tensor q, Tensor k, Tensor v, Tensor? rpb, int kh, int kw, bool causal_h, "
          "bool causal_w, float scale) -> (Tensor, Tensor)");
    m.def("na_window_bwd(Tensor q, Tensor k, Tensor v, Tensor? rpb, Tensor o, Tensor lse, Tensor d_o, "
          "int kh, int kw, bool causal_h, bool causal_w, float scale) -> (Tensor, Tensor, Tensor, Tensor)");
    m.def("natten2d(Tensor q, Tensor k, Tensor v, int kernel_size=7, float scale=1.0) -> Tensor");
    m.def("natten2d_dilated(Tensor q, Tensor k, Tensor v, int kernel_size, float scale, int dilation) -> Tensor");
    m.def("natten2d_window(Tensor q, Tensor k, Tensor v, Tensor? rpb, int kh, int kw, bool causal_h, "
          "bool causal_w, float scale) -> Tensor");
    m.def("natten1d_window(Tensor q, Tensor k, Tensor v, Tensor? rpb, int kernel_size, bool causal, "
          "float scale) -> Tensor");
    m.def("natten1d(Tensor q, Tensor k, Tensor v, int kernel_size=7, float scale=1.0) -> Tensor");
}

TORCH_LIBRARY_IMPL(enatten, CompositeExplicitAutograd, m) {
    m.impl("na2d_fwd", &na2d_fwd);
    m.impl("na2d_bwd", &na2d_bwd);
    m.impl("na1d_fwd", &na1d_fwd);
    m.impl("na1d_bwd", &na1d_bwd);
    m.impl("na2d_dilated_fwd", &na2d_dilated_fwd);
    m.impl("na2d_dilated_bwd", &na2d_dilated_bwd);
    m.impl("na_window_fwd", &na_window_fwd);
    m.impl("na_window_bwd", &na_window_bwd);
    m.impl("natten2d", &natten2d_plain);
    m.impl("natten2d_dilated", &natten2d_dilated_plain);
    m.impl("natten2d_window", &natten2d_window_plain);
    m.impl("natten1d_window", &natten1d_window_plain);
    m.impl("natten1d", &natten1d_plain);
}

TORCH_LIBRARY_IMPL(enatten, Autograd, m) {
    m.impl("natten2d", &natten2d_autograd);
    m.impl("natten2d_dilated", &natten2d_dilated_autograd);
    m.impl("natten2d_window", &natten2d_window_autograd);
    m.impl("natten1d_window", &natten1d_window_autograd);
    m.impl("natten1d", &natten1d_autograd);
}
