// Autograd formulas of the operators, in C++ on the Autograd key.
//
// A small layer's training step is a handful of kernels of a few microseconds; formulas registered from Python
// (torch.library.register_autograd) put two Python autograd Functions, their contexts and the interpreter lock of the
// backward thread around them, more than the kernels took.  The formulas are the reference's
// (mamtorch/kernel/v4/fullyconnected.py:30-64, mamtorch/kernel/v4/fullyconnected_fast.py:14-39): the forward saves its
// operands and index tensors, the backward calls the namespace's backward operator with the gradient of C alone.  Every
// call goes through the dispatcher, so that fake tensors and tracing see the operators and not their kernels.
#include <ATen/ATen.h>
#include <ATen/core/dispatch/Dispatcher.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/library.h>

#include <vector>

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::Function;
using torch::autograd::variable_list;
typedef std::vector<Tensor> Tensors;
typedef c10::optional<Tensor> MaybeTensor;

template <class Signature>
c10::TypedOperatorHandle<Signature> find(const char *name)
{
    return c10::Dispatcher::singleton().findSchemaOrThrow(name, "").typed<Signature>();
}

bool wants_grad(const Tensor &t) { return t.defined() && t.requires_grad(); }
bool wants_grad(const MaybeTensor &t) { return t.has_value() && wants_grad(*t); }
template <class... T>
bool recording(const T &...t)
{
    return at::GradMode::is_enabled() && (wants_grad(t) || ...);
}

// ---- fullyconnected(a, b) -> [C, argmax, argmin] of v1 and v4 ----
struct V1 {
    static constexpr const char *forward = "mamtorch_kernel_v1::fullyconnected";
    static constexpr const char *backward = "mamtorch_kernel_v1::fullyconnected_backward";
};
struct V4 {
    static constexpr const char *forward = "mamtorch_kernel_v4::fullyconnected";
    static constexpr const char *backward = "mamtorch_kernel_v4::fullyconnected_backward";
};

template <class Names>
Tensors exact_below(const Tensor &a, const Tensor &b)
{
    static const auto op = find<Tensors(Tensor, Tensor)>(Names::forward);
    at::AutoDispatchBelowADInplaceOrView below;
    return op.call(a, b);
}

template <class Names>
struct Exact : public Function<Exact<Names>> {
    static variable_list forward(AutogradContext *ctx, const Tensor &a, const Tensor &b)
    {
        Tensors out = exact_below<Names>(a, b);
        ctx->save_for_backward({a, b, out[1], out[2]});
        ctx->mark_non_differentiable({out[1], out[2]});
        ctx->set_materialize_grads(false);      // no zero-filled gradients for the index outputs
        return out;
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads)
    {
        static const auto op = find<Tensors(Tensor, Tensor, Tensor, Tensor, Tensor)>(Names::backward);
        if (!grads[0].defined()) return {Tensor(), Tensor()};
        const variable_list s = ctx->get_saved_variables();
        const Tensors g = op.call(s[0], s[1], grads[0].contiguous(), s[2], s[3]);
        return {g[0], g[1]};
    }
};

template <class Names>
Tensors exact(const Tensor &a, const Tensor &b)
{
    return recording(a, b) ? Exact<Names>::apply(a, b) : exact_below<Names>(a, b);
}

// ---- fullyconnected_wt(a, weight, bias, hand_over) -> [C, argmax, argmin, sel] ----
Tensors wt_below(const Tensor &a, const Tensor &weight, const MaybeTensor &bias, bool hand_over)
{
    static const auto op = find<Tensors(const Tensor &, const Tensor &, const MaybeTensor &, bool)>(
        "mamtorch_kernel_v4::fullyconnected_wt");
    at::AutoDispatchBelowADInplaceOrView below;
    return op.call(a, weight, bias, hand_over);
}

Tensor bias_grad(const Tensor &g)
{
    static const auto op = find<Tensor(const Tensor &)>("mamtorch_kernel_v4::bias_grad");
    return op.call(g);
}

struct Wt : public Function<Wt> {
    static variable_list forward(AutogradContext *ctx, const Tensor &a, const Tensor &weight, const MaybeTensor &bias,
                                 bool hand_over)
    {
        Tensors out = wt_below(a, weight, bias, hand_over);
        const bool operands = a.requires_grad() || weight.requires_grad();
        ctx->saved_data["operands"] = operands;
        ctx->saved_data["bias"] = bias.has_value() && bias->defined() && bias->requires_grad();
        if (operands)
            ctx->save_for_backward({a, weight, out[1], out[2], out[3]});
        ctx->mark_non_differentiable({out[1], out[2], out[3]});
        ctx->set_materialize_grads(false);
        return out;
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads)
    {
        typedef Tensors Backward(const Tensor &, const Tensor &, const Tensor &, const Tensor &, const Tensor &, const MaybeTensor &);
        static const auto op = find<Backward>("mamtorch_kernel_v4::fullyconnected_wt_backward");
        static const auto op_bias = find<Backward>("mamtorch_kernel_v4::fullyconnected_wt_backward_bias");
        variable_list out(4);
        const Tensor &g = grads[0];
        if (!g.defined()) return out;
        const bool bias = ctx->saved_data["bias"].toBool();
        if (ctx->saved_data["operands"].toBool()) {
            const variable_list s = ctx->get_saved_variables();
            const Tensors all = (bias ? op_bias : op).call(s[0], s[1], g.contiguous(), s[2], s[3], s[4]);
            for (size_t i = 0; i < all.size(); ++i) out[i] = all[i];
        } else if (bias) {
            out[2] = bias_grad(g);
        }
        return out;
    }
};

Tensors fullyconnected_wt(const Tensor &a, const Tensor &weight, const MaybeTensor &bias, bool hand_over)
{
    return recording(a, weight, bias) ? Wt::apply(a, weight, bias, hand_over) : wt_below(a, weight, bias, hand_over);
}

// ---- fullyconnected_ranges(a, weight, bias, range_len, with_indices) -> [C, argmax, argmin] ----
Tensors ranges_below(const Tensor &a, const Tensor &weight, const MaybeTensor &bias, int64_t range_len, bool with_indices)
{
    static const auto op = find<Tensors(const Tensor &, const Tensor &, const MaybeTensor &, int64_t, bool)>(
        "mamtorch_kernel_v4::fullyconnected_ranges");
    at::AutoDispatchBelowADInplaceOrView below;
    return op.call(a, weight, bias, range_len, with_indices);
}

struct Ranges : public Function<Ranges> {
    static variable_list forward(AutogradContext *ctx, const Tensor &a, const Tensor &weight, const MaybeTensor &bias,
                                 int64_t range_len, bool with_indices)
    {
        Tensors out = ranges_below(a, weight, bias, range_len, with_indices);
        ctx->saved_data["operands"] = a.requires_grad() || weight.requires_grad();
        ctx->saved_data["bias"] = bias.has_value() && bias->defined() && bias->requires_grad();
        ctx->saved_data["range_len"] = range_len;
        ctx->saved_data["with_indices"] = with_indices;
        ctx->save_for_backward({a, weight, out[1], out[2]});
        ctx->mark_non_differentiable({out[1], out[2]});
        ctx->set_materialize_grads(false);
        return out;
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads)
    {
        typedef Tensors Backward(const Tensor &, const Tensor &, const Tensor &, const Tensor &, const Tensor &, int64_t);
        static const auto op = find<Backward>("mamtorch_kernel_v4::fullyconnected_ranges_backward");
        static const auto op_bias = find<Backward>("mamtorch_kernel_v4::fullyconnected_ranges_backward_bias");
        variable_list out(5);
        const Tensor &g = grads[0];
        if (!g.defined()) return out;
        const bool bias = ctx->saved_data["bias"].toBool();
        if (ctx->saved_data["operands"].toBool()) {
            TORCH_CHECK(ctx->saved_data["with_indices"].toBool(),
                        "fullyconnected_ranges was run without indices; its gradient needs them");
            const variable_list s = ctx->get_saved_variables();
            const Tensors all =
                (bias ? op_bias : op).call(s[0], s[1], g.contiguous(), s[2], s[3], ctx->saved_data["range_len"].toInt());
            for (size_t i = 0; i < all.size(); ++i) out[i] = all[i];
        } else if (bias) {
            out[2] = bias_grad(g);
        }
        return out;
    }
};

Tensors fullyconnected_ranges(const Tensor &a, const Tensor &weight, const MaybeTensor &bias, int64_t range_len, bool with_indices)
{
    return recording(a, weight, bias) ? Ranges::apply(a, weight, bias, range_len, with_indices)
                                      : ranges_below(a, weight, bias, range_len, with_indices);
}

// ---- fullyconnected_fast(a, b), fullyconnected_fast_wt(a, weight, bias): values only; as in the reference the
// registered backward is the dense multiply-accumulate gradient ----
Tensor fast_below(const Tensor &a, const Tensor &b)
{
    static const auto op = find<Tensor(Tensor, Tensor)>("mamtorch_kernel_v4::fullyconnected_fast");
    at::AutoDispatchBelowADInplaceOrView below;
    return op.call(a, b);
}

struct Fast : public Function<Fast> {
    static Tensor forward(AutogradContext *ctx, const Tensor &a, const Tensor &b)
    {
        ctx->save_for_backward({a, b});
        return fast_below(a, b);
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads)
    {
        const variable_list s = ctx->get_saved_variables();
        return {grads[0].matmul(s[1].t()), s[0].t().matmul(grads[0])};
    }
};

Tensor fullyconnected_fast(const Tensor &a, const Tensor &b)
{
    return recording(a, b) ? Fast::apply(a, b) : fast_below(a, b);
}

Tensor fast_wt_below(const Tensor &a, const Tensor &weight, const MaybeTensor &bias)
{
    static const auto op =
        find<Tensor(const Tensor &, const Tensor &, const MaybeTensor &)>("mamtorch_kernel_v4::fullyconnected_fast_wt");
    at::AutoDispatchBelowADInplaceOrView below;
    return op.call(a, weight, bias);
}

struct FastWt : public Function<FastWt> {
    static Tensor forward(AutogradContext *ctx, const Tensor &a, const Tensor &weight, const MaybeTensor &bias)
    {
        ctx->save_for_backward({a, weight});
        ctx->saved_data["bias"] = bias.has_value() && bias->defined() && bias->requires_grad();
        return fast_wt_below(a, weight, bias);
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads)
    {
        const variable_list s = ctx->get_saved_variables();
        const Tensor &g = grads[0];
        variable_list out(3);
        if (s[0].requires_grad() || s[1].requires_grad()) {
            out[0] = g.matmul(s[1]);
            out[1] = g.t().matmul(s[0]);
        }
        if (ctx->saved_data["bias"].toBool()) out[2] = g.sum(0);
        return out;
    }
};

Tensor fullyconnected_fast_wt(const Tensor &a, const Tensor &weight, const MaybeTensor &bias)
{
    return recording(a, weight, bias) ? FastWt::apply(a, weight, bias) : fast_wt_below(a, weight, bias);
}

// ---- blend(mam, mac, bias, alpha, beta) ----
Tensor blend_below(const Tensor &mam, const Tensor &mac, const MaybeTensor &bias, double alpha, double beta)
{
    static const auto op =
        find<Tensor(const Tensor &, const Tensor &, const MaybeTensor &, double, double)>("mamtorch_kernel_v4::blend");
    at::AutoDispatchBelowADInplaceOrView below;
    return op.call(mam, mac, bias, alpha, beta);
}

struct Blend : public Function<Blend> {
    static Tensor forward(AutogradContext *ctx, const Tensor &mam, const Tensor &mac, const MaybeTensor &bias, double alpha,
                          double beta)
    {
        ctx->saved_data["alpha"] = alpha;
        ctx->saved_data["beta"] = beta;
        ctx->saved_data["mam"] = mam.requires_grad();
        ctx->saved_data["mac"] = mac.requires_grad();
        ctx->saved_data["bias"] = bias.has_value() && bias->defined() && bias->requires_grad();
        return blend_below(mam, mac, bias, alpha, beta);
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads)
    {
        variable_list out(5);
        const Tensor &g = grads[0];
        if (ctx->saved_data["mam"].toBool()) out[0] = g * ctx->saved_data["alpha"].toDouble();
        if (ctx->saved_data["mac"].toBool()) out[1] = g * ctx->saved_data["beta"].toDouble();
        if (ctx->saved_data["bias"].toBool()) out[2] = g.sum(0);
        return out;
    }
};

Tensor blend(const Tensor &mam, const Tensor &mac, const MaybeTensor &bias, double alpha, double beta)
{
    return recording(mam, mac, bias) ? Blend::apply(mam, mac, bias, alpha, beta) : blend_below(mam, mac, bias, alpha, beta);
}

// ---- apply_keep(weight, keep): its gradient is the same masking ----
Tensor keep_below(const Tensor &weight, const Tensor &keep)
{
    static const auto op = find<Tensor(const Tensor &, const Tensor &)>("mamtorch_kernel_v4::apply_keep");
    at::AutoDispatchBelowADInplaceOrView below;
    return op.call(weight, keep);
}

struct Keep : public Function<Keep> {
    static Tensor forward(AutogradContext *ctx, const Tensor &weight, const Tensor &keep)
    {
        ctx->save_for_backward({keep});
        return keep_below(weight, keep);
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads)
    {
        static const auto op = find<Tensor(const Tensor &, const Tensor &)>("mamtorch_kernel_v4::apply_keep");
        return {op.call(grads[0], ctx->get_saved_variables()[0]), Tensor()};
    }
};

Tensor apply_keep(const Tensor &weight, const Tensor &keep)
{
    return recording(weight) ? Keep::apply(weight, keep) : keep_below(weight, keep);
}

// ---- im2col and col2im: each other's adjoint ----
const c10::TypedOperatorHandle<Tensor(const Tensor &, int64_t, int64_t, int64_t, int64_t)> &im2col_op()
{
    static const auto op = find<Tensor(const Tensor &, int64_t, int64_t, int64_t, int64_t)>("mamtorch_kernel_v4::im2col");
    return op;
}

typedef Tensor Col2im(const Tensor &, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t);
const c10::TypedOperatorHandle<Col2im> &col2im_op()
{
    static const auto op = find<Col2im>("mamtorch_kernel_v4::col2im");
    return op;
}

struct ToColumns : public Function<ToColumns> {
    static Tensor forward(AutogradContext *ctx, const Tensor &x, int64_t k1, int64_t k2, int64_t s1, int64_t s2)
    {
        ctx->saved_data["geometry"] = std::vector<int64_t>{x.size(0), x.size(1), x.size(2), x.size(3), k1, k2, s1, s2};
        at::AutoDispatchBelowADInplaceOrView below;
        return im2col_op().call(x, k1, k2, s1, s2);
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads)
    {
        const std::vector<int64_t> v = ctx->saved_data["geometry"].toIntVector();
        variable_list out(5);
        out[0] = col2im_op().call(grads[0].contiguous(), v[0], v[1], v[2], v[3], v[4], v[5], v[6], v[7]);
        return out;
    }
};

struct FromColumns : public Function<FromColumns> {
    static Tensor forward(AutogradContext *ctx, const Tensor &cols, int64_t B, int64_t C, int64_t H, int64_t W, int64_t k1,
                          int64_t k2, int64_t s1, int64_t s2)
    {
        ctx->saved_data["window"] = std::vector<int64_t>{k1, k2, s1, s2};
        at::AutoDispatchBelowADInplaceOrView below;
        return col2im_op().call(cols, B, C, H, W, k1, k2, s1, s2);
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads)
    {
        const std::vector<int64_t> v = ctx->saved_data["window"].toIntVector();
        variable_list out(9);
        out[0] = im2col_op().call(grads[0].contiguous(), v[0], v[1], v[2], v[3]);
        return out;
    }
};

Tensor im2col(const Tensor &x, int64_t k1, int64_t k2, int64_t s1, int64_t s2)
{
    if (recording(x)) return ToColumns::apply(x, k1, k2, s1, s2);
    at::AutoDispatchBelowADInplaceOrView below;
    return im2col_op().call(x, k1, k2, s1, s2);
}

Tensor col2im(const Tensor &cols, int64_t B, int64_t C, int64_t H, int64_t W, int64_t k1, int64_t k2, int64_t s1, int64_t s2)
{
    if (recording(cols)) return FromColumns::apply(cols, B, C, H, W, k1, k2, s1, s2);
    at::AutoDispatchBelowADInplaceOrView below;
    return col2im_op().call(cols, B, C, H, W, k1, k2, s1, s2);
}

// ---- fullyconnected_wt_picks(a, weight, bias) -> [C, picks, sel] ----
Tensors picks_below(const Tensor &a, const Tensor &weight, const MaybeTensor &bias)
{
    static const auto op = find<Tensors(const Tensor &, const Tensor &, const MaybeTensor &)>(
        "mamtorch_kernel_v4::fullyconnected_wt_picks");
    at::AutoDispatchBelowADInplaceOrView below;
    return op.call(a, weight, bias);
}

struct Picks : public Function<Picks> {
    static variable_list forward(AutogradContext *ctx, const Tensor &a, const Tensor &weight, const MaybeTensor &bias)
    {
        Tensors out = picks_below(a, weight, bias);
        const bool operands = a.requires_grad() || weight.requires_grad();
        ctx->saved_data["operands"] = operands;
        ctx->saved_data["bias"] = bias.has_value() && bias->defined() && bias->requires_grad();
        if (operands) ctx->save_for_backward({a, weight, out[1], out[2]});
        ctx->mark_non_differentiable({out[1], out[2]});
        ctx->set_materialize_grads(false);
        return out;
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads)
    {
        static const auto op = find<Tensors(const Tensor &, const Tensor &, const Tensor &, const Tensor &, const Tensor &, bool)>(
            "mamtorch_kernel_v4::fullyconnected_wt_picks_backward");
        variable_list out(3);
        const Tensor &g = grads[0];
        if (!g.defined()) return out;
        const bool bias = ctx->saved_data["bias"].toBool();
        if (ctx->saved_data["operands"].toBool()) {
            const variable_list s = ctx->get_saved_variables();
            const Tensors all = op.call(s[0], s[1], g.contiguous(), s[2], s[3], bias);
            for (size_t i = 0; i < all.size(); ++i) out[i] = all[i];
        } else if (bias) {
            out[2] = bias_grad(g);
        }
        return out;
    }
};

Tensors fullyconnected_wt_picks(const Tensor &a, const Tensor &weight, const MaybeTensor &bias)
{
    return recording(a, weight, bias) ? Picks::apply(a, weight, bias) : picks_below(a, weight, bias);
}

Tensors exact_v1(Tensor a, Tensor b) { return exact<V1>(a, b); }
Tensors exact_v4(Tensor a, Tensor b) { return exact<V4>(a, b); }
Tensor fast_v4(Tensor a, Tensor b) { return fullyconnected_fast(a, b); }

}  // namespace

TORCH_LIBRARY_IMPL(mamtorch_kernel_v1, Autograd, m) { m.impl("fullyconnected", &exact_v1); }

TORCH_LIBRARY_IMPL(mamtorch_kernel_v4, Autograd, m)
{
    m.impl("fullyconnected", &exact_v4);
    m.impl("fullyconnected_fast", &fast_v4);
    m.impl("fullyconnected_wt", &fullyconnected_wt);
    m.impl("fullyconnected_wt_picks", &fullyconnected_wt_picks);
    m.impl("fullyconnected_fast_wt", &fullyconnected_fast_wt);
    m.impl("fullyconnected_ranges", &fullyconnected_ranges);
    m.impl("blend", &blend);
    m.impl("apply_keep", &apply_keep);
    m.impl("im2col", &im2col);
    m.impl("col2im", &col2im);
}
