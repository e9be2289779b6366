// Native autograd kernels of the row and fused training operators (AutogradCUDA).
//
// The operators, their schemas, fake implementations, device kernels and backward operators
// are registered from Python (ops/activation_execution.py, ops/fused_training.py). Their
// generated Python autograd functions cost more host time than the kernels take at small
// sizes: RMSNorm forward and backward of 512 x 1280 took 157 us for 22 us of kernels. These
// record the same graph from C++: same saved tensors, same backward operators. Differences
// in work only: gradients of the auxiliary outputs (saved projections, BF16 weights, rstd)
// are not materialized, so no zero tensors are filled for outputs that nothing reads
// (86 us per pass of the 16384 x 2048 x 5632 SwiGLU block).
//
// They dispatch below autograd and nothing else: fake tensors, tracing, functorch and
// saved-tensor hooks see the operators as before. A call that records nothing (no_grad, or no
// input that requires a gradient) goes straight to the operator's kernel, as the Python
// functions do: a node would refuse forward-mode tensors there. A backward under create_graph
// goes through the backward operator's own autograd kernel, which refuses to be differentiated.
#include <torch/csrc/autograd/custom_function.h>
#include <torch/library.h>

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::Function;
using torch::autograd::variable_list;

template <class Signature>
c10::TypedOperatorHandle<Signature> find(const char* name) {
  return c10::Dispatcher::singleton().findSchemaOrThrow(name, "").typed<Signature>();
}

// The operator below autograd, as a forward calls its kernel.
template <class Op, class... Args>
auto below(const Op& op, Args&&... args) {
  at::AutoDispatchBelowAutograd guard;
  return op.call(std::forward<Args>(args)...);
}
// Whether a call with these inputs records a node.
template <class... Inputs>
bool records(const Inputs&... inputs) {
  return at::GradMode::is_enabled() && (inputs.requires_grad() || ...);
}
// A backward operator: below autograd, unless its own gradient is being recorded.
template <class Op, class... Args>
auto backward_op(const Op& op, Args&&... args) {
  if (at::GradMode::is_enabled()) return op.call(std::forward<Args>(args)...);
  return below(op, std::forward<Args>(args)...);
}

// The incoming gradient, zeros when only auxiliary outputs were differentiated.
Tensor grad_or_zeros(const Tensor& grad, const Tensor& like, c10::SymIntArrayRef sizes) {
  return grad.defined() ? grad : at::zeros_symint(sizes, like.options());
}

struct SwigluFn : Function<SwigluFn> {
  static const auto& op() {
    static const auto handle = find<Tensor(const Tensor&, bool)>("warpstate::bf16_swiglu");
    return handle;
  }
  static Tensor forward(AutogradContext* ctx, const Tensor& packed, bool eager) {
    Tensor out = below(op(), packed, eager);
    ctx->save_for_backward({packed});
    ctx->saved_data["eager"] = eager;
    return out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    static auto op = find<Tensor(const Tensor&, const Tensor&, bool)>("warpstate::bf16_swiglu_backward");
    const auto saved = ctx->get_saved_variables();
    return {backward_op(op, saved[0], grads[0], ctx->saved_data["eager"].toBool()), Tensor()};
  }
};

struct RmsnormFn : Function<RmsnormFn> {
  static const auto& op() {
    static const auto handle =
        find<std::tuple<Tensor, Tensor>(const Tensor&, const Tensor&, double, bool)>(
            "warpstate::bf16_rmsnorm");
    return handle;
  }
  // The statistics go out beside the node's one output, a tensor without history: an output
  // marked non-differentiable would be refused by compiled autograd.
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& weight, double eps,
                        bool eager, Tensor* rstd_out) {
    ctx->set_materialize_grads(false);
    auto [y, rstd] = below(op(), x, weight, eps, eager);
    ctx->save_for_backward({x, weight, rstd});
    ctx->saved_data["eager"] = eager;
    *rstd_out = rstd;
    return y;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    static auto op = find<std::tuple<Tensor, Tensor>(const Tensor&, const Tensor&, const Tensor&,
                                                     const Tensor&, bool)>(
        "warpstate::bf16_rmsnorm_backward");
    const auto s = ctx->get_saved_variables();
    auto [dx, dw] = backward_op(op, s[0], s[1], s[2],
                                grad_or_zeros(grads[0], s[0], s[0].sym_sizes()),
                                ctx->saved_data["eager"].toBool());
    return {dx, dw, Tensor(), Tensor(), Tensor()};
  }
};

struct NormProjectionFn : Function<NormProjectionFn> {
  typedef std::tuple<Tensor, Tensor, Tensor, Tensor> Out;
  static const auto& op() {
    static const auto handle = find<Out(const Tensor&, const Tensor&, const Tensor&, double,
                                        c10::SymInt, c10::SymInt)>(
        "warpstate::fused_norm_projection");
    return handle;
  }
  static variable_list forward(AutogradContext* ctx, const Tensor& x, const Tensor& norm_weight,
                               const Tensor& weight, double eps, c10::SymInt gate_begin,
                               c10::SymInt gate_end) {
    ctx->set_materialize_grads(false);
    auto [out, rstd, normed, w] = below(op(), x, norm_weight, weight, eps, gate_begin, gate_end);
    ctx->save_for_backward({x, norm_weight, rstd, normed, w, out});
    ctx->saved_data["gate_begin"] = gate_begin;
    ctx->saved_data["gate_end"] = gate_end;
    return {out, rstd, normed, w};
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    typedef const Tensor& T;
    static auto op = find<std::tuple<Tensor, Tensor, Tensor>(T, T, T, T, T, T, T, c10::SymInt,
                                                             c10::SymInt)>(
        "warpstate::fused_norm_projection_backward");
    const auto s = ctx->get_saved_variables();
    auto [dx, dnorm, dw] =
        backward_op(op, grad_or_zeros(grads[0], s[5], s[5].sym_sizes()), s[0], s[1], s[2], s[3],
                    s[4], s[5], ctx->saved_data["gate_begin"].toSymInt(),
                    ctx->saved_data["gate_end"].toSymInt());
    return {dx, dnorm, dw, Tensor(), Tensor(), Tensor()};
  }
};

// dA and dW of a projection with rows a and BF16 weight w, from dOut.
variable_list projection_grads(const char* name, const Tensor& grad, const Tensor& a,
                               const Tensor& w) {
  typedef std::tuple<Tensor, Tensor> Out;
  const auto op = find<Out(const Tensor&, const Tensor&, const Tensor&)>(name);
  auto [da, dw] = backward_op(op, grad, a, w);
  return {da, dw};
}

struct ResidualProjectionFn : Function<ResidualProjectionFn> {
  static const auto& op() {
    static const auto handle =
        find<std::tuple<Tensor, Tensor>(const Tensor&, const Tensor&, const Tensor&)>(
            "warpstate::fused_residual_projection");
    return handle;
  }
  static variable_list forward(AutogradContext* ctx, const Tensor& a, const Tensor& weight,
                               const Tensor& residual) {
    ctx->set_materialize_grads(false);
    auto [out, w] = below(op(), a, weight, residual);
    ctx->save_for_backward({a, w});
    return {out, w};
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto s = ctx->get_saved_variables();
    const Tensor grad = grad_or_zeros(grads[0], s[0], {s[0].sym_size(0), s[1].sym_size(0)});
    variable_list g = projection_grads("warpstate::fused_residual_projection_backward", grad,
                                       s[0], s[1]);
    return {g[0], g[1], grad};
  }
};

struct LinearFn : Function<LinearFn> {
  static const auto& op() {
    static const auto handle = find<std::tuple<Tensor, Tensor>(const Tensor&, const Tensor&)>(
        "warpstate::fused_linear");
    return handle;
  }
  static variable_list forward(AutogradContext* ctx, const Tensor& a, const Tensor& weight) {
    ctx->set_materialize_grads(false);
    auto [out, w] = below(op(), a, weight);
    ctx->save_for_backward({a, w});
    return {out, w};
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto s = ctx->get_saved_variables();
    return projection_grads("warpstate::fused_linear_backward",
                            grad_or_zeros(grads[0], s[0], {s[0].sym_size(0), s[1].sym_size(0)}),
                            s[0], s[1]);
  }
};

typedef std::tuple<Tensor, Tensor, Tensor, Tensor, Tensor> FiveTensors;

// dH, dW_upgate and dW_down of the SwiGLU block from the saved (h, packed, act, W_ug, W_d).
variable_list swiglu_block_grads(const Tensor& grad, const variable_list& s) {
  typedef const Tensor& T;
  static auto op = find<std::tuple<Tensor, Tensor, Tensor>(T, T, T, T, T, T)>(
      "warpstate::fused_swiglu_block_backward");
  auto [dh, g_upgate, g_down] = backward_op(op, grad, s[0], s[1], s[2], s[3], s[4]);
  return {dh, g_upgate, g_down};
}

Tensor swiglu_block_grad(const variable_list& grads, const variable_list& s) {
  return grad_or_zeros(grads[0], s[0], {s[0].sym_size(0), s[4].sym_size(0)});
}

struct SwigluBlockFn : Function<SwigluBlockFn> {
  static const auto& op() {
    static const auto handle =
        find<FiveTensors(const Tensor&, const Tensor&, const Tensor&, const Tensor&)>(
            "warpstate::fused_swiglu_block");
    return handle;
  }
  static variable_list forward(AutogradContext* ctx, const Tensor& h, const Tensor& w_upgate,
                               const Tensor& w_down, const Tensor& residual) {
    ctx->set_materialize_grads(false);
    auto [out, packed, act, wug, wd] = below(op(), h, w_upgate, w_down, residual);
    ctx->save_for_backward({h, packed, act, wug, wd});
    return {out, packed, act, wug, wd};
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto s = ctx->get_saved_variables();
    const Tensor grad = swiglu_block_grad(grads, s);
    variable_list g = swiglu_block_grads(grad, s);
    return {g[0], g[1], g[2], grad};
  }
};

struct SwigluMlpFn : Function<SwigluMlpFn> {
  static const auto& op() {
    static const auto handle = find<FiveTensors(const Tensor&, const Tensor&, const Tensor&)>(
        "warpstate::fused_swiglu_mlp");
    return handle;
  }
  static variable_list forward(AutogradContext* ctx, const Tensor& h, const Tensor& w_upgate,
                               const Tensor& w_down) {
    ctx->set_materialize_grads(false);
    auto [out, packed, act, wug, wd] = below(op(), h, w_upgate, w_down);
    ctx->save_for_backward({h, packed, act, wug, wd});
    return {out, packed, act, wug, wd};
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto s = ctx->get_saved_variables();
    return swiglu_block_grads(swiglu_block_grad(grads, s), s);
  }
};

std::tuple<Tensor, Tensor> two(const variable_list& v) { return {v[0], v[1]}; }
std::tuple<Tensor, Tensor, Tensor, Tensor> four(const variable_list& v) {
  return {v[0], v[1], v[2], v[3]};
}
FiveTensors five(const variable_list& v) { return {v[0], v[1], v[2], v[3], v[4]}; }

Tensor swiglu(const Tensor& packed, bool eager) {
  if (!records(packed)) return below(SwigluFn::op(), packed, eager);
  return SwigluFn::apply(packed, eager);
}
std::tuple<Tensor, Tensor> rmsnorm(const Tensor& x, const Tensor& weight, double eps, bool eager) {
  if (!records(x, weight)) return below(RmsnormFn::op(), x, weight, eps, eager);
  Tensor rstd;
  Tensor y = RmsnormFn::apply(x, weight, eps, eager, &rstd);
  return {y, rstd};
}
std::tuple<Tensor, Tensor, Tensor, Tensor> norm_projection(const Tensor& x,
                                                           const Tensor& norm_weight,
                                                           const Tensor& weight, double eps,
                                                           c10::SymInt gate_begin,
                                                           c10::SymInt gate_end) {
  if (!records(x, norm_weight, weight))
    return below(NormProjectionFn::op(), x, norm_weight, weight, eps, gate_begin, gate_end);
  return four(NormProjectionFn::apply(x, norm_weight, weight, eps, gate_begin, gate_end));
}
std::tuple<Tensor, Tensor> residual_projection(const Tensor& a, const Tensor& weight,
                                               const Tensor& residual) {
  if (!records(a, weight, residual)) return below(ResidualProjectionFn::op(), a, weight, residual);
  return two(ResidualProjectionFn::apply(a, weight, residual));
}
std::tuple<Tensor, Tensor> linear(const Tensor& a, const Tensor& weight) {
  if (!records(a, weight)) return below(LinearFn::op(), a, weight);
  return two(LinearFn::apply(a, weight));
}
FiveTensors swiglu_block(const Tensor& h, const Tensor& w_upgate, const Tensor& w_down,
                         const Tensor& residual) {
  if (!records(h, w_upgate, w_down, residual))
    return below(SwigluBlockFn::op(), h, w_upgate, w_down, residual);
  return five(SwigluBlockFn::apply(h, w_upgate, w_down, residual));
}
FiveTensors swiglu_mlp(const Tensor& h, const Tensor& w_upgate, const Tensor& w_down) {
  if (!records(h, w_upgate, w_down)) return below(SwigluMlpFn::op(), h, w_upgate, w_down);
  return five(SwigluMlpFn::apply(h, w_upgate, w_down));
}

}  // namespace

TORCH_LIBRARY_IMPL(warpstate, AutogradCUDA, m) {
  m.impl("bf16_swiglu", &swiglu);
  m.impl("bf16_rmsnorm", &rmsnorm);
  m.impl("fused_norm_projection", &norm_projection);
  m.impl("fused_residual_projection", &residual_projection);
  m.impl("fused_linear", &linear);
  m.impl("fused_swiglu_block", &swiglu_block);
  m.impl("fused_swiglu_mlp", &swiglu_mlp);
}
