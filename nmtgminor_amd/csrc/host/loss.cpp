// Output projection and loss of GeneratorLoss in training, as one autograd node: the logits are kept once in the working
// dtype, turned into their gradient in place by the backward and contracted there (modules/generator_loss.py, whose Python
// function takes the calls whose logits do not fit the budget). The sum of the losses is a result of the node, so that its
// scalar gradient reaches the loss kernel as it is: no expansion to a row per label, and between the caller's read of the
// loss (the one synchronisation) and the first kernel of the backward lie 40 us of host work instead of 190.
#include "host.h"

namespace nmtg_host {

using torch::autograd::AutogradContext;
using torch::autograd::Function;
using torch::autograd::variable_list;

namespace {

struct LossCall {
  Tensor labels;
  double smoothing;
  int64_t padding_idx;
};

// [n, pitch], the first V columns of each row written; what lies behind them is never used
Tensor project(const Tensor& hidden, const Tensor& weight, const Tensor& bias, void* stream) {
  const int64_t n = hidden.size(0), e = hidden.size(1), v = weight.size(0), pitch = (v + 63) / 64 * 64;
  Tensor full = empty_like_sized(hidden, {n, pitch});
  check(api.gemm(0, 1, n, v, e, 1.f, ptr(hidden), e, 0, ptr(weight), e, 0, ptr(full), pitch, 0, 1, ptr(bias), nullptr, 0, dtype_code(hidden), stream),
        "nmtg_gemm");
  return full;
}

struct GeneratorNode : Function<GeneratorNode> {
  static variable_list forward(AutogradContext* ctx, const Tensor& hidden, const Tensor& weight, const optional<Tensor>& bias_arg, const LossCall* call) {
    const Tensor bias = bias_arg.has_value() ? *bias_arg : Tensor();
    const int64_t n = hidden.size(0), v = weight.size(0);
    Launch on(hidden);
    Tensor full = project(hidden, weight, bias, on.stream);
    Tensor losses = empty_as(hidden, {n}, at::kFloat), lse = empty_as(hidden, {n}, at::kFloat);
    check(api.xentropy_fwd(ptr(full), call->labels.data_ptr<int64_t>(), losses.data_ptr<float>(), lse.data_ptr<float>(), n, v, full.stride(0),
                           static_cast<float>(call->smoothing), call->padding_idx, dtype_code(full), on.stream), "nmtg_xentropy_fwd");
    Tensor total = losses.sum();
    ctx->saved_data["s"] = call->smoothing;
    ctx->saved_data["p"] = call->padding_idx;
    ctx->saved_data["b"] = bias.defined();
    ctx->saved_data["logits"] = full;
    ctx->save_for_backward({hidden, weight, bias, call->labels, lse});
    ctx->set_materialize_grads(false);
    return {losses, total};
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    variable_list r(4);
    if (!grads[0].defined() && !grads[1].defined()) return r;
    auto s = ctx->get_saved_variables();
    const Tensor &hidden = s[0], &weight = s[1], &bias = s[2], &labels = s[3], &lse = s[4];
    const int64_t n = hidden.size(0), e = hidden.size(1), v = weight.size(0);
    Launch on(hidden);
    // a second backward over the same graph finds the logits consumed and projects again
    Tensor full;
    auto kept = ctx->saved_data.find("logits");
    if (kept != ctx->saved_data.end()) {
      full = kept->second.toTensor();
      ctx->saved_data.erase(kept);
    } else {
      full = project(hidden, weight, bias, on.stream);
    }
    Tensor g = !grads[0].defined() ? grads[1].reshape({1}) : grads[1].defined() ? grads[0] + grads[1] : grads[0];
    g = contiguous(g.scalar_type() == at::kFloat ? g : g.to(at::kFloat));
    const bool one = g.numel() == 1 && n > 1, need_b = ctx->saved_data["b"].toBool() && ctx->needs_input_grad(2);
    const float smoothing = static_cast<float>(ctx->saved_data["s"].toDouble());
    const int64_t padding_idx = ctx->saved_data["p"].toInt(), pitch = full.stride(0);
    const int dtype = dtype_code(hidden);
    if (need_b) {
      r[2] = empty_like_sized(weight, {v});
      const Scratch part(hidden, api.xentropy_bwd_colsum_parts(n) * v * static_cast<int64_t>(sizeof(float)));
      check(api.xentropy_bwd_colsum(g.data_ptr<float>(), one ? 0 : 1, ptr(full), lse.data_ptr<float>(), labels.data_ptr<int64_t>(), ptr(full),
                                    ptr(r[2]), part.get<float>(), n, v, pitch, pitch, smoothing, padding_idx, dtype, on.stream),
            "nmtg_xentropy_bwd_colsum");
    } else {
      if (one) g = g.expand({n}).contiguous();
      check(api.xentropy_bwd(g.data_ptr<float>(), ptr(full), lse.data_ptr<float>(), labels.data_ptr<int64_t>(), ptr(full), n, v, pitch, pitch, 0, v,
                             smoothing, padding_idx, dtype, on.stream), "nmtg_xentropy_bwd");
    }
    auto product = [&](int trans_a, int64_t m, int64_t k, const Tensor& b, const Tensor& c) {
      const int64_t bytes = api.gemm_workspace_bytes(m, e, k, 1);
      const Scratch ws(hidden, bytes);
      check(api.gemm(trans_a, 0, m, e, k, 1.f, ptr(full), pitch, 0, ptr(b), e, 0, ptr(c), e, 0, 1, nullptr, ws.get(), bytes, dtype, on.stream),
            "nmtg_gemm");
    };
    if (ctx->needs_input_grad(1)) {
      r[1] = new_like(weight);
      product(1, v, n, hidden, r[1]);                              // [V, N] x [N, E]
    }
    if (ctx->needs_input_grad(0)) {
      r[0] = new_like(hidden);
      product(0, n, v, weight, r[0]);                              // [N, V] x [V, E], the classes split over the chip
    }
    return r;
  }
};

}  // namespace

void define_loss(pybind11::module_& m) {
  // -> (losses [N], their sum), or nothing where the call is not this one (no gradient, or logits beyond keep_bytes)
  m.def("generator_loss", [](const Tensor& hidden, const Tensor& weight, const optional<Tensor>& bias, const Tensor& labels, double smoothing,
                             int64_t padding_idx, int64_t keep_bytes) -> optional<std::tuple<Tensor, Tensor>> {
    const auto type = hidden.scalar_type();
    auto fits = [&](const Tensor& t, at::ScalarType want) { return t.is_cuda() && t.device() == hidden.device() && t.scalar_type() == want; };
    if (!hidden.is_cuda() || (type != at::kHalf && type != at::kBFloat16) || hidden.dim() != 2 || weight.dim() != 2 || labels.dim() != 1 ||
        !fits(weight, type) || !fits(labels, at::kLong) || (bias.has_value() && (!fits(*bias, type) || bias->dim() != 1)))
      return {};
    const int64_t n = hidden.size(0), v = weight.size(0);
    const bool grad = at::GradMode::is_enabled() &&
                      (hidden.requires_grad() || weight.requires_grad() || (bias.has_value() && bias->requires_grad()));
    if (!grad || n == 0 || v == 0 || labels.size(0) != n || weight.size(1) != hidden.size(1) || (bias.has_value() && bias->size(0) != v) ||
        n * ((v + 63) / 64 * 64) * 2 > keep_bytes)
      return {};
    const LossCall call{contiguous(labels), smoothing, padding_idx};
    auto r = GeneratorNode::apply(contiguous(hidden), contiguous(weight), bias.has_value() ? optional<Tensor>(contiguous(*bias)) : bias, &call);
    return std::make_tuple(r[0], r[1]);
  });
}

}  // namespace nmtg_host
