// Autograd nodes of the single operators (LayerNorm, feed-forward block, cross-entropy, packed attention): what the Python
// autograd functions of nmtgminor_amd/modules do, for tensors on the GPU, without the interpreter between the operator and
// its kernels in either direction.
#include "host.h"

namespace nmtg_host {

using torch::autograd::AutogradContext;
using torch::autograd::Function;
using torch::autograd::variable_list;

namespace {

Tensor saved(const optional<Tensor>& t) { return t.has_value() ? *t : Tensor(); }

// ---------------------------------------------------------------------------------------------------------- LayerNorm
struct LayerNormNode : Function<LayerNormNode> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& gamma, const Tensor& beta, double eps, bool memory_efficient) {
    Norm n = ln_fwd(x, gamma, beta, eps);
    ctx->saved_data["m"] = memory_efficient;
    ctx->save_for_backward({memory_efficient ? n.z : x, n.stats, gamma, memory_efficient ? beta : Tensor()});
    return n.z;
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    auto s = ctx->get_saved_variables();
    Tensor dz = contiguous(g[0]);
    if (dz.scalar_type() != s[2].scalar_type()) dz = dz.to(s[2].scalar_type());
    NormGrads r = ln_bwd(dz, s[0], s[1], s[2], s[3], ctx->saved_data["m"].toBool());
    return {r.dx, r.dgamma, r.dbeta, Tensor(), Tensor()};
  }
};

// ------------------------------------------------------------------------------------------------ dropout + residual
struct DropoutAddNode : Function<DropoutAddNode> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& residual, double p, bool training) {
    Tensor mask = dropout_add_(x, residual, p, training);
    ctx->saved_data["p"] = p;
    ctx->save_for_backward({mask});
    ctx->mark_dirty({x});
    return x;
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    auto s = ctx->get_saved_variables();
    if (!s[0].defined()) return {g[0], g[0], Tensor(), Tensor()};
    Tensor go = contiguous(g[0]);
    return {ctx->needs_input_grad(0) ? dropout_bwd(go, s[0], ctx->saved_data["p"].toDouble()) : Tensor(), g[0], Tensor(), Tensor()};
  }
};

// --------------------------------------------------------------------------------------------- two-layer feed-forward
struct MlpNode : Function<MlpNode> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& w1, const Tensor& w2, const optional<Tensor>& b1,
                        const optional<Tensor>& b2, const optional<Tensor>& mask, double p, int64_t act) {
    Mlp r = mlp_fwd(x, w1, w2, saved(b1), saved(b2), p, act, mask, act != NMTG_ACT_RELU);
    ctx->saved_data["p"] = p;
    ctx->saved_data["a"] = act;
    ctx->saved_data["b1"] = b1.has_value();
    ctx->saved_data["b2"] = b2.has_value();
    ctx->save_for_backward({x, w1, w2, r.post, r.pre, r.mask});
    return r.out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    auto s = ctx->get_saved_variables();
    auto need = [&](int i) { return ctx->needs_input_grad(i); };   // counts the tensors among the arguments: an absent bias does not
    const bool has_b1 = ctx->saved_data["b1"].toBool(), has_b2 = ctx->saved_data["b2"].toBool();
    MlpGrads r = mlp_bwd(contiguous(g[0]), s[0], s[1], s[2], s[3], s[4], s[5], ctx->saved_data["p"].toDouble(), ctx->saved_data["a"].toInt(),
                         need(0), need(1) || need(2), has_b1 && need(3), has_b2 && need(has_b1 ? 4 : 3));
    return {r.dx, r.dw1, r.dw2, r.db1, r.db2, Tensor(), Tensor(), Tensor()};
  }
};

// ------------------------------------------------------------------------------------------------------ cross-entropy
struct XentNode : Function<XentNode> {
  static Tensor forward(AutogradContext* ctx, const Tensor& logits, const Tensor& labels, double smoothing, int64_t padding_idx) {
    const int64_t n = logits.size(0), v = logits.size(1);
    Launch on(logits);
    Tensor losses = empty_as(logits, {n}, at::kFloat), lse = empty_as(logits, {n}, at::kFloat);
    check(api.xentropy_fwd(ptr(logits), labels.data_ptr<int64_t>(), losses.data_ptr<float>(), lse.data_ptr<float>(), n, v, logits.stride(0),
                           static_cast<float>(smoothing), padding_idx, dtype_code(logits), on.stream), "nmtg_xentropy_fwd");
    ctx->saved_data["s"] = smoothing;
    ctx->saved_data["p"] = padding_idx;
    ctx->save_for_backward({logits, lse, labels});
    return losses;
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    auto s = ctx->get_saved_variables();
    const Tensor &logits = s[0], &lse = s[1], &labels = s[2];
    Launch on(logits);
    const int64_t n = logits.size(0), v = logits.size(1);
    Tensor go = contiguous(g[0]);
    Tensor dz = empty_like_sized(logits, {n, v});
    check(api.xentropy_bwd(go.data_ptr<float>(), ptr(logits), lse.data_ptr<float>(), labels.data_ptr<int64_t>(), ptr(dz), n, v,
                           logits.stride(0), v, 0, v, static_cast<float>(ctx->saved_data["s"].toDouble()), ctx->saved_data["p"].toInt(),
                           dtype_code(logits), on.stream), "nmtg_xentropy_bwd");
    return {dz, Tensor(), Tensor(), Tensor()};
  }
};

// --------------------------------------------------------------------------------- attention over packed sequences
struct PackedNode : Function<PackedNode> {
  static Tensor forward(AutogradContext* ctx, const Tensor& qkv, const Tensor& cu, int64_t max_len, double p, double scale, bool causal,
                        Bits* drawn) {
    const int64_t total = qkv.size(0), h = qkv.size(2), d = qkv.size(3), b = cu.numel() - 1;
    Launch on(qkv);
    Tensor out = empty_like_sized(qkv, {total, h, d});
    Tensor lse = empty_as(qkv, {b, h, max_len}, at::kFloat);     // written and read for the rows of the sequences only
    Bits bits;
    if (p > 0.0) {
      bits.mode = 2;
      bits.words = empty_as(qkv, {std::max<int64_t>(api.flash_attn_dropout_bits_bytes(b, h, max_len, max_len), 16) / 4}, at::kInt);
      std::tie(bits.seed, bits.offset) = draw(qkv, 4 * b * h * ((max_len + 3) / 4) * ((max_len + 3) / 4));
    }
    const int64_t st = qkv.stride(0), sh = qkv.stride(2);
    const char* q = static_cast<const char*>(qkv.data_ptr());
    const int64_t slot = qkv.stride(1) * 2;
    check(api.flash_attn_fwd(q, q + slot, q + 2 * slot, ptr(out), cu.data_ptr<int32_t>(), cu.data_ptr<int32_t>(), lse.data_ptr<float>(), b, h,
                             d, max_len, max_len, st, sh, st, sh, st, sh, h * d, d, static_cast<float>(scale), causal ? 1 : 0,
                             static_cast<int>(bits.mode), static_cast<float>(p), nullptr, nullptr, ptr(bits.words), bits.seed, bits.offset,
                             dtype_code(qkv), on.stream), "nmtg_flash_attn_fwd");
    ctx->saved_data["n"] = max_len;
    ctx->saved_data["p"] = p;
    ctx->saved_data["s"] = scale;
    ctx->saved_data["c"] = causal;
    ctx->saved_data["seed"] = static_cast<int64_t>(bits.seed);
    ctx->saved_data["offset"] = static_cast<int64_t>(bits.offset);
    ctx->save_for_backward({qkv, out, lse, cu, bits.words});
    *drawn = bits;
    return out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    auto s = ctx->get_saved_variables();
    const Tensor &qkv = s[0], &out = s[1], &lse = s[2], &cu = s[3], &words = s[4];
    const int64_t h = qkv.size(2), d = qkv.size(3), b = cu.numel() - 1, max_len = ctx->saved_data["n"].toInt();
    Launch on(qkv);
    Tensor dout = g[0].stride(-1) == 1 ? g[0] : g[0].contiguous();
    Tensor dqkv = empty_like_sized(qkv, qkv.sizes());
    const Scratch sd(qkv, b * h * max_len * static_cast<int64_t>(sizeof(float)));
    const int64_t st = qkv.stride(0), sh = qkv.stride(2), slot = qkv.stride(1) * 2;
    const int64_t gt = dqkv.stride(0), gh = dqkv.stride(2), gslot = dqkv.stride(1) * 2;
    const char* q = static_cast<const char*>(qkv.data_ptr());
    char* dq = static_cast<char*>(dqkv.data_ptr());
    check(api.flash_attn_bwd(ptr(dout), q, q + slot, q + 2 * slot, ptr(out), lse.data_ptr<float>(), dq, dq + gslot, dq + 2 * gslot,
                             sd.get<float>(), cu.data_ptr<int32_t>(), cu.data_ptr<int32_t>(), b, h, d, max_len, max_len, dout.stride(0),
                             dout.stride(1), st, sh, st, sh, st, sh, h * d, d, gt, gh, gt, gh, gt, gh,
                             static_cast<float>(ctx->saved_data["s"].toDouble()), ctx->saved_data["c"].toBool() ? 1 : 0,
                             words.defined() ? 2 : 0, static_cast<float>(ctx->saved_data["p"].toDouble()), nullptr, ptr(words),
                             words.defined() ? 1 : 0, static_cast<uint64_t>(ctx->saved_data["seed"].toInt()),
                             static_cast<uint64_t>(ctx->saved_data["offset"].toInt()), dtype_code(qkv), on.stream), "nmtg_flash_attn_bwd");
    return {dqkv, Tensor(), Tensor(), Tensor(), Tensor(), Tensor(), Tensor()};
  }
};

}  // namespace

void define_autograd(pybind11::module_& m) {
  m.def("layer_norm", [](const Tensor& x, const Tensor& gamma, const Tensor& beta, double eps, bool memory_efficient) {
    TORCH_CHECK(gamma.is_cuda() && beta.is_cuda(), "expected a tensor in device memory (HIP); this op has no CPU path");
    TORCH_CHECK(beta.scalar_type() == gamma.scalar_type(), "ln_fwd: beta and gamma dtypes differ");
    TORCH_CHECK(gamma.sizes() == beta.sizes(), "ln_fwd: gamma and beta shapes differ");
    TORCH_CHECK(gamma.numel() > 0 && x.dim() > 0 && x.numel() % gamma.numel() == 0, "ln_fwd: hidden size mismatch");
    TORCH_CHECK(eps >= 0.0, "ln_fwd: epsilon must be >= 0");
    return LayerNormNode::apply(contiguous(x), contiguous(gamma), contiguous(beta), eps, memory_efficient);
  });
  m.def("dropout_add", [](const Tensor& x, const Tensor& residual, double p, bool training) {
    TORCH_CHECK(residual.is_cuda(), "expected a tensor in device memory (HIP); this op has no CPU path");
    TORCH_CHECK(x.scalar_type() == residual.scalar_type(), "fused_dropout_add: dtype mismatch");
    TORCH_CHECK(x.numel() == residual.numel(), "fused_dropout_add: size mismatch");
    return DropoutAddNode::apply(contiguous(x), contiguous(residual), p, training);
  });
  m.def("mlp", [](const Tensor& x, const Tensor& w1, const Tensor& w2, const optional<Tensor>& b1, const optional<Tensor>& b2,
                  const optional<Tensor>& mask, double p, int64_t act) {
    for (const Tensor* t : {&w1, &w2}) {
      TORCH_CHECK(t->is_cuda(), "expected a tensor in device memory (HIP); this op has no CPU path");
      TORCH_CHECK(t->scalar_type() == x.scalar_type() && t->dim() == 2, "mlp: weight shape / dtype mismatch");
    }
    TORCH_CHECK(x.scalar_type() == at::kHalf || x.scalar_type() == at::kBFloat16 || x.scalar_type() == at::kFloat,
                "mlp: fp32, fp16 and bf16 are supported (there is no fp64 kernel)");
    TORCH_CHECK(w1.size(1) == x.size(-1) && w2.size(1) == w1.size(0), "mlp: weight shape / dtype mismatch");
    optional<Tensor> b[2] = {b1, b2};
    for (int i = 0; i < 2; ++i)
      if (b[i].has_value()) {
        TORCH_CHECK(b[i]->is_cuda(), "expected a tensor in device memory (HIP); this op has no CPU path");
        TORCH_CHECK(b[i]->scalar_type() == x.scalar_type() && b[i]->numel() == (i ? w2 : w1).size(0), "mlp: bias shape / dtype mismatch");
        b[i] = contiguous(*b[i]);
      }
    const bool grad = at::GradMode::is_enabled() && (x.requires_grad() || w1.requires_grad() || w2.requires_grad() ||
                                                     (b1 && b1->requires_grad()) || (b2 && b2->requires_grad()));
    const bool dual = forward_mode() && (has_tangent(x) || has_tangent(w1) || has_tangent(w2) || has_tangent(saved(b[0])) || has_tangent(saved(b[1])));
    if (!grad && !dual)                              // nothing will be back-propagated: the pre-activations are not written
      return mlp_fwd(contiguous(x), contiguous(w1), contiguous(w2), saved(b[0]), saved(b[1]), p, act, mask, false).out;
    return MlpNode::apply(contiguous(x), contiguous(w1), contiguous(w2), b[0], b[1], mask, p, act);
  });
  m.def("xentropy", [](const Tensor& logits, const Tensor& labels, double smoothing, int64_t padding_idx) {
    return XentNode::apply(logits, contiguous(labels), smoothing, padding_idx);
  });
  m.def("packed_attention", [](const Tensor& qkv, const Tensor& cu, int64_t max_len, double p, double scale, bool causal) {
    Bits bits;
    Tensor out = PackedNode::apply(qkv, cu, max_len, p, scale, causal, &bits);
    return std::make_tuple(out, bits.mode, bits.seed, bits.offset, bits.words.defined() ? optional<Tensor>(bits.words) : optional<Tensor>());
  });
}

}  // namespace nmtg_host
