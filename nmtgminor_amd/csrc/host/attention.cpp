// The attention modules in training with their coverage on the tiled core, as one autograd node each: projections,
// attention, coverage, output projection. The extension's path kept scores, probabilities and mask bytes of
// [B * H, len_q, len_k] elements for the backward (0.9 GB at [512 x 32 x 1024]) and read them back three times; here the
// backward recomputes the scores, and the coverage is the one tensor of that size, written once.
// Self-attention [512 x 32 x 1024] bf16 with coverage, forward and backward: 1285 us on that path, 840 us here.
#include "host.h"

namespace nmtg_host {

using torch::autograd::AutogradContext;
using torch::autograd::Function;
using torch::autograd::variable_list;

namespace {

void keep_bits(AutogradContext* ctx, const Bits& b) {
  ctx->saved_data["mode"] = b.mode;
  ctx->saved_data["seed"] = static_cast<int64_t>(b.seed);
  ctx->saved_data["offset"] = static_cast<int64_t>(b.offset);
}
Bits kept_bits(AutogradContext* ctx, const Tensor& words) {
  return {ctx->saved_data["mode"].toInt(), static_cast<uint64_t>(ctx->saved_data["seed"].toInt()),
          static_cast<uint64_t>(ctx->saved_data["offset"].toInt()), words};
}

Tensor or_undefined(const optional<Tensor>& t) { return t.has_value() ? *t : Tensor(); }

// what travels beside the differentiable arguments
struct Call {
  Tensor pad, time;
  int64_t heads;
  double p;
  Coverage coverage;
};

struct SelfAttentionNode : Function<SelfAttentionNode> {
  static variable_list forward(AutogradContext* ctx, const Tensor& x, const Tensor& wi, const Tensor& wo, const optional<Tensor>& in_bias,
                               const optional<Tensor>& out_bias, const Call* call) {
    const int64_t heads = call->heads, d = x.size(2) / heads;
    const Tensor bi = or_undefined(in_bias), bo = or_undefined(out_bias), &pad = call->pad, &time = call->time;
    const double p = call->p;
    Launch on(x);
    Tensor lin = linear_fwd(x, wi, bi);
    Flash f = flash_fwd_batched(slot(lin, heads, 3, 0), slot(lin, heads, 3, 1), slot(lin, heads, 3, 2), pad, time, p,
                                1.0 / std::sqrt(static_cast<double>(d)), false, call->coverage);
    Tensor out = linear_fwd(f.out.view(x.sizes()), wo, bo);
    ctx->saved_data["heads"] = heads;
    ctx->saved_data["p"] = p;
    ctx->saved_data["bi"] = bi.defined();
    ctx->saved_data["bo"] = bo.defined();
    keep_bits(ctx, f.bits);
    ctx->save_for_backward({x, wi, wo, lin, f.out, f.lse, f.bits.words, pad, time});
    ctx->set_materialize_grads(false);
    ctx->mark_non_differentiable({f.probs});
    return {out, f.probs};
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    auto s = ctx->get_saved_variables();
    const Tensor &x = s[0], &wi = s[1], &wo = s[2], &lin = s[3], &cx = s[4], &lse = s[5], &words = s[6], &pad = s[7], &time = s[8];
    if (!grads[0].defined()) return variable_list(6);
    const int64_t heads = ctx->saved_data["heads"].toInt(), d = x.size(2) / heads;
    Launch on(x);
    auto need = [&](int i) { return ctx->needs_input_grad(i); };   // counts the tensors among the arguments: absent biases do not
    const bool has_bi = ctx->saved_data["bi"].toBool(), has_bo = ctx->saved_data["bo"].toBool();
    const bool need_bi = has_bi && need(3), need_bo = has_bo && need(has_bi ? 4 : 3);
    LinearGrads o = linear_bwd(contiguous(grads[0]), cx, wo, need(0) || need(1) || need_bi, need(2), need_bo);
    LinearGrads i;
    if (o.dx.defined()) {
      Tensor dlin = new_like(lin);
      if (cx.numel() > 0)
        flash_bwd_batched({cx.size(0), cx.size(0), cx.size(1), heads, d}, o.dx, slot_view(lin, heads, 3, 0), slot_view(lin, heads, 3, 1),
                          slot_view(lin, heads, 3, 2), cx, lse, slot_view(dlin, heads, 3, 0), slot_view(dlin, heads, 3, 1),
                          slot_view(dlin, heads, 3, 2), pad, time, ctx->saved_data["p"].toDouble(), 1.0 / std::sqrt(static_cast<double>(d)),
                          false, kept_bits(ctx, words));
      i = linear_bwd(dlin, x, wi, need(0), need(1), need_bi);
    }
    return {i.dx, i.dw, o.dw, i.db, o.db, Tensor()};
  }
};

struct CrossAttentionNode : Function<CrossAttentionNode> {
  static variable_list forward(AutogradContext* ctx, const Tensor& xq, const Tensor& xkv, const Tensor& wq, const Tensor& wkv, const Tensor& wo,
                               const optional<Tensor>& q_bias, const optional<Tensor>& kv_bias, const optional<Tensor>& out_bias, const Call* call) {
    const int64_t tq = xq.size(0), b = xq.size(1), heads = call->heads, d = xq.size(2) / heads;
    const Tensor bq = or_undefined(q_bias), bkv = or_undefined(kv_bias), bo = or_undefined(out_bias), &pad = call->pad;
    const double p = call->p;
    Launch on(xq);
    Tensor ql = linear_fwd(xq, wq, bq), kvl = linear_fwd(xkv, wkv, bkv);
    Flash f = flash_fwd_batched(ql.view({tq, b, heads, d}), slot(kvl, heads, 2, 0), slot(kvl, heads, 2, 1), pad, Tensor(), p,
                                1.0 / std::sqrt(static_cast<double>(d)), false, call->coverage);
    Tensor out = linear_fwd(f.out.view(xq.sizes()), wo, bo);
    ctx->saved_data["heads"] = heads;
    ctx->saved_data["p"] = p;
    ctx->saved_data["bq"] = bq.defined();
    ctx->saved_data["bkv"] = bkv.defined();
    ctx->saved_data["bo"] = bo.defined();
    keep_bits(ctx, f.bits);
    ctx->save_for_backward({xq, xkv, wq, wkv, wo, ql, kvl, f.out, f.lse, f.bits.words, pad});
    ctx->set_materialize_grads(false);
    ctx->mark_non_differentiable({f.probs});
    return {out, f.probs};
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    auto s = ctx->get_saved_variables();
    const Tensor &xq = s[0], &xkv = s[1], &wq = s[2], &wkv = s[3], &wo = s[4], &ql = s[5], &kvl = s[6], &cx = s[7], &lse = s[8], &words = s[9],
                 &pad = s[10];
    if (!grads[0].defined()) return variable_list(9);
    const int64_t heads = ctx->saved_data["heads"].toInt(), d = xq.size(2) / heads;
    Launch on(xq);
    auto need = [&](int i) { return ctx->needs_input_grad(i); };   // as above: queries, keys / values, weights q / kv / out, biases
    int at = 5;
    auto need_bias = [&](const char* name) { return ctx->saved_data[name].toBool() && need(at++); };
    const bool need_bq = need_bias("bq"), need_bkv = need_bias("bkv"), need_bo = need_bias("bo");
    const bool inner = need(0) || need(1) || need(2) || need(3) || need_bq || need_bkv;
    LinearGrads o = linear_bwd(contiguous(grads[0]), cx, wo, inner, need(4), need_bo), q, kv;
    if (inner) {
      Tensor dq = new_like(ql), dkv = new_like(kvl);
      if (cx.numel() > 0)
        flash_bwd_batched({cx.size(0), kvl.size(0), cx.size(1), heads, d}, o.dx, head_view(ql, heads), slot_view(kvl, heads, 2, 0),
                          slot_view(kvl, heads, 2, 1), cx, lse, head_view(dq, heads), slot_view(dkv, heads, 2, 0), slot_view(dkv, heads, 2, 1), pad,
                          Tensor(), ctx->saved_data["p"].toDouble(), 1.0 / std::sqrt(static_cast<double>(d)), false, kept_bits(ctx, words));
      else dkv.zero_();                            // no query position looked at the keys
      q = linear_bwd(dq, xq, wq, need(0), need(2), need_bq);
      kv = linear_bwd(dkv, xkv, wkv, need(1), need(3), need_bkv);
    }
    return {q.dx, kv.dx, q.dw, kv.dw, o.dw, q.db, kv.db, o.db, Tensor()};
  }
};

// a weight [out, in] of x's type, device and a matching width, or its bias [out]
void check_projection(const Tensor& x, const Tensor& w, const optional<Tensor>& b, int64_t out) {
  TORCH_CHECK(w.device() == x.device() && w.scalar_type() == x.scalar_type() && w.dim() == 2 && w.size(0) == out && w.size(1) == x.size(2),
              "attention: weight shape / dtype mismatch");
  TORCH_CHECK(!b.has_value() || (b->device() == x.device() && b->scalar_type() == x.scalar_type() && b->numel() == out),
              "attention: bias shape / dtype mismatch");
}
optional<Tensor> flat(const optional<Tensor>& t) { return t.has_value() ? optional<Tensor>(contiguous(*t)) : t; }

}  // namespace

void define_attention(pybind11::module_& m) {
  // -> [output, probabilities after dropout]
  m.def("self_attention", [](const Tensor& x, const Tensor& wi, const Tensor& wo, const optional<Tensor>& bi, const optional<Tensor>& bo,
                             const optional<Tensor>& mask, bool time_mask, int64_t heads, double p) {
    const int64_t t = x.size(0), b = x.size(1), e = x.size(2);
    check_projection(x, wi, bi, 3 * e);
    check_projection(x, wo, bo, e);
    const Call call{time_mask ? Tensor() : pad_bytes(mask, x, b, t), time_mask ? pad_bytes(mask, x, t, t) : Tensor(), heads, p,
                    Coverage::dropped};
    return SelfAttentionNode::apply(contiguous(x), contiguous(wi), contiguous(wo), flat(bi), flat(bo), &call);
  });
  // -> [output, probabilities before dropout, or after it with `dropped`]
  m.def("cross_attention", [](const Tensor& xq, const Tensor& xkv, const Tensor& wq, const Tensor& wkv, const Tensor& wo,
                              const optional<Tensor>& bq, const optional<Tensor>& bkv, const optional<Tensor>& bo, const optional<Tensor>& mask,
                              int64_t heads, double p, bool dropped) {
    const int64_t e = xq.size(2);
    TORCH_CHECK(xkv.device() == xq.device() && xkv.scalar_type() == xq.scalar_type() && xkv.dim() == 3 && xkv.size(1) == xq.size(1),
                "attention: queries and keys / values disagree");
    check_projection(xq, wq, bq, e);
    check_projection(xkv, wkv, bkv, 2 * e);
    check_projection(xq, wo, bo, e);
    const Call call{pad_bytes(mask, xq, xkv.size(1), xkv.size(0)), Tensor(), heads, p, dropped ? Coverage::dropped : Coverage::softmax};
    return CrossAttentionNode::apply(contiguous(xq), contiguous(xkv), contiguous(wq), contiguous(wkv), contiguous(wo), flat(bq), flat(bkv), flat(bo),
                                     &call);
  });
}

}  // namespace nmtg_host
