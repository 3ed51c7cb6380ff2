// The pre-norm encoder and decoder layers in their plain form (modules/transformer_layers.py decides which calls that is) as
// one autograd node each. The forward is called in pieces: the attention core of the self-attention is called between them
// through its Python name, flash_attn_cuda.fwd_batched (which comes back to flash_fwd_batched here); the backward runs from end
// to end.
//
// What the composition of single operators paid for and this does not: an autograd node, its saved tensors and an
// interpreter round trip per operator; the additions and copies autograd makes to sum the two gradients of every residual
// stream (the LayerNorm backward adds the stream's gradient to its own); a pass of its own for every
// residual addition (the next LayerNorm makes it on the way in); two reductions and two host synchronisations per layer for
// the clamp of non-finite values. Encoder layer [512 x 32 x 1024] bf16, forward + backward: 53 launches before, 33 now, six of
// them reductions of products too large to carry them (28 at [37 x 13 x 512]).
#include "host.h"

namespace nmtg_host {

using torch::autograd::AutogradContext;
using torch::autograd::Function;
using torch::autograd::variable_list;

namespace {

constexpr double kEps = 1e-5;                                     // of every LayerNorm of the layers

Tensor defined_or(const optional<Tensor>& t) { return t.has_value() ? *t : Tensor(); }

struct Rates { double attn, residual, ffn; };                     // dropout: attention weights, sub-layer outputs, feed-forward

// the flag of the fp16 clamp: cleared by the LayerNorm in front of the feed-forward block, see add_ln_fwd
Tensor guard_flag(const Tensor& x) { return x.scalar_type() == at::kHalf ? empty_as(x, {1}, at::kInt) : Tensor(); }

// ---- the feed-forward block, shared by both layers: x -> h = x + dropout(out), LayerNorm, feed-forward, dropout + add ----
struct FfnState { Tensor h, z, stats, keep, post, pre, mask, guard, out; };
FfnState ffn_fwd(const Tensor& y, const Tensor& residual, double p_in, const Tensor& g, const Tensor& b, const Tensor& w1, const Tensor& c1,
                 const Tensor& w2, const Tensor& c2, int64_t act, double p_ffn, double p_out, bool grad) {
  Tensor flag = guard_flag(y);
  AddNorm n = add_ln_fwd(y, residual, p_in, flag, g, b, kEps);
  Mlp m = mlp_fwd(n.z, w1, w2, c1, c2, p_ffn, act, {}, grad && act != NMTG_ACT_RELU);
  Tensor guard = dropout_add_guard_(m.out, n.h, p_out, flag, grad);
  return {n.h, n.z, n.stats, n.mask, m.post, m.pre, m.mask, guard, m.out};
}

// --------------------------------------------------------------------------------------------------------------- encoder
struct EncoderIn {
  Tensor x, z1, stats1, lin, ctx, lse, words, pad;
  int64_t heads, act, mode;
  uint64_t seed, offset;
  Rates p;
  bool grad;
};

struct EncoderNode : Function<EncoderNode> {
  // parameters: LayerNorm (2), in-projection (2), out-projection (2), LayerNorm (2), feed-forward (4)
  static Tensor forward(AutogradContext* ctx, EncoderIn* in, const Tensor& x, const Tensor& g1, const Tensor& b1, const Tensor& wi, const Tensor& bi,
                        const Tensor& wo, const Tensor& bo, const Tensor& g2, const Tensor& b2, const Tensor& w1, const Tensor& c1,
                        const Tensor& w2, const Tensor& c2) {
    Tensor y, keep;
    FfnState f = compute(*in, x, wo, bo, g2, b2, w1, c1, w2, c2, &keep);
    ctx->saved_data["heads"] = in->heads;
    ctx->saved_data["act"] = in->act;
    ctx->saved_data["mode"] = in->mode;
    ctx->saved_data["seed"] = static_cast<int64_t>(in->seed);
    ctx->saved_data["offset"] = static_cast<int64_t>(in->offset);
    ctx->saved_data["pa"] = in->p.attn;
    ctx->saved_data["pr"] = in->p.residual;
    ctx->saved_data["pf"] = in->p.ffn;
    ctx->save_for_backward({x, in->z1, in->stats1, in->lin, in->ctx, in->lse, in->words, in->pad, keep, f.h, f.z, f.stats, f.post, f.pre, f.mask,
                            f.guard, g1, wi, wo, g2, w1, w2});
    return f.out;
  }
  static FfnState compute(const EncoderIn& in, const Tensor& x, const Tensor& wo, const Tensor& bo, const Tensor& g2, const Tensor& b2,
                          const Tensor& w1, const Tensor& c1, const Tensor& w2, const Tensor& c2, Tensor* keep) {
    Tensor y = linear_fwd(in.ctx.view(in.x.sizes()), wo, bo);
    // the dropout of the attention's output is torch's own (its mask comes from torch's stream of random numbers)
    if (in.p.residual > 0.0) std::tie(y, *keep) = at::native_dropout(y, in.p.residual, true);
    return ffn_fwd(y, x, 0.0, g2, b2, w1, c1, w2, c2, in.act, in.p.ffn, in.p.residual, in.grad);
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    auto s = ctx->get_saved_variables();
    const Tensor &x = s[0], &z1 = s[1], &stats1 = s[2], &lin = s[3], &cx = s[4], &lse = s[5], &words = s[6], &pad = s[7], &keep = s[8], &h = s[9],
                 &z2 = s[10], &stats2 = s[11], &post = s[12], &pre = s[13], &mask = s[14], &guard = s[15], &g1 = s[16], &wi = s[17], &wo = s[18],
                 &g2 = s[19], &w1 = s[20], &w2 = s[21];
    const int64_t heads = ctx->saved_data["heads"].toInt();
    const double pa = ctx->saved_data["pa"].toDouble(), pr = ctx->saved_data["pr"].toDouble(), pf = ctx->saved_data["pf"].toDouble();
    Launch on(x);
    auto need = [&](int i) { return ctx->needs_input_grad(i); };   // 0: x, then the parameters in order
    Tensor g = contiguous(grads[0]);
    Tensor df = dropout_guard_bwd(g, guard, pr);
    MlpGrads m = mlp_bwd(df, z2, w1, w2, post, pre, mask, pf, ctx->saved_data["act"].toInt(), true, need(9) || need(11), need(10), need(12));
    AddNormGrads n2 = ln_bwd_add(m.dx, h, stats2, g2, g, guard, keep, pr);
    const Tensor& dy = keep.defined() ? n2.dy : n2.dx;
    LinearGrads o = linear_bwd(dy, cx, wo, true, need(5), need(6));
    Tensor dlin = new_like(lin);
    const int64_t t = x.size(0), b = x.size(1), d = x.size(2) / heads;
    Bits bits{ctx->saved_data["mode"].toInt(), static_cast<uint64_t>(ctx->saved_data["seed"].toInt()),
              static_cast<uint64_t>(ctx->saved_data["offset"].toInt()), words};
    flash_bwd_batched({t, t, b, heads, d}, o.dx, slot_view(lin, heads, 3, 0), slot_view(lin, heads, 3, 1), slot_view(lin, heads, 3, 2), cx, lse,
                      slot_view(dlin, heads, 3, 0), slot_view(dlin, heads, 3, 1), slot_view(dlin, heads, 3, 2), pad, Tensor(), pa,
                      1.0 / std::sqrt(static_cast<double>(d)), false, bits);
    LinearGrads i = linear_bwd(dlin, z1, wi, true, need(3), need(4));
    AddNormGrads n1 = ln_bwd_add(i.dx, x, stats1, g1, n2.dx, Tensor(), Tensor(), 0.0);
    return {Tensor(), n1.dx, n1.dgamma, n1.dbeta, i.dw, i.db, o.dw, o.db, n2.dgamma, n2.dbeta, m.dw1, m.db1, m.dw2, m.db2};
  }
};

// --------------------------------------------------------------------------------------------------------------- decoder
// Self-attention under a time mask, cross-attention whose coverage (the probabilities before dropout) is returned,
// feed-forward block.
struct DecoderIn {
  Tensor x, context, z1, stats1, lin, ctx, lse, words, time, pad;
  int64_t heads, act, mode;
  uint64_t seed, offset;
  Rates p;
  double p_cross;
  bool grad;
};

struct Cross { Tensor q_lin, kv_lin, softmax, dropped, mask, ctx, out; };
Cross cross_fwd(const Tensor& xq, const Tensor& xkv, const Tensor& wq, const Tensor& wkv, const Tensor& wo, const Tensor& mask, int64_t heads,
                double p, bool grad) {
  const int64_t tq = xq.size(0), tk = xkv.size(0), b = xq.size(1), e = xq.size(2), d = e / heads;
  Launch on(xq);
  Cross r;
  r.q_lin = new_like(xq);
  r.kv_lin = empty_like_sized(xkv, {tk, b, 2 * e});
  r.ctx = new_like(xq);
  r.out = new_like(xq);
  r.dropped = empty_like_sized(xq, {b * heads, tq, tk});
  // the kernels read mask bytes four or eight at a time: a view that starts at an odd address is copied
  const Tensor pad = mask.defined() && reinterpret_cast<uintptr_t>(ptr(mask)) % 8 != 0 ? mask.clone() : mask;
  // an inference call writes the probabilities only where one kernel makes them and the context (nmtg_encdec_attn_fwd)
  const bool probs_only = !grad && p == 0.0 && api.attn_scores_needed(tk, d, dtype_code(xq)) == 0;
  Scratch scores;
  if (!probs_only) scores = Scratch(xq, b * heads * tq * tk * static_cast<int64_t>(xq.element_size()));
  uint64_t seed = 0, offset = 0;
  if (grad) r.softmax = empty_like_sized(xq, {b * heads, tq, tk});
  if (p > 0.0) {
    r.mask = empty_as(xq, {b * heads, tq, tk}, at::kByte);
    std::tie(seed, offset) = draw(xq, r.mask.numel());
  }
  check(api.encdec_attn_fwd(ptr(xq), ptr(xkv), ptr(wq), ptr(wkv), ptr(wo), nullptr, nullptr, nullptr, static_cast<const uint8_t*>(ptr(pad)),
                            ptr(r.q_lin), ptr(r.kv_lin), scores.get(), ptr(r.softmax), ptr(r.dropped), static_cast<uint8_t*>(ptr(r.mask)),
                            p > 0.0 ? 2 : 0, static_cast<float>(p), seed, offset, ptr(r.ctx), ptr(r.out), tq, tk, b, e,
                            static_cast<int>(heads), dtype_code(xq), on.stream), "nmtg_encdec_attn_fwd");
  if (!grad) r.softmax = r.dropped;
  return r;
}

struct CrossGrads { Tensor dxq, dxkv, dwq, dwkv, dwo; };
CrossGrads cross_bwd(const Tensor& dy, const Cross& c, const Tensor& xq, const Tensor& xkv, const Tensor& wq, const Tensor& wkv, const Tensor& wo,
                     int64_t heads, double p) {
  const int64_t tq = xq.size(0), tk = xkv.size(0), b = xq.size(1), e = xq.size(2);
  Launch on(xq);
  CrossGrads r{new_like(xq), new_like(xkv), new_like(wq), new_like(wkv), new_like(wo)};
  const Scratch ws(xq, std::max<int64_t>(api.encdec_attn_bwd_workspace_bytes(tq, tk, b, e, static_cast<int>(heads)), 256));
  check(api.encdec_attn_bwd_from_probs(ptr(dy), ptr(c.ctx), ptr(c.dropped), ptr(c.softmax), ptr(c.q_lin), ptr(c.kv_lin), ptr(xq), ptr(xkv), ptr(wq),
                                       ptr(wkv), ptr(wo), static_cast<const uint8_t*>(ptr(c.mask)), static_cast<float>(p), ptr(r.dxq), ptr(r.dxkv),
                                       ptr(r.dwq), ptr(r.dwkv), ptr(r.dwo), nullptr, nullptr, ws.get(), ws.bytes, tq, tk, b, e,
                                       static_cast<int>(heads), dtype_code(xq), on.stream), "nmtg_encdec_attn_bwd_from_probs");
  return r;
}

struct DecoderSaved { Tensor keep1, h1, z2, stats2; Cross c; FfnState f; };
DecoderSaved decoder_compute(const DecoderIn& in, const Tensor& x, const Tensor& context, const Tensor& wo, const Tensor& bo, const Tensor& g2,
                             const Tensor& b2, const Tensor& wq, const Tensor& wkv, const Tensor& wc, const Tensor& g3, const Tensor& b3,
                             const Tensor& w1, const Tensor& c1, const Tensor& w2, const Tensor& c2) {
  DecoderSaved r;
  Tensor y = linear_fwd(in.ctx.view(in.x.sizes()), wo, bo);
  if (in.p.residual > 0.0) std::tie(y, r.keep1) = at::native_dropout(y, in.p.residual, true);     // see EncoderNode::compute
  AddNorm n = add_ln_fwd(y, x, 0.0, Tensor(), g2, b2, kEps);
  r.h1 = n.h;
  r.z2 = n.z;
  r.stats2 = n.stats;
  r.c = cross_fwd(n.z, context, wq, wkv, wc, in.pad, in.heads, in.p_cross, in.grad);
  r.f = ffn_fwd(r.c.out, n.h, in.p.residual, g3, b3, w1, c1, w2, c2, in.act, in.p.ffn, in.p.residual, in.grad);
  return r;
}

struct DecoderNode : Function<DecoderNode> {
  // parameters: LayerNorm (2), in-projection (2), out-projection (2), LayerNorm (2), cross q / kv / out (3), LayerNorm (2), feed-forward (4)
  static variable_list forward(AutogradContext* ctx, DecoderIn* in, const Tensor& x, const Tensor& context, const Tensor& g1, const Tensor& b1,
                               const Tensor& wi, const Tensor& bi, const Tensor& wo, const Tensor& bo, const Tensor& g2, const Tensor& b2,
                               const Tensor& wq, const Tensor& wkv, const Tensor& wc, const Tensor& g3, const Tensor& b3, const Tensor& w1,
                               const Tensor& c1, const Tensor& w2, const Tensor& c2) {
    DecoderSaved r = decoder_compute(*in, x, context, wo, bo, g2, b2, wq, wkv, wc, g3, b3, w1, c1, w2, c2);
    ctx->saved_data["heads"] = in->heads;
    ctx->saved_data["act"] = in->act;
    ctx->saved_data["mode"] = in->mode;
    ctx->saved_data["seed"] = static_cast<int64_t>(in->seed);
    ctx->saved_data["offset"] = static_cast<int64_t>(in->offset);
    ctx->saved_data["pa"] = in->p.attn;
    ctx->saved_data["pc"] = in->p_cross;
    ctx->saved_data["pr"] = in->p.residual;
    ctx->saved_data["pf"] = in->p.ffn;
    ctx->save_for_backward({x, context, in->z1, in->stats1, in->lin, in->ctx, in->lse, in->words, in->time, r.keep1, r.h1, r.z2, r.stats2, r.c.q_lin,
                            r.c.kv_lin, r.c.softmax, r.c.dropped, r.c.mask, r.c.ctx, r.f.h, r.f.z, r.f.stats, r.f.keep, r.f.post, r.f.pre, r.f.mask,
                            r.f.guard, g1, wi, wo, g2, wq, wkv, wc, g3, w1, w2});
    ctx->set_materialize_grads(false);                              // no zero-filled gradient of the coverage
    ctx->mark_non_differentiable({r.c.softmax});
    return {r.f.out, r.c.softmax};
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    if (!grads[0].defined()) return variable_list(20);
    auto s = ctx->get_saved_variables();
    const Tensor &x = s[0], &context = s[1], &z1 = s[2], &stats1 = s[3], &lin = s[4], &cx = s[5], &lse = s[6], &words = s[7], &time = s[8],
                 &keep1 = s[9], &h1 = s[10], &z2 = s[11], &stats2 = s[12];
    Cross c{s[13], s[14], s[15], s[16], s[17], s[18], Tensor()};
    const Tensor &h2 = s[19], &z3 = s[20], &stats3 = s[21], &keep2 = s[22], &post = s[23], &pre = s[24], &mask = s[25], &guard = s[26], &g1 = s[27],
                 &wi = s[28], &wo = s[29], &g2 = s[30], &wq = s[31], &wkv = s[32], &wc = s[33], &g3 = s[34], &w1 = s[35], &w2 = s[36];
    const int64_t heads = ctx->saved_data["heads"].toInt();
    const double pa = ctx->saved_data["pa"].toDouble(), pc = ctx->saved_data["pc"].toDouble(), pr = ctx->saved_data["pr"].toDouble(),
                 pf = ctx->saved_data["pf"].toDouble();
    Launch on(x);
    auto need = [&](int i) { return ctx->needs_input_grad(i); };   // 0: x, 1: context, then the parameters in order
    Tensor g = contiguous(grads[0]);
    Tensor df = dropout_guard_bwd(g, guard, pr);
    MlpGrads m = mlp_bwd(df, z3, w1, w2, post, pre, mask, pf, ctx->saved_data["act"].toInt(), true, need(15) || need(17), need(16), need(18));
    AddNormGrads n3 = ln_bwd_add(m.dx, h2, stats3, g3, g, guard, keep2, pr);
    CrossGrads r = cross_bwd(keep2.defined() ? n3.dy : n3.dx, c, z2, context, wq, wkv, wc, heads, pc);
    AddNormGrads n2 = ln_bwd_add(r.dxq, h1, stats2, g2, n3.dx, Tensor(), keep1, pr);
    LinearGrads o = linear_bwd(keep1.defined() ? n2.dy : n2.dx, cx, wo, true, need(6), need(7));
    Tensor dlin = new_like(lin);
    const int64_t t = x.size(0), b = x.size(1), d = x.size(2) / heads;
    Bits bits{ctx->saved_data["mode"].toInt(), static_cast<uint64_t>(ctx->saved_data["seed"].toInt()),
              static_cast<uint64_t>(ctx->saved_data["offset"].toInt()), words};
    flash_bwd_batched({t, t, b, heads, d}, o.dx, slot_view(lin, heads, 3, 0), slot_view(lin, heads, 3, 1), slot_view(lin, heads, 3, 2), cx, lse,
                      slot_view(dlin, heads, 3, 0), slot_view(dlin, heads, 3, 1), slot_view(dlin, heads, 3, 2), Tensor(), time, pa,
                      1.0 / std::sqrt(static_cast<double>(d)), false, bits);
    LinearGrads i = linear_bwd(dlin, z1, wi, true, need(4), need(5));
    AddNormGrads n1 = ln_bwd_add(i.dx, x, stats1, g1, n2.dx, Tensor(), Tensor(), 0.0);
    return {Tensor(), n1.dx, r.dxkv, n1.dgamma, n1.dbeta, i.dw, i.db, o.dw, o.db, n2.dgamma, n2.dbeta, r.dwq, r.dwkv, r.dwo, n3.dgamma, n3.dbeta,
            m.dw1, m.db1, m.dw2, m.db2};
  }
};

// One step of incremental decoding: x [1, B, E], self-attention over the n cached positions and the new one (which is written
// into row n of the buffers), cross-attention over the cached encoder keys / values, feed-forward block.
std::tuple<Tensor, Tensor> decoder_step(const Tensor& x, const Tensor& kbuf, const Tensor& vbuf, int64_t n, const Tensor& ck, const Tensor& cv,
                                        const Tensor& pad, const std::vector<Tensor>& w, int64_t heads, int64_t act) {
  const int64_t b = x.size(1), e = x.size(2), d = e / heads, tk = ck.size(0);
  const float scale = static_cast<float>(1.0 / std::sqrt(static_cast<double>(d)));
  Launch on(x);
  // few rows: LayerNorms, activation and last addition go with the products (8 launches and the clamp of fp16 instead of 13)
  auto whole = [](const Tensor& t) { return reinterpret_cast<uintptr_t>(ptr(t)) % 16 == 0; };
  bool fused = api.step_linear_ok(b, e, w[13].size(0)) != 0 && whole(x);
  for (int i : {0, 1, 2, 6, 7, 8, 11, 12, 13, 15}) fused = fused && whole(w[i]);
  Tensor lin = fused ? norm_step(x, Tensor(), w[0], w[1], kEps, Tensor(), w[2], w[3], NMTG_ACT_NONE).y : linear_step(ln_fwd(x, w[0], w[1], kEps).z, w[2], w[3]);
  Tensor cx = new_like(x);
  check(api.attn_decode_append(ptr(lin), 3 * e, ptr(kbuf), kbuf.stride(0), kbuf.stride(1), ptr(vbuf), vbuf.stride(0), vbuf.stride(1), ptr(cx), e, b,
                               heads, d, n, scale, dtype_code(x), on.stream), "nmtg_attn_decode_append");
  Tensor y = linear_step(cx, w[4], w[5]), q, h;
  if (fused) {
    StepNorm s = norm_step(y, x, w[6], w[7], kEps, Tensor(), w[8], Tensor(), NMTG_ACT_NONE);
    q = s.y;
    h = s.h;
  } else {
    AddNorm n2 = add_ln_fwd(y, x, 0.0, Tensor(), w[6], w[7], kEps);
    q = linear_step(n2.z, w[8], Tensor());
    h = n2.h;
  }
  Tensor coverage = empty_like_sized(x, {b * heads, 1, tk});
  check(api.attn_decode(ptr(q), e, ptr(ck), ck.stride(0), ck.stride(1), ptr(cv), cv.stride(0), cv.stride(1),
                        static_cast<const uint8_t*>(ptr(pad)), ptr(coverage), ptr(cx), e, b, heads, d, tk, scale, dtype_code(x), on.stream),
        "nmtg_attn_decode");
  y = linear_step(cx, w[10], Tensor());
  if (fused) {
    Tensor guard = guard_flag(x);
    StepNorm s = norm_step(y, h, w[11], w[12], kEps, guard, w[13], w[14], act);
    return {linear_add_step(s.y, w[15], w[16], s.h, guard), coverage};
  }
  return {ffn_fwd(y, h, 0.0, w[11], w[12], w[13], w[14], w[15], w[16], act, 0.0, 0.0, false).out, coverage};
}

// Whether an encoder layer's 12 or a decoder layer's 17 parameters (all present) have the shapes that x's last dimension asks
// for: what follows hands their addresses to kernels. Anything else is left to the operators, whose checks name it.
bool shapes_fit(int64_t e, const std::vector<optional<Tensor>>& p) {
  const bool decoder = p.size() == 17;
  if (!decoder && p.size() != 12) return false;
  size_t i = 0;
  auto vec = [&](int64_t n) { return p[i++]->numel() == n; };
  auto mat = [&](int64_t rows, int64_t cols) {
    const Tensor& t = *p[i++];
    return t.dim() == 2 && t.size(0) == rows && t.size(1) == cols;
  };
  if (!(vec(e) && vec(e) && mat(3 * e, e) && vec(3 * e) && mat(e, e) && vec(e) && vec(e) && vec(e))) return false;
  if (decoder && !(mat(e, e) && mat(2 * e, e) && mat(e, e) && vec(e) && vec(e))) return false;
  const int64_t inner = p[i]->dim() == 2 ? p[i]->size(0) : -1;
  return mat(inner, e) && vec(inner) && mat(e, inner) && vec(e);
}

using State = std::tuple<int64_t, uint64_t, uint64_t, optional<Tensor>, optional<Tensor>, optional<Tensor>>;
using Params = std::vector<Tensor>;

}  // namespace

void define_layers(pybind11::module_& m) {
  // LayerNorm and in-projection of the self-attention -> (z, stats, projection, q, k, v)
  m.def("layer_begin", [](const Tensor& input, const Tensor& g, const Tensor& b, const Tensor& wi, const Tensor& bi, int64_t heads) {
    at::AutoDispatchBelowADInplaceOrView off;
    TORCH_CHECK(heads > 0 && input.size(2) % heads == 0, "layer: ", heads, " heads do not divide ", input.size(2));
    Tensor x = contiguous(input);
    Norm n = ln_fwd(x, g, b, kEps);
    Tensor lin = linear_fwd(n.z, wi, bi);
    return std::make_tuple(n.z, n.stats, lin, slot(lin, heads, 3, 0), slot(lin, heads, 3, 1), slot(lin, heads, 3, 2));
  });
  m.def("flash_fwd_batched", [](const Tensor& q, const Tensor& k, const Tensor& v, const optional<Tensor>& pad, const optional<Tensor>& time, double p,
                                double scale, bool causal) {
    at::AutoDispatchBelowADInplaceOrView off;
    Flash f = flash_fwd_batched(q, k, v, defined_or(pad), defined_or(time), p, scale, causal);
    return std::make_tuple(f.out, f.lse, State(f.bits.mode, f.bits.seed, f.bits.offset, {},
                                               f.bits.words.defined() ? optional<Tensor>(f.bits.words) : optional<Tensor>(), {}));
  });
  // What the layers ask before they take this path: 0 = no (a parameter of another type, shape, layout or device, or none, or a
  // forward-mode tangent anywhere), 1 = yes, nothing will be back-propagated, 2 = yes, with gradients.
  m.def("layer_mode", [](const Tensor& x, const std::vector<optional<Tensor>>& inputs, const std::vector<optional<Tensor>>& params) {
    const bool forward = forward_mode();
    if (!x.is_cuda() || x.dim() != 3 || x.numel() == 0 || (x.scalar_type() != at::kHalf && x.scalar_type() != at::kBFloat16) ||
        (forward && has_tangent(x)))
      return 0;
    bool grad = x.requires_grad();
    for (const auto* list : {&inputs, &params})
      for (const auto& p : *list) {
        if (!p.has_value() || !p->defined() || p->device() != x.device() || p->scalar_type() != x.scalar_type() || !p->is_contiguous() ||
            (forward && has_tangent(*p)))
          return 0;
        grad = grad || p->requires_grad();
      }
    if (!shapes_fit(x.size(2), params)) return 0;
    return grad && at::GradMode::is_enabled() ? 2 : 1;
  });
  m.def("mask_bytes", [](const optional<Tensor>& mask, const Tensor& operand, int64_t rows, int64_t cols) {
    Tensor t = pad_bytes(mask, operand, rows, cols);
    return t.defined() ? optional<Tensor>(t) : optional<Tensor>();
  });
  // the rest of an encoder layer, from the context of its attention core
  m.def("encoder_end", [](const Tensor& x, const Tensor& z1, const Tensor& stats1, const Tensor& lin, const Tensor& cx, const Tensor& lse,
                          const State& state, const optional<Tensor>& pad, const Params& w, int64_t heads, int64_t act, double p_attn,
                          double p_residual, double p_ffn, bool grad) {
    EncoderIn in{x, z1, stats1, lin, cx, lse, defined_or(std::get<4>(state)), defined_or(pad), heads, act, std::get<0>(state), std::get<1>(state),
                 std::get<2>(state), {p_attn, p_residual, p_ffn}, grad};
    if (!grad) {
      at::AutoDispatchBelowADInplaceOrView off;
      Tensor keep;
      return EncoderNode::compute(in, x, w[4], w[5], w[6], w[7], w[8], w[9], w[10], w[11], &keep).out;
    }
    return EncoderNode::apply(&in, x, w[0], w[1], w[2], w[3], w[4], w[5], w[6], w[7], w[8], w[9], w[10], w[11]);
  });
  m.def("decoder_step", [](const Tensor& x, const Tensor& kbuf, const Tensor& vbuf, int64_t n, const Tensor& ck, const Tensor& cv,
                           const optional<Tensor>& pad, const Params& w, int64_t heads, int64_t act) {
    at::AutoDispatchBelowADInplaceOrView off;
    for (const Tensor* t : {&kbuf, &vbuf, &ck, &cv}) check_device(*t, x);
    check_device(defined_or(pad), x);
    auto r = decoder_step(contiguous(x), kbuf, vbuf, n, ck, cv, defined_or(pad), w, heads, act);
    return std::make_tuple(std::get<0>(r), std::get<1>(r), kbuf.narrow(0, 0, n + 1), vbuf.narrow(0, 0, n + 1));
  });
  // -> (output, coverage)
  m.def("decoder_end", [](const Tensor& x, const Tensor& context, const Tensor& z1, const Tensor& stats1, const Tensor& lin, const Tensor& cx,
                          const Tensor& lse, const State& state, const optional<Tensor>& time, const optional<Tensor>& pad, const Params& w,
                          int64_t heads, int64_t act, double p_attn, double p_cross, double p_residual, double p_ffn, bool grad) {
    DecoderIn in{x, context, z1, stats1, lin, cx, lse, defined_or(std::get<4>(state)), defined_or(time), defined_or(pad), heads, act,
                 std::get<0>(state), std::get<1>(state), std::get<2>(state), {p_attn, p_residual, p_ffn}, p_cross, grad};
    if (!grad) {
      at::AutoDispatchBelowADInplaceOrView off;
      DecoderSaved r = decoder_compute(in, x, context, w[4], w[5], w[6], w[7], w[8], w[9], w[10], w[11], w[12], w[13], w[14], w[15], w[16]);
      return std::make_tuple(r.f.out, r.c.softmax);
    }
    auto r = DecoderNode::apply(&in, x, context, w[0], w[1], w[2], w[3], w[4], w[5], w[6], w[7], w[8], w[9], w[10], w[11], w[12], w[13], w[14], w[15],
                                w[16]);
    return std::make_tuple(r[0], r[1]);
  });
}

}  // namespace nmtg_host
