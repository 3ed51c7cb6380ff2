// The operators of the host layer: argument preparation, result allocation and the call of the C entry point.
#include "host.h"
#include <dlfcn.h>

namespace nmtg_host {

Api api;

void bind(const std::string& path) {
  void* lib = dlopen(path.c_str(), RTLD_NOW | RTLD_LOCAL);
  TORCH_CHECK(lib != nullptr, "cannot load ", path, ": ", dlerror());
#define X(name)                                                                                     \
  api.name = reinterpret_cast<decltype(&nmtg_##name)>(dlsym(lib, "nmtg_" #name));                   \
  TORCH_CHECK(api.name != nullptr, path, " has no nmtg_" #name ": built from other sources");
  NMTG_HOST_API(X)
#undef X
}

void check(int rc, const char* what) {
  if (rc == 0) return;
  throw std::runtime_error(std::string(what) + ": " + api.last_error() + " (status " + std::to_string(rc) + ")");
}

int dtype_code(const Tensor& t) {
  switch (t.scalar_type()) {
    case at::kFloat: return NMTG_F32;
    case at::kHalf: return NMTG_F16;
    case at::kBFloat16: return NMTG_BF16;
    default: TORCH_CHECK(false, "unsupported dtype ", t.scalar_type());
  }
}

std::pair<uint64_t, uint64_t> draw(const Tensor& like, int64_t count) {
  at::Generator gen = at::globalContext().defaultGenerator(like.device());
  std::lock_guard<std::mutex> lock(gen.mutex());
  const uint64_t seed = gen.current_seed(), offset = gen.get_offset();
  gen.set_offset(offset + static_cast<uint64_t>((count + 3) / 4 * 4));
  return {seed, offset};
}

// ---------------------------------------------------------------------------------------------------------- LayerNorm
Norm ln_fwd(const Tensor& x, const Tensor& gamma, const Tensor& beta, double eps) {
  const int64_t h = gamma.numel(), rows = h ? x.numel() / h : 0;
  Launch on(x);
  Norm r{x.is_contiguous() ? empty_as(x, x.sizes(), gamma.scalar_type()) : at::empty_like(x, x.options().dtype(gamma.scalar_type())), empty_as(x, {2, rows}, at::kFloat)};
  float* mu = r.stats.data_ptr<float>();
  check(api.ln_fwd(ptr(x), ptr(gamma), ptr(beta), ptr(r.z), mu, mu + rows, rows, h, static_cast<float>(eps), dtype_code(x),
                   dtype_code(gamma), on.stream), "nmtg_ln_fwd");
  return r;
}

NormGrads ln_bwd(const Tensor& dz, const Tensor& x_or_z, const Tensor& stats, const Tensor& gamma, const Tensor& beta, bool memory_efficient) {
  const int64_t h = gamma.numel(), rows = stats.size(1);
  Launch on(dz);
  NormGrads r{new_like(x_or_z), new_like(gamma), new_like(gamma)};
  const int64_t parts = api.ln_bwd_parts(rows, h);
  const Scratch part(dz, 2 * parts * h * static_cast<int64_t>(sizeof(float)));
  float* pp = part.get<float>();
  const float* mu = stats.data_ptr<float>();
  check(api.ln_bwd(ptr(dz), ptr(x_or_z), mu, mu + rows, ptr(gamma), memory_efficient ? ptr(beta) : nullptr, ptr(r.dx), ptr(r.dgamma),
                   ptr(r.dbeta), pp, pp + parts * h, parts, rows, h, memory_efficient ? 1 : 0, dtype_code(x_or_z), dtype_code(gamma),
                   on.stream), "nmtg_ln_bwd");
  return r;
}

AddNorm add_ln_fwd(const Tensor& x, const Tensor& residual, double p, const Tensor& clear, const Tensor& gamma, const Tensor& beta, double eps) {
  const int64_t h = gamma.numel(), rows = x.numel() / h;
  Launch on(x);
  AddNorm r{new_like(x), new_like(x), empty_as(x, {2, rows}, at::kFloat), Tensor()};
  uint64_t seed = 0, offset = 0;
  if (p > 0.0) {
    r.mask = empty_as(x, x.sizes(), at::kByte);
    std::tie(seed, offset) = draw(x, x.numel());
  }
  float* mu = r.stats.data_ptr<float>();
  check(api.add_ln_fwd(ptr(x), ptr(residual), ptr(r.h), static_cast<uint8_t*>(ptr(r.mask)), p > 0.0 ? 2 : 0, static_cast<float>(p), seed, offset,
                       static_cast<int*>(ptr(clear)), ptr(gamma), ptr(beta), ptr(r.z), mu, mu + rows, rows, h, static_cast<float>(eps),
                       dtype_code(x), on.stream), "nmtg_add_ln_fwd");
  return r;
}

AddNormGrads ln_bwd_add(const Tensor& dz, const Tensor& x, const Tensor& stats, const Tensor& gamma, const Tensor& grad_residual,
                        const Tensor& guard, const Tensor& keep, double p) {
  const int64_t h = gamma.numel(), rows = stats.size(1);
  Launch on(dz);
  AddNormGrads r{new_like(x), Tensor(), new_like(gamma), new_like(gamma)};
  if (keep.defined()) r.dy = new_like(x);
  const int64_t parts = api.ln_bwd_parts(rows, h);
  const Scratch part(dz, 2 * parts * h * static_cast<int64_t>(sizeof(float)));
  float* pp = part.get<float>();
  const float* mu = stats.data_ptr<float>();
  check(api.ln_bwd_add(ptr(dz), ptr(x), mu, mu + rows, ptr(gamma), ptr(grad_residual), static_cast<const uint8_t*>(ptr(guard)),
                       static_cast<const uint8_t*>(ptr(keep)), static_cast<float>(p), ptr(r.dx), ptr(r.dy), ptr(r.dgamma), ptr(r.dbeta), pp,
                       pp + parts * h, parts, rows, h, dtype_code(x), on.stream), "nmtg_ln_bwd_add");
  return r;
}

// -------------------------------------------------------------------------------------------------- products and MLP
static Tensor linear_result(const Tensor& x, int64_t out) {
  auto sizes = x.sizes().vec();
  sizes.back() = out;
  return empty_like_sized(x, sizes);
}

Tensor linear_fwd(const Tensor& x, const Tensor& w, const Tensor& b) {
  const int64_t in = w.size(1), out = w.size(0), rows = x.numel() / in;
  Launch on(x);
  Tensor y = linear_result(x, out);
  check(api.gemm(0, 1, rows, out, in, 1.f, ptr(x), in, 0, ptr(w), in, 0, ptr(y), out, 0, 1, ptr(b), nullptr, 0, dtype_code(x), on.stream),
        "nmtg_gemm");
  return y;
}

Tensor linear_step(const Tensor& x, const Tensor& w, const Tensor& b) {
  const int64_t in = w.size(1), out = w.size(0);
  Launch on(x);
  Tensor y = linear_result(x, out);
  check(api.linear_step(x.numel() / in, out, in, ptr(x), ptr(w), ptr(b), ptr(y), dtype_code(x), on.stream), "nmtg_linear_step");
  return y;
}

StepNorm norm_step(const Tensor& x, const Tensor& residual, const Tensor& gamma, const Tensor& beta, double eps, const Tensor& clear, const Tensor& w,
                   const Tensor& b, int64_t act) {
  const int64_t in = w.size(1), out = w.size(0);
  Launch on(x);
  StepNorm r{linear_result(x, out), residual.defined() ? new_like(x) : Tensor()};
  check(api.step_linear(x.numel() / in, out, in, ptr(x), ptr(residual), ptr(gamma), ptr(beta), static_cast<float>(eps), ptr(r.h),
                        static_cast<int*>(ptr(clear)), ptr(w), ptr(b), static_cast<int>(act), nullptr, nullptr, ptr(r.y), dtype_code(x), on.stream),
        "nmtg_step_linear");
  return r;
}

Tensor linear_add_step(const Tensor& x, const Tensor& w, const Tensor& b, const Tensor& add, const Tensor& guard) {
  const int64_t in = w.size(1), out = w.size(0);
  Launch on(x);
  Tensor y = linear_result(x, out);
  check(api.step_linear(x.numel() / in, out, in, ptr(x), nullptr, nullptr, nullptr, 0.f, nullptr, nullptr, ptr(w), ptr(b), NMTG_ACT_NONE, ptr(add),
                        static_cast<int*>(ptr(guard)), ptr(y), dtype_code(x), on.stream), "nmtg_step_linear");
  return y;
}

static Scratch mlp_workspace(const Tensor& x, int layers, const int64_t* outs, int64_t rows, int64_t in) {
  return Scratch(x, std::max<int64_t>(api.mlp_bwd_dtype_workspace_bytes(layers, outs, rows, in, dtype_code(x)), 256));
}

LinearGrads linear_bwd(const Tensor& dy, const Tensor& x, const Tensor& w, bool want_x, bool want_w, bool want_b) {
  const int64_t out = w.size(0), in = w.size(1), rows = dy.numel() / out;
  Launch on(dy);
  LinearGrads r;
  if (want_x) { auto sizes = dy.sizes().vec(); sizes.back() = in; r.dx = empty_like_sized(dy, sizes); }
  if (want_w) r.dw = new_like(w);
  if (want_b) r.db = empty_like_sized(dy, {out});
  if (rows == 0) {                                  // no rows contribute zero gradients
    for (Tensor* t : {&r.dw, &r.db}) if (t->defined()) t->zero_();
    return r;
  }
  const Scratch ws = mlp_workspace(dy, 1, &out, rows, in);
  const void* weights[1] = {ptr(w)};
  void* dws[1] = {ptr(r.dw)};
  void* dbs[1] = {ptr(r.db)};
  check(api.mlp_bwd(1, ptr(x), weights, &out, rows, in, ptr(dy), nullptr, nullptr, nullptr, 0.f, NMTG_ACT_NONE, ptr(r.dx), dws, dbs, ws.get(),
                    ws.bytes, dtype_code(dy), on.stream), "nmtg_mlp_bwd");
  return r;
}

Mlp mlp_fwd(const Tensor& x, const Tensor& w1, const Tensor& w2, const Tensor& b1, const Tensor& b2, double p, int64_t act,
            const optional<Tensor>& mask, bool save_pre) {
  const int64_t in = w1.size(1), rows = x.numel() / in, inner = w1.size(0), out = w2.size(0), hidden = rows * inner;
  Launch on(x);
  auto sizes = x.sizes().vec();
  sizes.back() = out;
  Mlp r;
  r.out = empty_like_sized(x, sizes);
  r.post = empty_like_sized(x, {hidden});
  if (save_pre) r.pre = empty_like_sized(x, {hidden});
  int mode = 0;
  uint64_t seed = 0, offset = 0;
  if (p > 0.0) {
    if (mask.has_value()) {
      TORCH_CHECK(mask->scalar_type() == at::kByte && mask->numel() == hidden, "mlp: mask must be uint8 with one byte per hidden activation");
      check_device(*mask, x);
      r.mask = contiguous(*mask);
      mode = 1;
    } else {
      r.mask = empty_as(x, {hidden}, at::kByte);
      mode = 2;
      std::tie(seed, offset) = draw(x, hidden);
    }
  }
  const void* weights[2] = {ptr(w1), ptr(w2)};
  const void* biases[2] = {ptr(b1), ptr(b2)};
  const int64_t outs[2] = {inner, out};
  if (rows > 0)
    check(api.mlp_fwd(2, ptr(x), weights, biases, outs, rows, in, ptr(r.out), ptr(r.post), ptr(r.pre), static_cast<uint8_t*>(ptr(r.mask)), mode,
                      static_cast<float>(p), seed, offset, static_cast<int>(act), dtype_code(x), on.stream), "nmtg_mlp_fwd");
  return r;
}

MlpGrads mlp_bwd(const Tensor& dy, const Tensor& x, const Tensor& w1, const Tensor& w2, const Tensor& post, const Tensor& pre,
                 const Tensor& mask, double p, int64_t act, bool want_x, bool want_w, bool want_b1, bool want_b2) {
  const int64_t in = w1.size(1), rows = x.numel() / in, outs[2] = {w1.size(0), w2.size(0)};
  Launch on(dy);
  MlpGrads r;
  if (want_x) r.dx = new_like(x);
  if (want_w) { r.dw1 = new_like(w1); r.dw2 = new_like(w2); }
  if (want_b1) r.db1 = empty_like_sized(x, {outs[0]});
  if (want_b2) r.db2 = empty_like_sized(x, {outs[1]});
  if (rows == 0) {                                  // an empty batch contributes zero gradients
    for (Tensor* t : {&r.dw1, &r.dw2, &r.db1, &r.db2}) if (t->defined()) t->zero_();
    return r;
  }
  const Scratch ws = mlp_workspace(x, 2, outs, rows, in);
  const void* weights[2] = {ptr(w1), ptr(w2)};
  void* dws[2] = {ptr(r.dw1), ptr(r.dw2)};
  void* dbs[2] = {ptr(r.db1), ptr(r.db2)};
  check(api.mlp_bwd(2, ptr(x), weights, outs, rows, in, ptr(dy), ptr(post), ptr(pre), p > 0.0 ? static_cast<const uint8_t*>(ptr(mask)) : nullptr,
                    static_cast<float>(p), static_cast<int>(act), ptr(r.dx), dws, dbs, ws.get(), ws.bytes, dtype_code(x), on.stream),
        "nmtg_mlp_bwd");
  return r;
}

// ------------------------------------------------------------------------------------------------ dropout + residual
Tensor dropout_add_(const Tensor& x, const Tensor& residual, double p, bool training) {
  Launch on(x);
  Tensor mask;
  int mode = 0;
  uint64_t seed = 0, offset = 0;
  if (training && p > 0.0) {
    mask = empty_as(x, x.sizes(), at::kByte);
    mode = 2;
    std::tie(seed, offset) = draw(x, x.numel());
  }
  check(api.dropout_add_fwd(ptr(x), ptr(residual), static_cast<uint8_t*>(ptr(mask)), x.numel(), static_cast<float>(p), mode, seed, offset,
                            dtype_code(x), on.stream), "nmtg_dropout_add_fwd");
  return mask;
}

Tensor dropout_bwd(const Tensor& g, const Tensor& mask, double p) {
  Launch on(g);
  Tensor dx = new_like(g);
  check(api.dropout_add_bwd(ptr(g), static_cast<const uint8_t*>(mask.data_ptr()), ptr(dx), g.numel(), static_cast<float>(p), dtype_code(g),
                            on.stream), "nmtg_dropout_add_bwd");
  return dx;
}

Tensor dropout_add_guard_(const Tensor& x, const Tensor& residual, double p, const Tensor& flag, bool want_mask) {
  Launch on(x);
  Tensor mask;
  uint64_t seed = 0, offset = 0;
  if (p > 0.0) std::tie(seed, offset) = draw(x, x.numel());
  if (p > 0.0 || want_mask) mask = empty_as(x, x.sizes(), at::kByte);
  check(api.dropout_add_guard_fwd(ptr(x), ptr(residual), static_cast<uint8_t*>(ptr(mask)), x.numel(), static_cast<float>(p), p > 0.0 ? 2 : 0,
                                  seed, offset, static_cast<int*>(ptr(flag)), dtype_code(x), on.stream), "nmtg_dropout_add_guard_fwd");
  return mask;
}

Tensor dropout_guard_bwd(const Tensor& g, const Tensor& mask, double p) {
  Launch on(g);
  Tensor dx = new_like(g);
  check(api.dropout_add_guard_bwd(ptr(g), static_cast<const uint8_t*>(mask.data_ptr()), ptr(dx), g.numel(), static_cast<float>(p),
                                  dtype_code(g), on.stream), "nmtg_dropout_add_guard_bwd");
  return dx;
}

// ------------------------------------------------------------------------------------------------------ tiled attention
static Tensor bits_words(const Tensor& like, int64_t b, int64_t h, int64_t tq, int64_t tk) {
  return empty_as(like, {std::max<int64_t>(api.flash_attn_dropout_bits_bytes(b, h, tq, tk), 16) / 4}, at::kInt);
}
static Scratch info_words(const Tensor& like, int64_t bytes) { return Scratch(like, std::max<int64_t>(bytes, 4)); }

Tensor slot(const Tensor& lin, int64_t heads, int64_t parts, int64_t which) {
  const int64_t d = lin.size(2) / (heads * parts);
  return lin.as_strided({lin.size(0), lin.size(1), heads, d}, {lin.stride(0), lin.stride(1), parts * d, 1}, lin.storage_offset() + which * d);
}

Tensor pad_bytes(const optional<Tensor>& mask, const Tensor& operand, int64_t rows, int64_t cols) {
  if (!mask.has_value() || !mask->defined() || mask->numel() == 0) return Tensor();
  check_device(*mask, operand);
  TORCH_CHECK(mask->numel() == rows * cols, "mask must be [", rows, ", ", cols, "]");
  Tensor m = contiguous(*mask).view({rows, cols});
  if (m.scalar_type() == at::kBool) return m.view(at::kByte);          // a bool mask is its bytes
  return m.scalar_type() == at::kByte ? m : m.to(at::kByte);
}

Flash flash_fwd_batched(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& pad, const Tensor& time_mask, double p,
                        double scale, bool causal, Coverage coverage) {
  TORCH_CHECK((q.scalar_type() == at::kHalf || q.scalar_type() == at::kBFloat16) && k.scalar_type() == q.scalar_type() &&
              v.scalar_type() == q.scalar_type(), "flash_attn: q, k and v must share a 16-bit dtype");
  TORCH_CHECK(q.dim() == 4 && k.dim() == 4 && k.sizes() == v.sizes(), "flash_attn: q [len_q, B, H, D], k and v [len_k, B, H, D]");
  TORCH_CHECK(k.sizes().slice(1) == q.sizes().slice(1), "flash_attn: k and v must have q's batch, heads and head_dim");
  for (const Tensor* t : {&q, &k, &v}) {
    TORCH_CHECK(t->device() == q.device(), "expected a tensor in device memory (HIP); this op has no CPU path");
    TORCH_CHECK(t->stride(3) == 1, "flash_attn: the head dimension must be contiguous");
  }
  auto byte_mask = [&](const Tensor& m, int64_t rows, int64_t cols) {
    return m.device() == q.device() && m.scalar_type() == at::kByte && m.dim() == 2 && m.size(0) == rows && m.size(1) == cols && m.is_contiguous();
  };
  TORCH_CHECK(!pad.defined() || byte_mask(pad, q.size(1), k.size(0)), "flash_attn: key_padding_mask must be contiguous uint8 [batch, len_k]");
  TORCH_CHECK(!time_mask.defined() || byte_mask(time_mask, q.size(0), k.size(0)), "flash_attn: time_mask must be contiguous uint8 [len_q, len_k]");
  const int64_t tq = q.size(0), b = q.size(1), h = q.size(2), d = q.size(3), tk = k.size(0);
  Launch on(q);
  Flash r;
  r.out = empty_like_sized(q, {tq, b, h, d});
  r.lse = empty_as(q, {b, h, tq}, at::kFloat);
  Scratch kinfo, tinfo;
  if (pad.defined()) kinfo = info_words(q, api.flash_attn_key_info_bytes(b, tk));
  if (time_mask.defined()) tinfo = info_words(q, api.flash_attn_time_info_bytes(tq, tk));
  if (p > 0.0) {
    r.bits.words = bits_words(q, b, h, tq, tk);
    r.bits.mode = coverage == Coverage::none ? 2 : 3;
    std::tie(r.bits.seed, r.bits.offset) = draw(q, coverage == Coverage::none ? 4 * b * h * ((tq + 3) / 4) * ((tk + 3) / 4) : b * h * tq * tk);
  }
  if (coverage != Coverage::none) {
    r.probs = empty_like_sized(q, {b * h, tq, tk});
    check(api.flash_attn_batched_fwd_probs(
              ptr(q), ptr(k), ptr(v), ptr(r.out), static_cast<const uint8_t*>(ptr(pad)), kinfo.get(), static_cast<const uint8_t*>(ptr(time_mask)),
              tinfo.get(), r.lse.data_ptr<float>(), b, h, d, tq, tk, q.stride(0), q.stride(1), q.stride(2), k.stride(0), k.stride(1),
              k.stride(2), v.stride(0), v.stride(1), v.stride(2), r.out.stride(0), r.out.stride(1), r.out.stride(2), static_cast<float>(scale),
              causal ? 1 : 0, static_cast<int>(r.bits.mode), static_cast<float>(p), nullptr, nullptr, ptr(r.bits.words), r.bits.seed,
              r.bits.offset, dtype_code(q), on.stream, ptr(r.probs), coverage == Coverage::dropped ? 1 : 0),
          "nmtg_flash_attn_batched_fwd_probs");
    return r;
  }
  check(api.flash_attn_batched_fwd(ptr(q), ptr(k), ptr(v), ptr(r.out), static_cast<const uint8_t*>(ptr(pad)), kinfo.get(),
                                   static_cast<const uint8_t*>(ptr(time_mask)), tinfo.get(), r.lse.data_ptr<float>(), b, h, d, tq, tk,
                                   q.stride(0), q.stride(1), q.stride(2), k.stride(0), k.stride(1), k.stride(2), v.stride(0), v.stride(1),
                                   v.stride(2), r.out.stride(0), r.out.stride(1), r.out.stride(2), static_cast<float>(scale), causal ? 1 : 0,
                                   static_cast<int>(r.bits.mode), static_cast<float>(p), nullptr, nullptr, ptr(r.bits.words), r.bits.seed,
                                   r.bits.offset, dtype_code(q), on.stream), "nmtg_flash_attn_batched_fwd");
  return r;
}

View head_view(const Tensor& x, int64_t heads) { return {ptr(x), x.stride(0), x.stride(1), x.size(2) / heads}; }
View slot_view(const Tensor& lin, int64_t heads, int64_t parts, int64_t which) {
  const int64_t d = lin.size(2) / (heads * parts);
  return {static_cast<char*>(ptr(lin)) + which * d * static_cast<int64_t>(lin.element_size()), lin.stride(0), lin.stride(1), parts * d};
}

void flash_bwd_batched(const FlashShape& s, const Tensor& dout, const View& q, const View& k, const View& v, const Tensor& out, const Tensor& lse,
                       const View& dq, const View& dk, const View& dv, const Tensor& pad, const Tensor& time_mask, double p, double scale,
                       bool causal, const Bits& bits) {
  Launch on(out);
  Scratch kinfo, tinfo, sd(out, s.b * s.h * s.tq * static_cast<int64_t>(sizeof(float)));
  if (pad.defined()) kinfo = info_words(out, api.flash_attn_key_info_bytes(s.b, s.tk));
  if (time_mask.defined()) tinfo = info_words(out, api.flash_attn_time_info_bytes(s.tq, s.tk));
  check(api.flash_attn_batched_bwd(ptr(dout), q.data, k.data, v.data, ptr(out), lse.data_ptr<float>(), dq.data, dk.data, dv.data, sd.get<float>(),
                                   static_cast<const uint8_t*>(ptr(pad)), kinfo.get(), static_cast<const uint8_t*>(ptr(time_mask)), tinfo.get(),
                                   s.b, s.h, s.d, s.tq, s.tk, q.stride_t, q.stride_b, q.stride_h, k.stride_t, k.stride_b, k.stride_h, v.stride_t,
                                   v.stride_b, v.stride_h, out.stride(0), out.stride(1), out.stride(2), static_cast<float>(scale),
                                   causal ? 1 : 0, static_cast<int>(bits.mode), static_cast<float>(p), nullptr, ptr(bits.words),
                                   bits.words.defined() ? 1 : 0, bits.seed, bits.offset, dtype_code(out), on.stream),
        "nmtg_flash_attn_batched_bwd");
}

}  // namespace nmtg_host

PYBIND11_MODULE(_host, m) {
  m.def("bind", &nmtg_host::bind);
  nmtg_host::define_autograd(m);
  nmtg_host::define_layers(m);
  nmtg_host::define_optim(m);
  nmtg_host::define_attention(m);
  nmtg_host::define_loss(m);
}
