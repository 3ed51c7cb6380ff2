// Shared pieces of the native host layer (nmtgminor_amd/_host.so): the table of C entry points it calls, and the
// operators as functions from tensors to tensors (allocate the results, enqueue the kernels). ops.cpp implements them,
// autograd.cpp wraps them in autograd nodes, layers.cpp composes the transformer layers, attention.cpp the attention modules, loss.cpp the output
// projection with its loss, optim.cpp prepares the optimizer's passes.
//
// Why it exists: interpreter, ctypes and autograd bookkeeping of a call through the Python functions take several times what
// the kernels of a small batch take. Host time of a call on [64 x 512], LayerNorm / feed-forward block / dropout + add: forward
// 20 / 27 / 20 us there and 6 / 12 / 11 here, forward and backward 146 / 190 / 118 and 66 / 90 / 61 (about 40 of those are the
// autograd engine's way to its own thread and back).
#pragma once
#include <torch/extension.h>
#include <torch/csrc/autograd/forward_grad.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/core/CPUAllocator.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPCachingAllocator.h>
#include <c10/hip/HIPStream.h>
#include <optional>
#include <tuple>
#include <vector>

#include "../../../include/nmtg_hip.h"

namespace nmtg_host {

using at::Tensor;
using std::optional;

// The C entry points, resolved from the library that the Python side loaded (bind()).
#define NMTG_HOST_API(X)                                                                                              \
  X(last_error) X(ln_fwd) X(ln_bwd_parts) X(ln_bwd) X(dropout_add_fwd) X(dropout_add_bwd) X(xentropy_fwd)             \
  X(add_ln_fwd) X(ln_bwd_add) X(dropout_add_guard_fwd) X(dropout_add_guard_bwd) X(encdec_attn_fwd)                    \
  X(attn_decode) X(attn_decode_append) X(encdec_attn_bwd_workspace_bytes) X(encdec_attn_bwd_from_probs)               \
  X(attn_scores_needed)                                                                                               \
  X(xentropy_bwd) X(gemm) X(mlp_fwd) X(mlp_bwd_dtype_workspace_bytes) X(mlp_bwd) X(flash_attn_dropout_bits_bytes)     \
  X(flash_attn_fwd) X(flash_attn_bwd) X(flash_attn_key_info_bytes) X(flash_attn_time_info_bytes)                      \
  X(flash_attn_batched_fwd) X(flash_attn_batched_bwd) X(multi_tensor_adam) X(multi_tensor_clip)                       \
  X(multi_tensor_l2norm) X(multi_tensor_l2norm_workspace_bytes) X(flash_attn_batched_fwd_probs) X(linear_step) X(step_linear) X(step_linear_ok) X(gemm_workspace_bytes) \
  X(xentropy_bwd_colsum) X(xentropy_bwd_colsum_parts)

struct Api {
#define X(name) decltype(&nmtg_##name) name = nullptr;
  NMTG_HOST_API(X)
#undef X
};
extern Api api;
void bind(const std::string& path);

// The stream of a tensor's device, with that device made current for the scope.
struct Launch {
  c10::OptionalDeviceGuard guard;
  void* stream = nullptr;
  explicit Launch(const Tensor& t) {
    if (t.is_cuda()) {
      guard.reset_device(t.device());
      stream = c10::hip::getCurrentHIPStream(t.device().index()).stream();
    }
  }
};

void check(int rc, const char* what);
int dtype_code(const Tensor& t);
inline void* ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
inline void* ptr(const optional<Tensor>& t) { return t.has_value() ? ptr(*t) : nullptr; }
// A forward-mode dual: its tangent would be lost where the autograd node is passed by (the node itself refuses it). Duals exist
// while a level is open, which is asked first: a look at one tensor takes a lock of its own.
inline bool forward_mode() { return torch::autograd::ForwardADLevel::try_get_by_idx(0) != nullptr; }
inline bool has_tangent(const Tensor& t) { return t.defined() && t._fw_grad(/*level=*/0).defined(); }
inline Tensor contiguous(const Tensor& t) { return t.is_contiguous() ? t : t.contiguous(); }
// Results. A small batch is bound by this host work, and a layer's pass makes some 60 tensors: the allocator's own entry
// leaves out at::empty's way through the dispatcher. With it, Scratch and View (the six views of the attention's backward cost a
// dispatcher call each), enqueuing an encoder layer's pass of 8 positions went from 375 to 341 us, its backward from 206 to 179.
inline Tensor empty_as(const Tensor& like, at::IntArrayRef sizes, at::ScalarType type) {
  if (like.is_cuda()) return Tensor(at::detail::empty_cuda(sizes, type, like.device(), std::nullopt));
  return at::empty(sizes, like.options().dtype(type).requires_grad(false));
}
inline Tensor empty_like_sized(const Tensor& like, at::IntArrayRef sizes) { return empty_as(like, sizes, like.scalar_type()); }
inline Tensor new_like(const Tensor& like) { return like.is_contiguous() ? empty_as(like, like.sizes(), like.scalar_type()) : at::empty_like(like); }
// Memory of one call, on the stream and device that its Launch made current: no tensor around it, and given back to the
// allocator when the scope ends, for later work of that stream.
struct Scratch {
  int64_t bytes = 0;
  c10::DataPtr data;
  Scratch() = default;
  Scratch(const Tensor& like, int64_t n)
      : bytes(n), data((like.is_cuda() ? static_cast<c10::Allocator*>(c10::hip::HIPCachingAllocator::get()) : c10::GetCPUAllocator())->allocate(n)) {}
  template <typename T = void> T* get() const { return static_cast<T*>(data.get()); }
};
// (seed, offset) of the tensor's default generator, whose offset is advanced past `count` draws
std::pair<uint64_t, uint64_t> draw(const Tensor& like, int64_t count);

// ---- operators ------------------------------------------------------------------------------------------------------
struct Norm { Tensor z, stats; };                        // stats: fp32 [2, rows], mean then 1 / sigma
Norm ln_fwd(const Tensor& x, const Tensor& gamma, const Tensor& beta, double eps);
struct NormGrads { Tensor dx, dgamma, dbeta; };
NormGrads ln_bwd(const Tensor& dz, const Tensor& x_or_z, const Tensor& stats, const Tensor& gamma, const Tensor& beta, bool memory_efficient);

// h = residual + dropout(x), z = LayerNorm(h); mask undefined without dropout. clear: a device int set to 0, or undefined
struct AddNorm { Tensor h, z, stats, mask; };
AddNorm add_ln_fwd(const Tensor& x, const Tensor& residual, double p, const Tensor& clear, const Tensor& gamma, const Tensor& beta, double eps);
// backward of a LayerNorm on a residual stream: dx includes the stream's gradient; keep defined: dy = dx * keep / (1 - p) too
struct AddNormGrads { Tensor dx, dy, dgamma, dbeta; };
AddNormGrads ln_bwd_add(const Tensor& dz, const Tensor& x, const Tensor& stats, const Tensor& gamma, const Tensor& grad_residual,
                        const Tensor& guard, const Tensor& keep, double p);

Tensor linear_fwd(const Tensor& x, const Tensor& w, const Tensor& b);
Tensor linear_step(const Tensor& x, const Tensor& w, const Tensor& b);          // of a decoding step: few rows, no gradient
// the same on LayerNorm(x), or with a residual on LayerNorm(h), h = x + residual (see nmtg_step_linear)
struct StepNorm { Tensor y, h; };
StepNorm norm_step(const Tensor& x, const Tensor& residual, const Tensor& gamma, const Tensor& beta, double eps, const Tensor& clear, const Tensor& w,
                   const Tensor& b, int64_t act);
Tensor linear_add_step(const Tensor& x, const Tensor& w, const Tensor& b, const Tensor& add, const Tensor& guard);
struct LinearGrads { Tensor dx, dw, db; };
LinearGrads linear_bwd(const Tensor& dy, const Tensor& x, const Tensor& w, bool want_x, bool want_w, bool want_b);

struct Mlp { Tensor out, post, pre, mask; };
Mlp mlp_fwd(const Tensor& x, const Tensor& w1, const Tensor& w2, const Tensor& b1, const Tensor& b2, double p, int64_t act,
            const optional<Tensor>& mask, bool save_pre);
struct MlpGrads { Tensor dx, dw1, dw2, db1, db2; };
MlpGrads mlp_bwd(const Tensor& dy, const Tensor& x, const Tensor& w1, const Tensor& w2, const Tensor& post, const Tensor& pre,
                 const Tensor& mask, double p, int64_t act, bool want_x, bool want_w, bool want_b1, bool want_b2);

// x <- residual + dropout(x) in place; returns the keep-mask (undefined without dropout)
Tensor dropout_add_(const Tensor& x, const Tensor& residual, double p, bool training);
Tensor dropout_bwd(const Tensor& g, const Tensor& mask, double p);
// the same at the end of a layer, with the clamp of a stream that holds an inf or NaN (nmtg_dropout_add_guard_fwd); the mask
// comes back with want_mask or dropout. flag: a zeroed device int
Tensor dropout_add_guard_(const Tensor& x, const Tensor& residual, double p, const Tensor& flag, bool want_mask);
Tensor dropout_guard_bwd(const Tensor& g, const Tensor& mask, double p);

struct Bits { int64_t mode = 0; uint64_t seed = 0, offset = 0; Tensor words; };
// attention over a padded batch: q [Tq, B, H, D], k / v [Tk, B, H, D]
// coverage: the probabilities come back too ([B * H, Tq, Tk], before or after dropout), and the dropout mask is drawn in the
// extension modules' numbering
enum class Coverage { none, softmax, dropped };
struct Flash { Tensor out, lse, probs; Bits bits; };
Flash flash_fwd_batched(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& pad, const Tensor& time_mask, double p,
                        double scale, bool causal, Coverage coverage = Coverage::none);
// The same operand by its address and strides (in elements, D contiguous), for the backward, which hands out no views: of
// heads next to each other [T, B, H * D], or of one part of a projection (see slot)
struct View {
  void* data;
  int64_t stride_t, stride_b, stride_h;
};
View head_view(const Tensor& x, int64_t heads);
View slot_view(const Tensor& lin, int64_t heads, int64_t parts, int64_t which);
// out [Tq, B, H, D] contiguous, dout in its layout
struct FlashShape { int64_t tq, tk, b, h, d; };
void flash_bwd_batched(const FlashShape& shape, const Tensor& dout, const View& q, const View& k, const View& v, const Tensor& out, const Tensor& lse,
                       const View& dq, const View& dk, const View& dv, const Tensor& pad, const Tensor& time_mask, double p, double scale,
                       bool causal, const Bits& bits);
// q / k / v slots of a projection [T, B, H, parts, D]
Tensor slot(const Tensor& lin, int64_t heads, int64_t parts, int64_t which);
// a mask as contiguous bytes [rows, cols], on the device of the operand it belongs to (a kernel is handed its address)
Tensor pad_bytes(const optional<Tensor>& mask, const Tensor& operand, int64_t rows, int64_t cols);
inline void check_device(const Tensor& t, const Tensor& operand) {
  TORCH_CHECK(!t.defined() || t.device() == operand.device(), "expected a tensor on ", operand.device(), ", got one on ", t.device());
}

void define_autograd(pybind11::module_& m);
void define_layers(pybind11::module_& m);
void define_optim(pybind11::module_& m);
void define_attention(pybind11::module_& m);
void define_loss(pybind11::module_& m);

}  // namespace nmtg_host
