// Dropout + residual add, and its backward (masked scale), for gfx950.
//
// Stands in for fused_dropout_add_cuda.forward / backward of the reference
// (onmt/modules/extensions/dropout_add/fused_dropout_add_cuda_kernel.cu:19-95, kernels
// dropout.h:72-189). out = residual + x * keep / (1 - p), written in place into x; the keep mask
// is one byte per element (1 = keep). The mask either comes from the caller (replay / tests) or
// is drawn here from Philox4x32-10 keyed by (seed, offset, element index).
//
// Bandwidth bound: forward reads x and residual, writes x and 1 B/element of mask; backward
// reads g and the mask, writes dx. Each lane moves 16 bytes per access; the grid covers the
// tensor once (no grid-stride tail) so every CU streams contiguous 4 KiB wavefront chunks.
#include "common.hip.h"

namespace nmtg {
namespace {

constexpr int DA_THREADS = 256;
enum { DA_EVAL = 0, DA_MASK_IN = 1, DA_MASK_RNG = 2 };

template <typename T, int EPV, int MODE>
__global__ __launch_bounds__(DA_THREADS) void dropout_add_fwd_kernel(
    T* __restrict__ x, const T* __restrict__ residual, uint8_t* __restrict__ mask, int64_t n, float keep_p,
    float scale, uint64_t seed, uint64_t offset) {
  const int64_t first = (static_cast<int64_t>(blockIdx.x) * DA_THREADS + threadIdx.x) * EPV;
  if (first >= n) return;
  if (first + EPV <= n) {
    // all loads are issued before the first conversion, so the lane waits for memory once
    pack<T, EPV> rawx = load_raw<T, EPV>(x + first), rawr = load_raw<T, EPV>(residual + first);
    pack<uint8_t, EPV> rawm = {};
    if constexpr (MODE == DA_MASK_IN) rawm = load_raw<uint8_t, EPV>(mask + first);
    pin_raw(rawx); pin_raw(rawr); pin_raw(rawm);
    float xv[EPV], rv[EPV];
    unpack_raw<T, EPV>(rawx, xv);
    unpack_raw<T, EPV>(rawr, rv);
    if constexpr (MODE == DA_EVAL) {
#pragma unroll
      for (int j = 0; j < EPV; ++j) xv[j] += rv[j];
    } else {
      uint8_t keep[EPV];
      if constexpr (MODE == DA_MASK_IN) {
#pragma unroll
        for (int j = 0; j < EPV; ++j) keep[j] = rawm.v[j];
      } else {
        philox_keep<EPV>(Philox(seed), static_cast<uint64_t>(first), offset, keep_p, keep);
        store_bytes<EPV>(mask + first, keep);
      }
#pragma unroll
      for (int j = 0; j < EPV; ++j) xv[j] = rv[j] + (keep[j] ? xv[j] * scale : 0.f);
    }
    store_pack<T, EPV>(x + first, xv);
  } else {  // ragged tail: scalar
    for (int64_t e = first; e < n; ++e) {
      float xv = elem<T>::to_float(x[e]);
      const float rv = elem<T>::to_float(residual[e]);
      if constexpr (MODE == DA_EVAL) {
        xv += rv;
      } else {
        uint8_t keep[1];
        if constexpr (MODE == DA_MASK_IN) keep[0] = mask[e];
        else { philox_keep<1>(Philox(seed), static_cast<uint64_t>(e), offset, keep_p, keep); mask[e] = keep[0]; }
        xv = rv + (keep[0] ? xv * scale : 0.f);
      }
      x[e] = elem<T>::from_float(xv);
    }
  }
}

// ---------------------------------------------------------------------------------------------------------------------
// Dropout + residual add at the end of a layer, with the layer's guard on the way out: a layer clamps its outgoing stream
// to +-(largest finite value - 1000) when it holds an inf or NaN (the reference asks isinf(x).any() or isnan(x).any() on
// the host for that, two full passes and two synchronisations per layer). Here the element that is about to be stored is
// looked at in its register. For bf16 and fp32 the bound rounds to the largest finite value, so clamping an inf where it
// stands is the whole effect; for fp16 the bound (64504, stored as 64512) lies below the largest finite values, which are
// clamped too once any element of the tensor is not finite: the kernel raises `flag`, and guard_clamp_f16_kernel, behind
// it, returns at once unless it is raised. Bit 1 of an element's mask byte records that no gradient passes it (clamped or
// NaN). Bandwidth bound like the plain form: 22 us at [512 x 32 x 1024] bf16 with the mask drawn here, and none of the 39 us
// of the two reductions it replaces, nor a host round trip.
// ---------------------------------------------------------------------------------------------------------------------
template <typename T, int EPV, int MODE>
__device__ __forceinline__ void guard_pack(T* __restrict__ x, const T* __restrict__ residual, uint8_t* __restrict__ mask, int64_t first,
                                           float keep_p, float scale, uint64_t seed, uint64_t offset, int* __restrict__ flag) {
  pack<T, EPV> rawx = load_raw<T, EPV>(x + first), rawr = load_raw<T, EPV>(residual + first);
  pin_raw(rawx); pin_raw(rawr);
  float xv[EPV], rv[EPV];
  unpack_raw<T, EPV>(rawx, xv);
  unpack_raw<T, EPV>(rawr, rv);
  uint8_t keep[EPV];
  if constexpr (MODE == DA_MASK_RNG) {
    philox_keep<EPV>(Philox(seed), static_cast<uint64_t>(first), offset, keep_p, keep);
  } else {
#pragma unroll
    for (int j = 0; j < EPV; ++j) keep[j] = 1;
  }
#pragma unroll
  for (int j = 0; j < EPV; ++j) xv[j] = rv[j] + (keep[j] ? xv[j] * scale : 0.f);
  // one comparison per element (false for NaN); only a pack with an element at or beyond the largest finite value looks closer
  bool any = false;
#pragma unroll
  for (int j = 0; j < EPV; ++j) any = any || !(fabsf(xv[j]) < guard_limit<T>());
  if (any) {
    for (int j = 0; j < EPV; ++j) {
      T o = elem<T>::from_float(xv[j]);
      if (guard_element(o)) {
        keep[j] |= 2;
        if (flag != nullptr) *flag = 1;
      }
      x[first + j] = o;
      if (mask != nullptr) mask[first + j] = keep[j];
    }
    return;
  }
  store_pack<T, EPV>(x + first, xv);
  if (mask != nullptr) store_bytes<EPV>(mask + first, keep);
}

template <typename T, int EPV, int MODE>
__global__ __launch_bounds__(DA_THREADS) void dropout_add_guard_kernel(
    T* __restrict__ x, const T* __restrict__ residual, uint8_t* __restrict__ mask, int64_t n, float keep_p,
    float scale, uint64_t seed, uint64_t offset, int* __restrict__ flag) {
  const int64_t first = (static_cast<int64_t>(blockIdx.x) * DA_THREADS + threadIdx.x) * EPV;
  if (first >= n) return;
  if (first + EPV <= n) {
    guard_pack<T, EPV, MODE>(x, residual, mask, first, keep_p, scale, seed, offset, flag);
  } else {  // ragged tail: scalar
    for (int64_t e = first; e < n; ++e) guard_pack<T, 1, MODE>(x, residual, mask, e, keep_p, scale, seed, offset, flag);
  }
}

__global__ __launch_bounds__(DA_THREADS) void guard_clamp_f16_kernel(f16_t* __restrict__ x, uint8_t* __restrict__ mask, int64_t n,
                                                                     const int* __restrict__ flag) {
  if (*flag == 0) return;
  for (int64_t e = static_cast<int64_t>(blockIdx.x) * DA_THREADS + threadIdx.x; e < n; e += static_cast<int64_t>(gridDim.x) * DA_THREADS) {
    const uint16_t b = x[e].bits, mag = b & 0x7fffu;
    if (mag <= 0x7be0u) continue;                     // 64512, the bound as fp16 stores it
    if (mag <= 0x7c00u) x[e].bits = static_cast<uint16_t>((b & 0x8000u) | 0x7be0u);
    if (mask != nullptr) mask[e] |= 2;
  }
}

// GUARDED: mask bytes with bit 1 set (see above) pass no gradient either
template <typename T, int EPV, bool GUARDED>
__global__ __launch_bounds__(DA_THREADS) void masked_scale_kernel(
    const T* __restrict__ g, const uint8_t* __restrict__ mask, T* __restrict__ dx, int64_t n, float scale) {
  const int64_t first = (static_cast<int64_t>(blockIdx.x) * DA_THREADS + threadIdx.x) * EPV;
  if (first >= n) return;
  if (first + EPV <= n) {
    float gv[EPV];
    uint8_t keep[EPV];
    load_pack<T, EPV>(g + first, gv);
    load_bytes<EPV>(mask + first, keep);
#pragma unroll
    for (int j = 0; j < EPV; ++j) gv[j] = (GUARDED ? keep[j] == 1 : keep[j] != 0) ? gv[j] * scale : 0.f;
    store_pack<T, EPV>(dx + first, gv);
  } else {
    for (int64_t e = first; e < n; ++e)
      dx[e] = elem<T>::from_float((GUARDED ? mask[e] == 1 : mask[e] != 0) ? elem<T>::to_float(g[e]) * scale : 0.f);
  }
}

template <typename T>
int dropout_add_fwd_launch(void* x, const void* residual, uint8_t* mask, int64_t n, float p, int mode,
                           uint64_t seed, uint64_t offset, hipStream_t st) {
  const float keep_p = 1.f - p, scale = 1.f / (1.f - p);
  T* X = static_cast<T*>(x);
  const T* R = static_cast<const T*>(residual);
  constexpr int WIDE = 16 / sizeof(T);
  TraceScope trace("dropout_add_fwd", st);
  const bool wide = aligned16(x) && aligned16(residual) && (mode == DA_EVAL || aligned8(mask));
#define DA_LAUNCH(EPV, MODE)                                                                         \
  {                                                                                                  \
    const int64_t per_block = static_cast<int64_t>(DA_THREADS) * EPV;                                \
    const int64_t grid = (n + per_block - 1) / per_block;                                            \
    hipLaunchKernelGGL((dropout_add_fwd_kernel<T, EPV, MODE>), dim3(static_cast<unsigned>(grid)),    \
                       dim3(DA_THREADS), 0, st, X, R, mask, n, keep_p, scale, seed, offset);         \
  }
  if (wide) {
    if (mode == DA_EVAL) DA_LAUNCH(WIDE, DA_EVAL)
    else if (mode == DA_MASK_IN) DA_LAUNCH(WIDE, DA_MASK_IN)
    else DA_LAUNCH(WIDE, DA_MASK_RNG)
  } else {
    if (mode == DA_EVAL) DA_LAUNCH(1, DA_EVAL)
    else if (mode == DA_MASK_IN) DA_LAUNCH(1, DA_MASK_IN)
    else DA_LAUNCH(1, DA_MASK_RNG)
  }
#undef DA_LAUNCH
  return 0;
}

template <typename T, bool GUARDED>
int masked_scale_launch(const void* g, const uint8_t* mask, void* dx, int64_t n, float p, hipStream_t st) {
  const float scale = 1.f / (1.f - p);
  constexpr int WIDE = 16 / sizeof(T);
  const bool wide = aligned16(g) && aligned16(dx) && aligned8(mask);
  TraceScope trace("dropout_add_bwd", st);
  if (wide) {
    const int64_t per_block = static_cast<int64_t>(DA_THREADS) * WIDE;
    hipLaunchKernelGGL((masked_scale_kernel<T, WIDE, GUARDED>), dim3(static_cast<unsigned>((n + per_block - 1) / per_block)),
                       dim3(DA_THREADS), 0, st, static_cast<const T*>(g), mask, static_cast<T*>(dx), n, scale);
  } else {
    hipLaunchKernelGGL((masked_scale_kernel<T, 1, GUARDED>), dim3(static_cast<unsigned>((n + DA_THREADS - 1) / DA_THREADS)),
                       dim3(DA_THREADS), 0, st, static_cast<const T*>(g), mask, static_cast<T*>(dx), n, scale);
  }
  return 0;
}

template <typename T>
int guard_launch(void* x, const void* residual, uint8_t* mask, int64_t n, float p, int mode, uint64_t seed, uint64_t offset, int* flag,
                 hipStream_t st) {
  constexpr int WIDE = 16 / sizeof(T);
  T* X = static_cast<T*>(x);
  const T* R = static_cast<const T*>(residual);
  const float keep_p = 1.f - p, scale = mode == DA_MASK_RNG ? 1.f / (1.f - p) : 1.f;
  const bool wide = aligned16(x) && aligned16(residual) && (mask == nullptr || aligned8(mask));
  TraceScope trace("dropout_add_guard", st);
  auto go = [&](auto kern, int epv) {
    const int64_t per_block = static_cast<int64_t>(DA_THREADS) * epv;
    hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>((n + per_block - 1) / per_block)), dim3(DA_THREADS), 0, st, X, R, mask, n, keep_p,
                       scale, seed, offset, flag);
  };
  if (mode == DA_MASK_RNG) wide ? go(dropout_add_guard_kernel<T, WIDE, DA_MASK_RNG>, WIDE) : go(dropout_add_guard_kernel<T, 1, DA_MASK_RNG>, 1);
  else wide ? go(dropout_add_guard_kernel<T, WIDE, DA_EVAL>, WIDE) : go(dropout_add_guard_kernel<T, 1, DA_EVAL>, 1);
  return 0;
}

}  // namespace
// Behind the kernel that raises `flag`: the clamp of an fp16 stream that is not finite everywhere (also behind the decoding step's
// last product, gemm_skinny.hip).
void guard_clamp_f16(void* x, uint8_t* mask, int64_t n, const int* flag, hipStream_t st) {
  const int64_t blocks = (n + DA_THREADS * 8 - 1) / (DA_THREADS * 8), cap = num_cus();
  hipLaunchKernelGGL(guard_clamp_f16_kernel, dim3(static_cast<unsigned>(blocks < cap ? blocks : cap)), dim3(DA_THREADS), 0, st,
                     static_cast<f16_t*>(x), mask, n, flag);
}

}  // namespace nmtg

using namespace nmtg;

extern "C" int nmtg_dropout_add_guard_fwd(void* x, const void* residual, uint8_t* mask, int64_t n, float p, int mask_mode, uint64_t seed,
                                          uint64_t offset, int* flag, int dtype, void* stream) {
  NMTG_REQUIRE(n >= 0 && n < (int64_t(1) << 40), "dropout_add_guard_fwd: bad element count %lld", (long long)n);
  NMTG_REQUIRE(mask_mode == DA_EVAL || mask_mode == DA_MASK_RNG, "dropout_add_guard_fwd: bad mask_mode %d", mask_mode);
  if (n == 0) return 0;
  NMTG_REQUIRE(x && residual, "dropout_add_guard_fwd: null pointer argument");
  NMTG_REQUIRE(dtype != NMTG_F16 || flag != nullptr, "dropout_add_guard_fwd: fp16 needs a flag (a zeroed int on the device)");
  NMTG_REQUIRE(mask_mode == DA_EVAL || (mask != nullptr && p >= 0.f && p < 1.f), "dropout_add_guard_fwd: mask buffer and p in [0, 1) required");
  hipStream_t st = static_cast<hipStream_t>(stream);
  int rc = 0;
  NMTG_DISPATCH_DTYPE(dtype, T, rc = guard_launch<T>(x, residual, mask, n, p, mask_mode, seed, offset, flag, st));
  if (rc) return rc;
  if (dtype == NMTG_F16) guard_clamp_f16(x, mask, n, flag, st);
  NMTG_CHECK_LAUNCH("dropout_add_guard_fwd");
  return 0;
}

extern "C" int nmtg_dropout_add_guard_bwd(const void* grad_out, const uint8_t* mask, void* grad_x, int64_t n, float p, int dtype, void* stream) {
  NMTG_REQUIRE(n >= 0 && n < (int64_t(1) << 40), "dropout_add_guard_bwd: bad element count %lld", (long long)n);
  if (n == 0) return 0;
  NMTG_REQUIRE(grad_out && mask && grad_x, "dropout_add_guard_bwd: null pointer argument");
  NMTG_REQUIRE(p >= 0.f && p < 1.f, "dropout_add_guard_bwd: dropout probability %f outside [0, 1)", p);
  int rc = 0;
  NMTG_DISPATCH_DTYPE(dtype, T, rc = (masked_scale_launch<T, true>(grad_out, mask, grad_x, n, p, static_cast<hipStream_t>(stream))));
  if (rc) return rc;
  NMTG_CHECK_LAUNCH("dropout_add_guard_bwd");
  return 0;
}

extern "C" int nmtg_dropout_add_fwd(void* x, const void* residual, uint8_t* mask, int64_t n, float p,
                                    int mask_mode, uint64_t seed, uint64_t offset, int dtype, void* stream) {
  NMTG_REQUIRE(n >= 0 && n < (int64_t(1) << 40), "dropout_add_fwd: bad element count %lld", (long long)n);
  NMTG_REQUIRE(mask_mode >= DA_EVAL && mask_mode <= DA_MASK_RNG, "dropout_add_fwd: bad mask_mode %d", mask_mode);
  if (n == 0) return 0;
  NMTG_REQUIRE(x && residual, "dropout_add_fwd: null pointer argument");
  if (mask_mode != DA_EVAL) {
    NMTG_REQUIRE(mask != nullptr, "dropout_add_fwd: mask buffer required when dropout is applied");
    NMTG_REQUIRE(p >= 0.f && p < 1.f, "dropout_add_fwd: dropout probability %f outside [0, 1)", p);
  }
  int rc = 0;
  NMTG_DISPATCH_DTYPE(dtype, T, rc = dropout_add_fwd_launch<T>(x, residual, mask, n, p, mask_mode, seed, offset,
                                                                static_cast<hipStream_t>(stream)));
  if (rc) return rc;
  NMTG_CHECK_LAUNCH("dropout_add_fwd");
  return 0;
}

extern "C" int nmtg_dropout_add_bwd(const void* grad_out, const uint8_t* mask, void* grad_x, int64_t n, float p,
                                    int dtype, void* stream) {
  NMTG_REQUIRE(n >= 0 && n < (int64_t(1) << 40), "dropout_add_bwd: bad element count %lld", (long long)n);
  if (n == 0) return 0;
  NMTG_REQUIRE(grad_out && mask && grad_x, "dropout_add_bwd: null pointer argument");
  NMTG_REQUIRE(p >= 0.f && p < 1.f, "dropout_add_bwd: dropout probability %f outside [0, 1)", p);
  int rc = 0;
  NMTG_DISPATCH_DTYPE(dtype, T, rc = (masked_scale_launch<T, false>(grad_out, mask, grad_x, n, p, static_cast<hipStream_t>(stream))));
  if (rc) return rc;
  NMTG_CHECK_LAUNCH("dropout_add_bwd");
  return 0;
}
