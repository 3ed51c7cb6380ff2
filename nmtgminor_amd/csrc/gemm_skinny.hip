// C[m][n] = alpha * sum_k X[m][k] W[n][k] (+ bias[n]) for at most 64 rows m: the projections of a decoding step
// (one new position of a few dozen hypotheses against a [1024 x 1024] weight), which the reference runs as cuBLASLt
// calls like any other linear layer (onmt/modules/extensions/mlp_blaslt/linear.cpp:142-144).
//
// With so few rows the product is a read of W: 2 MB of weight against 64 KB of activations, and a 128 x 128 output
// tile leaves all but eight compute units idle while each of those walks the whole reduction. What counts is the
// latency of one block, so the reduction is spread over the wavefronts of a block instead: a block owns up to 32 output
// columns (sk_cols) and all (at most 32) rows, its eight wavefronts each take an eighth of k, load their slices of X and W
// straight into matrix-core operand layout (a lane's 16 bytes of its row: no LDS staging, every load of a 128-k chunk in
// flight at once), run v_mfma_f32_32x32x16 over them, and leave their 32 x 32 partial sums in LDS, where the block adds
// the eight of them up in a fixed order. A [1024 x 1024] weight is 128 blocks (8 columns) for up to 8 rows, 64 for more, of one
// load latency each.
#include "gemm.hip.h"

#include <algorithm>

namespace nmtg {
void guard_clamp_f16(void* x, uint8_t* mask, int64_t n, const int* flag, hipStream_t st);   // dropout_add.hip
namespace {

constexpr int SK_ROWS = 32, SK_WAVES = 8, SK_THREADS = 64 * SK_WAVES, SK_CHUNK = 128;
// Up to two row blocks where the caller allows it (GemmArgs::skinny_rows): a batch of 64 hypotheses re-reads W from L2 and
// still leaves the 128 x 128 tile far behind. Other calls of more than 32 rows stay with the tiles: the two sum the reduction
// in different orders, and in training a hidden activation within rounding of zero would pass the relu with the one and not
// with the other.
constexpr int SK_MAX_ROWS = 64;

// Columns per block: 32, and fewer of long rows of W, which one compute unit fetches slowly, while there is a compute unit for each
// block. More blocks read (and normalise, below) the same rows of X again, so the more rows the fewer. Steps of a
// decoder layer as a graph with at most 8192 / 16384 / 32768 elements of W per block: 5 rows, E = 512: 35.3 / 36.9 / 37.1 us (38.9 with 32
// columns throughout); 20 rows, E = 1024: 64.0 / 63.2 / 67.2 (70.6); 64 rows, E = 1024: 99.7 / 82.9 / 74.5 (77.7). The sums are the same.
// Products alone, each call on a weight that is in no cache, us with 32 / 16 / 8 columns on 256 compute units: [512 x 2048], 8 rows:
// 8.1 / 6.3 / 5.8; [2048 x 1024]: 5.5 / 4.7 / 4.5 (256 blocks of 8); [4096 x 1024]: 5.6 / 5.0 / 6.1 (512 of 8); [8192 x 1024]: 6.6 / 7.1 / 9.6;
// [32000 x 1024]: 20 / 23 / 29, 32 rows 28 / 38 / 59.
inline int sk_cols(int rows, int n, int k) {
  const int64_t most = rows <= 8 ? 8192 : rows <= SK_ROWS ? 16384 : 32768;
  const int64_t cus = num_cus(), row_blocks = (rows + SK_ROWS - 1) / SK_ROWS;
  int cols = 32;
  while (cols > 8 && static_cast<int64_t>(cols) * k > most && (n + static_cast<int64_t>(cols) / 2 - 1) / (cols / 2) * row_blocks <= cus) cols /= 2;
  return cols;
}

template <typename T>
__global__ __launch_bounds__(SK_THREADS) void gemm_skinny_kernel(const GemmArgs g, int cols) {
  __shared__ float part[SK_WAVES][16][64];               // partial tiles in accumulator layout
  const int tid = threadIdx.x, lane = tid & 63, half = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n0 = static_cast<int>(blockIdx.x) * cols;
  const T* X = static_cast<const T*>(g.A);
  const T* W = static_cast<const T*>(g.B);
  // this wavefront's share of k: whole 16-k steps, dealt out in chunks of 128 so that the loads in flight stay bounded
  const int steps = (g.K + 15) / 16, per = (steps + SK_WAVES - 1) / SK_WAVES;
  const int k_begin = wave * per * 16, k_end = min(g.K, (wave + 1) * per * 16);
  const int m0 = static_cast<int>(blockIdx.y) * SK_ROWS;
  const int m = m0 + (lane & 31), n = n0 + (lane & 31);
  const T* xrow = X + static_cast<int64_t>(m) * g.lda + 8 * half;
  const T* wrow = W + static_cast<int64_t>(n) * g.ldb + 8 * half;
  acc16_t acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.f;
  for (int k0 = k_begin; k0 < k_end; k0 += SK_CHUNK) {
    uint4 xf[SK_CHUNK / 16], wf[SK_CHUNK / 16];
#pragma unroll
    for (int s = 0; s < SK_CHUNK / 16; ++s) {
      const int k = k0 + 16 * s + 8 * half;               // K is a multiple of 8: a lane's 8 elements are all in or all out
      const bool in = k < k_end;
      xf[s] = in && m < g.M ? *reinterpret_cast<const uint4*>(xrow + k0 + 16 * s) : make_uint4(0, 0, 0, 0);
      wf[s] = in && (lane & 31) < cols && n < g.N ? *reinterpret_cast<const uint4*>(wrow + k0 + 16 * s) : make_uint4(0, 0, 0, 0);
    }
#pragma unroll
    for (int s = 0; s < SK_CHUNK / 16; ++s) mfma<T>::run(xf[s], wf[s], acc);   // acc[r], lane (j, half): row 8 (r / 4) + 4 half + r % 4, column j
  }
#pragma unroll
  for (int r = 0; r < 16; ++r) part[wave][r][lane] = acc[r];
  __syncthreads();
  // 1024 outputs, two per thread; the eight partial sums are added in wavefront order
  for (int o = tid; o < 16 * 64; o += SK_THREADS) {
    const int r = o >> 6, l = o & 63;
    float v = 0.f;
#pragma unroll
    for (int w = 0; w < SK_WAVES; ++w) v += part[w][r][l];
    const int row = m0 + 8 * (r / 4) + 4 * (l >> 5) + r % 4, col = n0 + (l & 31);
    if (row < g.M && (l & 31) < cols && col < g.N) {
      v *= g.alpha;
      if (g.bias != nullptr) v += elem<T>::to_float(static_cast<const T*>(g.bias)[col]);
      static_cast<T*>(g.C)[static_cast<int64_t>(row) * g.ldc + col] = elem<T>::from_float(v);
    }
  }
}

// ---- the products of a decoder layer's step with what stands around them (nmtg_step_linear) ----
// A step is a chain of launches of a few microseconds that depend on each other, so what counts is their number. In front:
// LayerNorm of x, or of h = x + residual, computed by every block for its rows (5 rows x 512: one row per wavefront) while its
// weights are on their way from memory; block 0 writes h. Behind: the activation, or the layer's last addition with its guard.
// Rounding points are those of the separate kernels (h, the normalised row, the product with its bias). The sums are in the same
// order but for the product in front of an activation, which the separate calls run on the tiled kernels and this one as eight
// partial sums over k: a step is evaluation, where no gradient depends on the side of a gate that a value rounds to. A beam of 5 at
// E = 512 in fp16: 13 launches and 50 us of kernels for a step, 9 and 39 with these.
enum { STEP_PRE_NONE = 0, STEP_PRE_NORM = 1, STEP_PRE_ADD_NORM = 2 };
enum { STEP_POST_ACT = 0, STEP_POST_ADD = 1 };
constexpr int STEP_MAX_NORM = 1024;                      // columns that a wavefront normalises out of its registers
struct StepArgs {
  const void *x, *residual, *gamma, *beta, *w, *bias, *add;
  void *h, *y;
  int *clear, *guard;      // set to 0 here for a later launch; raised where an element is not finite (fp16)
  int M, N, K, act, cols;
  float eps;
};
constexpr int step_row_bytes(int k) { return k * 2 + 16; }   // of a normalised row in LDS: 16 rows' chunks lie in different banks

// Every k of a wavefront in flight at once: 128 behind a normalisation (in <= 1024), 256 in front of an addition (inner <= 2048).
template <int POST> constexpr int step_chunk() { return POST == STEP_POST_ADD ? 256 : SK_CHUNK; }

template <typename T, int PRE, int POST>
__global__ __launch_bounds__(SK_THREADS) void step_linear_kernel(const StepArgs g) {
  extern __shared__ __align__(16) uint8_t step_lds[];
  float (*part)[16][64] = reinterpret_cast<float (*)[16][64]>(step_lds);                  // [SK_WAVES], as in gemm_skinny_kernel
  uint8_t* const rows_lds = step_lds + SK_WAVES * 16 * 64 * 4;                           // PRE: the normalised rows
  const int tid = threadIdx.x, lane = tid & 63, half = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n0 = static_cast<int>(blockIdx.x) * g.cols, m0 = static_cast<int>(blockIdx.y) * SK_ROWS;
  const int steps = (g.K + 15) / 16, per = (steps + SK_WAVES - 1) / SK_WAVES;
  const int k_begin = wave * per * 16, k_end = min(g.K, (wave + 1) * per * 16);
  const int m = m0 + (lane & 31), n = n0 + (lane & 31);
  const T* wrow = static_cast<const T*>(g.w) + static_cast<int64_t>(n) * g.K + 8 * half;
  const int nrows = min(g.M - m0, SK_ROWS);
  if (PRE != STEP_PRE_NONE && g.clear != nullptr && blockIdx.x == 0 && blockIdx.y == 0 && tid == 0) *g.clear = 0;
  constexpr int CHUNK = step_chunk<POST>();
  uint4 wf[CHUNK / 16];
  auto load_w = [&](int k0) {
#pragma unroll
    for (int s = 0; s < CHUNK / 16; ++s) {
      const int k = k0 + 16 * s + 8 * half;
      wf[s] = k < k_end && (lane & 31) < g.cols && n < g.N ? *reinterpret_cast<const uint4*>(wrow + k0 + 16 * s) : make_uint4(0, 0, 0, 0);
    }
  };
  load_w(k_begin);         // ahead of the normalisation: this is the memory latency that the block waits for

  if constexpr (PRE != STEP_PRE_NONE) {
    // wavefront w: rows w, w + 8, ...; a lane's 8 columns at 8 lane and 512 + 8 lane, as nmtg_ln_fwd deals them out
    const float rn = 1.f / static_cast<float>(g.K);
    const T *x = static_cast<const T*>(g.x), *res = static_cast<const T*>(g.residual);
    const int col[2] = {8 * lane, 512 + 8 * lane};
    pack<T, 8> gr[2], br[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int cc = col[i] < g.K ? col[i] : 0;
      gr[i] = load_raw<T, 8>(static_cast<const T*>(g.gamma) + cc);
      br[i] = load_raw<T, 8>(static_cast<const T*>(g.beta) + cc);
    }
    for (int r = wave; r < nrows; r += SK_WAVES) {
      const int64_t row = static_cast<int64_t>(m0 + r) * g.K;
      float xf[2][8];
      float sum = 0.f;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
#pragma unroll
        for (int j = 0; j < 8; ++j) xf[i][j] = 0.f;
        if (col[i] < g.K) {
          load_pack<T, 8>(x + row + col[i], xf[i]);
          if constexpr (PRE == STEP_PRE_ADD_NORM) {
            float rf[8];
            load_pack<T, 8>(res + row + col[i], rf);
            pack<T, 8> out;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
              out.v[j] = elem<T>::from_float(xf[i][j] + rf[j]);
              xf[i][j] = elem<T>::to_float(out.v[j]);
            }
            if (blockIdx.x == 0) *reinterpret_cast<pack<T, 8>*>(static_cast<T*>(g.h) + row + col[i]) = out;
          }
#pragma unroll
          for (int j = 0; j < 8; ++j) sum += xf[i][j];
        }
      }
      const float mean = wave_sum(sum) * rn;
      float m2 = 0.f;
#pragma unroll
      for (int i = 0; i < 2; ++i)
        if (col[i] < g.K) {
#pragma unroll
          for (int j = 0; j < 8; ++j) { const float d = xf[i][j] - mean; m2 += d * d; }
        }
      const float rs = rsqrtf(wave_sum(m2) * rn + g.eps);
#pragma unroll
      for (int i = 0; i < 2; ++i)
        if (col[i] < g.K) {
          float gf[8], bf[8], zf[8];
          unpack_raw<T, 8>(gr[i], gf);
          unpack_raw<T, 8>(br[i], bf);
#pragma unroll
          for (int j = 0; j < 8; ++j) zf[j] = as_fp32(gf[j] * (rs * (xf[i][j] - mean)) + bf[j]);
          store_pack<T, 8>(reinterpret_cast<T*>(rows_lds + r * step_row_bytes(g.K)) + col[i], zf);
        }
    }
    __syncthreads();
  }

  const T* xrow = PRE == STEP_PRE_NONE ? static_cast<const T*>(g.x) + static_cast<int64_t>(m) * g.K + 8 * half
                                       : reinterpret_cast<const T*>(rows_lds + min(lane & 31, nrows - 1) * step_row_bytes(g.K)) + 8 * half;
  acc16_t acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.f;
  for (int k0 = k_begin; k0 < k_end; k0 += CHUNK) {
    uint4 xf[CHUNK / 16];
    if (k0 != k_begin) load_w(k0);
#pragma unroll
    for (int s = 0; s < CHUNK / 16; ++s) {
      const int k = k0 + 16 * s + 8 * half;
      xf[s] = k < k_end && m < g.M ? *reinterpret_cast<const uint4*>(xrow + k0 + 16 * s) : make_uint4(0, 0, 0, 0);
    }
#pragma unroll
    for (int s = 0; s < CHUNK / 16; ++s) mfma<T>::run(xf[s], wf[s], acc);
  }
#pragma unroll
  for (int r = 0; r < 16; ++r) part[wave][r][lane] = acc[r];
  __syncthreads();
  auto outputs = [&](auto act_tag) {
    constexpr int ACT = decltype(act_tag)::value;
    for (int o = tid; o < 16 * 64; o += SK_THREADS) {
      const int r = o >> 6, l = o & 63;
      float v = 0.f;
#pragma unroll
      for (int w = 0; w < SK_WAVES; ++w) v += part[w][r][l];
      const int row = m0 + 8 * (r / 4) + 4 * (l >> 5) + r % 4, c = n0 + (l & 31);
      if (row < g.M && (l & 31) < g.cols && c < g.N) {
        if (g.bias != nullptr) v += elem<T>::to_float(static_cast<const T*>(g.bias)[c]);
        const int64_t at = static_cast<int64_t>(row) * g.N + c;
        T out = elem<T>::from_float(v);
        if constexpr (POST == STEP_POST_ADD) {
          out = elem<T>::from_float(as_fp32(elem<T>::to_float(static_cast<const T*>(g.add)[at]) + elem<T>::to_float(out)));
          if (guard_element(out) && g.guard != nullptr) *g.guard = 1;
        } else if constexpr (ACT != NMTG_ACT_NONE) {
          out = elem<T>::from_float(act_apply<ACT>(elem<T>::to_float(out), nullptr));
        }
        static_cast<T*>(g.y)[at] = out;
      }
    }
  };
  if constexpr (POST == STEP_POST_ACT) dispatch_act<false>(g.act, 0, outputs);
  else outputs(std::integral_constant<int, NMTG_ACT_NONE>{});
}

template <typename T, int PRE, int POST>
int step_launch(const StepArgs& g, hipStream_t st) {
  const int lds = SK_WAVES * 16 * 64 * 4 + (PRE != STEP_PRE_NONE ? std::min(g.M, SK_ROWS) * step_row_bytes(g.K) : 0);
  auto kern = step_linear_kernel<T, PRE, POST>;
  if (lds > 64 * 1024) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) return fail(NMTG_ERR_LAUNCH, "step_linear: cannot reserve %d bytes of LDS: %s", lds, hipGetErrorString(e));
  }
  const dim3 grid(static_cast<unsigned>((g.N + g.cols - 1) / g.cols), static_cast<unsigned>((g.M + SK_ROWS - 1) / SK_ROWS));
  TraceScope trace("step_linear", st);
  hipLaunchKernelGGL(kern, grid, dim3(SK_THREADS), lds, st, g);
  // fp16: the clamp of a spoilt stream takes every element, and so a launch of its own, as in dropout_add.hip. (By the block that
  // finishes last, with a fence, every step waited for the L2's write-back: the launch took 2 us longer than this one takes.)
  if constexpr (POST == STEP_POST_ADD && std::is_same<T, f16_t>::value) guard_clamp_f16(g.y, nullptr, static_cast<int64_t>(g.M) * g.N, g.guard, st);
  return 0;
}

}  // namespace

// Eligibility: row-major X and W (the NT layout), plain epilogue, one batch, 16-byte aligned rows. NMTG_GEMM_SKINNY=0
// sends these calls to the tiled kernels instead.
bool gemm_skinny_ok(int dtype, int layout, int epi, const GemmArgs& a) {
  if (switched_off("NMTG_GEMM_SKINNY")) return false;
  return (dtype == NMTG_F16 || dtype == NMTG_BF16) && layout == LAYOUT_NT && epi == EPI_PLAIN && a.batch == 1 && a.M >= 1 &&
         a.M <= (a.skinny_rows != 0 ? std::min<int>(a.skinny_rows, SK_MAX_ROWS) : SK_ROWS) && a.N >= 64 && a.K >= 8 && a.K % 8 == 0 && a.lda % 8 == 0 && a.ldb % 8 == 0 && aligned16(a.A) &&
         aligned16(a.B);
}

int gemm_skinny_run(int dtype, const GemmArgs& a, hipStream_t st) {
  const int cols = sk_cols(a.M, a.N, a.K);
  const dim3 grid(static_cast<unsigned>((a.N + cols - 1) / cols), static_cast<unsigned>((a.M + SK_ROWS - 1) / SK_ROWS));
  TraceScope trace("gemm_nt_skinny", st);
  if (dtype == NMTG_F16) hipLaunchKernelGGL((gemm_skinny_kernel<f16_t>), grid, dim3(SK_THREADS), 0, st, a, cols);
  else hipLaunchKernelGGL((gemm_skinny_kernel<bf16_t>), grid, dim3(SK_THREADS), 0, st, a, cols);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(NMTG_ERR_LAUNCH, "gemm: launch failed: %s", hipGetErrorString(e));
  return 0;
}

}  // namespace nmtg

using namespace nmtg;

extern "C" int nmtg_linear_step(int64_t rows, int64_t out, int64_t in, const void* x, const void* w, const void* bias, void* y, int dtype,
                                void* stream) {
  NMTG_REQUIRE(rows >= 0 && out >= 0 && in >= 0 && rows <= INT32_MAX && out <= INT32_MAX && in <= INT32_MAX, "linear_step: bad shape");
  GemmArgs g{};
  g.A = x; g.B = w; g.C = y; g.bias = bias;
  g.lda = in; g.ldb = in; g.ldc = out;
  g.M = static_cast<int>(rows); g.N = static_cast<int>(out); g.K = static_cast<int>(in);
  g.batch = 1;
  g.alpha = 1.f;
  g.skinny_rows = SK_MAX_ROWS;
  return gemm_run(dtype, LAYOUT_NT, EPI_PLAIN, g, nullptr, 0, static_cast<hipStream_t>(stream));
}

extern "C" int nmtg_step_linear_ok(int64_t rows, int64_t model, int64_t inner) {
  return rows >= 1 && rows <= SK_MAX_ROWS && model >= 64 && model <= STEP_MAX_NORM && model % 8 == 0 && inner >= 64 && inner % 8 == 0 &&
                 inner <= INT32_MAX && !switched_off("NMTG_GEMM_SKINNY")
             ? 1 : 0;
}

extern "C" int nmtg_step_linear(int64_t rows, int64_t out, int64_t in, const void* x, const void* residual, const void* gamma,
                                const void* beta, float eps, void* h, int* clear, const void* w, const void* bias, int act,
                                const void* add, int* guard, void* y, int dtype, void* stream) {
  NMTG_REQUIRE(dtype == NMTG_F16 || dtype == NMTG_BF16, "step_linear: fp16 or bf16 tensors required");
  NMTG_REQUIRE(rows >= 0 && rows <= SK_MAX_ROWS && out >= 1 && out <= INT32_MAX && in >= 8 && in % 8 == 0 && in <= INT32_MAX,
               "step_linear: bad shape rows=%lld out=%lld in=%lld", (long long)rows, (long long)out, (long long)in);
  NMTG_REQUIRE(act >= NMTG_ACT_NONE && act <= NMTG_ACT_AGELU, "step_linear: activation %d", act);
  if (rows == 0) return 0;
  NMTG_REQUIRE(x && w && y && aligned16(x) && aligned16(w), "step_linear: 16-byte aligned x and w required");
  NMTG_REQUIRE(gamma == nullptr ? residual == nullptr : (beta && in <= STEP_MAX_NORM && aligned16(gamma) && aligned16(beta)),
               "step_linear: the normalisation takes up to %d columns and 16-byte aligned parameters", STEP_MAX_NORM);
  NMTG_REQUIRE(residual == nullptr || (h && aligned16(residual) && aligned16(h)), "step_linear: 16-byte aligned residual and h required");
  NMTG_REQUIRE(add == nullptr || (gamma == nullptr && act == NMTG_ACT_NONE && (guard || dtype != NMTG_F16)),
               "step_linear: the addition follows a plain product, and in fp16 needs its guard");
  // Blocks write their columns of y, and those of the first columns h, while others still read the rows: in place only y = add,
  // whose elements are read and written by one thread.
  struct Span { const void* at; int64_t bytes; };
  const Span outs[2] = {{y, rows * out * 2}, {residual != nullptr ? h : nullptr, rows * in * 2}};
  const Span ins[7] = {{x, rows * in * 2}, {residual, rows * in * 2}, {w, out * in * 2}, {bias, out * 2}, {gamma, in * 2}, {gamma != nullptr ? beta : nullptr, in * 2},
                       {add != y ? add : nullptr, rows * out * 2}};
  auto meet = [](const Span& a, const Span& b) {
    const uintptr_t p = reinterpret_cast<uintptr_t>(a.at), q = reinterpret_cast<uintptr_t>(b.at);
    return p != 0 && q != 0 && p < q + static_cast<uintptr_t>(b.bytes) && q < p + static_cast<uintptr_t>(a.bytes);
  };
  for (const Span& o : outs)
    for (const Span& i : ins) NMTG_REQUIRE(!meet(o, i), "step_linear: y and h may not overlap what is read (y = add excepted)");
  NMTG_REQUIRE(!meet(outs[0], outs[1]), "step_linear: y and h may not overlap");
  StepArgs g{x, residual, gamma, beta, w, bias, add, h, y, clear, guard, static_cast<int>(rows), static_cast<int>(out), static_cast<int>(in), act,
             sk_cols(static_cast<int>(rows), static_cast<int>(out), static_cast<int>(in)), eps};
  hipStream_t st = static_cast<hipStream_t>(stream);
  auto run = [&](auto t) {
    using T = decltype(t);
    if (add != nullptr) return step_launch<T, STEP_PRE_NONE, STEP_POST_ADD>(g, st);
    if (gamma == nullptr) return step_launch<T, STEP_PRE_NONE, STEP_POST_ACT>(g, st);
    return residual == nullptr ? step_launch<T, STEP_PRE_NORM, STEP_POST_ACT>(g, st) : step_launch<T, STEP_PRE_ADD_NORM, STEP_POST_ACT>(g, st);
  };
  if (int rc = dtype == NMTG_F16 ? run(f16_t{}) : run(bf16_t{})) return rc;
  NMTG_CHECK_LAUNCH("step_linear");
  return 0;
}
