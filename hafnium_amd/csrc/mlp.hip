// Inference and training kernels of the learned SCF guess (a small MLP on
// gfx950): a BF16 MFMA GEMM with FP32 accumulation and a fused bias / SiLU
// epilogue, the SiLU backward, column sums (bias gradients), a weighted
// squared-error loss with its gradient, and the Adam update that keeps FP32
// master weights beside their BF16 copy.
//
// Arithmetic contract (mirrored by the CPU restatement the tests check it
// against): every GEMM operand is rounded to bf16 (round to nearest even)
// when it is loaded, products are accumulated in FP32, and everything
// outside the GEMMs runs in FP32.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <string>

#include "hfjk_internal.h"

namespace {

typedef float f4 __attribute__((ext_vector_type(4)));
typedef uint32_t u4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));

constexpr int kT = 256;
constexpr int kTileM = 32;
constexpr int kTileN = 32;
constexpr int kWaves = 8;  // per tile
constexpr int kGemmT = 64 * kWaves;

__device__ __forceinline__ uint16_t to_bf16(float x) {
  uint32_t u = __float_as_uint(x);
  if ((u & 0x7F800000u) == 0x7F800000u) return (uint16_t)((u >> 16) | ((u & 0xFFFFu) ? 0x40u : 0u));
  u += 0x7FFFu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}

__device__ __forceinline__ float silu(float z) { return z / (1.0f + expf(-z)); }

__device__ __forceinline__ float silu_slope(float z) {  // s (1 + z (1 - s)), s = 1 / (1 + e^-z)
  const float s = 1.0f / (1.0f + expf(-z));
  return s * (1.0f + z * (1.0f - s));
}

struct GemmArgs {
  int m, n, k;
  const void* a;
  int lda, ta;
  const int* a_rows;
  const void* b;
  int ldb, tb;
  const float* bias;
  float* c;
  int ldc;
  int accumulate;
  float* h;            // silu(C)
  const float* slope;  // C *= silu'(slope[i][j]), leading dimension ldc
  // The weighted squared error of C: grad, and the workgroup's part of the loss.
  const float* tgt;
  int ldt;
  const int* t_rows;
  const float* w;
  float scale;
  float* grad;
  float* loss_part;
};

// Eight consecutive k of one row (or column) of an operand as a lane holds
// them: element (i, k + e), k + e < kmax, i < imax, zero elsewhere. Stored row
// i (rows[i] when given) along k, or with trans k along i. load8 only loads
// (bf16 in pairs where `vec` and the row's end let it); operand8 rounds and
// masks once the values are needed.
template <typename T>
struct Raw8 {
  T x[8];
  u4 pair;  // bf16: elements 2 w and 2 w + 1 in word w, when `pairs`
  bool pairs;
};

template <typename T>
__device__ __forceinline__ void load8(const T* __restrict__ p, int ld, int trans, const int* __restrict__ rows, int i,
                                      int imax, int k, int kmax, bool vec, Raw8<T>& r) {
  // Rows and columns past the operand read its last ones and count as zero,
  // so that every load is unconditional. kmax, imax >= 1 here.
  const int ic = min(i, imax - 1);
  const T* src = trans ? p + ic : p + (long long)(rows ? rows[ic] : ic) * ld;
  r.pairs = !trans && vec && k + 8 <= kmax;
  if (r.pairs) {
    if constexpr (sizeof(T) == 2) {
      r.pair = *(const u4*)(src + k);
    } else {
      const f4 u = ((const f4*)(src + k))[0], v = ((const f4*)(src + k))[1];
#pragma unroll
      for (int e = 0; e < 4; ++e) r.x[e] = u[e], r.x[4 + e] = v[e];
    }
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int kc = min(k + e, kmax - 1);
      r.x[e] = trans ? src[(long long)(rows ? rows[kc] : kc) * ld] : src[kc];
    }
  }
}

template <typename T>
__device__ __forceinline__ bf8 operand8(const Raw8<T>& r, int i, int imax, int k, int kmax) {
  union {
    uint16_t u[8];
    bf8 b;
  } o;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    uint16_t v;
    if constexpr (sizeof(T) == 2)
      v = r.pairs ? (uint16_t)(r.pair[e >> 1] >> (e & 1) * 16) : r.x[e];
    else
      v = to_bf16(r.x[e]);
    o.u[e] = i < imax && k + e < kmax ? v : (uint16_t)0;
  }
  return o.b;
}

// The operands of a k step of a tile as the MFMA reads them (16 rows of A, 16
// more, 16 columns of B, 16 more), a step per wave, two rounds of them.
struct GemmSmem {
  bf8 step[2][kWaves][4][64];
  float losses[4];
};

// C[m][n] = op(A) op(B) (+ C) (+ bias) and the epilogues of GemmArgs.
// op(A) is m x k: A is stored m x k (ta = 0) or k x m (ta = 1), row-major
// with leading dimension lda; storage row r of A is read from row a_rows[r]
// when a_rows is given (a gather of minibatch rows). op(B) is k x n: B is
// stored k x n (tb = 0) or n x k (tb = 1).
// One 512-thread workgroup per 32 x 32 tile of C as 2 x 2
// v_mfma_f32_16x16x32_bf16 tiles (A[i][8 (l / 16) + e] in element e of lane
// l, i = l % 16; B likewise with j = l % 16; D register r of lane l =
// D[4 (l / 16) + r][l % 16]). The waves fetch every eighth 32-k step each,
// straight from global memory, and leave its operands in LDS; wave w < 4 then
// runs the chain of products of block (w / 2, w % 2), one step after another,
// while the next eight steps are on their way: an element's sum runs along k
// in order, whatever the tile or the number of waves.
//
// Bound by latency at the training sizes (256 x 256 x 288): 64 workgroups of
// one or two steps per wave, 8 to 9 us, where 64 x 64 tiles left 16 workgroups
// walking nine dependent steps of scalar loads and two barriers, 22 us. Larger
// products are bound by the loads of their operands, which the 64 x 64 tiles
// share twice as widely, in a serial order: 2048 x 384 x 384 28 -> 14 us,
// 4096^3 3.4 -> 1.7 ms, 288 x 256 x 65536 4.8 -> 0.70 ms; only gradients of
// very wide layers with few rows lose (65536 x 256 x 288, A transposed: 263 ->
// 302 us, nine steps in two rounds of eight).
template <typename TA, typename TB>
__device__ void gemm_tile(const GemmArgs& g, int tile_row, int tile_col, GemmSmem& sm) {
  const TA* a = (const TA*)g.a;
  const TB* b = (const TB*)g.b;
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int row0 = tile_row * kTileM, col0 = tile_col * kTileN;
  const bool avec = (((uintptr_t)a | (uintptr_t)g.lda * sizeof(TA)) & 15) == 0;
  const bool bvec = (((uintptr_t)b | (uintptr_t)g.ldb * sizeof(TB)) & 15) == 0;
  const int mi = wave >> 1 & 1, ni = wave & 1;
  const int steps = (g.k + 31) / 32;
  Raw8<TA> ra[2];
  Raw8<TB> rb[2];
  auto fetch = [&](int step) {
    const int k = 32 * step + 8 * (lane >> 4);
#pragma unroll
    for (int f = 0; f < 2; ++f) {
      load8(a, g.lda, g.ta, g.a_rows, row0 + f * 16 + (lane & 15), g.m, k, g.k, avec, ra[f]);
      load8(b, g.ldb, !g.tb, nullptr, col0 + f * 16 + (lane & 15), g.n, k, g.k, bvec, rb[f]);
    }
  };
  f4 acc = f4{0.f, 0.f, 0.f, 0.f};
  if (wave < steps) fetch(wave);
  for (int s0 = 0, round = 0; s0 < steps; s0 += kWaves, round ^= 1) {
    if (s0 + wave < steps) {
      const int k = 32 * (s0 + wave) + 8 * (lane >> 4);
#pragma unroll
      for (int f = 0; f < 2; ++f) {
        sm.step[round][wave][f][lane] = operand8(ra[f], row0 + f * 16 + (lane & 15), g.m, k, g.k);
        sm.step[round][wave][2 + f][lane] = operand8(rb[f], col0 + f * 16 + (lane & 15), g.n, k, g.k);
      }
    }
    // This round's operands are in LDS, and the round before is read: the next one may replace it.
    __syncthreads();
    if (s0 + kWaves + wave < steps) fetch(s0 + kWaves + wave);
    if (wave < 4) {
      auto product = [&](int s) {
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(sm.step[round][s][mi][lane], sm.step[round][s][2 + ni][lane], acc,
                                                      0, 0, 0);
      };
      if (steps - s0 >= kWaves) {
#pragma unroll
        for (int s = 0; s < kWaves; ++s) product(s);
      } else {
        for (int s = 0; s < steps - s0; ++s) product(s);
      }
    }
  }
  float loss = 0.f;
  if (wave < 4) {
    const int j = col0 + ni * 16 + (lane & 15);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = row0 + mi * 16 + 4 * (lane >> 4) + r;
      if (i >= g.m || j >= g.n) continue;
      float v = acc[r];
      const long long at = (long long)i * g.ldc + j;
      if (g.accumulate) v += g.c[at];
      if (g.bias) v += g.bias[j];
      if (g.slope) v *= silu_slope(g.slope[at]);
      g.c[at] = v;
      if (g.h) g.h[at] = silu(v);
      if (g.tgt) {
        const long long tr = g.t_rows ? g.t_rows[i] : i;
        const float d = v - g.tgt[tr * g.ldt + j];
        const float wj = g.w ? g.w[j] : 1.0f;
        loss += wj * d * d;
        g.grad[at] = 2.0f * g.scale * wj * d;
      }
    }
  }
  if (g.tgt) {
    for (int off = 32; off > 0; off >>= 1) loss += __shfl_xor(loss, off);
    if (lane == 0 && wave < 4) sm.losses[wave] = loss;
    __syncthreads();
    if (threadIdx.x == 0)
      g.loss_part[tile_row * ((g.n + kTileN - 1) / kTileN) + tile_col] =
          (sm.losses[0] + sm.losses[1]) + (sm.losses[2] + sm.losses[3]);
  }
}

// Tiles from `first` on.
template <typename TA, typename TB>
__global__ __launch_bounds__(kGemmT) void mlp_gemm_kernel(GemmArgs g, int first) {
  __shared__ GemmSmem sm;
  const int cols = (g.n + kTileN - 1) / kTileN, t = first + blockIdx.x;
  gemm_tile<TA, TB>(g, t / cols, t % cols, sm);
}

// out[j] = sum_i x[i][j] of 64 columns by 256 threads: 4 row phases, fixed order.
__device__ __forceinline__ void column_sums(int m, int n, const float* __restrict__ x, int ldx,
                                            float* __restrict__ out, int block, float (*part)[64]) {
  const int c = threadIdx.x & 63;
  const int phase = threadIdx.x >> 6;
  const int j = block * 64 + c;
  float s = 0.f;
  if (j < n && phase < 4) {
#pragma unroll 16
    for (int i = phase; i < m; i += 4) s += x[(long long)i * ldx + j];
  }
  if (phase < 4) part[phase][c] = s;
  __syncthreads();
  if (phase == 0 && j < n) out[j] = (part[0][c] + part[1][c]) + (part[2][c] + part[3][c]);
}

// One layer of the backward pass: the bias gradients (the first `sums`
// workgroups), the weight gradients (tiles below split) and the gradient of
// the layer's input, all of the same dz: 7 us in one launch, where the two
// products, the column sum and the SiLU backward took 22 + 22 + 7 + 3 us in
// four. Every sum has the order of the separate calls'.
__global__ __launch_bounds__(kGemmT) void mlp_backward_kernel(GemmArgs weights, GemmArgs input, int sums, int split,
                                                              float* __restrict__ bias, int first) {
  __shared__ GemmSmem sm;
  int t = first + blockIdx.x;
  if (t < sums) {
    column_sums(weights.k, weights.n, (const float*)weights.b, weights.ldb, bias, t, (float(*)[64]) & sm);
    return;
  }
  t -= sums;
  if (t < split) {
    const int cols = (weights.n + kTileN - 1) / kTileN;
    gemm_tile<float, float>(weights, t / cols, t % cols, sm);
  } else {
    t -= split;
    const int cols = (input.n + kTileN - 1) / kTileN;
    gemm_tile<float, uint16_t>(input, t / cols, t % cols, sm);
  }
}

// grad_z = grad_h * silu'(z), silu'(z) = s (1 + z (1 - s)), s = 1 / (1 + e^-z).
__global__ __launch_bounds__(kT) void silu_backward_kernel(long long count, const float* __restrict__ grad_h,
                                                           const float* __restrict__ z, float* __restrict__ grad_z) {
  for (long long e = (long long)blockIdx.x * kT + threadIdx.x; e < count; e += (long long)gridDim.x * kT) {
    grad_z[e] = grad_h[e] * silu_slope(z[e]);
  }
}

__global__ __launch_bounds__(kT) void column_sum_kernel(int m, int n, const float* __restrict__ x, int ldx,
                                                        float* __restrict__ out) {
  __shared__ float part[4][64];
  column_sums(m, n, x, ldx, out, blockIdx.x, part);
}

// Weighted squared error over y [m][n]: loss[0] = scale sum_ij w_j (y_ij - t_ij)^2,
// grad[i][j] = 2 scale w_j (y_ij - t_ij); target row i is t_rows[i] when
// given. One workgroup, fixed summation order.
__global__ __launch_bounds__(kT) void mse_kernel(int m, int n, const float* __restrict__ y, int ldy,
                                                 const float* __restrict__ tgt, int ldt, const int* __restrict__ t_rows,
                                                 const float* __restrict__ w, float scale, float* __restrict__ grad,
                                                 float* __restrict__ loss) {
  __shared__ float part[kT];
  float s = 0.f;
  const long long total = (long long)m * n;
  for (long long e = threadIdx.x; e < total; e += kT) {
    const int i = (int)(e / n), j = (int)(e % n);
    const long long tr = t_rows ? t_rows[i] : i;
    const float d = y[(long long)i * ldy + j] - tgt[tr * ldt + j];
    const float wj = w ? w[j] : 1.0f;
    s += wj * d * d;
    if (grad) grad[(long long)i * ldy + j] = 2.0f * scale * wj * d;
  }
  part[threadIdx.x] = s;
  __syncthreads();
  for (int half = kT / 2; half > 0; half >>= 1) {
    if (threadIdx.x < half) part[threadIdx.x] += part[threadIdx.x + half];
    __syncthreads();
  }
  if (threadIdx.x == 0) loss[0] = scale * part[0];
}

// Adam (decoupled weight decay): m, v moments; p -= lr_t m / (sqrt(v) + eps) + lr wd p;
// the bf16 copy of p is refreshed in the same pass.
// The host forms 1 - beta in double (1 - 0.999f in float loses 4 digits).
__global__ __launch_bounds__(kT) void adam_kernel(long long count, float* __restrict__ p, const float* __restrict__ g,
                                                  float* __restrict__ m1, float* __restrict__ m2,
                                                  uint16_t* __restrict__ p16, float lr_t, float beta1,
                                                  float one_minus_beta1, float beta2, float one_minus_beta2,
                                                  float eps, float decay, const float* __restrict__ loss_part,
                                                  int nparts, float scale, float* __restrict__ loss) {
  // The training step's loss, from the parts of the output tiles in a fixed order.
  if (loss_part != nullptr && blockIdx.x == 0 && threadIdx.x < 64) {
    float s = 0.f;
    for (int i = threadIdx.x; i < nparts; i += 64) s += loss_part[i];
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off);
    if (threadIdx.x == 0) loss[0] = scale * s;
  }
  for (long long e = (long long)blockIdx.x * kT + threadIdx.x; e < count; e += (long long)gridDim.x * kT) {
    const float gi = g[e];
    const float a = beta1 * m1[e] + one_minus_beta1 * gi;
    const float b = beta2 * m2[e] + one_minus_beta2 * gi * gi;
    m1[e] = a;
    m2[e] = b;
    float x = p[e];
    x -= lr_t * a / (sqrtf(b) + eps) + decay * x;
    p[e] = x;
    if (p16) p16[e] = to_bf16(x);
  }
}

__global__ __launch_bounds__(kT) void to_bf16_kernel(long long count, const float* __restrict__ src,
                                                     uint16_t* __restrict__ dst) {
  for (long long e = (long long)blockIdx.x * kT + threadIdx.x; e < count; e += (long long)gridDim.x * kT)
    dst[e] = to_bf16(src[e]);
}

struct MlpFailure {
  int code;
  std::string message;
};

[[noreturn]] void mfail(int code, const std::string& m) { throw MlpFailure{code, m}; }

void mcheck(hipError_t e, const char* what) {
  if (e != hipSuccess) mfail(HFJK_ERR_HIP, std::string(what) + ": " + hipGetErrorString(e));
}

template <typename F>
int mguard(hfjk_ctx* ctx, F&& body) {
  try {
    if (ctx == nullptr) mfail(HFJK_ERR_INPUT, "null context");
    mcheck(hipSetDevice(ctx->device), "hipSetDevice");
    body();
    return HFJK_OK;
  } catch (const MlpFailure& f) {
    hfjk_internal_set_error(f.message.c_str());
    return f.code;
  } catch (...) {
    hfjk_internal_set_error("unknown failure in an MLP routine");
    return HFJK_ERR_HIP;
  }
}

constexpr int kMaxRows = 65535 * 64;  // of a product: part of the entry points' contract

// launch(first, count) for all of `tiles` workgroups of kGemmT threads, at
// most 2^31 work-items at a time (a grid holds less than 2^32).
template <typename F>
void in_launches(int tiles, const char* what, F&& launch) {
  constexpr int kMost = (1 << 30) / (kGemmT / 2);
  for (int first = 0; first < tiles;) {
    const int count = std::min(kMost, tiles - first);
    launch(first, dim3((unsigned)count));
    mcheck(hipGetLastError(), what);
    first += count;
  }
}

// Float offsets of a training step's workspace: every layer's z and dz, the
// hidden layers' h, the loss parts of the output tiles.
constexpr int kMaxLayers = 16;
struct TrainLayout {
  long long z[kMaxLayers], h[kMaxLayers], dz[kMaxLayers], loss, total;
};

TrainLayout train_layout(int layers, const int* sizes, int m) {
  TrainLayout L{};
  long long at = 0;
  auto take = [&](long long n) {
    const long long here = at;
    at += (n + 63) / 64 * 64;
    return here;
  };
  for (int l = 0; l < layers && l < kMaxLayers; ++l) {
    const long long n = (long long)m * sizes[l + 1];
    L.z[l] = take(n);
    if (l + 1 < layers) L.h[l] = take(n);
  }
  for (int l = 0; l < layers && l < kMaxLayers; ++l) L.dz[l] = take((long long)m * sizes[l + 1]);
  L.loss = take((long long)((m + kTileM - 1) / kTileM) * ((sizes[layers] + kTileN - 1) / kTileN));
  L.total = at;
  return L;
}

}  // namespace

extern "C" {

int hfjk_mlp_gemm(hfjk_ctx* ctx, int m, int n, int k, const void* a, int a_bf16, int lda, int trans_a,
                  const int* a_rows, const void* b, int b_bf16, int ldb, int trans_b, const float* bias, float* c,
                  int ldc, int accumulate, float* h_silu, void* stream) {
  return mguard(ctx, [&] {
    if (m < 0 || n < 0 || k < 0) mfail(HFJK_ERR_INPUT, "hfjk_mlp_gemm: negative size");
    if (m == 0 || n == 0) return;
    if (a == nullptr || b == nullptr || c == nullptr) mfail(HFJK_ERR_INPUT, "hfjk_mlp_gemm: null operand");
    // Leading dimensions cover the stored rows (gathered row indices are the caller's contract).
    if (lda < (trans_a ? m : k) || ldb < (trans_b ? k : n) || ldc < n)
      mfail(HFJK_ERR_INPUT, "hfjk_mlp_gemm: a leading dimension is smaller than its row");
    if (h_silu == c) mfail(HFJK_ERR_INPUT, "hfjk_mlp_gemm: the activation output must not alias C");
    if (m > kMaxRows) mfail(HFJK_ERR_INPUT, "hfjk_mlp_gemm: more than 4194240 rows");
    GemmArgs g{};
    g.m = m;
    g.n = n;
    g.k = k;
    g.a = a;
    g.lda = lda;
    g.ta = trans_a ? 1 : 0;
    g.a_rows = a_rows;
    g.b = b;
    g.ldb = ldb;
    g.tb = trans_b ? 1 : 0;
    g.bias = bias;
    g.c = c;
    g.ldc = ldc;
    g.accumulate = accumulate ? 1 : 0;
    g.h = h_silu;
    const long long cols = (n + kTileN - 1) / kTileN, rows = (m + kTileM - 1) / kTileM;
    if (cols * rows > 0x7FFFFFFFLL) mfail(HFJK_ERR_INPUT, "hfjk_mlp_gemm: too many output tiles");
    hipStream_t s = (hipStream_t)stream;
    in_launches((int)(cols * rows), "mlp_gemm launch", [&](int first, dim3 grid) {
      if (a_bf16 && b_bf16)
        hipLaunchKernelGGL((mlp_gemm_kernel<uint16_t, uint16_t>), grid, dim3(kGemmT), 0, s, g, first);
      else if (a_bf16)
        hipLaunchKernelGGL((mlp_gemm_kernel<uint16_t, float>), grid, dim3(kGemmT), 0, s, g, first);
      else if (b_bf16)
        hipLaunchKernelGGL((mlp_gemm_kernel<float, uint16_t>), grid, dim3(kGemmT), 0, s, g, first);
      else
        hipLaunchKernelGGL((mlp_gemm_kernel<float, float>), grid, dim3(kGemmT), 0, s, g, first);
    });
  });
}

int hfjk_mlp_silu_backward(hfjk_ctx* ctx, long long count, const float* grad_h, const float* z, float* grad_z,
                           void* stream) {
  return mguard(ctx, [&] {
    if (count < 0 || (count > 0 && (grad_h == nullptr || z == nullptr || grad_z == nullptr)))
      mfail(HFJK_ERR_INPUT, "hfjk_mlp_silu_backward: null buffer");
    if (count == 0) return;
    hipLaunchKernelGGL(silu_backward_kernel, dim3(hfjk::grid_for(count)), dim3(kT), 0, (hipStream_t)stream, count,
                       grad_h, z, grad_z);
    mcheck(hipGetLastError(), "silu_backward launch");
  });
}

int hfjk_mlp_column_sum(hfjk_ctx* ctx, int m, int n, const float* x, int ldx, float* out, void* stream) {
  return mguard(ctx, [&] {
    if (m < 0 || n < 0 || ldx < n) mfail(HFJK_ERR_INPUT, "hfjk_mlp_column_sum: bad shape");
    if (n == 0) return;
    if (out == nullptr || (m > 0 && x == nullptr)) mfail(HFJK_ERR_INPUT, "hfjk_mlp_column_sum: null buffer");
    hipLaunchKernelGGL(column_sum_kernel, dim3((n + 63) / 64), dim3(kT), 0, (hipStream_t)stream, m, n, x, ldx, out);
    mcheck(hipGetLastError(), "column_sum launch");
  });
}

int hfjk_mlp_mse(hfjk_ctx* ctx, int m, int n, const float* y, int ldy, const float* target, int ldt,
                 const int* target_rows, const float* col_weights, float scale, float* grad, float* loss,
                 void* stream) {
  return mguard(ctx, [&] {
    if (m < 0 || n < 1 || ldy < n || ldt < n) mfail(HFJK_ERR_INPUT, "hfjk_mlp_mse: bad shape");
    if (loss == nullptr || (m > 0 && (y == nullptr || target == nullptr)))
      mfail(HFJK_ERR_INPUT, "hfjk_mlp_mse: null buffer");
    hipLaunchKernelGGL(mse_kernel, dim3(1), dim3(kT), 0, (hipStream_t)stream, m, n, y, ldy, target, ldt, target_rows,
                       col_weights, scale, grad, loss);
    mcheck(hipGetLastError(), "mse launch");
  });
}

int hfjk_mlp_adam(hfjk_ctx* ctx, long long count, float* params, const float* grads, float* moment1, float* moment2,
                  uint16_t* params_bf16, double lr, double lr_t, double beta1, double beta2, double eps,
                  double weight_decay, void* stream) {
  return mguard(ctx, [&] {
    if (count < 0 || (count > 0 && (params == nullptr || grads == nullptr || moment1 == nullptr ||
                                    moment2 == nullptr)))
      mfail(HFJK_ERR_INPUT, "hfjk_mlp_adam: null buffer");
    if (!(beta1 >= 0.0 && beta1 < 1.0 && beta2 >= 0.0 && beta2 < 1.0 && eps >= 0.0))
      mfail(HFJK_ERR_INPUT, "hfjk_mlp_adam: betas in [0, 1) and eps >= 0 are required");
    if (count == 0) return;
    hipLaunchKernelGGL(adam_kernel, dim3(hfjk::grid_for(count)), dim3(kT), 0, (hipStream_t)stream, count, params,
                       grads, moment1, moment2, params_bf16, (float)lr_t, (float)beta1, (float)(1.0 - beta1),
                       (float)beta2, (float)(1.0 - beta2), (float)eps, (float)(lr * weight_decay),
                       (const float*)nullptr, 0, 0.0f, (float*)nullptr);
    mcheck(hipGetLastError(), "adam launch");
  });
}

long long hfjk_mlp_train_workspace(int layers, const int* sizes, int m) {
  if (layers < 1 || layers > kMaxLayers || sizes == nullptr || m < 0) return 0;
  return train_layout(layers, sizes, m).total;
}

int hfjk_mlp_train_step(hfjk_ctx* ctx, int layers, const int* sizes, int m, const float* x, const int* rows,
                        const float* target, int ldt, const float* col_weights, double scale, float* params,
                        uint16_t* params_bf16, float* grads, float* moment1, float* moment2, double lr, double lr_t,
                        double beta1, double beta2, double eps, double weight_decay, float* workspace, float* loss,
                        void* stream) {
  return mguard(ctx, [&] {
    if (layers < 1 || layers > kMaxLayers || sizes == nullptr || m < 1)
      mfail(HFJK_ERR_INPUT, "hfjk_mlp_train_step: 1 to 16 layers and at least one row are required");
    for (int l = 0; l <= layers; ++l)
      if (sizes[l] < 1 || (l < layers && sizes[l] > kMaxRows) || m > kMaxRows)
        mfail(HFJK_ERR_INPUT, "hfjk_mlp_train_step: layer sizes are positive, rows and inputs at most 4194240");
    if (x == nullptr || target == nullptr || params == nullptr || params_bf16 == nullptr || grads == nullptr ||
        moment1 == nullptr || moment2 == nullptr || workspace == nullptr || loss == nullptr || ldt < sizes[layers])
      mfail(HFJK_ERR_INPUT, "hfjk_mlp_train_step: null buffer or a target narrower than the output");
    if (!(beta1 >= 0.0 && beta1 < 1.0 && beta2 >= 0.0 && beta2 < 1.0 && eps >= 0.0))
      mfail(HFJK_ERR_INPUT, "hfjk_mlp_train_step: betas in [0, 1) and eps >= 0 are required");
    hipStream_t s = (hipStream_t)stream;
    const TrainLayout L = train_layout(layers, sizes, m);
    auto tiles = [](int v) { return (v + kTileM - 1) / kTileM; };
    static_assert(kTileM == kTileN, "square tiles");
    for (int l = 0; l <= layers; ++l)
      if ((long long)tiles(m) * tiles(sizes[l]) > (1 << 29) ||
          (long long)tiles(sizes[l]) * tiles(sizes[std::min(l + 1, layers)]) > (1 << 29))
        mfail(HFJK_ERR_INPUT, "hfjk_mlp_train_step: too many output tiles");
    long long at[kMaxLayers + 1] = {0};  // W [k][n], then b [n], of every layer
    for (int l = 0; l < layers; ++l) at[l + 1] = at[l] + (long long)sizes[l] * sizes[l + 1] + sizes[l + 1];
    const int out = layers - 1;
    for (int l = 0; l < layers; ++l) {
      const int k = sizes[l], n = sizes[l + 1];
      GemmArgs g{};
      g.m = m;
      g.n = n;
      g.k = k;
      g.a = l == 0 ? (const void*)x : (const void*)(workspace + L.h[l - 1]);
      g.lda = k;
      g.a_rows = l == 0 ? rows : nullptr;
      g.b = params_bf16 + at[l];
      g.ldb = n;
      g.bias = params + at[l] + (long long)k * n;
      g.c = workspace + L.z[l];
      g.ldc = n;
      if (l < out) {
        g.h = workspace + L.h[l];
      } else {
        g.tgt = target;
        g.ldt = ldt;
        g.t_rows = rows;
        g.w = col_weights;
        g.scale = (float)scale;
        g.grad = workspace + L.dz[l];
        g.loss_part = workspace + L.loss;
      }
      in_launches(tiles(n) * tiles(m), "mlp forward launch", [&](int first, dim3 grid) {
        hipLaunchKernelGGL((mlp_gemm_kernel<float, uint16_t>), grid, dim3(kGemmT), 0, s, g, first);
      });
    }
    for (int l = out; l >= 0; --l) {
      const int k = sizes[l], n = sizes[l + 1];
      GemmArgs w{};
      w.m = k;
      w.n = n;
      w.k = m;
      w.a = l == 0 ? (const void*)x : (const void*)(workspace + L.h[l - 1]);
      w.lda = k;
      w.ta = 1;
      w.a_rows = l == 0 ? rows : nullptr;
      w.b = workspace + L.dz[l];
      w.ldb = n;
      w.c = grads + at[l];
      w.ldc = n;
      const int split = tiles(k) * tiles(n);
      GemmArgs d{};
      if (l > 0) {
        d.m = m;
        d.n = k;
        d.k = n;
        d.a = workspace + L.dz[l];
        d.lda = n;
        d.b = params_bf16 + at[l];
        d.ldb = n;
        d.tb = 1;
        d.c = workspace + L.dz[l - 1];
        d.ldc = k;
        d.slope = workspace + L.z[l - 1];
      }
      const int sums = (n + 63) / 64;
      in_launches(sums + split + (l > 0 ? tiles(m) * tiles(k) : 0), "mlp backward launch", [&](int first, dim3 grid) {
        hipLaunchKernelGGL(mlp_backward_kernel, grid, dim3(kGemmT), 0, s, w, d, sums, split,
                           grads + at[l] + (long long)k * n, first);
      });
    }
    const long long count = at[layers];
    hipLaunchKernelGGL(adam_kernel, dim3(hfjk::grid_for(count)), dim3(kT), 0, s, count, params, grads, moment1,
                       moment2, params_bf16, (float)lr_t, (float)beta1, (float)(1.0 - beta1), (float)beta2,
                       (float)(1.0 - beta2), (float)eps, (float)(lr * weight_decay), workspace + L.loss,
                       tiles(m) * tiles(sizes[layers]), (float)scale, loss);
    mcheck(hipGetLastError(), "adam launch");
  });
}

int hfjk_mlp_to_bf16(hfjk_ctx* ctx, long long count, const float* src, uint16_t* dst, void* stream) {
  return mguard(ctx, [&] {
    if (count < 0 || (count > 0 && (src == nullptr || dst == nullptr)))
      mfail(HFJK_ERR_INPUT, "hfjk_mlp_to_bf16: null buffer");
    if (count == 0) return;
    hipLaunchKernelGGL(to_bf16_kernel, dim3(hfjk::grid_for(count)), dim3(kT), 0, (hipStream_t)stream, count, src,
                       dst);
    mcheck(hipGetLastError(), "to_bf16 launch");
  });
}

}  // extern "C"
