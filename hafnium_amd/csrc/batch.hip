// Batched DF-J/K: many instances of uneven size in one launch per phase
// (charges, Coulomb, orbitals, half-transform, SYRK, reductions).
//
// A plan (hfjk_batch_create) derives every instance's shapes, splits and
// buffer offsets on the host; hfjk_batch_bind uploads it once into the
// caller's workspace; hfjk_batch_run only enqueues kernels (a counter reset
// kernel and one kernel per phase, persistent where the items are uneven), so a run can be captured in a
// hipGraph and replayed.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <string>
#include <vector>

#include "hfjk_internal.h"

struct hfjk_batch {
  hfjk_ctx* ctx = nullptr;
  int precision = HFJK_FP64;
  int tile = 0;  // half-transform column tile
  int ninst = 0;
  std::vector<hfjk::BatchInst> insts;
  std::vector<long long> prefix;  // [kPhCount][ninst + 1]
  long long b_total = 0;          // elements of one plane of the batch tensor
  long long c_total = 0, d_total = 0;
  long long ws64_total = 0;       // fp64 workspace elements
  long long cp_total = 0, x_total = 0, kp_total = 0;  // mode elements (per plane for bf16)
  size_t off_insts = 0, off_prefix = 0, off_counters = 0, off_ws64 = 0, off_cp = 0, off_x = 0, off_kp = 0;
  size_t bytes = 0;
  void* ws = nullptr;
  int grid_mfma = 0;
  // Second stream of builds with densities (bind creates it where the plan uses it): the Coulomb
  // half beside the half-transform.
  bool beside = false;
  hipStream_t side = nullptr;
  hipEvent_t fork = nullptr, join = nullptr;
  ~hfjk_batch() {
    if (fork != nullptr) (void)hipEventDestroy(fork);
    if (join != nullptr) (void)hipEventDestroy(join);
    if (side != nullptr) (void)hipStreamDestroy(side);
  }
};

namespace hfjk {
namespace {

constexpr int kGammaQb = 64;
constexpr long long kMaxGrid = 1 << 20;

// Aux functions of one item of b_charges_x_kernel.
constexpr int charges_per_item(int precision) { return precision == HFJK_BF16X3 ? 8 : 4; }

template <int PREC>
__device__ __forceinline__ void bload4(const void* b, long long plane, long long off, double out[4]) {
  if (PREC == HFJK_FP64) {
    const double2* src = (const double2*)((const double*)b + off);
    const double2 v0 = src[0], v1 = src[1];
    out[0] = v0.x;
    out[1] = v0.y;
    out[2] = v1.x;
    out[3] = v1.y;
  } else if (PREC == HFJK_FP32) {
    const float4 v = *(const float4*)((const float*)b + off);
    out[0] = v.x;
    out[1] = v.y;
    out[2] = v.z;
    out[3] = v.w;
  } else {
    const uint16_t* hi = (const uint16_t*)b + off;
    const ushort4 h = *(const ushort4*)hi;
    const ushort4 l = *(const ushort4*)(hi + plane);
    auto f = [](uint16_t x) { return __uint_as_float(((uint32_t)x) << 16); };
    out[0] = (double)(f(h.x) + f(l.x));
    out[1] = (double)(f(h.y) + f(l.y));
    out[2] = (double)(f(h.z) + f(l.z));
    out[3] = (double)(f(h.w) + f(l.w));
  }
}

__device__ __forceinline__ void rc_of(int tile, int& r, int& c) {
  int rr = (int)((sqrt(8.0 * (double)tile + 1.0) - 1.0) * 0.5);
  while ((rr + 1) * (rr + 2) / 2 <= tile) ++rr;
  while (rr * (rr + 1) / 2 > tile) --rr;
  r = rr;
  c = tile - rr * (rr + 1) / 2;
}

__device__ __forceinline__ uint16_t to_bf16(float x) {
  uint32_t u = __float_as_uint(x);
  if ((u & 0x7F800000u) == 0x7F800000u) return (uint16_t)((u >> 16) | ((u & 0xFFFFu) ? 0x40u : 0u));
  u += 0x7FFFu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}

__global__ __launch_bounds__(kThreads) void reset_kernel(unsigned long long* counters, int n) {
  for (int i = threadIdx.x; i < n; i += kThreads) counters[i] = 0ull;
}

// Phases whose items are uniform: one item per workgroup, dealt by the
// hardware (grids are capped at kMaxGrid and stride). Pulling them from the
// per-XCD counters cost 0.1 ms a phase by itself: every workgroup's last
// visits to the eight counters are serial atomics.
#define BATCH_LOOP(PHASE)                                                                          \
  const long long* pre = v.prefix + (long long)(PHASE) * (v.ninst + 1);                            \
  for (long long item = blockIdx.x; item < v.items[PHASE]; item += gridDim.x) {                    \
    const int inst = batch_find(pre, v.ninst, item);                                               \
    const BatchInst in = v.insts[inst];                                                            \
    const long long local = item - pre[inst];

#define BATCH_END }

// Packed weights of D (D on diagonal tiles, D + D^T elsewhere), one tile per item.
__global__ __launch_bounds__(kThreads) void b_weights_kernel(BatchView v, const double* __restrict__ d,
                                                             double* __restrict__ ws64) {
  BATCH_LOOP(kPhWeights)
  int r, c;
  rc_of((int)local, r, c);
  const double* di = d + in.d_off;
  double* w = ws64 + in.w_off + local * kTileElems;
  for (int v4 = 0; v4 < 4; ++v4) {
    const int e = threadIdx.x * 4 + v4;
    const int row = r * kTile + e / kTile;
    const int col = c * kTile + e % kTile;
    double value = 0.0;
    if (row < in.nao && col < in.nao) {
      value = di[(long long)row * in.nao + col];
      if (r != c) value += di[(long long)col * in.nao + row];
    }
    w[e] = value;
  }
  BATCH_END
}

// Charge partials: gp[tile][q] for a 64-q block, one (tile, q block) per item.
template <int PREC>
__global__ __launch_bounds__(kThreads) void b_gamma_kernel(BatchView v, const void* __restrict__ b, long long plane,
                                                           double* __restrict__ ws64) {
  __shared__ double red[kThreads / 64][kGammaQb];
  BATCH_LOOP(kPhGamma)
  const long long ntiles = in.p / kTileElems;
  const long long tile = local % ntiles;
  const int q0 = (int)(local / ntiles) * kGammaQb;
  const long long e = tile * kTileElems + threadIdx.x * 4;
  const double* w = ws64 + in.w_off + e;
  const double w0 = w[0], w1 = w[1], w2 = w[2], w3 = w[3];
  const int qn = min(kGammaQb, in.naux - q0);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int qi = 0; qi < qn; qi += 8) {
    double s[8];
#pragma unroll
    for (int x = 0; x < 8; ++x) {
      double bv[4];
      bload4<PREC>(b, plane, in.b_off + (long long)(q0 + min(qi + x, qn - 1)) * in.p + e, bv);
      s[x] = bv[0] * w0 + bv[1] * w1 + bv[2] * w2 + bv[3] * w3;
    }
    const double total = wave_sums8(s, lane);
    if ((lane & 7) == 0) red[wave][qi + (lane >> 3)] = total;
  }
  __syncthreads();
  if ((int)threadIdx.x < qn)
    ws64[in.gp_off + tile * in.naux + q0 + threadIdx.x] =
        red[0][threadIdx.x] + red[1][threadIdx.x] + red[2][threadIdx.x] + red[3][threadIdx.x];
  __syncthreads();
  BATCH_END
}

// gamma[q] = sum over tiles, 64 aux functions per item: wave g sums every
// fourth tile.
__global__ __launch_bounds__(kThreads) void b_gamma_reduce_kernel(BatchView v, double* __restrict__ ws64) {
  __shared__ double red[kThreads / 64][64];
  BATCH_LOOP(kPhGammaReduce)
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int q = (int)local * 64 + lane;
  const long long ntiles = in.p / kTileElems;
  const double* gp = ws64 + in.gp_off + min(q, in.naux - 1);
  double s = 0.0;
#pragma unroll 4
  for (long long t = wave; t < ntiles; t += kThreads / 64) s += gp[t * in.naux];
  red[wave][lane] = s;
  __syncthreads();
  if (wave == 0 && q < in.naux) ws64[in.g_off + q] = (red[0][lane] + red[1][lane]) + (red[2][lane] + red[3][lane]);
  __syncthreads();
  BATCH_END
}

// gamma[q] from a caller's flat charge vector (instance i at q_off), 64 per item.
__global__ __launch_bounds__(kThreads) void b_charges_load_kernel(BatchView v, const double* __restrict__ charges,
                                                                  double* __restrict__ ws64) {
  BATCH_LOOP(kPhGammaReduce)
  const int q = (int)local * 64 + threadIdx.x;
  if (threadIdx.x < 64 && q < in.naux) ws64[in.g_off + q] = charges[in.q_off + q];
  BATCH_END
}

// gamma[q] = <B[q], C C^T> = sum_{mu < nao, i < nocc} C[mu][i] X[q][mu][i] from the
// half-transformed X of the exchange (mode layout; BF16X3: hi + lo planes)
// and the caller's FP64 orbitals, charges_per_item aux functions per item.
// The rows [0, nao) of X[q] are one contiguous range of nao * ldo elements,
// streamed in 16-byte groups (ldo is a multiple of 32, so no group straddles
// two rows); columns past nocc are skipped (X is zero there). Bound by the
// pass over X: an item's aux functions share the loads of C, which at one
// aux function per item were 8 bytes from the cache for every 4 (BF16X3) or
// 8 bytes of X (128 BF16x3 instances to 220 functions: 3.31 -> 1.32 ms).
template <int PREC>
__global__ __launch_bounds__(kThreads) void b_charges_x_kernel(BatchView v, const double* __restrict__ c,
                                                               const void* __restrict__ xbase, long long x_plane,
                                                               double* __restrict__ ws64) {
  constexpr int V = PREC == HFJK_FP64 ? 2 : PREC == HFJK_FP32 ? 4 : 8;  // elements per 16-byte group
  constexpr int QB = charges_per_item(PREC);
  __shared__ double red[kThreads / 64][8];
  BATCH_LOOP(kPhCharges)
  const double* ci = c + in.c_off;
  const int q0 = (int)local * QB;
  const long long xstride = (long long)in.xrows * in.ldo;
  double s[8];
#pragma unroll
  for (int x = 0; x < 8; ++x) s[x] = 0.0;
  const int per_row = in.ldo / V;
  const int groups = in.nao * per_row;
  // Group g = mu * per_row + gi, stepped by the block size without a division.
  const int dm = kThreads / per_row, dg = kThreads % per_row;
  int mu = (int)threadIdx.x / per_row, gi = (int)threadIdx.x % per_row;
  for (int g = threadIdx.x; g < groups; g += kThreads) {
    const int i0 = gi * V;
    if (i0 < in.nocc) {
      const long long at = in.x_off + (long long)mu * in.ldo + i0;
      uint4 w[QB], wl[PREC == HFJK_BF16X3 ? QB : 1];
#pragma unroll
      for (int x = 0; x < QB; ++x) {
        const long long here = at + min(q0 + x, in.naux - 1) * xstride;
        if constexpr (PREC == HFJK_FP64) {
          w[x] = *(const uint4*)((const double*)xbase + here);
        } else if constexpr (PREC == HFJK_FP32) {
          w[x] = *(const uint4*)((const float*)xbase + here);
        } else {
          w[x] = *(const uint4*)((const uint16_t*)xbase + here);
          wl[x] = *(const uint4*)((const uint16_t*)xbase + here + x_plane);
        }
      }
      const double* crow = ci + (long long)mu * in.nocc + i0;
      double cv[V];
#pragma unroll
      for (int e = 0; e < V; ++e) cv[e] = crow[min(e, in.nocc - 1 - i0)];
#pragma unroll
      for (int x = 0; x < QB; ++x) {
        const uint32_t hw[4] = {w[x].x, w[x].y, w[x].z, w[x].w};
#pragma unroll
        for (int e = 0; e < V; ++e) {
          double xe;
          if constexpr (PREC == HFJK_FP64) {
            xe = __hiloint2double((int)hw[2 * e + 1], (int)hw[2 * e]);
          } else if constexpr (PREC == HFJK_FP32) {
            xe = (double)__uint_as_float(hw[e]);
          } else {
            const uint4& l = wl[x];
            const uint32_t lw[4] = {l.x, l.y, l.z, l.w};
            const uint32_t sh = (e & 1) * 16;
            xe = (double)(__uint_as_float(((hw[e >> 1] >> sh) & 0xFFFFu) << 16) +
                          __uint_as_float(((lw[e >> 1] >> sh) & 0xFFFFu) << 16));
          }
          if (i0 + e < in.nocc) s[x] += cv[e] * xe;
        }
      }
    }
    mu += dm;
    gi += dg;
    if (gi >= per_row) {
      gi -= per_row;
      ++mu;
    }
  }
  const int lane = threadIdx.x & 63;
  const double total = wave_sums8(s, lane);
  if ((lane & 7) == 0) red[threadIdx.x >> 6][lane >> 3] = total;
  __syncthreads();
  const int x = threadIdx.x;
  if (x < QB && q0 + x < in.naux) ws64[in.g_off + q0 + x] = red[0][x] + red[1][x] + red[2][x] + red[3][x];
  __syncthreads();
  BATCH_END
}

// Part of the packed J of one tile: sum over the jq aux functions of the
// item's slice of gamma[q] B[q][tile], eight of them in flight. The slices
// give a batch of few tiles enough workgroups (12 water clusters, 480 tiles:
// 0.88 ms in one slice, 0.39 ms in slices of 64; 128 BF16x3 instances to 220
// functions 3.71 -> 3.26 ms, 4.7 TB/s).
template <int PREC>
__global__ __launch_bounds__(kThreads) void b_coulomb_kernel(BatchView v, const void* __restrict__ b, long long plane,
                                                             double* __restrict__ ws64) {
  BATCH_LOOP(kPhCoulomb)
  const long long ntiles = in.p / kTileElems;
  const int slice = (int)(local / ntiles);
  const long long e = (local - slice * ntiles) * kTileElems + threadIdx.x * 4;
  double acc[4] = {0.0, 0.0, 0.0, 0.0};
  const double* g = ws64 + in.g_off;
  const int q1 = min((slice + 1) * in.jq, in.naux);
  int q = slice * in.jq;
  for (; q + 8 <= q1; q += 8) {
    double bv[8][4];
#pragma unroll
    for (int x = 0; x < 8; ++x) bload4<PREC>(b, plane, in.b_off + (long long)(q + x) * in.p + e, bv[x]);
#pragma unroll
    for (int x = 0; x < 8; ++x) {
      const double gq = g[q + x];
      for (int k = 0; k < 4; ++k) acc[k] += gq * bv[x][k];
    }
  }
  for (; q < q1; ++q) {
    double bv[4];
    bload4<PREC>(b, plane, in.b_off + (long long)q * in.p + e, bv);
    const double gq = g[q];
    for (int k = 0; k < 4; ++k) acc[k] += gq * bv[k];
  }
  double* jp = ws64 + in.jp_off + (long long)slice * in.p + e;
  for (int k = 0; k < 4; ++k) jp[k] = acc[k];
  BATCH_END
}

// J [nao][nao] from the slices of the packed J, one tile per item: the tile
// and, through LDS, its mirror.
__global__ __launch_bounds__(kThreads) void b_coulomb_unpack_kernel(BatchView v, const double* __restrict__ ws64,
                                                                    double* __restrict__ j) {
  __shared__ double tile[kTile][kTile + 1];
  BATCH_LOOP(kPhCoulombUnpack)
  int r, c;
  rc_of((int)local, r, c);
  const double* jp = ws64 + in.jp_off + local * kTileElems + threadIdx.x * 4;
  double sum[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 4
  for (int slice = 0; slice < in.jsplit; ++slice)
    for (int k = 0; k < 4; ++k) sum[k] += jp[(long long)slice * in.p + k];
  double* ji = j + in.d_off;
  const int tr = threadIdx.x / 8, tc = threadIdx.x % 8 * 4;
  for (int k = 0; k < 4; ++k) {
    const int row = r * kTile + tr, col = c * kTile + tc + k;
    if (row < in.nao && col < in.nao) ji[(long long)row * in.nao + col] = sum[k];
    tile[tr][tc + k] = sum[k];
  }
  __syncthreads();
  if (r != c) {
    for (int k = 0; k < 4; ++k) {
      const int row = c * kTile + tr, col = r * kTile + tc + k;
      if (row < in.nao && col < in.nao) ji[(long long)row * in.nao + col] = tile[tc + k][tr];
    }
  }
  __syncthreads();
  BATCH_END
}

// Padded orbitals in the mode's layout and the (all +1) column signs.
template <int PREC>
__global__ __launch_bounds__(kThreads) void b_orbitals_kernel(BatchView v, const double* __restrict__ c,
                                                              double* __restrict__ ws64, void* __restrict__ cbase,
                                                              long long c_plane) {
  BATCH_LOOP(kPhOrbitals)
  const int npad = in.nt * kTile;
  if (local == 0)
    for (int i = threadIdx.x; i < in.ldo; i += kThreads) ws64[in.sg_off + i] = i < in.nocc ? 1.0 : 0.0;
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const long long idx = (local * 4 + u) * kThreads + threadIdx.x;
    if (idx < (long long)npad * in.ldo) {
      const double* ci = c + in.c_off;
      if (PREC == HFJK_BF16X3) {
        const int i = (int)(idx / npad), k = (int)(idx % npad);  // Ct[i][k]
        const float x = (k < in.nao && i < in.nocc) ? (float)ci[(long long)k * in.nocc + i] : 0.0f;
        uint16_t* hi = (uint16_t*)cbase + in.cp_off;
        const uint16_t h = to_bf16(x);
        hi[idx] = h;
        hi[idx + c_plane] = to_bf16(x - __uint_as_float(((uint32_t)h) << 16));
      } else {
        const int k = (int)(idx / in.ldo), i = (int)(idx % in.ldo);  // C[k][i], in the operand order
        const double x = (k < in.nao && i < in.nocc) ? ci[(long long)k * in.nocc + i] : 0.0;
        const ColumnGroups cg = in.cg;
        if (i / 16 < cg.groups * cg.blocks + cg.tail) {
          if (PREC == HFJK_FP64)
            ((double*)cbase)[in.cp_off + fragment_index<double>(cg, npad, k, i)] = x;
          else
            ((float*)cbase)[in.cp_off + fragment_index<float>(cg, npad, k, i)] = (float)x;
        }
      }
    }
  }
  BATCH_END
}

#undef BATCH_LOOP
#undef BATCH_END

}  // namespace

dim3 batch_grid(long long items) { return dim3((unsigned)std::max(1LL, std::min(items, kMaxGrid))); }

namespace {
dim3 grid_of(const BatchView& v, int phase) { return batch_grid(v.items[phase]); }
}  // namespace

hipError_t launch_batch_reset(BatchView v, hipStream_t s) {
  hipLaunchKernelGGL(reset_kernel, dim3(1), dim3(kThreads), 0, s, v.counters, kPhCount * 8);
  return hipGetLastError();
}

hipError_t launch_batch_coulomb(BatchView v, int precision, const void* b, long long b_plane, const double* d,
                                double* ws64, double* j, hipStream_t s) {
  const dim3 blk(kThreads);
  hipLaunchKernelGGL(b_weights_kernel, grid_of(v, kPhWeights), blk, 0, s, v, d, ws64);
  if (precision == HFJK_FP64) {
    hipLaunchKernelGGL(b_gamma_kernel<HFJK_FP64>, grid_of(v, kPhGamma), blk, 0, s, v, b, b_plane, ws64);
    hipLaunchKernelGGL(b_gamma_reduce_kernel, grid_of(v, kPhGammaReduce), blk, 0, s, v, ws64);
    hipLaunchKernelGGL(b_coulomb_kernel<HFJK_FP64>, grid_of(v, kPhCoulomb), blk, 0, s, v, b, b_plane, ws64);
  } else if (precision == HFJK_FP32) {
    hipLaunchKernelGGL(b_gamma_kernel<HFJK_FP32>, grid_of(v, kPhGamma), blk, 0, s, v, b, b_plane, ws64);
    hipLaunchKernelGGL(b_gamma_reduce_kernel, grid_of(v, kPhGammaReduce), blk, 0, s, v, ws64);
    hipLaunchKernelGGL(b_coulomb_kernel<HFJK_FP32>, grid_of(v, kPhCoulomb), blk, 0, s, v, b, b_plane, ws64);
  } else {
    hipLaunchKernelGGL(b_gamma_kernel<HFJK_BF16X3>, grid_of(v, kPhGamma), blk, 0, s, v, b, b_plane, ws64);
    hipLaunchKernelGGL(b_gamma_reduce_kernel, grid_of(v, kPhGammaReduce), blk, 0, s, v, ws64);
    hipLaunchKernelGGL(b_coulomb_kernel<HFJK_BF16X3>, grid_of(v, kPhCoulomb), blk, 0, s, v, b, b_plane, ws64);
  }
  hipLaunchKernelGGL(b_coulomb_unpack_kernel, grid_of(v, kPhCoulombUnpack), blk, 0, s, v, ws64, j);
  return hipGetLastError();
}

hipError_t launch_batch_coulomb_occ(BatchView v, int precision, const void* b, long long b_plane, const double* c,
                                    const void* xbase, long long x_plane, double* ws64, double* j,
                                    hipStream_t s) {
  const dim3 blk(kThreads);
  if (precision == HFJK_FP64) {
    hipLaunchKernelGGL(b_charges_x_kernel<HFJK_FP64>, grid_of(v, kPhCharges), blk, 0, s, v, c, xbase, x_plane, ws64);
    hipLaunchKernelGGL(b_coulomb_kernel<HFJK_FP64>, grid_of(v, kPhCoulomb), blk, 0, s, v, b, b_plane, ws64);
  } else if (precision == HFJK_FP32) {
    hipLaunchKernelGGL(b_charges_x_kernel<HFJK_FP32>, grid_of(v, kPhCharges), blk, 0, s, v, c, xbase, x_plane, ws64);
    hipLaunchKernelGGL(b_coulomb_kernel<HFJK_FP32>, grid_of(v, kPhCoulomb), blk, 0, s, v, b, b_plane, ws64);
  } else {
    hipLaunchKernelGGL(b_charges_x_kernel<HFJK_BF16X3>, grid_of(v, kPhCharges), blk, 0, s, v, c, xbase, x_plane, ws64);
    hipLaunchKernelGGL(b_coulomb_kernel<HFJK_BF16X3>, grid_of(v, kPhCoulomb), blk, 0, s, v, b, b_plane, ws64);
  }
  hipLaunchKernelGGL(b_coulomb_unpack_kernel, grid_of(v, kPhCoulombUnpack), blk, 0, s, v, ws64, j);
  return hipGetLastError();
}

hipError_t launch_batch_coulomb_charges(BatchView v, int precision, const void* b, long long b_plane,
                                        const double* charges, double* ws64, double* j, hipStream_t s) {
  const dim3 blk(kThreads);
  hipLaunchKernelGGL(b_charges_load_kernel, grid_of(v, kPhGammaReduce), blk, 0, s, v, charges, ws64);
  if (precision == HFJK_FP64)
    hipLaunchKernelGGL(b_coulomb_kernel<HFJK_FP64>, grid_of(v, kPhCoulomb), blk, 0, s, v, b, b_plane, ws64);
  else if (precision == HFJK_FP32)
    hipLaunchKernelGGL(b_coulomb_kernel<HFJK_FP32>, grid_of(v, kPhCoulomb), blk, 0, s, v, b, b_plane, ws64);
  else
    hipLaunchKernelGGL(b_coulomb_kernel<HFJK_BF16X3>, grid_of(v, kPhCoulomb), blk, 0, s, v, b, b_plane, ws64);
  hipLaunchKernelGGL(b_coulomb_unpack_kernel, grid_of(v, kPhCoulombUnpack), blk, 0, s, v, ws64, j);
  return hipGetLastError();
}

hipError_t launch_batch_orbitals(BatchView v, int precision, const double* c, double* ws64, void* cbase,
                                 long long c_plane, hipStream_t s) {
  const dim3 blk(kThreads);
  if (precision == HFJK_FP64)
    hipLaunchKernelGGL(b_orbitals_kernel<HFJK_FP64>, grid_of(v, kPhOrbitals), blk, 0, s, v, c, ws64, cbase, c_plane);
  else if (precision == HFJK_FP32)
    hipLaunchKernelGGL(b_orbitals_kernel<HFJK_FP32>, grid_of(v, kPhOrbitals), blk, 0, s, v, c, ws64, cbase, c_plane);
  else
    hipLaunchKernelGGL(b_orbitals_kernel<HFJK_BF16X3>, grid_of(v, kPhOrbitals), blk, 0, s, v, c, ws64, cbase, c_plane);
  return hipGetLastError();
}

}  // namespace hfjk

// ---------------------------------------------------------------- C ABI

namespace {

// The phases' item counts of a plan.
void fill_items(hfjk::BatchView& v, const std::vector<long long>& prefix) {
  for (int ph = 0; ph < hfjk::kPhCount; ++ph) v.items[ph] = prefix[(size_t)ph * (v.ninst + 1) + v.ninst];
}

// Bytes of B from which the Coulomb half runs beside the half-transform (its two passes over B then
// take ten times the 40 us of fork and join).
constexpr double kBesideBytes = 1e9;

size_t al256(size_t v) { return (v + 255) & ~size_t(255); }

}  // namespace

extern "C" {

int hfjk_batch_create(hfjk_ctx* ctx, const hfjk_batch_instance* instances, int ninst, int precision, int tile,
                      hfjk_batch** out) {
  if (out != nullptr) *out = nullptr;
  if (ctx == nullptr || out == nullptr || (ninst > 0 && instances == nullptr) || ninst < 1) {
    hfjk_internal_set_error("hfjk_batch_create needs a context, an output pointer and at least one instance");
    return HFJK_ERR_INPUT;
  }
  if (precision != HFJK_FP64 && precision != HFJK_FP32 && precision != HFJK_BF16X3) {
    hfjk_internal_set_error("precision must be HFJK_FP64, HFJK_FP32 or HFJK_BF16X3");
    return HFJK_ERR_INPUT;
  }
  if (tile != 0 && tile != 32 && tile != 64 && tile != 128 && tile != 256) {
    hfjk_internal_set_error("the half-transform column tile is 0, 32, 64, 128 or 256");
    return HFJK_ERR_INPUT;
  }
  hfjk_batch* bt = new (std::nothrow) hfjk_batch();
  if (bt == nullptr) {
    hfjk_internal_set_error("host allocation failed");
    return HFJK_ERR_HIP;
  }
  bt->ctx = ctx;
  bt->precision = precision;
  bt->ninst = ninst;
  bt->insts.resize(ninst);
  int max_ldo = 32;
  for (int i = 0; i < ninst; ++i) max_ldo = std::max(max_ldo, hfjk::occ_ld(std::max(instances[i].nocc, 1)));
  bt->tile = tile != 0 ? tile : (max_ldo <= 32 ? 32 : max_ldo <= 64 ? 64 : 128);
  const int es = precision == HFJK_FP64 ? 8 : precision == HFJK_FP32 ? 4 : 2;  // bf16: per plane
  long long w64 = 0, cp = 0, xx = 0, kp = 0, qq = 0;
  hipDeviceProp_t prop;
  if (hipGetDeviceProperties(&prop, ctx->device) != hipSuccess) prop.multiProcessorCount = 256;
  const int cus = std::max(8, prop.multiProcessorCount);
  double batch_us = 0.0;
  long long x_steps = 0;  // k steps of four units of the FP64 / FP32 half-transform
  for (int i = 0; i < ninst; ++i) {
    double whole_us;
    const long long nt = hfjk::n_tiles(std::max(1, instances[i].nao));
    x_steps += (std::max(1, instances[i].naux) * nt + 3) / 4 * nt * ((std::max(1, instances[i].nocc) + 127) / 128);
    if (instances[i].nao > 0 && instances[i].nao <= 46000)
      batch_us += hfjk::syrk_instance_us(precision, instances[i].naux, instances[i].nao, instances[i].nocc, true, whole_us);
  }
  // Coulomb slices of at least 64 aux functions, 16 workgroups per CU over the batch.
  long long tile_aux = 0;
  for (int i = 0; i < ninst; ++i) {
    const long long nt = hfjk::n_tiles(std::min(std::max(1, instances[i].nao), 46000));
    tile_aux += nt * (nt + 1) / 2 * std::max(1, instances[i].naux);
  }
  const int jq = (int)std::min(1LL << 30, std::max(64LL, (tile_aux / (16LL * cus) + 7) / 8 * 8));
  const double item_us = std::min(1700.0, std::max(40.0, batch_us / (2.0 * cus) / 4.0));
  for (int i = 0; i < ninst; ++i) {
    const hfjk_batch_instance& src = instances[i];
    if (src.nao < 1 || src.naux < 1 || src.nocc < 1 || src.nocc > src.nao || src.nao > 46000 ||
        src.b_offset < 0 || src.b_offset % hfjk::kTileElems != 0 || src.c_offset < 0 || src.d_offset < 0) {
      delete bt;
      hfjk_internal_set_error(("instance " + std::to_string(i) +
                               " needs 1 <= nocc <= nao <= 46000, naux >= 1, a tensor offset that is a multiple"
                               " of 1024 and non-negative offsets").c_str());
      return HFJK_ERR_INPUT;
    }
    hfjk::BatchInst& in = bt->insts[i];
    in.nao = src.nao;
    in.naux = src.naux;
    in.nocc = src.nocc;
    in.ldo = hfjk::occ_ld(src.nocc);
    in.nt = hfjk::n_tiles(src.nao);
    in.xrows = hfjk::x_rows(src.nao);
    // SYRK tile: 128 rows, on the direct-LDS ring where the instance's X offsets fit it. (Small
    // instances compute mostly padding in 128-row tiles, but the ring runs the 128-row tile near
    // the MFMA peak, about twice the rate of the 64-row register-staged tile, so it wins on the
    // whole batch; the 64-row tile serves only instances too large for the ring.)
    {
      const bool fits_ring = in.ldo <= 2048 && (long long)in.xrows * in.ldo * es < (1LL << 31);
      in.st = fits_ring || precision == HFJK_BF16X3 ? hfjk::syrk_tile() : 64;
      const long long nb = (in.xrows + in.st - 1) / in.st;
      in.npairs = (int)(nb * (nb + 1) / 2);
      in.se = fits_ring && precision != HFJK_BF16X3 ? hfjk::syrk_row_block(src.nao) : in.st;
    }
    // BF16x3 half-transform column tile: the smallest of 32 / 64 / 128 that covers the instance's
    // columns, at most the batch's tile (whose multiples then cover them); a batch tile of 256
    // applies to every instance. FP64 / FP32: column groups of at most the batch's tile.
    in.bn = bt->tile == 256 ? 256 : std::min(in.ldo <= 32 ? 32 : in.ldo <= 64 ? 64 : 128, bt->tile);
    in.cg = hfjk::column_groups(src.nocc, in.ldo, bt->tile);
    // Splits: about 8192 k per item, and where the batch is small enough that the longest such
    // item would outlast the others, as many as bring an instance's slowest tile down to a quarter
    // of the batch's mean load per workgroup slot (12 water clusters: 4 rounds of items instead of
    // a first round that holds 1.7 ms items, 2.07 -> 0.8 ms). Eight rounds of one instance's items
    // are enough: its partials stay below 0.6 GB, where items of 1.7 ms would take 7.5 GB at nao
    // 3000 / naux 5000 / nocc 300.
    double whole_us;
    hfjk::syrk_instance_us(precision, src.naux, src.nao, src.nocc, in.se != 64, whole_us);
    const long long by_k = std::min(64LL, ((long long)src.naux * in.ldo + 8191) / 8192);
    const long long by_load = std::min<long long>(std::min<long long>(src.naux, 16LL * cus / in.npairs),
                                                  (long long)std::ceil(whole_us / item_us));
    in.nsplit = (int)std::max(1LL, std::max(by_k, by_load));
    in.bm = 128;
    if (precision == HFJK_BF16X3) {
      // Items cover enough aux functions for about 32 pipelined k tiles (small instances have
      // few k tiles per aux function).
      in.qg = bt->tile == 256 ? 1 : std::max(1, std::min(src.naux, 32 / in.nt));
      in.nbm = (in.xrows + in.bm - 1) / in.bm;
      in.nbn = (in.ldo + in.bn - 1) / in.bn;
    } else {
      // Items of about 32 k steps of four units, fewer where the batch holds too few of them for
      // four items per workgroup.
      in.qg = 4 * (int)std::max(1LL, std::min(32LL, x_steps / (8LL * cus)) / in.nt);
      in.nbm = 1;
      in.nbn = in.cg.groups + (in.cg.tail > 0 ? 1 : 0);
    }
    in.p = hfjk::packed_elems(src.nao);
    in.b_off = src.b_offset;
    in.c_off = src.c_offset;
    in.d_off = src.d_offset;
    in.q_off = qq;
    qq += src.naux;
    bt->b_total = std::max(bt->b_total, src.b_offset + (long long)src.naux * in.p);
    bt->c_total = std::max(bt->c_total, src.c_offset + (long long)src.nao * src.nocc);
    bt->d_total = std::max(bt->d_total, src.d_offset + (long long)src.nao * src.nao);
    const long long ntiles = in.p / hfjk::kTileElems;
    auto take64 = [&](long long n) { const long long at = w64; w64 += (n + 31) / 32 * 32; return at; };
    in.w_off = take64(in.p);
    in.jsplit = (src.naux + jq - 1) / jq;
    in.jq = ((src.naux + in.jsplit - 1) / in.jsplit + 7) / 8 * 8;
    in.jsplit = (src.naux + in.jq - 1) / in.jq;
    in.jp_off = take64((long long)in.jsplit * in.p);
    in.gp_off = take64(ntiles * src.naux);
    in.g_off = take64(src.naux);
    in.sg_off = take64(in.ldo);
    in.cp_off = cp;
    cp += (long long)in.nt * hfjk::kTile * in.ldo + 64;
    in.x_off = xx;
    xx += (long long)src.naux * in.xrows * in.ldo + 64;
    in.kp_off = kp;
    kp += (long long)in.nsplit * in.npairs * in.st * in.st;
  }
  bt->ws64_total = w64;
  bt->cp_total = cp;
  bt->x_total = xx;
  bt->kp_total = kp;
  // Items per instance and phase.
  bt->prefix.assign((size_t)hfjk::kPhCount * (ninst + 1), 0);
  for (int i = 0; i < ninst; ++i) {
    const hfjk::BatchInst& in = bt->insts[i];
    const long long ntiles = in.p / hfjk::kTileElems;
    long long items[hfjk::kPhCount];
    items[hfjk::kPhWeights] = ntiles;
    items[hfjk::kPhGamma] = ntiles * ((in.naux + 63) / 64);
    items[hfjk::kPhGammaReduce] = (in.naux + 63) / 64;
    items[hfjk::kPhCoulomb] = ntiles * in.jsplit;
    items[hfjk::kPhCoulombUnpack] = ntiles;
    items[hfjk::kPhOrbitals] = ((long long)in.nt * hfjk::kTile * in.ldo + 4 * hfjk::kThreads - 1) / (4 * hfjk::kThreads);
    const long long x_units = (long long)in.naux * (precision == HFJK_FP64 ? hfjk::xform_units_per_aux<double>(in.nao)
                                                    : precision == HFJK_FP32 ? hfjk::xform_units_per_aux<float>(in.nao)
                                                                             : 1);
    items[hfjk::kPhXform] = (x_units + in.qg - 1) / in.qg * in.nbm * in.nbn;
    // Instances whose X offsets fit the ring's 32-bit lane offsets run on it, in a phase of
    // their own.
    const bool ring = in.ldo <= 2048 && (long long)in.xrows * in.ldo * es < (1LL << 31);
    items[hfjk::kPhSyrk] = ring ? 0 : (long long)in.npairs * in.nsplit;
    items[hfjk::kPhSyrkRing] = ring ? (long long)in.npairs * in.nsplit : 0;
    // Strips of 512 elements of every lower tile.
    items[hfjk::kPhSyrkReduce] = (long long)in.npairs * (in.st * in.st / (2 * hfjk::kThreads));
    const int per_item = hfjk::charges_per_item(precision);
    items[hfjk::kPhCharges] = (in.naux + per_item - 1) / per_item;
    for (int ph = 0; ph < hfjk::kPhCount; ++ph) {
      const size_t base = (size_t)ph * (ninst + 1);
      bt->prefix[base + i + 1] = bt->prefix[base + i] + items[ph];
    }
  }
  // Workspace layout.
  size_t off = 0;
  bt->off_insts = off;
  off = al256(off + sizeof(hfjk::BatchInst) * ninst);
  bt->off_prefix = off;
  off = al256(off + sizeof(long long) * bt->prefix.size());
  bt->off_counters = off;
  off = al256(off + sizeof(unsigned long long) * hfjk::kPhCount * 8);
  bt->off_ws64 = off;
  off = al256(off + sizeof(double) * (size_t)w64);
  const int planes = precision == HFJK_BF16X3 ? 2 : 1;
  bt->off_cp = off;
  off = al256(off + (size_t)es * planes * cp);
  bt->off_x = off;
  off = al256(off + (size_t)es * planes * xx);
  bt->off_kp = off;
  off = al256(off + (size_t)(precision == HFJK_FP64 ? 8 : 4) * kp);
  bt->bytes = off;
  bt->grid_mfma = ((2 * cus + 7) / 8) * 8;
  bt->beside = (double)bt->b_total * (precision == HFJK_FP64 ? 8 : 4) > kBesideBytes;
  *out = bt;
  return HFJK_OK;
}

int hfjk_batch_workspace_bytes(const hfjk_batch* batch, size_t* bytes) {
  if (batch == nullptr || bytes == nullptr) {
    hfjk_internal_set_error("null batch or output pointer");
    return HFJK_ERR_INPUT;
  }
  *bytes = batch->bytes;
  return HFJK_OK;
}

int hfjk_batch_sizes(const hfjk_batch* batch, long long* tensor_elems, long long* orbital_elems,
                     long long* matrix_elems) {
  if (batch == nullptr) {
    hfjk_internal_set_error("null batch");
    return HFJK_ERR_INPUT;
  }
  if (tensor_elems) *tensor_elems = batch->b_total;
  if (orbital_elems) *orbital_elems = batch->c_total;
  if (matrix_elems) *matrix_elems = batch->d_total;
  return HFJK_OK;
}

int hfjk_batch_bind(hfjk_batch* batch, void* workspace, size_t bytes, void* stream) {
  if (batch == nullptr || workspace == nullptr) {
    hfjk_internal_set_error("null batch or workspace");
    return HFJK_ERR_INPUT;
  }
  if (bytes < batch->bytes || ((uintptr_t)workspace & 255) != 0) {
    hfjk_internal_set_error(("the batch needs a 256-byte aligned workspace of " + std::to_string(batch->bytes) +
                             " bytes").c_str());
    return HFJK_ERR_WORKSPACE;
  }
  hipStream_t s = (hipStream_t)stream;
  char* ws = (char*)workspace;
  hipError_t e = hipSetDevice(batch->ctx->device);
  if (e == hipSuccess)
    e = hipMemcpyAsync(ws + batch->off_insts, batch->insts.data(), sizeof(hfjk::BatchInst) * batch->ninst,
                       hipMemcpyHostToDevice, s);
  if (e == hipSuccess)
    e = hipMemcpyAsync(ws + batch->off_prefix, batch->prefix.data(), sizeof(long long) * batch->prefix.size(),
                       hipMemcpyHostToDevice, s);
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  if (e == hipSuccess && batch->beside && batch->side == nullptr) {
    if (batch->fork == nullptr) e = hipEventCreateWithFlags(&batch->fork, hipEventDisableTiming);
    if (e == hipSuccess && batch->join == nullptr) e = hipEventCreateWithFlags(&batch->join, hipEventDisableTiming);
    if (e == hipSuccess) e = hipStreamCreateWithFlags(&batch->side, hipStreamNonBlocking);
  }
  if (e != hipSuccess) {
    hfjk_internal_set_error((std::string("uploading the batch plan: ") + hipGetErrorString(e)).c_str());
    return HFJK_ERR_HIP;
  }
  batch->ws = workspace;
  return HFJK_OK;
}

int hfjk_batch_run(hfjk_batch* batch, const void* tensor, const double* orbitals, const double* density,
                   double* coulomb, double* exchange, void* stream) {
  if (batch == nullptr || batch->ws == nullptr) {
    hfjk_internal_set_error("the batch is not bound to a workspace (hfjk_batch_bind)");
    return HFJK_ERR_INPUT;
  }
  if (tensor == nullptr || orbitals == nullptr || coulomb == nullptr || exchange == nullptr) {
    hfjk_internal_set_error("hfjk_batch_run needs the tensor, orbitals and both outputs");
    return HFJK_ERR_INPUT;
  }
  hipStream_t s = (hipStream_t)stream;
  char* ws = (char*)batch->ws;
  hfjk::BatchView v;
  v.insts = (const hfjk::BatchInst*)(ws + batch->off_insts);
  v.prefix = (const long long*)(ws + batch->off_prefix);
  v.counters = (unsigned long long*)(ws + batch->off_counters);
  v.ninst = batch->ninst;
  fill_items(v, batch->prefix);
  double* ws64 = (double*)(ws + batch->off_ws64);
  void* cbase = ws + batch->off_cp;
  void* xbase = ws + batch->off_x;
  void* kbase = ws + batch->off_kp;
  const int prec = batch->precision;
  hipError_t e = hipSetDevice(batch->ctx->device);
  if (e == hipSuccess) e = hfjk::launch_batch_reset(v, s);
  // With densities the Coulomb half needs nothing of the exchange: it streams B beside the
  // matrix-core-bound half-transform, whose waves leave register room for its own (128 FP64
  // instances to 220 functions 45.9 -> 42.2 ms; 96 to 220, FP32 3.66 -> 3.44, BF16x3 3.85 -> 3.59).
  const bool beside = density != nullptr && batch->side != nullptr;
  hipStream_t cs = beside ? batch->side : s;
  if (e == hipSuccess && beside) e = hipEventRecord(batch->fork, s);
  if (e == hipSuccess && beside) e = hipStreamWaitEvent(cs, batch->fork, 0);
  const bool forked = e == hipSuccess && beside;
  if (e == hipSuccess && density != nullptr)
    e = hfjk::launch_batch_coulomb(v, prec, tensor, batch->b_total, density, ws64, coulomb, cs);
  // Once forked, s waits for the side stream whatever fails: the caller may free J and the
  // workspace on return, and a capture must not end with a stream of its own.
  const hipError_t recorded = forked ? hipEventRecord(batch->join, cs) : hipSuccess;
  if (e == hipSuccess) e = recorded;
  if (e == hipSuccess)
    e = hfjk::launch_batch_orbitals(v, prec, orbitals, ws64, cbase, batch->cp_total, s);
  if (e == hipSuccess)
    e = hfjk::launch_batch_xform(v, prec, batch->tile, tensor, batch->b_total, cbase, batch->cp_total, xbase,
                                 batch->x_total, batch->grid_mfma, s);
  // Without densities D = C C^T: the charges come from X (one pass over X instead of one over B).
  if (e == hipSuccess && density == nullptr)
    e = hfjk::launch_batch_coulomb_occ(v, prec, tensor, batch->b_total, orbitals, xbase, batch->x_total, ws64,
                                       coulomb, s);
  if (e == hipSuccess)
    e = hfjk::launch_batch_syrk(v, prec, xbase, batch->x_total, ws64, kbase, batch->grid_mfma, s);
  if (e == hipSuccess) e = hfjk::launch_batch_syrk_reduce(v, prec, kbase, exchange, s);
  if (forked && recorded == hipSuccess) {
    const hipError_t joined = hipStreamWaitEvent(s, batch->join, 0);
    if (e == hipSuccess) e = joined;
  }
  if (e != hipSuccess) {
    hfjk_internal_set_error((std::string("batched launch: ") + hipGetErrorString(e)).c_str());
    return HFJK_ERR_HIP;
  }
  return HFJK_OK;
}

int hfjk_batch_coulomb_charges(hfjk_batch* batch, const void* tensor, const double* charges, double* coulomb,
                               void* stream) {
  if (batch == nullptr || batch->ws == nullptr) {
    hfjk_internal_set_error("the batch is not bound to a workspace (hfjk_batch_bind)");
    return HFJK_ERR_INPUT;
  }
  if (tensor == nullptr || charges == nullptr || coulomb == nullptr) {
    hfjk_internal_set_error("hfjk_batch_coulomb_charges needs the tensor, the charges and the output");
    return HFJK_ERR_INPUT;
  }
  hipStream_t s = (hipStream_t)stream;
  char* ws = (char*)batch->ws;
  hfjk::BatchView v;
  v.insts = (const hfjk::BatchInst*)(ws + batch->off_insts);
  v.prefix = (const long long*)(ws + batch->off_prefix);
  v.counters = (unsigned long long*)(ws + batch->off_counters);
  v.ninst = batch->ninst;
  fill_items(v, batch->prefix);
  double* ws64 = (double*)(ws + batch->off_ws64);
  hipError_t e = hipSetDevice(batch->ctx->device);
  if (e == hipSuccess) e = hfjk::launch_batch_reset(v, s);
  if (e == hipSuccess)
    e = hfjk::launch_batch_coulomb_charges(v, batch->precision, tensor, batch->b_total, charges, ws64, coulomb, s);
  if (e != hipSuccess) {
    hfjk_internal_set_error((std::string("batched launch: ") + hipGetErrorString(e)).c_str());
    return HFJK_ERR_HIP;
  }
  return HFJK_OK;
}

int hfjk_batch_destroy(hfjk_batch* batch) {
  delete batch;
  return HFJK_OK;
}

}  // extern "C"
