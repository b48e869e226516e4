// Batched symmetric eigensolver for the lowest eigenpairs in six launches
// (the Fock diagonalisation of a batched SCF, where rocSOLVER's batched divide
// and conquer is about 1500 small launches per call):
//   1. Householder reduction to tridiagonal form, T = Q^T A Q (Golub and
//      Van Loan, "Matrix Computations", algorithm 8.3.1), the reflector
//      vectors kept in the rows of A above the diagonal;
//   2. the nvec lowest eigenvalues of T by multisection (bisection with
//      several points per round) on the Sturm count of the LDL^T recurrence
//      (ibid. section 8.4.1; the pivot guard of LAPACK's dstebz);
//   3. their eigenvectors by inverse iteration on T with a partially
//      pivoted tridiagonal LU (as LAPACK's dlagtf / dlagts), equal
//      eigenvalues' shifts separated by 10 eps |T|, then made orthonormal
//      (Cholesky QR twice, or Gram-Schmidt twice past 64 vectors);
//   4. back-transformation x = Q y by the stored reflectors.
// A is row-major and symmetric; on return its rows 0 .. nvec - 1 are the
// eigenvectors of the nvec lowest eigenvalues and w[0 .. nvec) holds those
// eigenvalues in ascending order (rows nvec .. n - 1 of A hold scratch).
#include <algorithm>
#include <cfloat>
#include <cmath>
#include <string>

#include "hfjk_internal.h"

namespace {

typedef unsigned int u2 __attribute__((ext_vector_type(2)));

constexpr int kEigThreads = 512;
constexpr int kEigWaves = kEigThreads / 64;
constexpr int kEigMaxN = 512;
constexpr int kEigRegVecs = 64;             // nvec up to this: vectors stay in registers, Cholesky QR
constexpr int kGs = 65;                     // row stride of the Gram matrix and its inverse factor in LDS

// Workspace doubles per matrix: d, e, beta (n each) and the nvec eigenvectors [nvec][n].
__host__ __device__ inline long long eig_work_per(int n, int nvec) { return 3LL * n + (long long)nvec * n; }

// Sum over the workgroup (every thread passes its part; all get the total).
__device__ __forceinline__ double wg_sum(double v, double* red) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  __syncthreads();  // red is free (its previous readers are done)
  if (lane == 0) red[wave] = v;
  __syncthreads();
  double s = 0.0;
#pragma unroll
  for (int k = 0; k < kEigWaves; ++k) s += red[k];
  return s;
}

using hfjk::dpp_d;
using hfjk::wave_sums8;

// Sum over the wave, every lane gets it (shuffles across rows, DPP within a row).
__device__ inline double wave_sum(double v) {
  v += __shfl_xor(v, 32);
  v += __shfl_xor(v, 16);
  v += dpp_d<0x140>(v);
  v += dpp_d<0x141>(v);
  v += dpp_d<0x4E>(v);
  v += dpp_d<0xB1>(v);
  return v;
}

// Sum over the workgroup with one barrier: red must not be written again before a later barrier
// (callers alternate two buffers between barriers).
__device__ __forceinline__ double wg_sum1(double v, double* red) {
  v = wave_sum(v);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  double s = 0.0;
#pragma unroll
  for (int k = 0; k < kEigWaves; ++k) s += red[k];
  return s;
}

__device__ inline double readlane_d(double x, int l) {
  const long long b = __double_as_longlong(x);
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)b, l);
  const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(b >> 32), l);
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// 1 / q from the hardware estimate and one Newton step (the Sturm count needs only the signs
// of a recurrence that is stable under small relative perturbations).
__device__ inline double recip(double q) {
  const double r = __builtin_amdgcn_rcp(q);
  return fma(r, fma(-q, r, 1.0), r);
}

// A deterministic start vector entry in (-1, 1).
__device__ double start_entry(int j, int i) {
  unsigned h = (unsigned)(j * 73856093) ^ (unsigned)(i * 19349663) ^ 0x9e3779b9u;
  h ^= h >> 16;
  h *= 0x7feb352du;
  h ^= h >> 15;
  h *= 0x846ca68bu;
  h ^= h >> 16;
  return (double)(h & 0xFFFFFFu) / (double)0x800000 - 1.0;
}

constexpr int kOutOfRange = 1 << 30;  // a byte offset beyond any matrix of at most 512 x 512 doubles

__device__ inline double buf_ld(__amdgpu_buffer_rsrc_t rsrc, int off) {
  return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(rsrc, off, 0, 0));
}
__device__ inline void buf_st(__amdgpu_buffer_rsrc_t rsrc, double v, int off) {
  __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u2, v), rsrc, off, 0, 0);
}

// R rows j0, j0 + 8, ... of one pass, CB chunks each, without branches (so that the compiler
// keeps the per-row sums in place): rows past m load the last row and store out of range,
// lanes off the lower triangle enter the sums with a zero factor.
template <int NC, int CB, int R>
__device__ __forceinline__ void tri_batch(__amdgpu_buffer_rsrc_t rsrc, int boff, int n, int m, int j0, int lane,
                                          const double (&pvc)[NC], const double (&pwc)[NC], const double (&vc)[NC],
                                          double (&acc)[NC], const double* pv, const double* pw, const double* vv,
                                          double v0, double* nxt, double* prow, double* lsink, int lane_off,
                                          int last_off) {
  double val[R][CB];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int roff = boff + min(j0 + r * kEigWaves, m - 1) * n * 8;
#pragma unroll
    for (int c = 0; c < CB; ++c) val[r][c] = buf_ld(rsrc, roff + (c == NC - 1 ? last_off : lane_off) + 512 * c);
  }
  double rs[8];
#pragma unroll
  for (int r = 0; r < 8; ++r) rs[r] = 0.0;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int j = j0 + r * kEigWaves;
    const bool live = j < m;
    const int jc = min(j, m - 1);
    const int jm = live ? j : -1;  // lanes i <= jm are in the lower triangle of a live row
    const double vj = live ? (jc == 0 ? v0 : vv[jc]) : 0.0;
    const double pvj = pv[1 + jc], pwj = pw[1 + jc];
    const int roff = live ? boff + j * n * 8 : kOutOfRange;
#pragma unroll
    for (int c = 0; c < CB; ++c) {
      const int i = lane + 64 * c;
      const double a = val[r][c] - pvj * pwc[c] - pwj * pvc[c];
      buf_st(rsrc, a, roff + (c == NC - 1 ? last_off : lane_off) + 512 * c);
      if (c + 2 < CB) {  // below the diagonal in every row of the batch (a batch spans < 64 rows)
        acc[c] = fma(a, vj, acc[c]);
        rs[r] = fma(a, vc[c], rs[r]);  // the sums of rows past m are not used
      } else {
        acc[c] = fma(a, i <= jm ? vj : 0.0, acc[c]);
        rs[r] = fma(a, i < jm ? vc[c] : 0.0, rs[r]);
      }
      if (c == 0) *(live && lane == 0 ? nxt + j : lsink + lane) = a;
    }
  }
  const double tot = wave_sums8(rs, lane);
  if ((lane & 7) == 0) {
    const int r = lane >> 3, j = j0 + r * kEigWaves;
    if (r < R && j < m) prow[j] = tot;
  }
}

template <int NC, int CB, int R>
__device__ __forceinline__ void tri_batch_cb(int cb, __amdgpu_buffer_rsrc_t rsrc, int boff, int n, int m, int j0,
                                             int lane, const double (&pvc)[NC], const double (&pwc)[NC],
                                             const double (&vc)[NC], double (&acc)[NC], const double* pv,
                                             const double* pw, const double* vv, double v0, double* nxt, double* prow,
                                             double* lsink, int lane_off, int last_off) {
  if constexpr (CB <= NC) {
    if (cb == CB)
      tri_batch<NC, CB, R>(rsrc, boff, n, m, j0, lane, pvc, pwc, vc, acc, pv, pw, vv, v0, nxt, prow, lsink, lane_off,
                           last_off);
    else
      tri_batch_cb<NC, CB + 1, R>(cb, rsrc, boff, n, m, j0, lane, pvc, pwc, vc, acc, pv, pw, vv, v0, nxt, prow, lsink,
                                  lane_off, last_off);
  }
}

// The Householder vector of a column x (ss = |x|^2, x0 its first entry): v = x but v0, beta and the
// entry that the reflection leaves.
__device__ __forceinline__ void reflector(double ss, double x0, double& bk, double& ek, double& v0) {
  const double sigma = ss - x0 * x0;
  bk = 0.0;
  ek = x0;
  v0 = x0;
  if (sigma > 0.0) {
    const double norm = sqrt(ss);
    const double alpha = x0 > 0.0 ? -norm : norm;
    v0 = x0 - alpha;
    bk = 2.0 / (sigma + v0 * v0);
    ek = alpha;
  }
}

// One pass over the lower triangle of the m x m trailing block (rows and columns c0 .. n - 1 of
// A, at byte offset boff of the buffer rsrc, which covers A): applies the previous step's rank-2
// update A -= v' w'^T + w' v'^T (pv, pw indexed from row c0 - 1) and forms the product of the
// updated block with v (v[0] is v0): the column part sum_{j >= i} a_ji v_j into partw[i], the
// row part sum_{i < j} a_ji v_i into prow[j]; column c0 of the result also goes to nxt. Wave
// `wave` takes rows wave, wave + 8, ..., R rows per batch, each batch as many 64-column chunks as
// its last row reaches. Buffer loads and stores keep the VALU work per chunk to the arithmetic:
// the chunk's offset is an immediate, and lanes of the last chunk past the row end get an
// offset outside the buffer (loads read zero, stores are dropped). Lanes above the diagonal load
// and store the upper triangle of the block, which no pass reads.
template <int NC>
__device__ __forceinline__ void tri_pass(__amdgpu_buffer_rsrc_t rsrc, int boff, int n, int m, int wave, int lane,
                                         const double* pv, const double* pw, const double* vv, double v0,
                                         double* nxt, double* partw, double* prow, double* lsink) {
  constexpr int R = NC <= 4 ? 8 : 4;
  double pvc[NC], pwc[NC], vc[NC], acc[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int i = lane + 64 * c;
    pvc[c] = i < m ? pv[1 + i] : 0.0;
    pwc[c] = i < m ? pw[1 + i] : 0.0;
    vc[c] = i == 0 ? v0 : i < m ? vv[i] : 0.0;
    acc[c] = 0.0;
  }
  const int lane_off = lane * 8;
  const int last_off = lane + 64 * (NC - 1) < m ? lane * 8 : kOutOfRange;  // last chunk, less 512 (NC - 1)
  for (int j0 = wave; j0 < m; j0 += kEigWaves * R) {
    const int cb = (min(j0 + kEigWaves * (R - 1), m - 1) >> 6) + 1;
    tri_batch_cb<NC, 1, R>(cb, rsrc, boff, n, m, j0, lane, pvc, pwc, vc, acc, pv, pw, vv, v0, nxt, prow, lsink,
                           lane_off, last_off);
  }
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int i = lane + 64 * c;
    if (i < m) partw[i] = acc[c];
  }
}

// y[q] = Y[j0 + q] for the wave's eight vectors (zero past nvec or n).
template <int NC>
__device__ inline void load_vecs(double (&y)[8][NC], const double* Y, int n, int nvec, int j0, int lane) {
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const int j = min(j0 + q, nvec - 1);
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int r = lane + 64 * c;
      const double v = Y[(long long)j * n + min(r, n - 1)];
      y[q][c] = (j0 + q < nvec && r < n) ? v : 0.0;
    }
  }
}

template <int NC>
__device__ inline void store_vecs(const double (&y)[8][NC], double* Y, int n, int nvec, int j0, int lane) {
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    if (j0 + q < nvec) {
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const int r = lane + 64 * c;
        if (r < n) Y[(long long)(j0 + q) * n + r] = y[q][c];
      }
    }
  }
}

// Rows j0 .. j0 + 7 of the Gram matrix G = Y Y^T against columns 0 .. min(j0 + 7, nvec - 1)
// into gm (lower triangle), the wave's own vectors in y, the others read from Y.
template <int NC>
__device__ __forceinline__ void gram_rows(const double (&y)[8][NC], const double* Y, int n, int nvec, int j0, int lane,
                          double* gm) {
  constexpr int OB = NC <= 2 ? 8 : NC <= 4 ? 4 : 2;  // other vectors per batch of loads
  const int kend = min(j0 + 8, nvec);
  for (int kb = 0; kb < kend; kb += OB) {
    double ob[OB][NC];
#pragma unroll
    for (int o = 0; o < OB; ++o) {
      const int kk = min(kb + o, nvec - 1);
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const int r = lane + 64 * c;
        const double v = Y[(long long)kk * n + min(r, n - 1)];
        ob[o][c] = r < n ? v : 0.0;
      }
    }
#pragma unroll
    for (int g = 0; g < 8 * OB; g += 8) {
      double s[8];
#pragma unroll
      for (int x = 0; x < 8; ++x) {
        const int q = (g + x) / OB, o = (g + x) % OB;
        double a = 0.0;
#pragma unroll
        for (int c = 0; c < NC; ++c) a += y[q][c] * ob[o][c];
        s[x] = a;
      }
      const double tot = wave_sums8(s, lane);
      if ((lane & 7) == 0) {
        const int x = lane >> 3;
        const int q = (g + x) / OB, o = (g + x) % OB;
        const int j = j0 + q, kk = kb + o;
        if (j < nvec && kk <= j) gm[j * kGs + kk] = tot;
      }
    }
  }
}

// y <- rows j0 .. j0 + 7 of Linv Y (Linv lower triangular in li), Y read from memory.
template <int NC>
__device__ __forceinline__ void tri_product(double (&y)[8][NC], const double* Y, int n, int nvec, int j0, int lane,
                            const double* li) {
  constexpr int OB = NC <= 2 ? 8 : NC <= 4 ? 4 : 2;
#pragma unroll
  for (int q = 0; q < 8; ++q)
#pragma unroll
    for (int c = 0; c < NC; ++c) y[q][c] = 0.0;
  const int kend = min(j0 + 8, nvec);
  for (int kb = 0; kb < kend; kb += OB) {
    double ob[OB][NC];
#pragma unroll
    for (int o = 0; o < OB; ++o) {
      const int kk = min(kb + o, nvec - 1);
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const int r = lane + 64 * c;
        const double v = Y[(long long)kk * n + min(r, n - 1)];
        ob[o][c] = r < n ? v : 0.0;
      }
    }
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int j = j0 + q;
#pragma unroll
      for (int o = 0; o < OB; ++o) {
        const int kk = kb + o;
        const double coef = (j < nvec && kk <= j) ? li[j * kGs + kk] : 0.0;
#pragma unroll
        for (int c = 0; c < NC; ++c) y[q][c] += coef * ob[o][c];
      }
    }
  }
}

// li = L^{-1} of G = L L^T (G in the lower triangle of gm, nv <= 64) by elimination of [G | 1]: with
// G = U D U^T, U^{-1} is what the eliminations make of the unit matrix and L^{-1} = D^{-1/2} U^{-1}.
// Thread (i, c) = (t / 8, t % 8) holds the entries of row i in columns c, c + 8, ... of both; the
// owners of row k publish it and one barrier a step suffices with two buffers. A non-positive pivot
// is raised to DBL_MIN.
__device__ void cholesky_inverse(const double* gm, double* li, double (*rows)[2 * kEigRegVecs], int nv) {
  const int i = threadIdx.x >> 3, c = threadIdx.x & 7;
  double g[8], x[8];
#pragma unroll
  for (int m = 0; m < 8; ++m) {
    const int col = c + 8 * m;
    g[m] = i < nv && col < nv ? gm[max(i, col) * kGs + min(i, col)] : 0.0;
    x[m] = i == col ? 1.0 : 0.0;
  }
  for (int k = 0; k < nv; ++k) {
    double* row = rows[k & 1];
    if (i == k) {
#pragma unroll
      for (int m = 0; m < 8; ++m) {
        row[c + 8 * m] = g[m];
        row[kEigRegVecs + c + 8 * m] = x[m];
      }
    }
    __syncthreads();
    const double piv = fmax(row[k], DBL_MIN);
    if (i > k) {
      const double f = row[i] / piv;
#pragma unroll
      for (int m = 0; m < 8; ++m) {
        g[m] = fma(-f, row[c + 8 * m], g[m]);
        x[m] = fma(-f, row[kEigRegVecs + c + 8 * m], x[m]);
      }
    } else if (i == k) {
      const double r = 1.0 / sqrt(piv);
#pragma unroll
      for (int m = 0; m < 8; ++m) li[k * kGs + c + 8 * m] = x[m] * r;
    }
  }
}

// Orthonormalisation (Cholesky QR twice) of Y for nvec <= 64, each wave's eight vectors held in
// registers.
template <int NC>
__device__ __forceinline__ void orthonormalise(double* Y, double* gm, double* li, double (*rows)[2 * kEigRegVecs], int n,
                                               int nvec, int wave, int lane) {
  const int j0 = 8 * wave;
  double y[8][NC];
  load_vecs<NC>(y, Y, n, nvec, j0, lane);
  for (int pass = 0; pass < 2; ++pass) {
    if (j0 < nvec) gram_rows<NC>(y, Y, n, nvec, j0, lane, gm);
    __syncthreads();
    cholesky_inverse(gm, li, rows, nvec);
    __syncthreads();
    if (j0 < nvec) tri_product<NC>(y, Y, n, nvec, j0, lane, li);
    __syncthreads();  // every wave has read Y
    store_vecs<NC>(y, Y, n, nvec, j0, lane);
    __syncthreads();
  }
}

// Y <- H_0 H_1 ... H_{n-3} Y, reflector k = I - beta_k u u^T with u in row k of A (columns k + 1 ..
// n - 1): one vector per row of 16 lanes, so that a dot product ends in DPP steps alone. A
// workgroup is one wave with four vectors: the reflectors are a serial chain, and the vectors of
// all matrices side by side fill the chip (eight vectors in each wave of one workgroup per matrix
// took 0.2 ms of its 0.6). Reflectors come RB at a time through LDS, the next RB in flight in
// registers, from the L2 of the XCD that wrote them (one reflector ahead, from any XCD, a step
// waited 2.9 us).
template <int NC, int RB>
__device__ __forceinline__ void back_transform(const double* A, const double* lbeta, double (*lu)[kEigMaxN], double* Y,
                                               int n, int nvec, int j, int lane) {
  if (n < 3) return;
  constexpr int NL = (NC + 3) / 4;
  const int l16 = lane & 15;
  double y[NC], un[RB][NL];
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int r = 16 * c + l16;
    const double v = Y[(long long)min(j, nvec - 1) * n + min(r, n - 1)];
    y[c] = r < n ? v : 0.0;
  }
  auto load_block = [&](int k0) {  // reflectors k0, k0 - 1, ...
#pragma unroll
    for (int q = 0; q < RB; ++q) {
      const int k = max(k0 - q, 0);
#pragma unroll
      for (int c = 0; c < NL; ++c) un[q][c] = A[(long long)k * n + min(max(64 * c + lane, k + 1), n - 1)];
    }
  };
  load_block(n - 3);
  for (int k0 = n - 3; k0 >= 0; k0 -= RB) {
    __syncthreads();
#pragma unroll
    for (int q = 0; q < RB; ++q)
#pragma unroll
      for (int c = 0; c < NL; ++c) {
        const int r = 64 * c + lane;
        lu[q][r] = r > k0 - q && r < n ? un[q][c] : 0.0;
      }
    __syncthreads();
    if (k0 >= RB) load_block(k0 - RB);
#pragma unroll 1
    for (int q = 0; q < min(RB, k0 + 1); ++q) {
      double u[NC];
#pragma unroll
      for (int c = 0; c < NC; ++c) u[c] = lu[q][16 * c + l16];
      double s0 = 0.0, s1 = 0.0;
#pragma unroll
      for (int c = 0; c < NC; c += 2) {
        s0 = fma(u[c], y[c], s0);
        if (c + 1 < NC) s1 = fma(u[c + 1], y[c + 1], s1);
      }
      double s = s0 + s1;
      s += dpp_d<0x140>(s);
      s += dpp_d<0x141>(s);
      s += dpp_d<0x4E>(s);
      s += dpp_d<0xB1>(s);
      const double f = -lbeta[k0 - q] * s;
#pragma unroll
      for (int c = 0; c < NC; ++c) y[c] = fma(f, u[c], y[c]);
    }
  }
  if (j < nvec) {
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int r = 16 * c + l16;
      if (r < n) Y[(long long)j * n + r] = y[c];
    }
  }
}

// Workgroup part * (count rounded up to 8) + matrix, so that a matrix stays on the XCD of its
// tridiagonalisation (workgroup = matrix).
__global__ __launch_bounds__(64) void eig_back_kernel(int n, int nvec, int count, const double* __restrict__ a_all,
                                                       double* __restrict__ work_all) {
  __shared__ double lu[8][kEigMaxN], lbeta[kEigMaxN];
  const int lane = threadIdx.x;
  const int stride = (count + 7) & ~7;
  const int matrix = blockIdx.x % stride, part = blockIdx.x / stride;
  if (matrix >= count) return;
  const double* A = a_all + (long long)matrix * n * n;
  double* work = work_all + (long long)matrix * eig_work_per(n, nvec);
  double* Y = work + 3 * n;
  for (int i = lane; i < n; i += 64) lbeta[i] = work[2 * n + i];
  __syncthreads();
  const int j = 4 * part + (lane >> 4);
  switch ((n + 63) >> 6) {
    case 1: back_transform<4, 8>(A, lbeta, lu, Y, n, nvec, j, lane); break;
    case 2: back_transform<8, 8>(A, lbeta, lu, Y, n, nvec, j, lane); break;
    case 3: back_transform<12, 8>(A, lbeta, lu, Y, n, nvec, j, lane); break;
    case 4: back_transform<16, 8>(A, lbeta, lu, Y, n, nvec, j, lane); break;
    case 5: back_transform<20, 8>(A, lbeta, lu, Y, n, nvec, j, lane); break;
    case 6: back_transform<24, 4>(A, lbeta, lu, Y, n, nvec, j, lane); break;
    case 7: back_transform<28, 4>(A, lbeta, lu, Y, n, nvec, j, lane); break;
    default: back_transform<32, 4>(A, lbeta, lu, Y, n, nvec, j, lane); break;
  }
}

// The vectors to the first rows of A, whose reflectors every wave is done with.
__global__ __launch_bounds__(kEigThreads) void eig_store_kernel(int n, int nvec, double* __restrict__ a_all,
                                                                 const double* __restrict__ work_all,
                                                                 int* __restrict__ info) {
  double* A = a_all + (long long)blockIdx.x * n * n;
  const double* Y = work_all + (long long)blockIdx.x * eig_work_per(n, nvec) + 3 * n;
#pragma unroll 8
  for (int f = threadIdx.x; f < nvec * n; f += kEigThreads) A[f] = Y[f];
  if (threadIdx.x == 0) info[blockIdx.x] = 0;
}

// The trailing block that stays on the chip: its first 256 rows in the
// workgroup's registers, wave w rows w, w + 8, ... as 64-column chunks of the
// lower triangle (80 chunks, 160 registers), the last 32 rows in LDS.
constexpr int kResident = 288;
constexpr int kResidentBatches = 4;  // of 64 rows, in registers
constexpr int kResidentTail = kResident - 64 * kResidentBatches;
constexpr int kResidentCols = (kResident + 63) / 64;

// One chunk of R rows of the pass below: element updates, and the column part
// of the product; the row part too unless DIAG, the chunk that holds the
// diagonal, which is kept with both its triangles.
template <bool DIAG, int R, typename Load, typename Store>
__device__ __forceinline__ void resident_chunk(const double (&pvj)[R], const double (&pwj)[R], const double (&vj)[R],
                                               double pv, double pw, double v, double& acc, double (&rs)[8],
                                               Load load, Store store) {
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const double a = fma(-pwj[r], pv, fma(-pvj[r], pw, load(r)));
    store(r, a);
    acc = fma(a, vj[r], acc);
    if constexpr (!DIAG) rs[r] = fma(a, v, rs[r]);
  }
}

// Householder reduction to tridiagonal form on the lower triangle. Step k
// reflects column k below the diagonal; its rank-2 update of the trailing
// block is applied in the next step's single pass over the block, which also
// forms that step's product with the trailing block. nxt holds column k of the
// matrix as the previous pass left it; lv / lw hold v and w of the current and
// the previous step. The reflector vectors go to the upper triangle.
//
// One workgroup per matrix, so a step is bound by its own chain (two workgroup
// sums, three barriers) and by the pass. From memory the pass of the 288 x 288
// block moves 1.2 MB through one CU's L2 port and waits for it in every batch,
// 8.3 us a step; on the chip it is arithmetic alone, 4.9 us (a 288 x 288 matrix
// 2.4 -> 1.4 ms). Larger matrices take the pass from memory until the trailing
// block is that small.
__global__ __launch_bounds__(kEigThreads) void eig_tridiagonal_kernel(int n, int nvec, double* __restrict__ a_all,
                                                                       double* __restrict__ work_all) {
  __shared__ double part[kEigWaves][kEigMaxN];
  __shared__ double lv[2][kEigMaxN], lw[2][kEigMaxN], nxt[kEigMaxN], prow[kEigMaxN];
  __shared__ double tail[kResidentTail][64 * kResidentCols];
  __shared__ double red2[2][kEigWaves];
  __shared__ double lsink[64];
  __shared__ double last;
  const int t = threadIdx.x;
  const int lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  double* A = a_all + (long long)blockIdx.x * n * n;
  double* d = work_all + (long long)blockIdx.x * eig_work_per(n, nvec);
  double* e = d + n;
  double* beta = d + 2 * n;
  const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(A, 0, n * n * 8, 0x00020000);
  for (int i = t; i < n; i += kEigThreads) {
    nxt[i] = A[(long long)i * n];
    lv[1][i] = 0.0;
    lw[1][i] = 0.0;
  }
  __syncthreads();
  const int M = min(n, kResident);
  const int s0 = n - M;
  for (int k = 0; k < s0; ++k) {
    const int m = n - k - 1;
    const int c0 = k + 1;
    const int cur = k & 1;
    double* vv = lv[cur];
    double* ww = lw[cur];
    const double* pv = lv[cur ^ 1];
    const double* pw = lw[cur ^ 1];
    const double pv0 = pv[0], pw0 = pw[0];
    double sq = 0.0;
    if (t < m) {
      const double x = nxt[1 + t] - pv[1 + t] * pw0 - pw[1 + t] * pv0;
      vv[t] = x;
      sq = x * x;
    }
    const double x0 = nxt[1] - pv[1] * pw0 - pw[1] * pv0;
    const double dk = nxt[0] - 2.0 * pv0 * pw0;
    const double ss = wg_sum1(sq, red2[0]);
    double bk, ek, v0;
    reflector(ss, x0, bk, ek, v0);
    if (t == 0) {
      d[k] = dk;
      e[k] = ek;
      beta[k] = bk;
      vv[0] = v0;
    }
    const int boff = (c0 * n + c0) * 8;
    if (m <= 64 * 5)
      tri_pass<5>(rsrc, boff, n, m, wave, lane, pv, pw, vv, v0, nxt, part[wave], prow, lsink);
    else if (m <= 64 * 6)
      tri_pass<6>(rsrc, boff, n, m, wave, lane, pv, pw, vv, v0, nxt, part[wave], prow, lsink);
    else if (m <= 64 * 7)
      tri_pass<7>(rsrc, boff, n, m, wave, lane, pv, pw, vv, v0, nxt, part[wave], prow, lsink);
    else
      tri_pass<8>(rsrc, boff, n, m, wave, lane, pv, pw, vv, v0, nxt, part[wave], prow, lsink);
    __syncthreads();
    double p = 0.0, pdv = 0.0, vi = 0.0;
    if (t < m) {
      double sacc = 0.0;
#pragma unroll
      for (int g = 0; g < kEigWaves; ++g) sacc += part[g][t];
      p = bk * (sacc + prow[t]);
      vi = t == 0 ? v0 : vv[t];
      pdv = p * vi;
      A[(long long)k * n + c0 + t] = vi;  // the reflector vector, row k above the diagonal
    }
    const double K = 0.5 * bk * wg_sum1(pdv, red2[1]);
    if (t < m) ww[t] = p - K * vi;
    __syncthreads();
  }

  // The rest on the chip, rows and columns counted from s0 (the pending v and w are too).
  double val[4 * kResidentBatches * (kResidentBatches + 1)];
#pragma unroll
  for (int b = 0; b < kResidentBatches; ++b)
#pragma unroll
    for (int r = 0; r < 8; ++r)
#pragma unroll
      for (int c = 0; c <= b; ++c) {
        const int j = 64 * b + 8 * r + wave, i = 64 * c + lane;
        const double x = A[(long long)(s0 + min(max(i, j), M - 1)) * n + s0 + min(min(i, j), M - 1)];
        val[4 * b * (b + 1) + r * (b + 1) + c] = j < M && i < M ? x : 0.0;
      }
  for (int r = wave; r < kResidentTail; r += kEigWaves)
    for (int c = 0; c < kResidentCols; ++c) {
      const int j = 64 * kResidentBatches + r, i = 64 * c + lane;
      const double x = A[(long long)(s0 + min(max(i, j), M - 1)) * n + s0 + min(min(i, j), M - 1)];
      tail[r][i] = j < M && i < M ? x : 0.0;
    }
  for (int i = M + t; i < 64 * kResidentCols; i += kEigThreads)  // lanes past the block count as zero
    lv[0][i] = lv[1][i] = lw[0][i] = lw[1][i] = 0.0;
  __syncthreads();
  for (int kk = 0; kk + 2 < M; ++kk) {
    const int c0 = kk + 1;
    const int cur = (s0 + kk) & 1;
    double* vv = lv[cur];
    double* ww = lw[cur];
    const double* pv = lv[cur ^ 1];
    const double* pw = lw[cur ^ 1];
    const double pv0 = pv[kk], pw0 = pw[kk];
    double sq = 0.0;
    if (t < M) {
      const double x = t > kk ? nxt[t] - pv[t] * pw0 - pw[t] * pv0 : 0.0;
      vv[t] = x;
      sq = x * x;
    }
    const double x0 = nxt[c0] - pv[c0] * pw0 - pw[c0] * pv0;
    const double dk = nxt[kk] - 2.0 * pv0 * pw0;
    const double ss = wg_sum1(sq, red2[0]);
    double bk, ek, v0;
    reflector(ss, x0, bk, ek, v0);
    if (t == c0) {  // readers of vv before the next barrier take v0 at c0
      d[s0 + kk] = dk;
      e[s0 + kk] = ek;
      beta[s0 + kk] = bk;
      vv[c0] = v0;
    }
    const int cc = c0 >> 6, cl = c0 & 63;
    double acc[kResidentCols];
#pragma unroll
    for (int c = 0; c < kResidentCols; ++c) acc[c] = 0.0;
    double lpv[kResidentCols], lpw[kResidentCols], lvv[kResidentCols];
#pragma unroll
    for (int c = 0; c < kResidentCols; ++c) {
      lpv[c] = pv[64 * c + lane];
      lpw[c] = pw[64 * c + lane];
      lvv[c] = vv[64 * c + lane];
    }
#pragma unroll
    for (int c = 0; c < kResidentCols; ++c) {
      asm volatile("" : "+v"(lvv[c]));  // loads before the selects
      lvv[c] = 64 * c + lane == c0 ? v0 : lvv[c];
    }
    // v, w and the new v of a batch's rows, from the lanes that hold them.
    auto row_scalars = [&](int b, auto& pvj, auto& pwj, auto& vj) {
      constexpr int R = sizeof(pvj) / sizeof(double);
#pragma unroll
      for (int r = 0; r < R; ++r) {
        pvj[r] = readlane_d(lpv[b], 8 * r + wave);
        pwj[r] = readlane_d(lpw[b], 8 * r + wave);
        vj[r] = readlane_d(lvv[b], 8 * r + wave);
      }
    };
    auto store_sums = [&](const double (&rs)[8], int j0) {
      const double tot = wave_sums8(rs, lane);
      const int j = j0 + (lane & 56) + wave;
      if ((lane & 7) == 0 && j < M) prow[j] = tot;
    };
#pragma unroll
    for (int b = 0; b < kResidentBatches; ++b) {
      if (64 * b + 63 >= c0 && 64 * b < M) {
        double pvj[8], pwj[8], vj[8], rs[8];
        row_scalars(b, pvj, pwj, vj);
#pragma unroll
        for (int r = 0; r < 8; ++r) rs[r] = 0.0;
#pragma unroll
        for (int c = 0; c <= b; ++c) {
          if (64 * c + 63 >= c0) {
            auto load = [&](int r) { return val[4 * b * (b + 1) + r * (b + 1) + c]; };
            auto store = [&](int r, double a) { val[4 * b * (b + 1) + r * (b + 1) + c] = a; };
            if (c == b)
              resident_chunk<true, 8>(pvj, pwj, vj, lpv[c], lpw[c], lvv[c], acc[c], rs, load, store);
            else
              resident_chunk<false, 8>(pvj, pwj, vj, lpv[c], lpw[c], lvv[c], acc[c], rs, load, store);
            if (c == cc && lane == cl) {
#pragma unroll
              for (int r = 0; r < 8; ++r) nxt[64 * b + 8 * r + wave] = load(r);
            }
          }
        }
        if (b > 0 && 64 * b > c0) store_sums(rs, 64 * b);
      }
    }
    if (M > 64 * kResidentBatches) {
      constexpr int R = kResidentTail / kEigWaves, b = kResidentBatches;
      double pvj[R], pwj[R], vj[R], rs[8];
      row_scalars(b, pvj, pwj, vj);
#pragma unroll
      for (int r = 0; r < 8; ++r) rs[r] = 0.0;
#pragma unroll
      for (int c = 0; c <= b; ++c) {
        if (64 * c + 63 >= c0) {
          auto load = [&](int r) { return tail[8 * r + wave][64 * c + lane]; };
          double* here = &tail[wave][64 * c + lane];
          double now[R];
#pragma unroll
          for (int r = 0; r < R; ++r) now[r] = here[8 * r * 64 * kResidentCols];
          auto get = [&](int r) { return now[r]; };
          auto store = [&](int r, double a) { here[8 * r * 64 * kResidentCols] = a; };
          if (c == b)
            resident_chunk<true, R>(pvj, pwj, vj, lpv[c], lpw[c], lvv[c], acc[c], rs, get, store);
          else
            resident_chunk<false, R>(pvj, pwj, vj, lpv[c], lpw[c], lvv[c], acc[c], rs, get, store);
          if (c == cc && lane == cl) {
#pragma unroll
            for (int r = 0; r < R; ++r) nxt[64 * b + 8 * r + wave] = load(r);
          }
        }
      }
      if (64 * b > c0) store_sums(rs, 64 * b);
    }
#pragma unroll
    for (int c = 0; c < kResidentCols; ++c)
      if (64 * c + lane < M) part[wave][64 * c + lane] = acc[c];
    __syncthreads();
    double p = 0.0, pdv = 0.0, vi = 0.0;
    const bool mine = t > kk && t < M;
    if (mine) {
      double sacc = 0.0;
#pragma unroll
      for (int g = 0; g < kEigWaves; ++g) sacc += part[g][t];
      p = bk * (t >= 64 && (t & ~63) > c0 ? sacc + prow[t] : sacc);
      vi = t == c0 ? v0 : vv[t];
      pdv = p * vi;
      A[(long long)(s0 + kk) * n + s0 + t] = vi;  // the reflector vector, above the diagonal
    }
    const double K = 0.5 * bk * wg_sum1(pdv, red2[1]);
    if (t < M) ww[t] = mine ? p - K * vi : 0.0;
    __syncthreads();
  }
#pragma unroll
  for (int b = 0; b < kResidentBatches; ++b)
#pragma unroll
    for (int r = 0; r < 8; ++r)
      if (64 * b + 8 * r + wave == M - 1 && lane == ((M - 1) & 63)) last = val[4 * b * (b + 1) + r * (b + 1) + b];
  if (M > 64 * kResidentBatches && t == 0) last = tail[M - 1 - 64 * kResidentBatches][M - 1];
  __syncthreads();
  if (t == 0) {
    if (n >= 3) {
      const int cur = (n - 3) & 1;
      const double v0 = lv[cur][M - 2], v1 = lv[cur][M - 1], w0 = lw[cur][M - 2], w1 = lw[cur][M - 1];
      d[n - 2] = nxt[M - 2] - 2.0 * v0 * w0;
      e[n - 2] = nxt[M - 1] - v1 * w0 - w1 * v0;
      d[n - 1] = last - 2.0 * v1 * w1;
    } else if (n == 2) {
      d[0] = A[0];
      e[0] = A[2];
      d[1] = A[3];
    } else {
      d[0] = A[0];
    }
    if (n >= 2) beta[n - 2] = 0.0;
    e[n - 1] = 0.0;
    beta[n - 1] = 0.0;
  }
}

__global__ void eig_no_vectors_kernel(int count, int* __restrict__ info) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < count) info[i] = 0;
}

// Gershgorin interval, |T| and the pivot guard of the tridiagonal matrix, by every wave for itself.
struct TriBounds {
  double lo, hi, tnorm, pivmin;
};
__device__ TriBounds tri_bounds(const double* d, const double* e, int n, int lane) {
  double lo = DBL_MAX, hi = -DBL_MAX, emax = 0.0;
  for (int i = lane; i < n; i += 64) {
    const double ei = i + 1 < n ? e[i] : 0.0, r = (i > 0 ? fabs(e[i - 1]) : 0.0) + fabs(ei);
    lo = fmin(lo, d[i] - r);
    hi = fmax(hi, d[i] + r);
    emax = fmax(emax, ei * ei);
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    lo = fmin(lo, __shfl_xor(lo, o));
    hi = fmax(hi, __shfl_xor(hi, o));
    emax = fmax(emax, __shfl_xor(emax, o));
  }
  const double tnorm = fmax(fabs(lo), fabs(hi));
  return TriBounds{lo - 2.0 * DBL_EPSILON * tnorm - DBL_MIN, hi + 2.0 * DBL_EPSILON * tnorm + DBL_MIN,
                   fmax(tnorm, DBL_MIN), DBL_MIN * fmax(1.0, emax)};
}

// The nvec lowest eigenvalues by multisection, LANES lanes each, which count at
// LANES points of the interval: it shrinks LANES + 1 times per round. Bound by
// the chain of the Sturm recurrence, n steps a round, while the waves find
// SIMDs of their own: a wave per value then takes the fewest rounds (about ten;
// 60 values of a 288 x 288 matrix: 0.13 ms). Past that by the operations, of
// which eight lanes and 17 rounds take a quarter (256 matrices of 400 x 400, 80
// values: 1.95 ms by whole waves). d and e^2 come from LDS eight steps ahead.
constexpr int kValueWaves = 4;
constexpr long long kValueFill = 4096;  // values from which eight lanes take one
template <int LANES>
__global__ __launch_bounds__(64 * kValueWaves) void eig_values_kernel(int n, int nvec, double* __restrict__ w_all,
                                                                       const double* __restrict__ work_all) {
  constexpr int VALUES = 64 / LANES;  // of a wave
  __shared__ double2 t2[kEigMaxN + 8];  // (d_i, e_{i-1}^2)
  const int lane = threadIdx.x & 63;
  const int parts = (nvec + kValueWaves * VALUES - 1) / (kValueWaves * VALUES);
  const int matrix = blockIdx.x / parts, part = blockIdx.x % parts;
  const double* d = work_all + (long long)matrix * eig_work_per(n, nvec);
  const double* e = d + n;
  for (int i = threadIdx.x; i < n + 8; i += 64 * kValueWaves) {
    const double ep = i > 0 && i < n ? e[i - 1] : 0.0;
    t2[i] = make_double2(i < n ? d[i] : 0.0, ep * ep);
  }
  __syncthreads();
  const TriBounds tb = tri_bounds(d, e, n, lane);
  const int j = (part * kValueWaves + (threadIdx.x >> 6)) * VALUES + lane / LANES;
  if (j >= nvec) return;
  const int point = lane % LANES, group = lane - point;
  constexpr double sections = LANES + 1;
  const double tol = 0.5 * DBL_EPSILON * tb.tnorm;
  double a = tb.lo, b = tb.hi;
  for (int it = 0; it < 200; ++it) {
    if (b - a <= 2.0 * DBL_EPSILON * fmax(fabs(a), fabs(b)) + tol) break;
    const double x = a + (b - a) * (double)(point + 1) / sections;
    // count of negative pivots; the first step's e^2 is 0, so its previous pivot does not matter
    int cnt = 0;
    double q = 1.0;
    for (int i0 = 0; i0 < n; i0 += 8) {
      double2 v[8];
#pragma unroll
      for (int s = 0; s < 8; ++s) v[s] = t2[i0 + s];
#pragma unroll
      for (int s = 0; s < 8; ++s) {
        q = (v[s].x - x) - v[s].y * recip(q);
        if (fabs(q) < tb.pivmin) q = -tb.pivmin;
        cnt += i0 + s < n && q < 0.0;
      }
    }
    // The first point with count > j bounds the eigenvalue from above. (The lanes of a value are in
    // the loop together; others may have left it.)
    const unsigned long long above = __ballot(cnt > j) >> group & (~0ull >> (64 - LANES));
    const int sf = above ? __builtin_ctzll(above) : LANES;
    const double na = sf == 0 ? a : a + (b - a) * (double)sf / sections;
    const double nb = sf == LANES ? b : a + (b - a) * (double)(sf + 1) / sections;
    a = na;
    b = nb;
  }
  if (point == 0) w_all[(long long)matrix * n + j] = 0.5 * (a + b);
}

// Eigenvectors of T, one lane each: the shifts of equal eigenvalues are separated by 10 eps |T|
// (so that their iterations differ), two inverse iterations from a seeded start with a partially
// pivoted LU of T - lambda I. A workgroup is one wave with as many vectors as their factors leave
// room for in LDS, [n][vectors]; every recurrence over n is a serial chain, and from LDS it waits
// 0.1 us where the same factors in memory cost 0.5 us for each eight steps. U's superdiagonals
// are stored too unless COMPACT, which forms them again from T, the swaps and the multipliers: that
// adds to the chain (12 matrices of 288 x 288, 60 vectors: 0.08 ms of 1.92 in the whole solver), but
// two fifths of the vectors in flight were the time of a batch that fills the chip (256 matrices of
// 400 x 400, 80 vectors: 3.4 ms of 16.4).
template <bool COMPACT>
constexpr int kVectorBytes = COMPACT ? 25 : 41;  // LDS per vector and row: doubles and the swap flag
constexpr int kVectorLds = 48 * 1024;
template <bool COMPACT>
__global__ __launch_bounds__(64) void eig_vectors_kernel(int n, int nvec, int per, const double* __restrict__ w_all,
                                                          double* __restrict__ work_all) {
  extern __shared__ double vec_lds[];
  __shared__ double ld[kEigMaxN], le[kEigMaxN], lam_all[kEigMaxN];
  const int lane = threadIdx.x;
  const int parts = (nvec + per - 1) / per;
  const int matrix = blockIdx.x / parts, part = blockIdx.x % parts;
  const double* d = work_all + (long long)matrix * eig_work_per(n, nvec);
  const double* e = d + n;
  double* Y = work_all + (long long)matrix * eig_work_per(n, nvec) + 3 * n;  // [nvec][n]
  const double* w = w_all + (long long)matrix * n;
  const int j0 = part * per;
  const int jn = min(per, nvec - j0);
  for (int i = lane; i < n; i += 64) {
    ld[i] = d[i];
    le[i] = i + 1 < n ? e[i] : 0.0;
  }
  for (int i = lane; i < j0 + jn; i += 64) lam_all[i] = w[i];
  const double tnorm = tri_bounds(d, e, n, lane).tnorm;
  __syncthreads();
  if (lane == 0) {
    double prev = lam_all[0];
    for (int j = 1; j < j0 + jn; ++j) {
      double lam = lam_all[j];
      if (lam - prev < 10.0 * DBL_EPSILON * tnorm) lam = prev + 10.0 * DBL_EPSILON * tnorm;
      lam_all[j] = lam;
      prev = lam;
    }
  }
  __syncthreads();
  double* inv = vec_lds;  // 1 / pivot
  double* mul = inv + (long long)n * per;
  double* yv = mul + (long long)n * per;
  double* u1 = yv + (long long)n * per;  // U's two superdiagonals
  double* u2 = u1 + (long long)n * per;
  unsigned char* swp = (unsigned char*)(COMPACT ? u1 : u2 + (long long)n * per);
  if (lane < jn) {
    const int j = j0 + lane;
    const double lam = lam_all[j];
    const double tiny = DBL_EPSILON * tnorm;
    double p0 = ld[0] - lam, p1 = n > 1 ? le[0] : 0.0;
    for (int k = 0; k + 1 < n; ++k) {
      const double c = le[k];                                              // below the diagonal
      const double a1 = ld[k + 1] - lam, b1 = k + 2 < n ? le[k + 1] : 0.0;  // the next row
      const bool swap = fabs(c) > fabs(p0);
      if (!swap && fabs(p0) < tiny) p0 = p0 < 0.0 ? -tiny : tiny;
      const double piv = swap ? c : p0, rest = swap ? p0 : c;
      const double mult = rest / piv;
      const int at = k * per + lane;
      inv[at] = 1.0 / piv;
      if constexpr (!COMPACT) {
        u1[at] = swap ? a1 : p1;
        u2[at] = swap ? b1 : 0.0;
      }
      mul[at] = mult;
      swp[at] = swap;
      p0 = swap ? p1 - mult * a1 : a1 - mult * p1;
      p1 = swap ? -mult * b1 : b1;
    }
    if (fabs(p0) < tiny) p0 = p0 < 0.0 ? -tiny : tiny;
    inv[(n - 1) * per + lane] = 1.0 / p0;
    swp[(n - 1) * per + lane] = false;  // no row below to swap with
    if constexpr (!COMPACT) {
      u1[(n - 1) * per + lane] = 0.0;
      u2[(n - 1) * per + lane] = 0.0;
    }
    double scale = 1.0;
#pragma unroll
    for (int iter = 0; iter < 2; ++iter) {
      // Forward elimination of the right-hand side (the seeded start, or the previous iterate
      // times scale), then back substitution; scale makes the result unit length.
      double carry = iter == 0 ? start_entry(j, 0) : yv[lane] * scale;
      for (int k0 = 0; k0 + 1 < n; k0 += 8) {
        double lmv[8], yn[8];
        bool sw[8];
#pragma unroll
        for (int s = 0; s < 8; ++s) {
          const int k = min(k0 + s, n - 2);
          lmv[s] = mul[k * per + lane];
          sw[s] = swp[k * per + lane];
          yn[s] = iter == 0 ? start_entry(j, k + 1) : yv[(k + 1) * per + lane] * scale;
        }
#pragma unroll
        for (int s = 0; s < 8; ++s) {
          const int k = k0 + s;
          if (k + 1 < n) {
            const double yk = sw[s] ? yn[s] : carry, yk1 = sw[s] ? carry : yn[s];
            yv[k * per + lane] = yk;
            carry = yk1 - lmv[s] * yk;
          }
        }
      }
      yv[(n - 1) * per + lane] = carry;
      double nrm = 0.0, x1 = 0.0, x2 = 0.0;  // x_{i+1}, x_{i+2}
      for (int i0 = n - 1; i0 >= 0; i0 -= 8) {
        double yy[8], a1[8], a2[8], rr[8];
        bool sw = COMPACT && swp[i0 * per + lane];
#pragma unroll
        for (int s = 0; s < 8; ++s) {
          const int i = max(i0 - s, 0), at = i * per + lane, before = max(i - 1, 0) * per + lane;
          yy[s] = yv[at];
          rr[s] = inv[at];
          if constexpr (!COMPACT) {
            a1[s] = u1[at];
            a2[s] = u2[at];
            continue;
          }
          // Row i of U: the row below where they were swapped, else row i of T less its elimination
          // (which touches its superdiagonal only if the row it came from had been swapped). le[n - 1]
          // is 0.
          const bool swb = i > 0 && swp[before];
          const double kept = swb ? -mul[before] * le[i] : le[i];
          a1[s] = sw ? ld[min(i + 1, n - 1)] - lam : kept;
          a2[s] = sw ? le[min(i + 1, n - 1)] : 0.0;
          sw = swb;
        }
#pragma unroll
        for (int s = 0; s < 8; ++s) {
          const int i = i0 - s;
          if (i >= 0) {
            const double xi = (yy[s] - a1[s] * x1 - a2[s] * x2) * rr[s];
            yv[i * per + lane] = xi;
            nrm += xi * xi;
            x2 = x1;
            x1 = xi;
          }
        }
      }
      scale = nrm > 0.0 ? 1.0 / sqrt(nrm) : 0.0;
    }
    lam_all[lane] = scale;  // the eigenvalues are in registers by now
  }
  __syncthreads();
  for (int q = 0; q < jn; ++q)
    for (int i = lane; i < n; i += 64) Y[(long long)(j0 + q) * n + i] = yv[i * per + q] * lam_all[q];
}

// Orthonormalisation of the vectors, one workgroup per matrix.
__global__ __launch_bounds__(kEigThreads) void eig_orthonormal_kernel(int n, int nvec, double* __restrict__ work_all) {
  __shared__ double part[kEigMaxN];
  __shared__ double gm[kEigRegVecs * kGs], li[kEigRegVecs * kGs], rows[2][2 * kEigRegVecs];
  __shared__ double red[kEigWaves];
  const int t = threadIdx.x;
  const int lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  double* Y = work_all + (long long)blockIdx.x * eig_work_per(n, nvec) + 3 * n;  // [nvec][n]
  if (nvec <= kEigRegVecs) {
    switch ((n + 63) >> 6) {
      case 1: orthonormalise<1>(Y, gm, li, rows, n, nvec, wave, lane); break;
      case 2: orthonormalise<2>(Y, gm, li, rows, n, nvec, wave, lane); break;
      case 3: orthonormalise<3>(Y, gm, li, rows, n, nvec, wave, lane); break;
      case 4: orthonormalise<4>(Y, gm, li, rows, n, nvec, wave, lane); break;
      case 5: orthonormalise<5>(Y, gm, li, rows, n, nvec, wave, lane); break;
      case 6: orthonormalise<6>(Y, gm, li, rows, n, nvec, wave, lane); break;
      case 7: orthonormalise<7>(Y, gm, li, rows, n, nvec, wave, lane); break;
      default: orthonormalise<8>(Y, gm, li, rows, n, nvec, wave, lane); break;
    }
  } else {
    // Gram-Schmidt in order: vector j minus its components along vectors 0 .. j - 1 (dots by
    // waves, one earlier vector each), twice, then unit length.
    for (int j = 1; j < nvec; ++j) {
      double* y = Y + (long long)j * n;
      for (int pass = 0; pass < 2; ++pass) {
        for (int k = wave; k < j; k += kEigWaves) {
          const double* z = Y + (long long)k * n;
          double sdot = 0.0;
          for (int i = lane; i < n; i += 64) sdot += z[i] * y[i];
#pragma unroll
          for (int o = 32; o >= 1; o >>= 1) sdot += __shfl_xor(sdot, o);
          if (lane == 0) part[k] = sdot;
        }
        __syncthreads();
        for (int i = t; i < n; i += kEigThreads) {
          double v = y[i];
          for (int k = 0; k < j; ++k) v -= part[k] * Y[(long long)k * n + i];
          y[i] = v;
        }
        __syncthreads();
      }
      double sq = 0.0;
      for (int i = t; i < n; i += kEigThreads) sq += y[i] * y[i];
      const double nrm = wg_sum(sq, red);
      const double inv = nrm > 0.0 ? 1.0 / sqrt(nrm) : 0.0;
      for (int i = t; i < n; i += kEigThreads) y[i] *= inv;
      __syncthreads();
    }
  }
}

}  // namespace

extern "C" {

long long hfjk_eigh_lowest_batched_work(int n, int count, int nvec) {
  if (n < 1 || count < 0 || nvec < 0) return 0;
  return (long long)count * eig_work_per(n, nvec);
}

int hfjk_eigh_lowest_batched(hfjk_ctx* ctx, int n, int count, int nvec, double* a, double* w, double* work, int* info,
                             void* stream) {
  if (ctx == nullptr) {
    hfjk_internal_set_error("null context");
    return HFJK_ERR_INPUT;
  }
  if (n < 1 || n > kEigMaxN || count < 0 || nvec < 0 || nvec > n) {
    hfjk_internal_set_error(("hfjk_eigh_lowest_batched needs 1 <= n <= " + std::to_string(kEigMaxN) +
                             ", count >= 0 and 0 <= nvec <= n")
                                .c_str());
    return HFJK_ERR_INPUT;
  }
  if (count == 0) return HFJK_OK;
  if (a == nullptr || w == nullptr || work == nullptr || info == nullptr) {
    hfjk_internal_set_error("hfjk_eigh_lowest_batched needs device buffers");
    return HFJK_ERR_INPUT;
  }
  hipError_t err = hipSetDevice(ctx->device);
  if (err == hipSuccess) {
    if (nvec == 0) {
      hipLaunchKernelGGL(eig_no_vectors_kernel, dim3((unsigned)((count + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
                         count, info);
      err = hipGetLastError();
    }
    const auto per_wave = [&](int bytes) { return std::max(1, std::min(std::min(nvec, 64), kVectorLds / (bytes * n))); };
    const int per = nvec > 0 ? per_wave(kVectorBytes<false>) : 1, compact = nvec > 0 ? per_wave(kVectorBytes<true>) : 1;
    // A grid holds less than 2^32 work-items and the values take a wave per vector: 2^31 / 64 vectors at a
    // time (a multiple of 8 matrices, the XCDs' turn).
    const int most = std::max(8, (1 << 25) / std::max(nvec, 8) & ~7);
    for (int first = 0; nvec > 0 && first < count && err == hipSuccess; first += most) {
      const int now = std::min(most, count - first);
      double* ai = a + (long long)first * n * n;
      double* wi = w + (long long)first * n;
      double* ti = work + first * eig_work_per(n, nvec);
      const hipStream_t s = (hipStream_t)stream;
      hipLaunchKernelGGL(eig_tridiagonal_kernel, dim3((unsigned)now), dim3(kEigThreads), 0, s, n, nvec, ai, ti);
      if ((long long)now * nvec < kValueFill)
        hipLaunchKernelGGL(eig_values_kernel<64>, dim3((unsigned)(now * ((nvec + kValueWaves - 1) / kValueWaves))),
                           dim3(64 * kValueWaves), 0, s, n, nvec, wi, ti);
      else
        hipLaunchKernelGGL(eig_values_kernel<8>, dim3((unsigned)(now * ((nvec + 8 * kValueWaves - 1) / (8 * kValueWaves)))),
                           dim3(64 * kValueWaves), 0, s, n, nvec, wi, ti);
      // Two rounds of the three workgroups that a CU holds: past that a batch is bound by the vectors
      // in flight (64 matrices of 288 x 288 with 60 vectors lose 0.1 ms to COMPACT, 300 gain 0.4).
      if ((long long)now * nvec < 6LL * ctx->cus * per)
        hipLaunchKernelGGL(eig_vectors_kernel<false>, dim3((unsigned)(now * ((nvec + per - 1) / per))), dim3(64),
                           (size_t)kVectorBytes<false> * n * per, s, n, nvec, per, wi, ti);
      else
        hipLaunchKernelGGL(eig_vectors_kernel<true>, dim3((unsigned)(now * ((nvec + compact - 1) / compact))), dim3(64),
                           (size_t)kVectorBytes<true> * n * compact, s, n, nvec, compact, wi, ti);
      hipLaunchKernelGGL(eig_orthonormal_kernel, dim3((unsigned)now), dim3(kEigThreads), 0, s, n, nvec, ti);
      hipLaunchKernelGGL(eig_back_kernel, dim3((unsigned)((now + 7) / 8 * 8 * ((nvec + 3) / 4))), dim3(64), 0, s, n,
                         nvec, now, ai, ti);
      hipLaunchKernelGGL(eig_store_kernel, dim3((unsigned)now), dim3(kEigThreads), 0, s, n, nvec, ai, ti, info + first);
      err = hipGetLastError();
    }
  }
  if (err != hipSuccess) {
    hfjk_internal_set_error((std::string("eigensolver launch: ") + hipGetErrorString(err)).c_str());
    return HFJK_ERR_HIP;
  }
  return HFJK_OK;
}

}  // extern "C"
