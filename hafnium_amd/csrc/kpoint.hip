// k-point DF-J/K kernels (FP64, complex values as interleaved double2).
//
// Coulomb: the charges c_P = sum_k w_k sum_xw conj(B_k[P][x][w]) D_k[x][w]
// over the zero-transfer blocks (one workgroup per (k, P), a fixed-order
// reduction), then J_k = sum_P s_k[P] c_P B_k[P] streamed once over the
// blocks (one thread per matrix element, coalesced over elements).
//
// Exchange of one transfer block B = B[k1, k2] (general complex [naux][n][n])
// against a Hermitian D(k2) = V diag(l) V^dagger: with C = V |l|^1/2 sqrt(w)
// ([n][r] complex) the realified operands
//   Bh[P] = [[Re B, -Im B], [Im B, Re B]]   ([2n][2n] real),
//   Ch    = [Re C; Im C]                    ([2n][r] real)
// give Xh[P] = Bh[P] Ch = [Re X; Im X] for X = B[P] C, with no redundant
// products. The existing FP64 half-transform (direct-LDS ring over a full
// row-major B) and the signed SYRK then form
//   Kh = sum_P s[P] Xh[P] diag(sign l) Xh[P]^T ([2n][2n] symmetric),
// and K += (Kh_TL + Kh_BR) + i (Kh_BL - Kh_TR) is the block's
// sum_P s[P] B[P] D B[P]^dagger. Per-aux signs s[P] scale the SYRK's second
// operand per aux function.
#include <algorithm>

#include "hfjk_internal.h"

namespace hfjk {
namespace {

__device__ __forceinline__ double2 cmul(double2 a, double2 b) {
  return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}

// Fixed-order sum of one value per thread over a 256-thread workgroup.
__device__ __forceinline__ double block_sum(double v, double* red) {
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  const double out = red[0] + red[1] + red[2] + red[3];
  __syncthreads();
  return out;
}

// inner[k][P] = w[k] sum_xw conj(B_k[P][xw]) D_k[xw]; one workgroup per (k, P).
__global__ __launch_bounds__(kThreads) void kp_inner_kernel(const double2* __restrict__ b, long long kstride,
                                                            int naux, long long nn, const double2* __restrict__ d,
                                                            const double* __restrict__ w, double2* __restrict__ inner) {
  __shared__ double red[4];
  const int k = blockIdx.x / naux;
  const int p = blockIdx.x % naux;
  const double2* bp = b + (long long)k * kstride + (long long)p * nn;
  const double2* dk = d + (long long)k * nn;
  double re = 0.0, im = 0.0;
  for (long long i = threadIdx.x; i < nn; i += kThreads) {
    const double2 x = bp[i], y = dk[i];
    re += x.x * y.x + x.y * y.y;
    im += x.x * y.y - x.y * y.x;
  }
  re = block_sum(re, red);
  im = block_sum(im, red);
  if (threadIdx.x == 0) inner[(long long)k * naux + p] = make_double2(w[k] * re, w[k] * im);
}

// charges[P] = sum_k inner[k][P], k in order.
__global__ __launch_bounds__(kThreads) void kp_charges_kernel(const double2* __restrict__ inner, int nk, int naux,
                                                              double2* __restrict__ charges) {
  const int p = blockIdx.x * kThreads + threadIdx.x;
  if (p >= naux) return;
  double2 acc = make_double2(0.0, 0.0);
  for (int k = 0; k < nk; ++k) {
    const double2 v = inner[(long long)k * naux + p];
    acc.x += v.x;
    acc.y += v.y;
  }
  charges[p] = acc;
}

// J_k[xw] = sum_P s_k[P] charges[P] B_k[P][xw]; grid (element blocks, nk): 32
// elements per workgroup, eight thread groups sharing the aux functions
// (combined in a fixed order; one thread per element walking all of them left
// most of the device idle: 59 us at nao 28, naux 212, eight k-points).
constexpr int kCoulombElems = 32;

__global__ __launch_bounds__(kThreads) void kp_coulomb_kernel(const double2* __restrict__ b, long long kstride,
                                                              int naux, long long nn, const double* __restrict__ sig,
                                                              long long sig_kstride, const double2* __restrict__ charges,
                                                              double2* __restrict__ j) {
  constexpr int kParts = kThreads / kCoulombElems;
  __shared__ double2 red[kParts][kCoulombElems];
  const int k = blockIdx.y;
  const double2* bk = b + (long long)k * kstride;
  const double* sk = sig + (long long)k * sig_kstride;
  const int e = threadIdx.x % kCoulombElems, part = threadIdx.x / kCoulombElems;
  for (long long i0 = (long long)blockIdx.x * kCoulombElems; i0 < nn; i0 += (long long)gridDim.x * kCoulombElems) {
    const long long i = i0 + e;
    double2 acc = make_double2(0.0, 0.0);
    if (i < nn) {
#pragma unroll 4
      for (int p = part; p < naux; p += kParts) {
        const double2 c = charges[p];
        const double s = sk[p];
        const double2 v = cmul(make_double2(s * c.x, s * c.y), bk[(long long)p * nn + i]);
        acc.x += v.x;
        acc.y += v.y;
      }
    }
    red[part][e] = acc;
    __syncthreads();
    if (part == 0 && i < nn) {
      for (int q = 1; q < kParts; ++q) {
        acc.x += red[q][e].x;
        acc.y += red[q][e].y;
      }
      j[(long long)k * nn + i] = acc;
    }
    __syncthreads();
  }
}

// Bh[P][r][c] ([npad2][npad2], zero past 2n) of a complex [naux][n][n] block.
__global__ __launch_bounds__(kThreads) void kp_realify_kernel(const double2* __restrict__ b, int naux, int n,
                                                              int npad2, double* __restrict__ out) {
  const long long plane = (long long)npad2 * npad2;
  const long long total = (long long)naux * plane;
  for (long long idx = (long long)blockIdx.x * kThreads + threadIdx.x; idx < total;
       idx += (long long)gridDim.x * kThreads) {
    const long long p = idx / plane;
    const int r = (int)((idx % plane) / npad2);
    const int c = (int)(idx % npad2);
    double v = 0.0;
    if (r < 2 * n && c < 2 * n) {
      const int rr = r < n ? r : r - n, cc = c < n ? c : c - n;
      const double2 z = b[(p * n + rr) * n + cc];
      v = (r < n) == (c < n) ? z.x : (r < n ? -z.y : z.y);
    }
    out[idx] = v;
  }
}

// Ch^T [ldo][npad2] and the column signs [ldo] from the eigenpairs of the
// column-major view of a Hermitian row-major D (that view is conj(D), so its
// eigenvectors u give D's as conj(u)). Columns: the nneg most negative then
// the npos most positive eigenvalues (ascending order in w); scale
// sqrt(weight |l|); zero past r = nneg + npos and past 2n.
__global__ __launch_bounds__(kThreads) void kp_factor_kernel(const double2* __restrict__ u, const double* __restrict__ w,
                                                             int n, int nneg, int npos, double weight, int npad2,
                                                             int ldo, double* __restrict__ ct, double* __restrict__ sg) {
  const long long total = (long long)ldo * npad2;
  const int r = nneg + npos;
  for (long long idx = (long long)blockIdx.x * kThreads + threadIdx.x; idx < total;
       idx += (long long)gridDim.x * kThreads) {
    const int i = (int)(idx / npad2);
    const int k = (int)(idx % npad2);
    double v = 0.0;
    if (i < r && k < 2 * n) {
      const int jj = i < nneg ? i : n - npos + (i - nneg);
      const double scale = sqrt(weight * fabs(w[jj]));
      const double2 z = u[(long long)jj * n + (k < n ? k : k - n)];
      v = k < n ? scale * z.x : -scale * z.y;
    }
    ct[idx] = v;
    if (k == 0) sg[i] = i < nneg ? -1.0 : 1.0;
  }
}

// K[u][v] (+)= (Kh[u][v] + Kh[n+u][n+v]) + i (Kh[n+u][v] - Kh[u][n+v]); Kh is [2n][2n].
__global__ __launch_bounds__(kThreads) void kp_fold_kernel(const double* __restrict__ kh, int n, int accumulate,
                                                           double2* __restrict__ k) {
  const long long nn = (long long)n * n;
  const long long m = 2LL * n;
  for (long long idx = (long long)blockIdx.x * kThreads + threadIdx.x; idx < nn;
       idx += (long long)gridDim.x * kThreads) {
    const long long u = idx / n, v = idx % n;
    const double re = kh[u * m + v] + kh[(n + u) * m + n + v];
    const double im = kh[(n + u) * m + v] - kh[u * m + n + v];
    if (accumulate) {
      const double2 old = k[idx];
      k[idx] = make_double2(old.x + re, old.y + im);
    } else {
      k[idx] = make_double2(re, im);
    }
  }
}

// c (+)= alpha a b for complex row-major [n][n], one triple per blockIdx.y; one thread per output element.
__global__ __launch_bounds__(kThreads) void kp_zgemm_kernel(const double2* __restrict__ a, const double2* __restrict__ b,
                                                            int n, double alpha, int accumulate,
                                                            double2* __restrict__ c) {
  const long long nn = (long long)n * n;
  a += blockIdx.y * nn;
  b += blockIdx.y * nn;
  c += blockIdx.y * nn;
  for (long long idx = (long long)blockIdx.x * kThreads + threadIdx.x; idx < nn;
       idx += (long long)gridDim.x * kThreads) {
    const long long r = idx / n, col = idx % n;
    double2 acc = make_double2(0.0, 0.0);
    for (int q = 0; q < n; ++q) {
      const double2 v = cmul(a[r * n + q], b[(long long)q * n + col]);
      acc.x += v.x;
      acc.y += v.y;
    }
    acc.x *= alpha;
    acc.y *= alpha;
    if (accumulate) {
      const double2 old = c[idx];
      acc.x += old.x;
      acc.y += old.y;
    }
    c[idx] = acc;
  }
}

// Pivoted Cholesky of every k's positive semidefinite density, D = L L^H, one
// workgroup per k (one launch for all columns of all k instead of zheevd's
// hundreds of small kernels per k, 0.55 ms each): column c takes the largest
// remaining diagonal p (ties: lowest index), L[:, c] = (D[:, p] - sum_{j<c}
// L[:, j] conj(L[p][j])) / sqrt(d_p). Bound by the latency of a column.
constexpr int kCholThreads = 512;

__global__ __launch_bounds__(kCholThreads) void kp_cholesky_kernel(const double2* __restrict__ density, int n,
                                                                   double2* __restrict__ lmat,
                                                                   double* __restrict__ diag_all,
                                                                   KpState* __restrict__ state) {
  __shared__ double wval[kCholThreads / 64];
  __shared__ int widx[kCholThreads / 64];
  __shared__ double s_best;
  __shared__ int s_at;
  __shared__ double2 prow[kCholThreads];  // conj(L[p][j0 .. j0 + kCholThreads))
  const long long nn = (long long)n * n;
  const double2* d = density + blockIdx.x * nn;
  double2* l = lmat + blockIdx.x * nn;
  double* diag = diag_all + (long long)blockIdx.x * n;
  const int t = threadIdx.x;
  for (int i = t; i < n; i += kCholThreads) diag[i] = d[(long long)i * n + i].x;
  double cut = 0.0;
  int rank = n;
  for (int c = 0; c <= n; ++c) {
    __syncthreads();  // diag is written
    double best = -1.0;
    int at = -1;
    for (int i = t; i < n; i += kCholThreads)
      if (diag[i] > best) {
        best = diag[i];
        at = i;
      }
    for (int off = 32; off > 0; off >>= 1) {
      const double ov = __shfl_xor(best, off);
      const int oi = __shfl_xor(at, off);
      if (ov > best || (ov == best && oi >= 0 && (at < 0 || oi < at))) {
        best = ov;
        at = oi;
      }
    }
    if ((t & 63) == 0) {
      wval[t >> 6] = best;
      widx[t >> 6] = at;
    }
    __syncthreads();
    if (t == 0) {
      for (int w = 1; w < kCholThreads / 64; ++w)
        if (wval[w] > best || (wval[w] == best && widx[w] >= 0 && (at < 0 || widx[w] < at))) {
          best = wval[w];
          at = widx[w];
        }
      s_best = best;
      s_at = at;
    }
    __syncthreads();
    const double piv = s_best;
    const int p = s_at;
    if (c == 0) cut = 1e-14 * piv;
    if (c == n || p < 0 || !(piv > cut)) {
      rank = c;
      break;
    }
    const double inv = 1.0 / sqrt(piv);
    // Rows in strides of the workgroup; the pivot's row of L through LDS.
    for (int i0 = 0; i0 < n; i0 += kCholThreads) {
      const int i = i0 + t;
      double2 v = make_double2(0.0, 0.0);
      if (i < n) v = d[(long long)i * n + p];
      for (int j0 = 0; j0 < c; j0 += kCholThreads) {
        __syncthreads();
        if (j0 + t < c) {
          const double2 q = l[(long long)(j0 + t) * n + p];
          prow[t] = make_double2(q.x, -q.y);
        }
        __syncthreads();
        const int top = min(kCholThreads, c - j0);
        if (i < n) {
#pragma unroll 4
          for (int j = 0; j < top; ++j) {
            const double2 m = cmul(l[(long long)(j0 + j) * n + i], prow[j]);
            v.x -= m.x;
            v.y -= m.y;
          }
        }
      }
      if (i < n) {
        v.x *= inv;
        v.y *= inv;
        l[(long long)c * n + i] = v;
        diag[i] = i == p ? 0.0 : diag[i] - (v.x * v.x + v.y * v.y);
      }
    }
  }
  if (t == 0) state[blockIdx.x].rank = rank;
}

// Per k: max |D - D^H|, max |D| and the largest row sum of |D - L L^H|, which
// bounds its largest eigenvalue (atomic max of bits). A workgroup per row, so
// that a thread's chain is one pass over the rank.
__global__ __launch_bounds__(kThreads) void kp_residual_kernel(const double2* __restrict__ density, int n,
                                                               const double2* __restrict__ lmat,
                                                               KpState* __restrict__ state) {
  __shared__ double part[kThreads / 64];
  const long long nn = (long long)n * n;
  const double2* d = density + blockIdx.y * nn;
  const double2* l = lmat + blockIdx.y * nn;
  KpState* st = state + blockIdx.y;
  const int rank = st->rank;
  double asym = 0.0, mag = 0.0, worst = 0.0;
  for (int r = blockIdx.x; r < n; r += gridDim.x) {
    double sum = 0.0;
    for (int c = threadIdx.x; c < n; c += kThreads) {
      double2 a = d[(long long)r * n + c];
      const double2 t = d[(long long)c * n + r];
      asym = fmax(asym, hypot(a.x - t.x, a.y + t.y));
      mag = fmax(mag, hypot(a.x, a.y));
#pragma unroll 4
      for (int j = 0; j < rank; ++j) {
        const double2 u = l[(long long)j * n + r], v = l[(long long)j * n + c];
        const double2 m = cmul(u, make_double2(v.x, -v.y));
        a.x -= m.x;
        a.y -= m.y;
      }
      sum += fabs(a.x) + fabs(a.y);
    }
    for (int off = 32; off > 0; off >>= 1) sum += __shfl_xor(sum, off);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = sum;
    __syncthreads();
    sum = (part[0] + part[1]) + (part[2] + part[3]);
    // Not fmax, which would drop a NaN: a NaN must fail the host's test.
    worst = sum > worst || sum != sum ? sum : worst;
    __syncthreads();
  }
  if (threadIdx.x >= 64) worst = 0.0;  // every thread has it
  unsigned long long* out[3] = {&st->asym, &st->mag, &st->residual};
  double v[3] = {asym, mag, worst};
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    unsigned long long bits = (unsigned long long)__double_as_longlong(fabs(v[k]));
    for (int off = 32; off > 0; off >>= 1) {
      const unsigned long long o = __shfl_xor(bits, off);
      bits = o > bits ? o : bits;
    }
    if ((threadIdx.x & 63) == 0 && bits != 0) atomicMax(out[k], bits);
  }
}

__global__ __launch_bounds__(kThreads) void kp_clear_kernel(KpState* __restrict__ st, int nk) {
  for (int k = threadIdx.x; k < nk; k += kThreads) st[k] = KpState{0, 0, 0, 0, 0};
}

// Operand fragments of [Re X, Im X] = B [..]: a complex row of B is 2 n reals
// (re, im, re, im, ..), so the column of Re X_j is (Re C_0j, -Im C_0j, Re C_1j,
// ..) and that of Im X_j (Im C_0j, Re C_0j, ..), C = sqrt(weight) L. Columns
// [0, hb) are Re, [hb, 2 hb) Im, zero past the rank; and the column signs of
// the SYRKs of Re K and (shifted by hb) Im K.
__global__ __launch_bounds__(kThreads) void kp_fragments_kernel(const double2* __restrict__ lmat,
                                                                const KpState* __restrict__ state,
                                                                const double* __restrict__ weights, int n, int hb,
                                                                int kpad, ColumnGroups cg, double* __restrict__ frag,
                                                                double* __restrict__ sym, double* __restrict__ cross) {
  const int kp = blockIdx.y;
  const int rank = state[kp].rank;
  const double scale = sqrt(weights[kp]);
  const double2* l = lmat + (long long)kp * n * n;
  double* out = frag + (long long)kp * kpad * 2 * hb;
  const long long total = (long long)kpad * 2 * hb;
  for (long long idx = (long long)blockIdx.x * kThreads + threadIdx.x; idx < total;
       idx += (long long)gridDim.x * kThreads) {
    const int i = (int)(idx / kpad), k = (int)(idx % kpad);
    const int j = i < hb ? i : i - hb;
    double v = 0.0;
    if (k < 2 * n && j < rank) {
      const double2 z = l[(long long)j * n + k / 2];
      if (i < hb)
        v = k % 2 ? -z.y : z.x;
      else
        v = k % 2 ? z.x : z.y;
    }
    out[fragment_index<double>(cg, kpad, k, i)] = scale * v;
    if (kp == 0 && k == 0) {
      sym[i] = 1.0;
      cross[i] = i < hb ? -1.0 : 1.0;
    }
  }
}

// H = S + i A of a real row-major D (S, A its symmetric and antisymmetric parts), complex row-major.
__global__ __launch_bounds__(kThreads) void hermitian_of_real_kernel(const double* __restrict__ d, int n,
                                                                     double2* __restrict__ h) {
  const long long nn = (long long)n * n;
  for (long long idx = (long long)blockIdx.x * kThreads + threadIdx.x; idx < nn;
       idx += (long long)gridDim.x * kThreads) {
    const long long r = idx / n, c = idx % n;
    const double a = d[idx], b = d[c * n + r];
    h[idx] = make_double2(0.5 * (a + b), 0.5 * (a - b));
  }
}

// Columns [j0, j0 + rb) of the retained eigenpairs of H (the nneg lowest,
// then the npos highest; u column-major from zheevd of the view conj(H), so
// H's eigenvectors are conj(u)) as the real orbitals of the non-symmetric
// exchange: c [n][2 hb] = [Re V |l|^1/2 (rb columns), 0, Im V |l|^1/2, 0]
// with hb the half width, and the column signs of its two SYRKs:
// sym = (sign l, +1, sign l, +1), cross = (-sign l, +1, +sign l, +1).
__global__ __launch_bounds__(kThreads) void general_factor_kernel(const double2* __restrict__ u,
                                                                  const double* __restrict__ w, int n, int nneg,
                                                                  int npos, int j0, int rb, int hb,
                                                                  double* __restrict__ c, double* __restrict__ sym,
                                                                  double* __restrict__ cross) {
  const int ld = 2 * hb;
  const long long total = (long long)n * ld;
  for (long long idx = (long long)blockIdx.x * kThreads + threadIdx.x; idx < total;
       idx += (long long)gridDim.x * kThreads) {
    const int m = (int)(idx / ld);
    const int col = (int)(idx % ld);
    const int half = col >= hb ? 1 : 0;
    const int i = col - half * hb;
    double v = 0.0;
    double sg = 1.0;
    if (i < rb) {
      const int k = j0 + i;  // index among the retained pairs
      const int jj = k < nneg ? k : n - npos + (k - nneg);
      const double l = w[jj];
      const double2 z = u[(long long)jj * n + m];
      const double scale = sqrt(fabs(l));
      v = half ? -scale * z.y : scale * z.x;
      sg = l < 0.0 ? -1.0 : 1.0;
    }
    c[idx] = v;
    if (m == 0) {
      sym[col] = sg;
      cross[col] = i < rb ? (half ? sg : -sg) : 1.0;
    }
  }
}

}  // namespace

hipError_t launch_kp_charges(const void* b, long long kstride, int nk, int naux, int nao, const void* density,
                             const double* weights, void* inner, void* charges, hipStream_t s) {
  const long long nn = (long long)nao * nao;
  hipLaunchKernelGGL(kp_inner_kernel, dim3((unsigned)((long long)nk * naux)), dim3(kThreads), 0, s,
                     (const double2*)b, kstride, naux, nn, (const double2*)density, weights, (double2*)inner);
  hipError_t err = hipGetLastError();
  if (err != hipSuccess) return err;
  hipLaunchKernelGGL(kp_charges_kernel, dim3((unsigned)((naux + kThreads - 1) / kThreads)), dim3(kThreads), 0, s,
                     (const double2*)inner, nk, naux, (double2*)charges);
  return hipGetLastError();
}

hipError_t launch_kp_coulomb(const void* b, long long kstride, int nk, int naux, int nao, const double* sig,
                             long long sig_kstride, const void* charges, void* out, hipStream_t s) {
  const long long nn = (long long)nao * nao;
  const unsigned gx = (unsigned)std::min<long long>((nn + kCoulombElems - 1) / kCoulombElems, 1 << 16);
  hipLaunchKernelGGL(kp_coulomb_kernel, dim3(gx, (unsigned)nk), dim3(kThreads), 0, s, (const double2*)b, kstride,
                     naux, nn, sig, sig_kstride, (const double2*)charges, (double2*)out);
  return hipGetLastError();
}

hipError_t launch_kp_realify(const void* b, int naux, int nao, double* out, hipStream_t s) {
  const int npad2 = n_tiles(2 * nao) * kTile;
  hipLaunchKernelGGL(kp_realify_kernel, dim3(grid_for((long long)naux * npad2 * npad2)), dim3(kThreads), 0, s,
                     (const double2*)b, naux, nao, npad2, out);
  return hipGetLastError();
}

hipError_t launch_kp_factor(const void* eigvecs, const double* eigvals, int nao, int nneg, int npos, double weight,
                            int ldo, double* ct, double* signs, hipStream_t s) {
  const int npad2 = n_tiles(2 * nao) * kTile;
  hipLaunchKernelGGL(kp_factor_kernel, dim3(grid_for((long long)ldo * npad2)), dim3(kThreads), 0, s,
                     (const double2*)eigvecs, eigvals, nao, nneg, npos, weight, npad2, ldo, ct, signs);
  return hipGetLastError();
}

hipError_t launch_kp_fold(const double* kh, int nao, bool accumulate, void* k, hipStream_t s) {
  hipLaunchKernelGGL(kp_fold_kernel, dim3(grid_for((long long)nao * nao)), dim3(kThreads), 0, s, kh, nao,
                     accumulate ? 1 : 0, (double2*)k);
  return hipGetLastError();
}

hipError_t launch_kp_madelung(const void* overlap, const void* density, int nk, int nao, double alpha, void* tmp,
                              void* out, hipStream_t s) {
  const dim3 grid((unsigned)grid_for((long long)nao * nao), (unsigned)nk);
  hipLaunchKernelGGL(kp_zgemm_kernel, grid, dim3(kThreads), 0, s, (const double2*)overlap, (const double2*)density,
                     nao, 1.0, 0, (double2*)tmp);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(kp_zgemm_kernel, grid, dim3(kThreads), 0, s, (const double2*)tmp, (const double2*)overlap, nao,
                     alpha, 1, (double2*)out);
  return hipGetLastError();
}

hipError_t launch_kp_cholesky(const void* density, int nk, int nao, void* l, KpState* st, hipStream_t s) {
  hipLaunchKernelGGL(kp_clear_kernel, dim3(1), dim3(kThreads), 0, s, st, nk);
  // The diagonals live behind L.
  double* diag = (double*)((double2*)l + (long long)nk * nao * nao);
  hipLaunchKernelGGL(kp_cholesky_kernel, dim3((unsigned)nk), dim3(kCholThreads), 0, s, (const double2*)density, nao,
                     (double2*)l, diag, st);
  const unsigned gx = (unsigned)std::min(nao, 1024);
  hipLaunchKernelGGL(kp_residual_kernel, dim3(gx, (unsigned)nk), dim3(kThreads), 0, s, (const double2*)density, nao,
                     (const double2*)l, st);
  return hipGetLastError();
}

hipError_t launch_kp_fragments(const void* l, const KpState* st, const double* weights, int nk, int nao, int hb,
                               double* frag, double* sym, double* cross, hipStream_t s) {
  const int kpad = n_tiles(2 * nao) * kTile;
  const dim3 grid((unsigned)grid_for((long long)kpad * 2 * hb), (unsigned)nk);
  hipLaunchKernelGGL(kp_fragments_kernel, grid, dim3(kThreads), 0, s, (const double2*)l, st, weights, nao, hb, kpad,
                     column_groups(2 * hb, 2 * hb, 0), frag, sym, cross);
  return hipGetLastError();
}

hipError_t launch_hermitian_of_real(const double* d, int nao, void* h, hipStream_t s) {
  hipLaunchKernelGGL(hermitian_of_real_kernel, dim3(grid_for((long long)nao * nao)), dim3(kThreads), 0, s, d, nao,
                     (double2*)h);
  return hipGetLastError();
}

hipError_t launch_general_factor(const void* eigvecs, const double* eigvals, int nao, int nneg, int npos, int j0,
                                 int rb, int hb, double* c, double* sym, double* cross, hipStream_t s) {
  hipLaunchKernelGGL(general_factor_kernel, dim3(grid_for((long long)nao * 2 * hb)), dim3(kThreads), 0, s,
                     (const double2*)eigvecs, eigvals, nao, nneg, npos, j0, rb, hb, c, sym, cross);
  return hipGetLastError();
}

}  // namespace hfjk
