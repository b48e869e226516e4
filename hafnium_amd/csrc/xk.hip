// Exchange kernels for gfx950 (CDNA4): the half-transform X[P] = B[P] C and
// the symmetric rank-k update K = sum_P X[P] S X[P]^T, on MFMA, in three
// arithmetics (FP64, FP32, BF16x3).
//
// Structure shared by all of them:
//  * workgroups of 4 waves of 64 (8 for the 256 x 256 tiles), each k step's
//    loads in flight while the MFMAs of the step before run;
//  * the SYRK grid is XCD-aware: workgroups are dispatched round-robin over
//    the 8 XCDs, so linear id b runs on XCD b % 8, and every tile of one
//    aux-slice split s is mapped to the same XCD. The slice of X that those
//    tiles stream is then fetched from HBM into one L2 instead of eight.
//
// MFMA lane layouts (measured on gfx950):
//  * v_mfma_f64_16x16x4f64 : A[i][k] in lane i + 16 k, B[k][j] in lane j + 16 k,
//    D register r of lane l = D[l / 16 + 4 r][l % 16];
//  * v_mfma_f32_16x16x4f32 : same A/B, D register r of lane l = D[4 (l / 16) + r][l % 16];
//  * v_mfma_f32_16x16x32_bf16 : A[i][8 (l / 16) + e] in element e of lane l with
//    i = l % 16, B[8 (l / 16) + e][j] likewise with j = l % 16; D as f32 16x16x4.
//
// FP64/FP32 operands are single elements per lane, so a packed B tile is read
// directly or transposed by addressing alone. BF16x3 operands are 8
// consecutive k per lane, so tiles stored transposed are transposed in
// registers (4 x 4 blocks) on their way into a [row][k] LDS tile.
#include <algorithm>
#include <functional>
#include <type_traits>
#include <vector>

#include "hfjk_internal.h"

namespace hfjk {
namespace {

typedef double d4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ long long tidx(int r, int c) { return (long long)r * (r + 1) / 2 + c; }

__device__ __forceinline__ void tile_of(int tile, int& r, int& c) {
  int rr = (int)((sqrt(8.0 * (double)tile + 1.0) - 1.0) * 0.5);
  while ((rr + 1) * (rr + 2) / 2 <= tile) ++rr;
  while (rr * (rr + 1) / 2 > tile) --rr;
  r = rr;
  c = tile - rr * (rr + 1) / 2;
}

__device__ __forceinline__ uint16_t bf16_of(float x) {
  uint32_t u = __float_as_uint(x);
  if ((u & 0x7F800000u) == 0x7F800000u) return (uint16_t)((u >> 16) | ((u & 0xFFFFu) ? 0x40u : 0u));
  u += 0x7FFFu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}

__device__ __forceinline__ float f32_of(uint16_t h) { return __uint_as_float(((uint32_t)h) << 16); }

// Logical index of linear workgroup b of a W-workgroup 1-D grid: XCD x
// (b % 8) receives the consecutive logical range [x W/8, (x+1) W/8), so
// neighbouring tiles (which share operands) share one L2.
__device__ __forceinline__ int xcd_remap(int b, int w) {
  const int full = w & ~7;
  if (b >= full) return b;
  return (b & 7) * (full >> 3) + (b >> 3);
}

template <typename T>
struct Op;

template <>
struct Op<double> {
  typedef d4 acc_t;
  typedef double2 vec2;
  static __device__ __forceinline__ acc_t mma(double a, double b, acc_t c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int lane, int r) { return (lane >> 4) + 4 * r; }
};

template <>
struct Op<float> {
  typedef f4 acc_t;
  typedef float2 vec2;
  static __device__ __forceinline__ acc_t mma(float a, float b, acc_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int lane, int r) { return 4 * (lane >> 4) + r; }
};

// Zero a vector unless `keep`, component by component (a select of whole
// vectors is lowered through a private-memory copy).
__device__ __forceinline__ uint2 mask2(bool keep, uint2 v) {
  const uint32_t m = keep ? 0xFFFFFFFFu : 0u;
  return make_uint2(v.x & m, v.y & m);
}

__device__ __forceinline__ uint4 mask4(bool keep, uint4 v) {
  const uint32_t m = keep ? 0xFFFFFFFFu : 0u;
  return make_uint4(v.x & m, v.y & m, v.z & m, v.w & m);
}

// 8 bf16 from LDS as one 16-byte load, reinterpreted as the MFMA operand.
__device__ __forceinline__ bf8 lds_bf8(const uint16_t* p) {
  const uint4 v = *(const uint4*)p;
  return __builtin_bit_cast(bf8, v);
}

__device__ __forceinline__ f4 mma3(bf8 ah, bf8 al, bf8 bh, bf8 bl, f4 acc) {
  acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al, bh, acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bl, acc, 0, 0, 0);
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bh, acc, 0, 0, 0);
}

// ------------------------------------------------------------------ FP64 / FP32 half-transform
//
// X[q][m][i] = sum_k B[q][m][k] C[k][i] from the tiled packed B. The rows of
// every aux function in blocks of 16 MI form one list of units; each wave of a
// workgroup computes its own unit for the NI 16-column blocks of a column
// group, so all waves carry the same columns and no wave waits for another's
// padding. MI is 1 in FP64 (with 2, accumulators, two B tiles and C's operands
// spill) and 2 in FP32. One layout tile column per k step:
// * B goes from global memory straight into the MFMA operand registers, the
//   next step's tile while this one computes. Element e = EV eg + ee of a
//   lane's 8 per 16 rows is k = 4 EV eg + EV g + ee (g = lane / 16, EV
//   elements per 16 bytes), so a tile stored as (r, kt) is read as 16-byte
//   groups along its rows and one stored as (kt, r) as 128-byte runs of its
//   columns, without a transpose.
// * C, in the order the MFMA operand reads it (launch_prepare_orbitals),
//   goes by direct-LDS loads into one of two stage buffers shared by the
//   waves: one barrier per step, 16-byte conflict-free LDS reads.
//
// Bound by the MFMAs: 8 MI NI of them per step and wave, 64 cycles each in FP64
// (32 in FP32), against 4 KB of B and a shared 4 NI KB (2 NI KB) of C.
// It replaces 64 / 128-row tiles staged through registers into padded LDS
// (two barriers per step, waves idle on the padding of their quadrant): 128
// uneven instances 31.6 -> 22.0 ms, nao 288 / naux 1356 / nocc 60 320 -> 248
// us, nao 501 / naux 1800 / nocc 90 2.15 -> 1.43 ms (FP64), nao 709 / naux
// 2503 / nocc 117 in FP32 3.38 -> 2.98 ms.
template <typename T>
struct XFrag {
  static constexpr int EV = 16 / (int)sizeof(T);  // elements per 16-byte group
  static constexpr int NG = 8 / EV;               // groups per lane and 16 rows of a tile
  static constexpr int KG = 4 * EV;               // k per group over the four lane groups
  static constexpr int BLOCK = kTile * 16;        // elements of one 16-column block of a k tile
  static constexpr int LOADS = BLOCK * (int)sizeof(T) / 1024;  // 1 KB loads per block
  static constexpr int MI = sizeof(T) == 8 ? 1 : 2;   // 16-row blocks per unit
  typedef T unit __attribute__((ext_vector_type(16 / sizeof(T))));
};

// s_waitcnt vmcnt(VM) lgkmcnt(0) (gfx9 encoding: vmcnt in bits 3:0 and 15:14).
template <int VM>
__device__ __forceinline__ void wait_vm_lgkm0() {
  static_assert(VM >= 0 && VM < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((VM & 15) | ((VM >> 4) << 14) | (0x7 << 4));
}

// Workgroup barrier without a memory fence (a fence would wait for every
// load in flight, the stages ahead included). The clobber keeps the compiler
// from moving memory accesses across it.
__device__ __forceinline__ void barrier_nofence() { asm volatile("s_barrier" ::: "memory"); }

typedef __attribute__((address_space(3))) void lds_void_t;

// Units [u0, u1) (unit q nu + r, nu = ceil(nao / 16 MI)) of the column group
// whose fragments start at cf: b = the packed B of aux function 0, x = X of
// aux function 0 at the group's first column. zero_block: X's 16 columns
// after the group are written as zeros (the padding of ldo past an odd number
// of blocks). Rows past the last unit are not written. The whole workgroup
// calls it; on return its LDS reads have returned and no load is in flight.
template <typename T, int NI>
__device__ __forceinline__ void xform_units(const T* __restrict__ b, long long p, int nt, const T* __restrict__ cf,
                                            T* __restrict__ x, int xrows, int ldo, int u0, int u1, int nao,
                                            bool zero_block, T* lds0, T* lds1) {
  typedef XFrag<T> F;
  typedef typename F::unit unit;
  constexpr int MI = F::MI;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int waves = blockDim.x >> 6;
  const int row16 = lane & 15, grp = lane >> 4;
  const int nu = xform_units_per_aux<T>(nao);

  int steps = ((u1 - u0 + waves - 1) / waves) * nt;
  int u = u0 + wave;
  int q = u / nu, r = u - q * nu, kt = 0;
  int qc = u0 / nu, rc = u0 - qc * nu;  // a unit whose tiles may be read (u0 < u1)
  if (u < u1) {
    qc = q;
    rc = r;
  }

  auto load_c = [&](int k, T* stage) {
    const T* src = cf + (long long)k * NI * F::BLOCK + lane * F::EV;
    for (int c = wave; c < NI * F::LOADS; c += waves)
      __builtin_amdgcn_global_load_lds((const void*)(src + c * 64 * F::EV), (lds_void_t*)(stage + c * 64 * F::EV), 16,
                                       0, 0);
  };
  auto load_a = [&](int qq, int rr, int k, unit (&a)[MI][F::NG]) {
    const T* bq = b + (long long)qq * p;
    const int tr = rr * MI / 2, half = rr * MI % 2;  // layout tile row, its 16-row half
    if (tr >= k) {
      const T* src = bq + tidx(tr, k) * kTileElems + (half * 16 + row16) * kTile + grp * F::EV;
#pragma unroll
      for (int mi = 0; mi < MI; ++mi)
#pragma unroll
        for (int eg = 0; eg < F::NG; ++eg) a[mi][eg] = *(const unit*)(src + mi * 16 * kTile + eg * F::KG);
    } else {
      const T* src = bq + tidx(k, tr) * kTileElems + grp * F::EV * kTile + half * 16 + row16;
#pragma unroll
      for (int eg = 0; eg < F::NG; ++eg)
#pragma unroll
        for (int ee = 0; ee < F::EV; ++ee)
#pragma unroll
          for (int mi = 0; mi < MI; ++mi)
            a[mi][eg][ee] = src[(eg * F::KG + ee) * kTile + mi * 16];
    }
  };

  typename Op<T>::acc_t acc[MI][NI];
  auto clear = [&]() {
#pragma unroll
    for (int mi = 0; mi < MI; ++mi)
#pragma unroll
      for (int ni = 0; ni < NI; ++ni)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[mi][ni][e] = (T)0;
  };
  auto group = [&](const T* stage, int eg, const unit (&a)[MI][F::NG]) {
    unit bv[NI];
#pragma unroll
    for (int ni = 0; ni < NI; ++ni) bv[ni] = *(const unit*)(stage + ((eg * NI + ni) * 64 + lane) * F::EV);
#pragma unroll
    for (int ee = 0; ee < F::EV; ++ee)
#pragma unroll
      for (int mi = 0; mi < MI; ++mi)
#pragma unroll
        for (int ni = 0; ni < NI; ++ni) acc[mi][ni] = Op<T>::mma(a[mi][eg][ee], bv[ni][ee], acc[mi][ni]);
  };

  // Step: this wave's loads for it have landed and its LDS reads of the step
  // before have returned; after the barrier that holds for every wave, so the
  // other buffer takes the next step's C while this step computes.
  auto step = [&](const T* cur, T* next, unit (&a)[MI][F::NG], unit (&an)[MI][F::NG]) {
    wait_vm_lgkm0<0>();
    barrier_nofence();
    const bool last = kt + 1 == nt;
    int un = u, qn = q, rn = r;
    if (u < u1) {
      qc = q;
      rc = r;
    }
    const int kn = last ? 0 : kt + 1;
    if (last) {
      un += waves;
      rn += waves;
      while (rn >= nu) {
        rn -= nu;
        ++qn;
      }
    }
    // (A wave without a next unit reads this one's tile again: a conditional load would end in
    // register copies, and those in a wait.)
    if (steps > 1) load_c(kn, next);
    const bool more = un < u1;
    load_a(more ? qn : qc, more ? rn : rc, kn, an);
    if (u < u1) {
      // k past nao holds zeros.
      const int kleft = nao - kt * kTile;
#pragma unroll
      for (int eg = 0; eg < F::NG; ++eg)
        if (eg * F::KG < kleft) group(cur, eg, a);
      if (last) {
        T* dst = x + ((long long)q * xrows + r * 16 * MI) * ldo + row16;
#pragma unroll
        for (int mi = 0; mi < MI; ++mi)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            T* at = dst + (long long)(mi * 16 + Op<T>::row(lane, e)) * ldo;
#pragma unroll
            for (int ni = 0; ni < NI; ++ni) at[ni * 16] = acc[mi][ni][e];
            if (zero_block) at[NI * 16] = (T)0;
          }
        clear();
      }
    }
    u = un;
    q = qn;
    r = rn;
    kt = kn;
    return --steps > 0;
  };

  unit a0[MI][F::NG], a1[MI][F::NG];
  clear();
  load_c(0, lds0);
  load_a(qc, rc, 0, a0);
  while (step(lds0, lds1, a0, a1) && step(lds1, lds0, a1, a0)) {
  }
}

// Workgroup: `per` units of one column group (wg % ngroups), NI blocks wide
// except the last group's `tail`, which a launch of its own handles.
template <typename T, int NI>
__global__ __launch_bounds__(kThreads, NI <= 4 ? 3 : 2) void xform_units_kernel(
    const T* __restrict__ b, long long p, int nt, const T* __restrict__ cf, long long group_elems, int ngroups,
    T* __restrict__ x, int xrows, int ldo, int units, int per, int nao, int zero_block, int nwg) {
  __shared__ __attribute__((aligned(16))) T lds0[NI * XFrag<T>::BLOCK];
  __shared__ __attribute__((aligned(16))) T lds1[NI * XFrag<T>::BLOCK];
  const int logical = xcd_remap(blockIdx.x, nwg);
  const int g = logical % ngroups;
  const int u0 = logical / ngroups * per;
  xform_units<T, NI>(b, p, nt, cf + g * group_elems, x + g * NI * 16, xrows, ldo, u0, min(u0 + per, units), nao,
                     zero_block != 0 && g == ngroups - 1, lds0, lds1);
}

// Plain row-major rows times per-group operand fragments (FP64): rows of
// `len` doubles, `rows` per block, block b0 + i with the fragments of group
// (b0 + i) % ngroup; x[(i rows + row) ldo + column] for the NI blocks from
// column 0 of x on. The structure of xform_units with the operand read
// directly; k past len repeats the row's start against zero fragments.
template <int NI>
__global__ __launch_bounds__(kThreads, NI <= 4 ? 3 : 2) void rows_units_kernel(
    const double* __restrict__ b, long long rows, int len, int b0, int ngroup, const double* __restrict__ cf,
    long long group_elems, double* __restrict__ x, int ldo, int wgs_per_block) {
  typedef XFrag<double> F;
  typedef F::unit unit;
  __shared__ __attribute__((aligned(16))) double lds0[NI * F::BLOCK];
  __shared__ __attribute__((aligned(16))) double lds1[NI * F::BLOCK];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int row16 = lane & 15, grp = lane >> 4;
  const int blk = blockIdx.x / wgs_per_block;
  const long long row0 = ((long long)(blockIdx.x % wgs_per_block) * 4 + wave) * 16;
  const double* cg = cf + (b0 + blk) % ngroup * group_elems;
  const double* src = b + ((long long)(b0 + blk) * rows + min(row0 + row16, rows - 1)) * len;
  const int nt = (len + kTile - 1) / kTile;

  auto load_c = [&](int k, double* stage) {
    const double* p = cg + (long long)k * NI * F::BLOCK + lane * F::EV;
    for (int c = wave; c < NI * F::LOADS; c += 4)
      __builtin_amdgcn_global_load_lds((const void*)(p + c * 64 * F::EV), (lds_void_t*)(stage + c * 64 * F::EV), 16, 0,
                                       0);
  };
  auto load_a = [&](int kt, unit (&a)[F::NG]) {
#pragma unroll
    for (int eg = 0; eg < F::NG; ++eg) {
      const int k = kt * kTile + eg * F::KG + grp * F::EV;
      a[eg] = *(const unit*)(src + (k < len ? k : 0));
    }
  };
  Op<double>::acc_t acc[NI];
#pragma unroll
  for (int ni = 0; ni < NI; ++ni)
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[ni][e] = 0.0;
  int kt = 0;
  auto step = [&](const double* cur, double* next, unit (&a)[F::NG], unit (&an)[F::NG]) {
    wait_vm_lgkm0<0>();
    barrier_nofence();
    if (kt + 1 < nt) load_c(kt + 1, next);
    load_a(min(kt + 1, nt - 1), an);
#pragma unroll
    for (int eg = 0; eg < F::NG; ++eg)
      if (kt * kTile + eg * F::KG < len) {
        unit bv[NI];
#pragma unroll
        for (int ni = 0; ni < NI; ++ni) bv[ni] = *(const unit*)(cur + ((eg * NI + ni) * 64 + lane) * F::EV);
#pragma unroll
        for (int ee = 0; ee < F::EV; ++ee)
#pragma unroll
          for (int ni = 0; ni < NI; ++ni) acc[ni] = Op<double>::mma(a[eg][ee], bv[ni][ee], acc[ni]);
      }
    return ++kt < nt;
  };
  unit a0[F::NG], a1[F::NG];
  load_c(0, lds0);
  load_a(0, a0);
  while (step(lds0, lds1, a0, a1) && step(lds1, lds0, a1, a0)) {
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const long long row = row0 + Op<double>::row(lane, e);
    if (row >= rows) continue;
    double* at = x + ((long long)blk * rows + row) * ldo + row16;
#pragma unroll
    for (int ni = 0; ni < NI; ++ni) at[ni * 16] = acc[ni][e];
  }
}

// ------------------------------------------------------------------ BF16x3 half-transform

constexpr int kRowK = 40;  // bf16 LDS row: 32 k + 8 pad (80 bytes, 16-byte aligned rows)

// X in BF16x3: workgroup tile 128 rows (four layout tile rows) x BN columns,
// waves 2 x 2 each (64 x BN/2). A is staged [m][k]; C^T (stored [i][k])
// is staged [i][k].
template <int BN>
struct Xform16Smem {
  uint16_t Ah[128][kRowK];
  uint16_t Al[128][kRowK];
  uint16_t Bh[BN][kRowK];
  uint16_t Bl[BN][kRowK];
};

// One 128 x BN tile of X_q in BF16x3: hq/lq = the packed hi/lo planes of
// B_q, xhi/xlo = X_q's hi/lo rows (xrows rows of ldo).
template <int BN>
__device__ __forceinline__ void xform16_tile(const uint16_t* __restrict__ hq, const uint16_t* __restrict__ lq, int nt,
                                             const uint16_t* __restrict__ cthi, const uint16_t* __restrict__ ctlo,
                                             int npad, int ldo, uint16_t* __restrict__ xhi,
                                             uint16_t* __restrict__ xlo, int xrows, int mb, int nb,
                                             Xform16Smem<BN>& sm) {
  constexpr int MI = 4;            // 64 rows per wave
  constexpr int NI = BN / 2 / 16;  // BN/2 columns per wave
  constexpr int CCH = BN * 4 / kThreads > 0 ? BN * 4 / kThreads : 1;  // 16-byte chunks of C^T per plane
  auto& Ah = sm.Ah;
  auto& Al = sm.Al;
  auto& Bh = sm.Bh;
  auto& Bl = sm.Bl;
  const int n0 = nb * BN;
  const int t = threadIdx.x;
  const int lane = t & 63;
  const int wave = t >> 6;
  const int wm = wave & 1;
  const int wn = wave >> 1;

  f4 acc[MI][NI];
#pragma unroll
  for (int mi = 0; mi < MI; ++mi)
#pragma unroll
    for (int ni = 0; ni < NI; ++ni) acc[mi][ni] = f4{0.f, 0.f, 0.f, 0.f};

  // Each thread owns one 4 x 4 block of one of the four layout tiles.
  const int th = t >> 6;            // tile row within the block: r = 4 mb + th
  const int a0 = ((t & 63) >> 3) * 4;
  const int b0 = (t & 7) * 4;
  const int r_own = 4 * mb + th;
  uint2 rah[4], ral[4];
  uint4 rch[CCH], rcl[CCH];

  // Loads are unconditional (from a valid clamped address); the masks (bitwise,
  // which keeps the prefetch arrays in registers) are applied in store(), so
  // the wait for the loads falls at the end of the k step, not at its start.
  const bool own = r_own < nt;
  auto load = [&](int kt) {
    const int rc = own ? r_own : 0;
    const long long base = (rc >= kt ? tidx(rc, kt) : tidx(kt, rc)) * kTileElems + a0 * kTile + b0;
#pragma unroll
    for (int rr = 0; rr < 4; ++rr) {
      rah[rr] = *(const uint2*)(hq + base + rr * kTile);
      ral[rr] = *(const uint2*)(lq + base + rr * kTile);
    }
#pragma unroll
    for (int v = 0; v < CCH; ++v) {
      const int chunk = t + kThreads * v;  // BN rows x 4 chunks of 8 bf16
      const int jj = chunk >> 2;
      const int k8 = (chunk & 3) * 8;
      const int col = n0 + jj;
      const bool ok = chunk < BN * 4 && col < ldo;
      const long long off = ok ? (long long)col * npad + kt * kTile + k8 : 0;
      rch[v] = *(const uint4*)(cthi + off);
      rcl[v] = *(const uint4*)(ctlo + off);
    }
  };
  auto store = [&](int kt) {
#pragma unroll
    for (int rr = 0; rr < 4; ++rr) {
      rah[rr] = mask2(own, rah[rr]);
      ral[rr] = mask2(own, ral[rr]);
    }
#pragma unroll
    for (int v = 0; v < CCH; ++v) {
      const int chunk = t + kThreads * v;
      const bool ok = chunk < BN * 4 && n0 + (chunk >> 2) < ldo;
      rch[v] = mask4(ok, rch[v]);
      rcl[v] = mask4(ok, rcl[v]);
    }
    const bool direct = r_own >= kt;  // also true for r_own >= nt (zeros)
    if (direct) {
      // element (a, b) is B[m = r*32 + a][k = kt*32 + b]
#pragma unroll
      for (int rr = 0; rr < 4; ++rr) {
        *(uint2*)&Ah[th * kTile + a0 + rr][b0] = rah[rr];
        *(uint2*)&Al[th * kTile + a0 + rr][b0] = ral[rr];
      }
    } else {
      // element (a, b) is B[k = kt*32 + a][m = r*32 + b]: transpose the 4 x 4 block
#pragma unroll
      for (int cc = 0; cc < 4; ++cc) {
        uint2 h, l;
        const int sh = (cc & 1) * 16;
        auto pick = [&](const uint2& v) -> uint32_t { return ((cc < 2 ? v.x : v.y) >> sh) & 0xFFFFu; };
        h.x = pick(rah[0]) | (pick(rah[1]) << 16);
        h.y = pick(rah[2]) | (pick(rah[3]) << 16);
        l.x = pick(ral[0]) | (pick(ral[1]) << 16);
        l.y = pick(ral[2]) | (pick(ral[3]) << 16);
        *(uint2*)&Ah[th * kTile + b0 + cc][a0] = h;
        *(uint2*)&Al[th * kTile + b0 + cc][a0] = l;
      }
    }
#pragma unroll
    for (int v = 0; v < CCH; ++v) {
      const int chunk = t + kThreads * v;
      if (chunk < BN * 4) {
        const int jj = chunk >> 2;
        const int k8 = (chunk & 3) * 8;
        *(uint4*)&Bh[jj][k8] = rch[v];
        *(uint4*)&Bl[jj][k8] = rcl[v];
      }
    }
  };

  load(0);
  store(0);
  __syncthreads();
  for (int kt = 0; kt < nt; ++kt) {
    if (kt + 1 < nt) load(kt + 1);
    const int kq = 8 * (lane >> 4);
    bf8 ah[MI], al[MI];
#pragma unroll
    for (int mi = 0; mi < MI; ++mi) {
      ah[mi] = lds_bf8(&Ah[wm * 64 + mi * 16 + (lane & 15)][kq]);
      al[mi] = lds_bf8(&Al[wm * 64 + mi * 16 + (lane & 15)][kq]);
    }
#pragma unroll
    for (int ni = 0; ni < NI; ++ni) {
      const bf8 bh = lds_bf8(&Bh[wn * (BN / 2) + ni * 16 + (lane & 15)][kq]);
      const bf8 bl = lds_bf8(&Bl[wn * (BN / 2) + ni * 16 + (lane & 15)][kq]);
#pragma unroll
      for (int mi = 0; mi < MI; ++mi) acc[mi][ni] = mma3(ah[mi], al[mi], bh, bl, acc[mi][ni]);
    }
    __syncthreads();
    if (kt + 1 < nt) {
      store(kt + 1);
      __syncthreads();
    }
  }
#pragma unroll
  for (int mi = 0; mi < MI; ++mi)
#pragma unroll
    for (int ni = 0; ni < NI; ++ni) {
      const int col = n0 + wn * (BN / 2) + ni * 16 + (lane & 15);
      if (col < ldo) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int row = mb * 128 + wm * 64 + mi * 16 + 4 * (lane >> 4) + r;
          if (row < xrows) {
            const float v = acc[mi][ni][r];
            const uint16_t h = bf16_of(v);
            const long long off = (long long)row * ldo + col;
            xhi[off] = h;
            xlo[off] = bf16_of(v - f32_of(h));
          }
        }
      }
    }
}

// xform16_tile for each aux function q in [q0, q1) (the batched kernel's
// items): hq/lq = the packed hi/lo planes of aux function 0 (q's at stride
// p), xhi/xlo = X of aux function 0 (q's at stride xrows * ldo). The (q, k
// tile) steps run as one pipeline, the next step's loads issued before the
// current step's MFMAs across aux functions too, and each q's tile is
// written after its last k tile. With SKIP the MFMAs of 16-row blocks at or
// past nrow and of 16-column blocks at or past ncol are left out (B and C
// are zero there, so X is the same); each wave decides for its own blocks.
template <int BN, bool SKIP>
__device__ __forceinline__ void xform16_tiles(const uint16_t* __restrict__ hq, const uint16_t* __restrict__ lq,
                                              long long p, int nt, const uint16_t* __restrict__ cthi,
                                              const uint16_t* __restrict__ ctlo, int npad, int ldo,
                                              uint16_t* __restrict__ xhi, uint16_t* __restrict__ xlo, int xrows,
                                              int mb, int nb, int q0, int q1, Xform16Smem<BN>& sm, int nrow,
                                              int ncol) {
  constexpr int MI = 4;            // 64 rows per wave
  constexpr int NI = BN / 2 / 16;  // BN/2 columns per wave
  constexpr int CCH = BN * 4 / kThreads > 0 ? BN * 4 / kThreads : 1;  // 16-byte chunks of C^T per plane
  auto& Ah = sm.Ah;
  auto& Al = sm.Al;
  auto& Bh = sm.Bh;
  auto& Bl = sm.Bl;
  const int n0 = nb * BN;
  const int t = threadIdx.x;
  const int lane = t & 63;
  const int wave = t >> 6;
  const int wm = wave & 1;
  const int wn = wave >> 1;

  f4 acc[MI][NI];
#pragma unroll
  for (int mi = 0; mi < MI; ++mi)
#pragma unroll
    for (int ni = 0; ni < NI; ++ni) acc[mi][ni] = f4{0.f, 0.f, 0.f, 0.f};

  // Each thread owns one 4 x 4 block of one of the four layout tiles.
  const int th = t >> 6;
  const int a0 = ((t & 63) >> 3) * 4;
  const int b0 = (t & 7) * 4;
  const int r_own = 4 * mb + th;
  uint2 rah[4], ral[4];
  uint4 rch[CCH], rcl[CCH];
  const bool own = r_own < nt;
  auto load = [&](int q, int kt) {
    const int rc = own ? r_own : 0;
    const long long base = (long long)q * p + (rc >= kt ? tidx(rc, kt) : tidx(kt, rc)) * kTileElems + a0 * kTile + b0;
#pragma unroll
    for (int rr = 0; rr < 4; ++rr) {
      rah[rr] = *(const uint2*)(hq + base + rr * kTile);
      ral[rr] = *(const uint2*)(lq + base + rr * kTile);
    }
#pragma unroll
    for (int v = 0; v < CCH; ++v) {
      const int chunk = t + kThreads * v;  // BN rows x 4 chunks of 8 bf16
      const int jj = chunk >> 2;
      const int k8 = (chunk & 3) * 8;
      const int col = n0 + jj;
      const bool ok = chunk < BN * 4 && col < ldo;
      const long long off = ok ? (long long)col * npad + kt * kTile + k8 : 0;
      rch[v] = *(const uint4*)(cthi + off);
      rcl[v] = *(const uint4*)(ctlo + off);
    }
  };
  auto store = [&](int kt) {
#pragma unroll
    for (int rr = 0; rr < 4; ++rr) {
      rah[rr] = mask2(own, rah[rr]);
      ral[rr] = mask2(own, ral[rr]);
    }
#pragma unroll
    for (int v = 0; v < CCH; ++v) {
      const int chunk = t + kThreads * v;
      const bool ok = chunk < BN * 4 && n0 + (chunk >> 2) < ldo;
      rch[v] = mask4(ok, rch[v]);
      rcl[v] = mask4(ok, rcl[v]);
    }
    const bool direct = r_own >= kt;  // also true for r_own >= nt (zeros)
    if (direct) {
#pragma unroll
      for (int rr = 0; rr < 4; ++rr) {
        *(uint2*)&Ah[th * kTile + a0 + rr][b0] = rah[rr];
        *(uint2*)&Al[th * kTile + a0 + rr][b0] = ral[rr];
      }
    } else {
#pragma unroll
      for (int cc = 0; cc < 4; ++cc) {
        uint2 h, l;
        const int sh = (cc & 1) * 16;
        auto pick = [&](const uint2& v) -> uint32_t { return ((cc < 2 ? v.x : v.y) >> sh) & 0xFFFFu; };
        h.x = pick(rah[0]) | (pick(rah[1]) << 16);
        h.y = pick(rah[2]) | (pick(rah[3]) << 16);
        l.x = pick(ral[0]) | (pick(ral[1]) << 16);
        l.y = pick(ral[2]) | (pick(ral[3]) << 16);
        *(uint2*)&Ah[th * kTile + b0 + cc][a0] = h;
        *(uint2*)&Al[th * kTile + b0 + cc][a0] = l;
      }
    }
#pragma unroll
    for (int v = 0; v < CCH; ++v) {
      const int chunk = t + kThreads * v;
      if (chunk < BN * 4) {
        const int jj = chunk >> 2;
        const int k8 = (chunk & 3) * 8;
        *(uint4*)&Bh[jj][k8] = rch[v];
        *(uint4*)&Bl[jj][k8] = rcl[v];
      }
    }
  };

  // Wave-uniform block masks of SKIP.
  bool rv[MI], cv[NI];
  {
    const int wu = __builtin_amdgcn_readfirstlane(t >> 6);
#pragma unroll
    for (int mi = 0; mi < MI; ++mi) rv[mi] = !SKIP || mb * 128 + (wu & 1) * 64 + mi * 16 < nrow;
#pragma unroll
    for (int ni = 0; ni < NI; ++ni) cv[ni] = !SKIP || n0 + (wu >> 1) * (BN / 2) + ni * 16 < ncol;
  }

  const int steps = (q1 - q0) * nt;
  if (steps <= 0) return;
  load(q0, 0);
  store(0);
  __syncthreads();
  int q = q0, kt = 0;
  for (int step = 0; step < steps; ++step) {
    const int nq = kt + 1 < nt ? q : q + 1;
    const int nkt = kt + 1 < nt ? kt + 1 : 0;
    if (step + 1 < steps) load(nq, nkt);
    const int kq = 8 * (lane >> 4);
    bf8 ah[MI], al[MI];
#pragma unroll
    for (int mi = 0; mi < MI; ++mi) {
      ah[mi] = lds_bf8(&Ah[wm * 64 + mi * 16 + (lane & 15)][kq]);
      al[mi] = lds_bf8(&Al[wm * 64 + mi * 16 + (lane & 15)][kq]);
    }
#pragma unroll
    for (int ni = 0; ni < NI; ++ni) {
      if (!cv[ni]) continue;
      const bf8 bh = lds_bf8(&Bh[wn * (BN / 2) + ni * 16 + (lane & 15)][kq]);
      const bf8 bl = lds_bf8(&Bl[wn * (BN / 2) + ni * 16 + (lane & 15)][kq]);
#pragma unroll
      for (int mi = 0; mi < MI; ++mi)
        if (rv[mi]) acc[mi][ni] = mma3(ah[mi], al[mi], bh, bl, acc[mi][ni]);
    }
    __syncthreads();
    if (kt == nt - 1) {
      // This aux function's tile is complete: write it and start the next one from zero.
      const long long xq = (long long)q * xrows * ldo;
#pragma unroll
      for (int mi = 0; mi < MI; ++mi)
#pragma unroll
        for (int ni = 0; ni < NI; ++ni) {
          const int col = n0 + wn * (BN / 2) + ni * 16 + (lane & 15);
          if (col < ldo) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const int row = mb * 128 + wm * 64 + mi * 16 + 4 * (lane >> 4) + r;
              if (row < xrows) {
                const float v = acc[mi][ni][r];
                const uint16_t h = bf16_of(v);
                const long long off = xq + (long long)row * ldo + col;
                xhi[off] = h;
                xlo[off] = bf16_of(v - f32_of(h));
              }
            }
          }
          acc[mi][ni] = f4{0.f, 0.f, 0.f, 0.f};
        }
    }
    if (step + 1 < steps) {
      store(nkt);
      __syncthreads();
    }
    q = nq;
    kt = nkt;
  }
}

template <int BN>
__global__ __launch_bounds__(kThreads) void xform_bf16x3_kernel(
    const uint16_t* __restrict__ bhi, const uint16_t* __restrict__ blo, long long p, int nt,
    const uint16_t* __restrict__ cthi, const uint16_t* __restrict__ ctlo, int npad, int ldo,
    uint16_t* __restrict__ xhi, uint16_t* __restrict__ xlo, int xrows, int qbase, int nblocks_n, int nblocks_m,
    int nwg) {
  __shared__ __attribute__((aligned(16))) Xform16Smem<BN> sm;
  const int logical = xcd_remap(blockIdx.x, nwg);
  const int nb = logical % nblocks_n;
  const int mb = (logical / nblocks_n) % nblocks_m;  // 128-row block
  const int q = qbase + logical / (nblocks_n * nblocks_m);
  const long long xbase = (long long)q * xrows * ldo;
  xform16_tile<BN>(bhi + (long long)q * p, blo + (long long)q * p, nt, cthi, ctlo, npad, ldo, xhi + xbase,
                   xlo + xbase, xrows, mb, nb, sm);
}

// ------------------------------------------------------------------ Coulomb charges from X
//
// gamma_q = <B_q, C C^T> = sum_{m, i} X_q[m][i] C[m][i]: once X is
// half-transformed, the charges of D = C C^T cost one pass over X instead of
// one over B. C is the zero-padded orbital copy in X's row layout
// ([npad][ldo]; FP64 for X in FP64, FP32 otherwise). Workgroup (q, g) sums
// rows [kChargeRows g, kChargeRows (g + 1)) of X_q into parts[q][g];
// charge_reduce_kernel adds the parts in a fixed order.
// F: 0 = X in FP64, 1 = FP32, 2 = BF16x3 (hi plane, then lo plane `plane`
// elements later), 3 = BF16x3 interleaved (each row as ldo / 32 blocks of 32
// hi then 32 lo values).
constexpr int kChargeRows = 128;

// V consecutive X values from element idx (16 bytes of the plane, or of each
// plane for BF16x3), as doubles.
template <int F>
struct XVec {
  static constexpr int V = F == 0 ? 2 : F == 1 ? 4 : 8;
  // Element (row m, column i) of X_q: F 0-2 row-major [xrows][ldo] per plane; F 3 (BF16x3
  // interleaved) [xrows][ldo / 32][64], hi then lo per 32-column block.
  static __device__ __forceinline__ long long index(long long xq, int m, int i, int ldo) {
    if constexpr (F == 3)
      return 2 * xq + (long long)m * 2 * ldo + (i >> 5) * 64 + (i & 31);
    else
      return xq + (long long)m * ldo + i;
  }
  static __device__ __forceinline__ void load(const void* __restrict__ x, long long plane, long long idx,
                                              double (&out)[V]) {
    if constexpr (F == 0) {
      const double2 v = *(const double2*)((const double*)x + idx);
      out[0] = v.x;
      out[1] = v.y;
    } else if constexpr (F == 1) {
      const float4 v = *(const float4*)((const float*)x + idx);
      out[0] = v.x;
      out[1] = v.y;
      out[2] = v.z;
      out[3] = v.w;
    } else {
      const uint16_t* h = (const uint16_t*)x;
      const uint4 hv = *(const uint4*)(h + idx);
      const uint4 lv = *(const uint4*)(h + idx + (F == 3 ? 32 : plane));
      const uint32_t hw[4] = {hv.x, hv.y, hv.z, hv.w};
      const uint32_t lw[4] = {lv.x, lv.y, lv.z, lv.w};
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const uint16_t hb = (uint16_t)(hw[e >> 1] >> ((e & 1) * 16));
        const uint16_t lb = (uint16_t)(lw[e >> 1] >> ((e & 1) * 16));
        out[e] = (double)f32_of(hb) + (double)f32_of(lb);
      }
    }
  }
};

// V consecutive padded orbital values from element idx, as doubles.
template <typename TC, int V>
__device__ __forceinline__ void load_orbitals(const TC* __restrict__ c, long long idx, double (&out)[V]) {
  if constexpr (sizeof(TC) == 8) {
#pragma unroll
    for (int e = 0; e < V; e += 2) {
      const double2 v = *(const double2*)(c + idx + e);
      out[e] = v.x;
      out[e + 1] = v.y;
    }
  } else {
#pragma unroll
    for (int e = 0; e < V; e += 4) {
      const float4 v = *(const float4*)(c + idx + e);
      out[e] = v.x;
      out[e + 1] = v.y;
      out[e + 2] = v.z;
      out[e + 3] = v.w;
    }
  }
}

// One (aux function, row group) item per workgroup iteration; the grid may
// be smaller than the item count (a capped grid leaves room on every CU for
// the SYRK it runs beside).
template <int F>
__global__ __launch_bounds__(kThreads) void charges_from_x_kernel(const void* __restrict__ x, long long plane, int nao,
                                                                   int xrows, int ldo, const void* __restrict__ cpad,
                                                                   int ngroups, long long nitems,
                                                                   double* __restrict__ parts) {
  typedef typename std::conditional<F == 0, double, float>::type TC;
  const TC* __restrict__ c = (const TC*)cpad;
  __shared__ double red[kThreads / 64];
  for (long long item = blockIdx.x; item < nitems; item += gridDim.x) {
    const int q = (int)(item / ngroups);
    const int g = (int)(item - (long long)q * ngroups);
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const long long xq = (long long)q * xrows * ldo;
    const int m_end = min(nao, (g + 1) * kChargeRows);
    constexpr int V = XVec<F>::V;
    double part = 0.0;
    // Rows [m_begin, m_end) of X_q are one contiguous range of
    // (m_end - m_begin) * ldo elements (F 3: of both parts): the workgroup
    // streams it in 16-byte groups (ldo is a multiple of 32, so no group
    // straddles two rows), group f of thread t being f = t + kThreads j. The
    // padding is zero, so the loop body has no branch and the loads of
    // successive groups overlap.
    const int m_begin = g * kChargeRows;
    const int per_row = ldo / V;
    const int ngroups_blk = (m_end - m_begin) * per_row;
    const int step_m = kThreads / per_row;
    const int step_g = kThreads - step_m * per_row;
    int m = m_begin + (int)threadIdx.x / per_row;
    int gi = (int)threadIdx.x % per_row;  // group within the row
#pragma unroll 4
    for (int f = threadIdx.x; f < ngroups_blk; f += kThreads) {
      const int i0 = gi * V;
      double xv[V], cv[V];
      XVec<F>::load(x, plane, XVec<F>::index(xq, m, i0, ldo), xv);
      load_orbitals<TC, V>(c, (long long)m * ldo + i0, cv);
#pragma unroll
      for (int e = 0; e < V; ++e) part += xv[e] * cv[e];
      m += step_m;
      gi += step_g;
      if (gi >= per_row) {
        gi -= per_row;
        ++m;
      }
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) part += __shfl_xor(part, off);
    if (lane == 0) red[wave] = part;
    __syncthreads();
    if (threadIdx.x == 0) {
      double sum = 0.0;
#pragma unroll
      for (int w = 0; w < kThreads / 64; ++w) sum += red[w];
      parts[item] = sum;
    }
    __syncthreads();
  }
}

// gamma[q] = sum_g parts[q][g], in a fixed order.
__global__ __launch_bounds__(kThreads) void charge_reduce_kernel(const double* __restrict__ parts, int naux,
                                                                  int ngroups, double* __restrict__ gamma) {
  const int q = blockIdx.x * kThreads + threadIdx.x;
  if (q >= naux) return;
  double sum = 0.0;
  for (int g = 0; g < ngroups; ++g) sum += parts[(long long)q * ngroups + g];
  gamma[q] = sum;
}

// Orbitals [nao][nocc] float64 -> transposed split Ct[ldo][npad], zero-padded:
// ILV = false: the hi plane, then the lo plane; ILV = true: each row as
// npad / 32 blocks of 64 (32 hi, then the same 32 lo), the layout of the
// bf16 full copy of B.
template <bool ILV>
__global__ __launch_bounds__(kThreads) void orbitals_bf16x3_kernel(const double* __restrict__ c, int nao, int nocc,
                                                                    int npad, int ldo, uint16_t* __restrict__ hi,
                                                                    uint16_t* __restrict__ lo) {
  const long long total = (long long)npad * ldo;
  for (long long idx = (long long)blockIdx.x * kThreads + threadIdx.x; idx < total;
       idx += (long long)gridDim.x * kThreads) {
    const int i = (int)(idx / npad);
    const int k = (int)(idx % npad);
    const float v = (k < nao && i < nocc) ? (float)c[(long long)k * nocc + i] : 0.0f;
    const uint16_t h = bf16_of(v);
    if constexpr (ILV) {
      const long long o = (long long)i * 2 * npad + (k >> 5) * 64 + (k & 31);
      hi[o] = h;
      hi[o + 32] = bf16_of(v - f32_of(h));
    } else {
      hi[idx] = h;
      lo[idx] = bf16_of(v - f32_of(h));
    }
  }
}

// ------------------------------------------------------------------ SYRK

constexpr int kSyrkTile = 128;

// Split s and tile pair of linear workgroup b (XCD-aware, nsplit % 8 == 0).
__device__ __forceinline__ void syrk_coords(int b, int npairs, int& s, int& pair) {
  const int xcd = b & 7;
  const int slot = b >> 3;
  s = xcd + 8 * (slot / npairs);
  pair = slot % npairs;
}

// Partial slots of split s and the aux functions of slot c. run = 0 (FP64):
// one slot per split, [s naux / nsplit, (s + 1) naux / nsplit). run > 0 (the
// FP32-accumulating modes): slot c holds aux functions [c run, (c + 1) run),
// and split s takes slots [s nslot / nsplit, (s + 1) nslot / nsplit), so an
// FP32 accumulator never sums more than run aux functions whatever the
// split count.
__device__ __forceinline__ void slot_range(int s, int nsplit, int naux, int run, int& cb, int& ce) {
  if (run == 0) {
    cb = s;
    ce = s + 1;
    return;
  }
  const int nslot = (naux + run - 1) / run;
  cb = (int)((long long)s * nslot / nsplit);
  ce = (int)((long long)(s + 1) * nslot / nsplit);
}

__device__ __forceinline__ void slot_aux(int c, int nsplit, int naux, int run, int& qb, int& qe) {
  if (run == 0) {
    qb = (int)((long long)c * naux / nsplit);
    qe = (int)((long long)(c + 1) * naux / nsplit);
    return;
  }
  qb = c * run;
  qe = min(naux, qb + run);
}

template <typename T>
struct SyrkSmem {
  T As[kSyrkTile][kTile + 1];
  T Bs[kSyrkTile][kTile + 1];
};

// FP64 / FP32: one TS x TS tile (row block mb, column block nb; TS = 128, or
// 64 for the small instances of a batch) of sum_{q in [qb, qe)} X_q S X_q^T
// into dst[TS][TS]; x = the instance's X.
template <typename T, int TS = kSyrkTile>
__device__ __forceinline__ void syrk_tile(const T* __restrict__ x, int qb, int qe, int xrows, int ldo,
                                          const double* __restrict__ signs, int mb, int nb, T* __restrict__ dst,
                                          SyrkSmem<T>& sm) {
  static_assert(TS == 64 || TS == 128, "SYRK tiles are 64 or 128 rows");
  constexpr int MI = TS / 32, NI = TS / 32;  // wave tile TS/2 x TS/2
  constexpr int NV = TS / 16;                // 2-element chunks per thread and operand
  auto& As = sm.As;
  auto& Bs = sm.Bs;
  const int t = threadIdx.x;
  const int lane = t & 63;
  const int wave = t >> 6;
  const int wm = wave & 1;
  const int wn = wave >> 1;
  typename Op<T>::acc_t acc[MI][NI];
#pragma unroll
  for (int mi = 0; mi < MI; ++mi)
#pragma unroll
    for (int ni = 0; ni < NI; ++ni)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[mi][ni][r] = (T)0;

  // TS rows x 32 columns per operand = 16 TS 2-element chunks: TS / 16 per
  // thread. The prefetch only copies loaded values into registers; the row
  // masks and the column signs are applied in store(), so the wait for the
  // loads falls at the end of the k step, behind its MFMAs, not at its start.
  typename Op<T>::vec2 ra[NV], rb[NV];
  T sg[2];
  const int nchunk = ldo / kTile;
  const int mrows = min(TS, xrows - mb * TS);
  const int nrows = min(TS, xrows - nb * TS);
  auto load = [&](int q, int i0) {
    const T* xm = x + ((long long)q * xrows + mb * TS) * ldo + i0;
    const T* xn = x + ((long long)q * xrows + nb * TS) * ldo + i0;
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      const int chunk = t + kThreads * v;
      const int row = chunk >> 4;
      const int c2 = (chunk & 15) * 2;
      ra[v] = *(const typename Op<T>::vec2*)(xm + (long long)(row < mrows ? row : 0) * ldo + c2);
      rb[v] = *(const typename Op<T>::vec2*)(xn + (long long)(row < nrows ? row : 0) * ldo + c2);
    }
    // Every chunk of a thread has the same column pair c2 = (t & 15) * 2.
    sg[0] = (T)signs[i0 + (t & 15) * 2];
    sg[1] = (T)signs[i0 + (t & 15) * 2 + 1];
  };
  auto store = [&]() {
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      const int chunk = t + kThreads * v;
      const int row = chunk >> 4;
      const int c2 = (chunk & 15) * 2;
      const T sm = row < mrows ? (T)1 : (T)0;
      const T sn = row < nrows ? (T)1 : (T)0;
      As[row][c2] = ra[v].x * sm;
      As[row][c2 + 1] = ra[v].y * sm;
      Bs[row][c2] = rb[v].x * (sn * sg[0]);
      Bs[row][c2 + 1] = rb[v].y * (sn * sg[1]);
    }
  };

  const int steps = (qe - qb) * nchunk;
  if (steps > 0) {
    load(qb, 0);
    store();
  }
  __syncthreads();
  for (int step = 0; step < steps; ++step) {
    const int nxt = step + 1;
    if (nxt < steps) load(qb + nxt / nchunk, (nxt % nchunk) * kTile);
#pragma unroll
    for (int kk = 0; kk < kTile; kk += 4) {
      const int k = kk + (lane >> 4);
      T af[MI], bf[NI];
#pragma unroll
      for (int mi = 0; mi < MI; ++mi) af[mi] = As[wm * (TS / 2) + mi * 16 + (lane & 15)][k];
#pragma unroll
      for (int ni = 0; ni < NI; ++ni) bf[ni] = Bs[wn * (TS / 2) + ni * 16 + (lane & 15)][k];
#pragma unroll
      for (int mi = 0; mi < MI; ++mi)
#pragma unroll
        for (int ni = 0; ni < NI; ++ni) acc[mi][ni] = Op<T>::mma(af[mi], bf[ni], acc[mi][ni]);
    }
    __syncthreads();
    if (nxt < steps) {
      store();
      __syncthreads();
    }
  }
#pragma unroll
  for (int mi = 0; mi < MI; ++mi)
#pragma unroll
    for (int ni = 0; ni < NI; ++ni) {
      const int col = wn * (TS / 2) + ni * 16 + (lane & 15);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = wm * (TS / 2) + mi * 16 + Op<T>::row(lane, r);
        dst[row * TS + col] = acc[mi][ni][r];
      }
    }
}

template <typename T>
__global__ __launch_bounds__(kThreads) void syrk_kernel(const T* __restrict__ x, int naux, int xrows, int ldo,
                                                         const double* __restrict__ signs, int nsplit, int npairs,
                                                         int run, T* __restrict__ partial) {
  __shared__ SyrkSmem<T> sm;
  int s, pair;
  syrk_coords(blockIdx.x, npairs, s, pair);
  int mb, nb;
  tile_of(pair, mb, nb);
  int cb, ce;
  slot_range(s, nsplit, naux, run, cb, ce);
  for (int c = cb; c < ce; ++c) {
    int qb, qe;
    slot_aux(c, nsplit, naux, run, qb, qe);
    syrk_tile<T>(x, qb, qe, xrows, ldo, signs, mb, nb,
                 partial + ((long long)c * npairs + pair) * (kSyrkTile * kSyrkTile), sm);
  }
}

// ---------------------------------------------- SYRK over direct LDS loads
//
// FP64 / FP32 SYRK whose operand rows go from global memory straight into
// LDS (global_load_lds_dwordx4, gfx950), through a ring of kDmaStages stages:
// the loads of the next two k steps are in flight while one step computes
// and the first operands of the following step are read, no registers
// stage them, and each k step has one barrier.
//
// A stage holds CH chunks of k of the 128 rows of both operands as
// 1 KB chunks (one load instruction of one wave; lane l fills bytes
// [16 l, 16 l + 16)): chunk = 16 rows x 4 groups of 16 bytes along k, lane l
// carrying row l % 16 and group l / 16. The MFMA side reads a chunk back
// with one 16-byte LDS read per lane, lane l again getting row l % 16, group
// l / 16 (a contiguous, conflict-free 1 KB read). Element e of the group
// feeds MFMA e: that MFMA sums over k = E (l / 16) + e, a permutation of the
// chunk's k that both operands share, so the E MFMAs together sum all of it.
//
// CH = 2 (32 KB stages, 128 KB ring): one workgroup per CU, so one wave per
// SIMD, which measured at most 86 % of the FP64 MFMA rate even without any
// memory traffic. CH = 1 (16 KB stages, 64 KB ring, no sign table): two
// workgroups per CU, two waves per SIMD that fill each other's barrier and
// LDS-read gaps (99 % in the same measurement).
constexpr int kDmaStages = 4;
constexpr int kDmaMaxLdo = 2048;

template <typename T, int CH>
struct SyrkDma {
  static constexpr int E = 16 / (int)sizeof(T);       // elements per 16-byte group
  static constexpr int CHUNK = 1024 / (int)sizeof(T);  // elements per 1 KB chunk
  static constexpr int KC = 4 * E;                      // k per chunk
  static constexpr int KS = CH * KC;                    // k per stage (CH chunks per 16-row block)
  static constexpr int STAGE = 16 * CH * CHUNK;         // 2 operands x 8 row blocks x CH chunks
  static constexpr int LOADS = 4 * CH;                  // load instructions per wave per stage
  typedef T unit __attribute__((ext_vector_type(16 / sizeof(T))));
};

// The ring: acc += sum over `steps` k steps of (A rows) x (B rows)^T, the
// 128 rows of each operand read at step k from src(k, operand) plus this
// lane's byte offsets off[] (operand A = chunks of waves 0-1, B = waves 2-3).
// With SIGNED, the B operand's k values are scaled by sgn[sign_at(k) + k']
// times scale_at(k) (one factor per step).
//
// Wave (wm, wn) computes the 16 x 16 blocks (wm + 2 mi, wn + 2 ni) of the
// tile, and the MFMAs of block (mi, ni) run only where bit 4 mi + ni of its
// wave-uniform mask is set (the skipped accumulators stay as they were): tiles
// at the edge of the matrix skip their padding, diagonal SYRK tiles their
// upper triangle. Interleaving the blocks over the waves rather than giving
// each a 64 x 64 quadrant spreads what is left over the four SIMDs: a
// diagonal tile takes 10 of 16 blocks' time and one with 2 of 8 row blocks 4
// of 16, where quadrants took 16 and 8. An FP64 MFMA holds its SIMD for 64
// cycles, an FP32 one for 32, so the branches around them are free.
template <typename T, bool SIGNED, int CH, typename Src, typename SignAt, typename ScaleAt>
__device__ __forceinline__ void dma_ring(const Src& src, const int (&off)[4 * CH], int steps,
                                         const T* __restrict__ sgn, const SignAt& sign_at, const ScaleAt& scale_at,
                                         typename Op<T>::acc_t (&acc)[4][4], unsigned mask) {
  typedef SyrkDma<T, CH> D;
  typedef typename D::unit unit;
  constexpr int E = D::E;
  constexpr int LOADS = D::LOADS;
  __shared__ __attribute__((aligned(16))) T st0[D::STAGE];
  __shared__ __attribute__((aligned(16))) T st1[D::STAGE];
  __shared__ __attribute__((aligned(16))) T st2[D::STAGE];
  __shared__ __attribute__((aligned(16))) T st3[D::STAGE];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave & 1;
  const int wn = wave >> 1;
  const int operand = wave >> 1;  // the chunks of waves 0-1 are A's, of waves 2-3 B's

  auto issue = [&](int step, T* stage) {
    const T* base = src(step, operand);
#pragma unroll
    for (int v = 0; v < LOADS; ++v)
      __builtin_amdgcn_global_load_lds((const void*)((const char*)base + (unsigned)off[v]),
                                       (lds_void_t*)(stage + (wave * LOADS + v) * D::CHUNK), 16, 0, 0);
  };

  // Operands of one chunk (16 rows x KC k per 16-row block) of a stage, with
  // the column signs applied to the B side.
  auto read_chunk = [&](const T* stage, int step, int c, unit (&a)[4], unit (&b)[4]) {
#pragma unroll
    for (int mi = 0; mi < 4; ++mi) a[mi] = *(const unit*)(stage + ((((wm + 2 * mi) * CH + c) * 64 + lane) * E));
#pragma unroll
    for (int ni = 0; ni < 4; ++ni)
      b[ni] = *(const unit*)(stage + D::STAGE / 2 + ((((wn + 2 * ni) * CH + c) * 64 + lane) * E));
    if constexpr (SIGNED) {
      const unit sg = *(const unit*)(sgn + sign_at(step) + c * D::KC + (lane >> 4) * E) * scale_at(step);
#pragma unroll
      for (int ni = 0; ni < 4; ++ni) b[ni] *= sg;
    }
  };
  auto mma_chunk = [&](const unit (&a)[4], const unit (&b)[4]) {
#pragma unroll
    for (int e = 0; e < E; ++e)
#pragma unroll
      for (int mi = 0; mi < 4; ++mi)
#pragma unroll
        for (int ni = 0; ni < 4; ++ni) {
          if (!((mask >> (4 * mi + ni)) & 1u)) continue;
          acc[mi][ni] = Op<T>::mma(a[mi][e], b[ni][e], acc[mi][ni]);
        }
  };

  // Step k: wait until this wave's loads of stage k + 1 have landed (those
  // of stage k + 2 stay in flight) and every LDS read issued so far has
  // returned; after the barrier every wave's loads of stages k and k + 1 are
  // in LDS and nobody reads stage k - 1 any more, so its buffer takes the
  // loads of step k + 3. The first chunk of stage k is already in registers
  // (read during step k - 1). With CH = 2 the step reads its second chunk,
  // runs the first chunk's MFMAs, reads the first chunk of stage k + 1, then
  // runs the second chunk's MFMAs; with CH = 1 it reads stage k + 1's chunk
  // into the other register set while the MFMAs of stage k run. Either way
  // no MFMA waits for an LDS read after the barrier.
  // Past the last step the loads repeat the last stage into buffers nobody
  // reads and the MFMAs are skipped, so there are only the seven load sites
  // below, each naming its stage buffer statically: the compiler then tells
  // the stages being read from the ones being loaded and adds no wait of its
  // own.
  unit a0[4], b0[4], a1[4], b1[4];
  // odd: which register set holds stage k's first chunk (CH = 1 alternates).
  auto step_body = [&](int k, const T* cur, const T* next, T* free, bool odd) {
    // Keep the previous step's MFMAs ahead of the wait: issued before it,
    // they keep the matrix pipe busy while the wave waits at the barrier.
    __builtin_amdgcn_sched_barrier(0);
    wait_vm_lgkm0<LOADS>();
    barrier_nofence();
    issue(min(k + 3, steps - 1), free);
    if (k < steps) {
      if constexpr (CH == 2) {
        read_chunk(cur, k, 1, a1, b1);
        mma_chunk(a0, b0);
        read_chunk(next, k + 1, 0, a0, b0);
        mma_chunk(a1, b1);
      } else if (!odd) {
        read_chunk(next, k + 1, 0, a1, b1);
        mma_chunk(a0, b0);
      } else {
        read_chunk(next, k + 1, 0, a0, b0);
        mma_chunk(a1, b1);
      }
    }
  };

  if (steps > 0) {
    issue(0, st0);
    issue(min(1, steps - 1), st1);
    issue(min(2, steps - 1), st2);
    wait_vm_lgkm0<2 * LOADS>();
    barrier_nofence();
    read_chunk(st0, 0, 0, a0, b0);
    for (int k = 0; k < steps; k += kDmaStages) {
      step_body(k, st0, st1, st3, false);
      step_body(k + 1, st1, st2, st0, true);
      step_body(k + 2, st2, st3, st1, false);
      step_body(k + 3, st3, st0, st2, true);
    }
    // No load may still be writing this workgroup's LDS when it returns.
    wait_vm_lgkm0<0>();
  }
}

// Mask of dma_ring for wave (wm, wn): blocks below row block nrb and column
// block ncb of the tile and, with `lower`, on or below its diagonal.
__device__ __forceinline__ unsigned block_mask(int wm, int wn, int nrb, int ncb, bool lower) {
  unsigned m = 0;
#pragma unroll
  for (int mi = 0; mi < 4; ++mi)
#pragma unroll
    for (int ni = 0; ni < 4; ++ni) {
      const int r = wm + 2 * mi, c = wn + 2 * ni;
      m |= (unsigned)(r < nrb && c < ncb && (!lower || c <= r)) << (4 * mi + ni);
    }
  return m;
}

// The masked blocks of a wave's accumulators into a row-major 128 x 128 tile.
template <typename T>
__device__ __forceinline__ void store_tile(T* __restrict__ dst, const typename Op<T>::acc_t (&acc)[4][4], int wm,
                                           int wn, int lane, unsigned mask) {
#pragma unroll
  for (int mi = 0; mi < 4; ++mi)
#pragma unroll
    for (int ni = 0; ni < 4; ++ni) {
      if (!((mask >> (4 * mi + ni)) & 1u)) continue;
      const int col = (wn + 2 * ni) * 16 + (lane & 15);
#pragma unroll
      for (int r = 0; r < 4; ++r)
        dst[((wm + 2 * mi) * 16 + Op<T>::row(lane, r)) * kSyrkTile + col] = acc[mi][ni][r];
    }
}

// SIGNED = false: every sign is +1 on the occupied columns (the padded
// columns of X are zero), so the sign table is neither built nor applied.
// Only the blocks of the lower triangle that hold rows of K are computed and
// written.
template <typename T, bool SIGNED, int CH>
__global__ __launch_bounds__(kThreads, 1) void syrk_dma_kernel(
    const T* __restrict__ x, int naux, int nao, int xrows, int ldo, const double* __restrict__ signs,
    const double* __restrict__ auxsign, int shift, int nsplit, int npairs, int run, T* __restrict__ partial) {
  typedef SyrkDma<T, CH> D;
  constexpr int E = D::E;
  constexpr int LOADS = D::LOADS;
  __shared__ __attribute__((aligned(16))) T sgn[SIGNED ? kDmaMaxLdo : 1];

  int s, pair;
  syrk_coords(blockIdx.x, npairs, s, pair);
  int mb, nb;
  tile_of(pair, mb, nb);
  int cb, ce;
  slot_range(s, nsplit, naux, run, cb, ce);
  const int t = threadIdx.x;
  const int lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int wm = wave & 1;
  const int wn = wave >> 1;

  if (SIGNED)
    for (int i = t; i < ldo; i += kThreads) sgn[i] = (T)signs[i];

  // Byte offsets (within one aux function's X, from k = i0) of this lane's
  // group in the wave's LOADS chunks: chunks LOADS wave .. LOADS wave +
  // LOADS - 1 of the 16 CH of a stage (the first 8 CH operand A = row block
  // mb, the rest operand B = row block nb; chunk = CH * (16-row block) + k
  // part). Rows past xrows (the last 128-row block may hold only 64) read
  // row 0 instead: their products land in K rows and columns past nao, which
  // are never read.
  int off[LOADS];
#pragma unroll
  for (int v = 0; v < LOADS; ++v) {
    const int ch = wave * LOADS + v;
    const int blk = ch >= 8 * CH ? nb : mb;
    int row = blk * kSyrkTile + ((ch / CH) % 8) * 16 + (lane & 15);
    row = row < xrows ? row : 0;
    off[v] = (row * ldo + (ch % CH) * D::KC + (lane >> 4) * E) * (int)sizeof(T);
  }
  const int nch = ldo / D::KS;
  auto sign_at = [&](int step) { return (step % nch) * D::KS; };
  const int nblk = (nao + 15) / 16;
  const unsigned mask = block_mask(wm, wn, nblk - 8 * mb, nblk - 8 * nb, mb == nb);

  for (int c = cb; c < ce; ++c) {
    int qb, qe;
    slot_aux(c, nsplit, naux, run, qb, qe);
    const int steps = (qe - qb) * nch;
    // Step k covers k values i0 = (k % nch) KS of aux function qb + k / nch;
    // the second operand reads columns i0 + shift (mod ldo).
    auto src = [&](int step, int operand) -> const T* {
      const int qq = step / nch;
      int i0 = (step - qq * nch) * D::KS;
      if (operand) i0 = (i0 + shift) % ldo;
      return x + (long long)(qb + qq) * xrows * ldo + i0;
    };
    // Per-aux signs (the signature of an indefinite metric), when given.
    auto scale_at = [&](int step) -> T { return auxsign != nullptr ? (T)auxsign[qb + step / nch] : (T)1; };

    typename Op<T>::acc_t acc[4][4];
#pragma unroll
    for (int mi = 0; mi < 4; ++mi)
#pragma unroll
      for (int ni = 0; ni < 4; ++ni)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[mi][ni][r] = (T)0;

    // The sign table is written, and every wave's LDS reads of the previous
    // slot's ring have returned (each ring ends waiting for them), so the
    // stage buffers may take this slot's loads.
    __syncthreads();
    dma_ring<T, SIGNED, CH>(src, off, steps, sgn, sign_at, scale_at, acc, mask);

    T* dst = partial + ((long long)c * npairs + pair) * (kSyrkTile * kSyrkTile);
    store_tile<T>(dst, acc, wm, wn, lane, mask);
  }
}

// One tile (mb, nb) of sum_{q in [qb, qe)} X_q X_q^T on the ring: rows from
// mb edge, columns from nb edge (edge a multiple of 16 up to 128), the first
// kcols columns of X (all signs +1, the others are zero), stored row-major
// with 128 columns into dst; 16-row blocks at or past nrow (X's rows past nao) and blocks above the
// diagonal of a diagonal tile are neither computed nor written. The whole
// workgroup calls it; its LDS reads of an earlier call must have returned (a
// workgroup barrier between calls).
template <typename T, int CH>
__device__ __forceinline__ void syrk_ring_tile(const T* __restrict__ x, int xrows, int ldo, int kcols, int mb, int nb,
                                               int edge, int qb, int qe, T* __restrict__ dst, int nrow) {
  typedef SyrkDma<T, CH> D;
  constexpr int E = D::E;
  constexpr int LOADS = D::LOADS;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave & 1;
  const int wn = wave >> 1;
  // Lane byte offsets within one aux function's X, as in syrk_dma_kernel;
  // rows past xrows read row 0 (their products land in rows never read).
  int off[LOADS];
#pragma unroll
  for (int v = 0; v < LOADS; ++v) {
    const int ch = wave * LOADS + v;
    const int blk = ch >= 8 * CH ? nb : mb;
    int row = blk * edge + ((ch / CH) % 8) * 16 + (lane & 15);
    row = row < xrows ? row : 0;
    off[v] = (row * ldo + (ch % CH) * D::KC + (lane >> 4) * E) * (int)sizeof(T);
  }
  const int nch = (kcols + D::KS - 1) / D::KS;  // ldo is a multiple of KS
  auto src = [&](int step, int operand) -> const T* {
    (void)operand;
    const int qq = step / nch;
    return x + (long long)(qb + qq) * xrows * ldo + (step - qq * nch) * D::KS;
  };
  auto sign_at = [&](int) { return 0; };
  auto scale_at = [&](int) -> T { return (T)1; };
  typename Op<T>::acc_t acc[4][4];
#pragma unroll
  for (int mi = 0; mi < 4; ++mi)
#pragma unroll
    for (int ni = 0; ni < 4; ++ni)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[mi][ni][r] = (T)0;
  const int nblk = (nrow + 15) / 16;
  const int eb = edge / 16;
  const unsigned mask = block_mask(wm, wn, min(eb, nblk - eb * mb), min(eb, nblk - eb * nb), mb == nb);
  dma_ring<T, false, CH>(src, off, (qe - qb) * nch, (const T*)nullptr, sign_at, scale_at, acc, mask);
  store_tile<T>(dst, acc, wm, wn, lane, mask);
}

// The SYRK of unsigned columns (every sign +1) on the two-workgroups-per-CU
// ring. (The signed kernel's sign table, shift and per-aux signs cost
// registers that the FP64 accumulators leave no room for.)
template <typename T>
__global__ __launch_bounds__(kThreads, 2) void syrk_ring_kernel(const T* __restrict__ x, int naux, int nao, int xrows,
                                                                 int ldo, int kcols, int edge, int nsplit, int npairs,
                                                                 int run, T* __restrict__ partial) {
  int s, pair;
  syrk_coords(blockIdx.x, npairs, s, pair);
  int mb, nb;
  tile_of(pair, mb, nb);
  int cb, ce;
  slot_range(s, nsplit, naux, run, cb, ce);
  for (int c = cb; c < ce; ++c) {
    int qb, qe;
    slot_aux(c, nsplit, naux, run, qb, qe);
    __syncthreads();  // the previous slot's LDS reads have returned
    syrk_ring_tile<T, 1>(x, xrows, ldo, kcols, mb, nb, edge, qb, qe,
                         partial + ((long long)c * npairs + pair) * (kSyrkTile * kSyrkTile), nao);
  }
}

// FP64 / FP32 half-transform on the ring, from a full row-major copy of B
// (bfull[q][npad][npad], both triangles) and C^T (ct[ldo][npad], zero past
// nocc and past nao): X_q[m][i] = sum_k B_q[m][k] C^T[i][k], one 128 x 128
// tile (row block mb, column block nb) of one aux function per workgroup.
// Both operands are rows along k, as in the SYRK, so the ring is the same.
// X rows past npad (xrows may exceed it by up to 32) are written as zeros.
template <typename T, int CH>
__global__ __launch_bounds__(kThreads, CH == 1 ? 2 : 1) void xform_dma_kernel(
    const T* __restrict__ bfull, int nao, int npad, const T* __restrict__ ct, int ldo, T* __restrict__ x, int xrows,
    int qbase, int nblocks_n, int nblocks_m, int nwg) {
  typedef SyrkDma<T, CH> D;
  constexpr int E = D::E;
  constexpr int LOADS = D::LOADS;
  const int logical = xcd_remap(blockIdx.x, nwg);
  const int nb = logical % nblocks_n;
  const int mb = (logical / nblocks_n) % nblocks_m;
  const int q = qbase + logical / (nblocks_n * nblocks_m);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave & 1;
  const int wn = wave >> 1;

  // Lane offsets: operand A rows m of B_q (clamped below npad), operand B
  // rows i of C^T (clamped below ldo); both have row stride npad.
  int off[LOADS];
#pragma unroll
  for (int v = 0; v < LOADS; ++v) {
    const int ch = wave * LOADS + v;
    const bool is_b = ch >= 8 * CH;
    int row = (is_b ? nb : mb) * kSyrkTile + ((ch / CH) % 8) * 16 + (lane & 15);
    row = row < (is_b ? ldo : npad) ? row : 0;
    off[v] = (row * npad + (ch % CH) * D::KC + (lane >> 4) * E) * (int)sizeof(T);
  }
  const T* bq = bfull + (long long)q * npad * npad;
  auto src = [&](int step, int operand) -> const T* { return (operand ? ct : bq) + step * D::KS; };
  auto no_sign = [](int) { return 0; };
  auto no_scale = [](int) { return (T)1; };

  typename Op<T>::acc_t acc[4][4];
#pragma unroll
  for (int mi = 0; mi < 4; ++mi)
#pragma unroll
    for (int ni = 0; ni < 4; ++ni)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[mi][ni][r] = (T)0;

  // Blocks past nao stay zero, blocks past ldo are not written.
  const unsigned mask = block_mask(wm, wn, (nao + 15) / 16 - 8 * mb, ldo / 16 - 8 * nb, false);
  dma_ring<T, false, CH>(src, off, npad / D::KS, (const T*)nullptr, no_sign, no_scale, acc, mask);

  T* xq = x + (long long)q * xrows * ldo;
#pragma unroll
  for (int mi = 0; mi < 4; ++mi)
#pragma unroll
    for (int ni = 0; ni < 4; ++ni) {
      const int col = nb * kSyrkTile + (wn + 2 * ni) * 16 + (lane & 15);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = mb * kSyrkTile + (wm + 2 * mi) * 16 + Op<T>::row(lane, r);
        if (row < xrows && col < ldo) xq[(long long)row * ldo + col] = row < npad ? acc[mi][ni][r] : (T)0;
      }
    }
}

// Full row-major copy of tiled packed B in T: out[q][r][c] = B_q[r][c] for
// r, c < npad (both triangles; zero past nao, as the packed padding). One
// workgroup per stored 32 x 32 tile (tr >= tc) of one aux function, in a
// grid-stride loop: the tile is read once, contiguously, written to block
// (tr, tc) and, through LDS, transposed into block (tc, tr), so every global
// access is a run of 32 consecutive elements.
template <typename T>
__global__ __launch_bounds__(kThreads) void expand_full_kernel(const double* __restrict__ packed, long long p,
                                                                int naux, int ntp, int npad, T* __restrict__ out) {
  __shared__ T tile[kTile][kTile + 1];
  const long long jobs = (long long)naux * ntp;
  for (long long job = blockIdx.x; job < jobs; job += gridDim.x) {
    const int q = (int)(job / ntp);
    const int t = (int)(job - (long long)q * ntp);
    int tr = (int)((sqrt(8.0 * (double)t + 1.0) - 1.0) * 0.5);
    while ((tr + 1) * (tr + 2) / 2 <= t) ++tr;
    while (tr * (tr + 1) / 2 > t) --tr;
    const int tc = t - tr * (tr + 1) / 2;
    const double* src = packed + q * p + (long long)t * kTileElems;
    T* oq = out + (long long)q * npad * npad;
    for (int e = threadIdx.x; e < kTileElems; e += kThreads) {
      const int i = e / kTile, j = e % kTile;
      const T v = (T)src[e];
      tile[i][j] = v;
      oq[(long long)(tr * kTile + i) * npad + tc * kTile + j] = v;
    }
    if (tr != tc) {
      __syncthreads();
      for (int e = threadIdx.x; e < kTileElems; e += kThreads) {
        const int i = e / kTile, j = e % kTile;
        oq[(long long)(tc * kTile + i) * npad + tr * kTile + j] = tile[j][i];
      }
    }
    __syncthreads();
  }
}

// The orbitals C [nao][nocc] in the forms a build needs, each where its
// pointer is given, in one pass over the zero-padded [npad][ldo] matrix: the
// matrix itself (pad), its transpose (ct), the MFMA operand order of the
// packed half-transform (frag), and the column signs (+1 by default).
template <typename T>
__global__ __launch_bounds__(kThreads) void prepare_orbitals_kernel(const double* __restrict__ c, int nao, int nocc,
                                                                     int npad, int ldo, T* __restrict__ pad,
                                                                     T* __restrict__ ct, T* __restrict__ frag,
                                                                     ColumnGroups cg, const double* __restrict__ signs_in,
                                                                     double* __restrict__ signs) {
  const long long total = (long long)npad * ldo;
  for (long long idx = (long long)blockIdx.x * kThreads + threadIdx.x; idx < total;
       idx += (long long)gridDim.x * kThreads) {
    const int k = (int)(idx / ldo), i = (int)(idx % ldo);
    const T v = (T)((k < nao && i < nocc) ? c[(long long)k * nocc + i] : 0.0);
    if (pad != nullptr) pad[idx] = v;
    if (ct != nullptr) ct[(long long)i * npad + k] = v;
    if (frag != nullptr && i / 16 < cg.groups * cg.blocks + cg.tail) frag[fragment_index<T>(cg, npad, k, i)] = v;
    if (signs != nullptr && k == 0) signs[i] = i < nocc ? (signs_in != nullptr ? signs_in[i] : 1.0) : 0.0;
  }
}

struct Syrk16Smem {
  uint16_t Ah[kSyrkTile][kRowK];
  uint16_t Al[kSyrkTile][kRowK];
  uint16_t Bh[kSyrkTile][kRowK];
  uint16_t Bl[kSyrkTile][kRowK];
};

// BF16x3: one 128 x 128 FP32 tile of sum_{q in [qb, qe)} X_q S X_q^T.
__device__ __forceinline__ void syrk16_tile(const uint16_t* __restrict__ xhi, const uint16_t* __restrict__ xlo,
                                            int qb, int qe, int xrows, int ldo, const double* __restrict__ signs,
                                            int mb, int nb, float* __restrict__ dst, Syrk16Smem& sm) {
  constexpr int MI = 4, NI = 4;
  auto& Ah = sm.Ah;
  auto& Al = sm.Al;
  auto& Bh = sm.Bh;
  auto& Bl = sm.Bl;
  const int t = threadIdx.x;
  const int lane = t & 63;
  const int wave = t >> 6;
  const int wm = wave & 1;
  const int wn = wave >> 1;
  f4 acc[MI][NI];
#pragma unroll
  for (int mi = 0; mi < MI; ++mi)
#pragma unroll
    for (int ni = 0; ni < NI; ++ni) acc[mi][ni] = f4{0.f, 0.f, 0.f, 0.f};

  // 128 rows x 32 bf16 per plane = 512 16-byte chunks: 2 per thread per plane.
  // As in the FP64/FP32 SYRK, the prefetch only copies: row masks and sign
  // flips are applied in store(), at the end of the k step.
  uint4 rah[2], ral[2], rbh[2], rbl[2];
  double rsg[8];
  const int nchunk = ldo / kTile;
  const int mrows = min(kSyrkTile, xrows - mb * kSyrkTile);
  const int nrows = min(kSyrkTile, xrows - nb * kSyrkTile);
  // Every chunk of a thread has the same column block c8 = (t & 3) * 8.
  const int c8 = (t & 3) * 8;
  auto load = [&](int q, int i0) {
    const long long om = ((long long)q * xrows + mb * kSyrkTile) * ldo + i0;
    const long long on = ((long long)q * xrows + nb * kSyrkTile) * ldo + i0;
#pragma unroll
    for (int v = 0; v < 2; ++v) {
      const int row = (t + kThreads * v) >> 2;
      const long long am = om + (long long)(row < mrows ? row : 0) * ldo + c8;
      const long long an = on + (long long)(row < nrows ? row : 0) * ldo + c8;
      rah[v] = *(const uint4*)(xhi + am);
      ral[v] = *(const uint4*)(xlo + am);
      rbh[v] = *(const uint4*)(xhi + an);
      rbl[v] = *(const uint4*)(xlo + an);
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) rsg[e] = signs[i0 + c8 + e];
  };
  auto store = [&]() {
    // A negative sign flips the sign bit of the element in both planes.
    const uint32_t f0 = (rsg[0] < 0.0 ? 0x8000u : 0u) | (rsg[1] < 0.0 ? 0x80000000u : 0u);
    const uint32_t f1 = (rsg[2] < 0.0 ? 0x8000u : 0u) | (rsg[3] < 0.0 ? 0x80000000u : 0u);
    const uint32_t f2 = (rsg[4] < 0.0 ? 0x8000u : 0u) | (rsg[5] < 0.0 ? 0x80000000u : 0u);
    const uint32_t f3 = (rsg[6] < 0.0 ? 0x8000u : 0u) | (rsg[7] < 0.0 ? 0x80000000u : 0u);
#pragma unroll
    for (int v = 0; v < 2; ++v) {
      const int row = (t + kThreads * v) >> 2;
      const bool okm = row < mrows;
      const bool okn = row < nrows;
      uint4 h = rbh[v], l = rbl[v];
      h.x ^= f0;
      h.y ^= f1;
      h.z ^= f2;
      h.w ^= f3;
      l.x ^= f0;
      l.y ^= f1;
      l.z ^= f2;
      l.w ^= f3;
      *(uint4*)&Ah[row][c8] = mask4(okm, rah[v]);
      *(uint4*)&Al[row][c8] = mask4(okm, ral[v]);
      *(uint4*)&Bh[row][c8] = mask4(okn, h);
      *(uint4*)&Bl[row][c8] = mask4(okn, l);
    }
  };

  const int steps = (qe - qb) * nchunk;
  if (steps > 0) {
    load(qb, 0);
    store();
  }
  __syncthreads();
  for (int step = 0; step < steps; ++step) {
    const int nxt = step + 1;
    if (nxt < steps) load(qb + nxt / nchunk, (nxt % nchunk) * kTile);
    const int kq = 8 * (lane >> 4);
    bf8 ah[MI], al[MI];
#pragma unroll
    for (int mi = 0; mi < MI; ++mi) {
      ah[mi] = lds_bf8(&Ah[wm * 64 + mi * 16 + (lane & 15)][kq]);
      al[mi] = lds_bf8(&Al[wm * 64 + mi * 16 + (lane & 15)][kq]);
    }
#pragma unroll
    for (int ni = 0; ni < NI; ++ni) {
      const bf8 bh = lds_bf8(&Bh[wn * 64 + ni * 16 + (lane & 15)][kq]);
      const bf8 bl = lds_bf8(&Bl[wn * 64 + ni * 16 + (lane & 15)][kq]);
#pragma unroll
      for (int mi = 0; mi < MI; ++mi) acc[mi][ni] = mma3(ah[mi], al[mi], bh, bl, acc[mi][ni]);
    }
    __syncthreads();
    if (nxt < steps) {
      store();
      __syncthreads();
    }
  }
#pragma unroll
  for (int mi = 0; mi < MI; ++mi)
#pragma unroll
    for (int ni = 0; ni < NI; ++ni) {
      const int col = wn * 64 + ni * 16 + (lane & 15);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = wm * 64 + mi * 16 + 4 * (lane >> 4) + r;
        dst[row * kSyrkTile + col] = acc[mi][ni][r];
      }
    }
}

__global__ __launch_bounds__(kThreads) void syrk_bf16x3_kernel(const uint16_t* __restrict__ xhi,
                                                                const uint16_t* __restrict__ xlo, int naux,
                                                                int xrows, int ldo, const double* __restrict__ signs,
                                                                int nsplit, int npairs, int run,
                                                                float* __restrict__ partial) {
  __shared__ __attribute__((aligned(16))) Syrk16Smem sm;
  int s, pair;
  syrk_coords(blockIdx.x, npairs, s, pair);
  int mb, nb;
  tile_of(pair, mb, nb);
  int cb, ce;
  slot_range(s, nsplit, naux, run, cb, ce);
  for (int c = cb; c < ce; ++c) {
    int qb, qe;
    slot_aux(c, nsplit, naux, run, qb, qe);
    syrk16_tile(xhi, xlo, qb, qe, xrows, ldo, signs, mb, nb,
                partial + ((long long)c * npairs + pair) * (kSyrkTile * kSyrkTile), sm);
  }
}

// ------------------------------------------------------------------ BF16x3 on the direct-LDS ring
//
// The bf16 form of the ring: a 1 KB chunk (16 rows x 32 k of bf16, lane l
// carrying row l % 16 and k 8 (l / 16) .. + 8) is exactly one operand of
// v_mfma_f32_16x16x32_bf16, read back by lane l as one 16-byte LDS read. A
// stage holds 32 chunks: for each operand (A = the 128 rows of the first
// block, B = those of the second) its 8 row blocks in the hi and the lo
// plane, 32 KB; four stages fill 128 KB, one workgroup per CU. Wave w loads
// chunks 8 w .. 8 w + 7 (chunk = 16 operand + 2 block + plane), so waves
// 0-1 load A and waves 2-3 B. Each k step of 32 runs 48 MFMAs per wave
// (hi.hi + hi.lo + lo.hi on 4 x 4 output blocks) and reads the next stage's
// operands into the second register set meanwhile; the barrier and wait
// structure is the FP64/FP32 ring's (one barrier per step, the loads of
// two steps ahead in flight).
constexpr int kRing16Loads = 8;              // load instructions per wave per stage
constexpr int kRing16Stage = 32 * 512;       // uint16 elements per stage (32 KB)

struct Ops16 {
  bf8 ah[4], al[4], bh[4], bl[4];
};

// src(step, operand, plane): the uint16 base of operand `operand`'s `plane`
// at step `step`, to which this lane's byte offsets off[v] (row and k part)
// are added. With SIGNED, the B operand's elements are xored with the
// 16-bit masks sgn[sign_at(step) + k'] (0x8000 flips the sign).
template <bool SIGNED, typename Src, typename SignAt>
__device__ __forceinline__ void dma_ring16(const Src& src, const int (&off)[kRing16Loads], int steps,
                                           const uint16_t* __restrict__ sgn, const SignAt& sign_at,
                                           f4 (&acc)[4][4]) {
  __shared__ __attribute__((aligned(16))) uint16_t st0[kRing16Stage];
  __shared__ __attribute__((aligned(16))) uint16_t st1[kRing16Stage];
  __shared__ __attribute__((aligned(16))) uint16_t st2[kRing16Stage];
  __shared__ __attribute__((aligned(16))) uint16_t st3[kRing16Stage];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave & 1;
  const int wn = wave >> 1;
  const int operand = wave >> 1;

  auto issue = [&](int step, uint16_t* stage) {
    const uint16_t* hi = src(step, operand, 0);
    const uint16_t* lo = src(step, operand, 1);
#pragma unroll
    for (int v = 0; v < kRing16Loads; ++v) {
      const uint16_t* base = (v & 1) ? lo : hi;
      __builtin_amdgcn_global_load_lds((const void*)((const char*)base + (unsigned)off[v]),
                                       (lds_void_t*)(stage + (wave * kRing16Loads + v) * 512), 16, 0, 0);
    }
  };
  auto chunk = [&](const uint16_t* stage, int op, int blk, int plane) -> bf8 {
    return lds_bf8(stage + ((op * 16 + blk * 2 + plane) * 512 + lane * 8));
  };
  auto read = [&](const uint16_t* stage, int step, Ops16& o) {
#pragma unroll
    for (int mi = 0; mi < 4; ++mi) {
      o.ah[mi] = chunk(stage, 0, wm * 4 + mi, 0);
      o.al[mi] = chunk(stage, 0, wm * 4 + mi, 1);
    }
#pragma unroll
    for (int ni = 0; ni < 4; ++ni) {
      o.bh[ni] = chunk(stage, 1, wn * 4 + ni, 0);
      o.bl[ni] = chunk(stage, 1, wn * 4 + ni, 1);
    }
    if constexpr (SIGNED) {
      const uint4 m = *(const uint4*)(sgn + sign_at(step) + (lane >> 4) * 8);
#pragma unroll
      for (int ni = 0; ni < 4; ++ni) {
        uint4 h = __builtin_bit_cast(uint4, o.bh[ni]);
        uint4 l = __builtin_bit_cast(uint4, o.bl[ni]);
        h.x ^= m.x; h.y ^= m.y; h.z ^= m.z; h.w ^= m.w;
        l.x ^= m.x; l.y ^= m.y; l.z ^= m.z; l.w ^= m.w;
        o.bh[ni] = __builtin_bit_cast(bf8, h);
        o.bl[ni] = __builtin_bit_cast(bf8, l);
      }
    }
  };
  auto mma = [&](const Ops16& o) {
#pragma unroll
    for (int mi = 0; mi < 4; ++mi)
#pragma unroll
      for (int ni = 0; ni < 4; ++ni) acc[mi][ni] = mma3(o.ah[mi], o.al[mi], o.bh[ni], o.bl[ni], acc[mi][ni]);
  };

  Ops16 r0, r1;
  auto step_body = [&](int k, const uint16_t* next, uint16_t* free, bool odd) {
    __builtin_amdgcn_sched_barrier(0);
    wait_vm_lgkm0<kRing16Loads>();
    barrier_nofence();
    issue(min(k + 3, steps - 1), free);
    if (k < steps) {
      if (!odd) {
        read(next, k + 1, r1);
        mma(r0);
      } else {
        read(next, k + 1, r0);
        mma(r1);
      }
    }
  };
  if (steps > 0) {
    issue(0, st0);
    issue(min(1, steps - 1), st1);
    issue(min(2, steps - 1), st2);
    wait_vm_lgkm0<2 * kRing16Loads>();
    barrier_nofence();
    read(st0, 0, r0);
    for (int k = 0; k < steps; k += 4) {
      step_body(k, st1, st3, false);
      step_body(k + 1, st2, st0, true);
      step_body(k + 2, st3, st1, false);
      step_body(k + 3, st0, st2, true);
    }
    wait_vm_lgkm0<0>();
  }
}

// BF16x3 SYRK over the ring: the tile (mb, nb) of sum_q X_q S X_q^T from the
// hi/lo planes of X ([naux][xrows][ldo] each), partial slots as in the FP32
// SYRK (one per run of `run` aux functions). With SIGNED the sign masks of
// the columns sit in LDS. `shift` rotates the second operand's columns by
// that many (a multiple of 32): sum_k X[m][k] S_k X[n][(k + shift) mod ldo].
template <bool SIGNED>
__global__ __launch_bounds__(kThreads, 1) void syrk16_dma_kernel(const uint16_t* __restrict__ xhi,
                                                                 const uint16_t* __restrict__ xlo, int naux, int xrows,
                                                                 int ldo, const double* __restrict__ signs, int shift,
                                                                 int nsplit, int npairs, int run,
                                                                 float* __restrict__ partial) {
  __shared__ __attribute__((aligned(16))) uint16_t sgn[SIGNED ? kDmaMaxLdo : 8];
  int s, pair;
  syrk_coords(blockIdx.x, npairs, s, pair);
  int mb, nb;
  tile_of(pair, mb, nb);
  int cb, ce;
  slot_range(s, nsplit, naux, run, cb, ce);
  const int t = threadIdx.x;
  const int lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int wm = wave & 1;
  const int wn = wave >> 1;
  if (SIGNED)
    for (int i = t; i < ldo; i += kThreads) sgn[i] = signs[i] < 0.0 ? (uint16_t)0x8000 : (uint16_t)0;

  // Lane byte offsets within one aux function's plane: load v of this wave is
  // chunk 8 wave + v = 16 operand + 2 block + plane.
  int off[kRing16Loads];
#pragma unroll
  for (int v = 0; v < kRing16Loads; ++v) {
    const int ch = wave * kRing16Loads + v;
    const int blk = (ch >> 1) & 7;
    int row = ((ch >> 4) ? nb : mb) * kSyrkTile + blk * 16 + (lane & 15);
    row = row < xrows ? row : 0;
    off[v] = (row * ldo + (lane >> 4) * 8) * 2;
  }
  const int nch = ldo / 32;
  auto sign_at = [&](int step) { return (step % nch) * 32; };
  for (int c = cb; c < ce; ++c) {
    int qb, qe;
    slot_aux(c, nsplit, naux, run, qb, qe);
    auto src = [&](int step, int operand, int plane) -> const uint16_t* {
      const int qq = step / nch;
      int i0 = (step - qq * nch) * 32;
      if (operand) i0 = (i0 + shift) % ldo;
      return (plane ? xlo : xhi) + (long long)(qb + qq) * xrows * ldo + i0;
    };
    f4 acc[4][4];
#pragma unroll
    for (int mi = 0; mi < 4; ++mi)
#pragma unroll
      for (int ni = 0; ni < 4; ++ni) acc[mi][ni] = f4{0.f, 0.f, 0.f, 0.f};
    __syncthreads();  // sign masks written; the previous slot's LDS reads have returned
    dma_ring16<SIGNED>(src, off, (qe - qb) * nch, sgn, sign_at, acc);
    float* dst = partial + ((long long)c * npairs + pair) * (kSyrkTile * kSyrkTile);
#pragma unroll
    for (int mi = 0; mi < 4; ++mi)
#pragma unroll
      for (int ni = 0; ni < 4; ++ni) {
        const int col = wn * 64 + ni * 16 + (lane & 15);
#pragma unroll
        for (int r = 0; r < 4; ++r) dst[(wm * 64 + mi * 16 + 4 * (lane >> 4) + r) * kSyrkTile + col] = acc[mi][ni][r];
      }
  }
}

// One 128 x 128 tile (mb, nb) of sum_{q in [qb, qe)} X_q X_q^T in BF16x3 on
// the ring (all column signs +1) from X's hi/lo planes, stored row-major
// into dst. Called by the whole workgroup, a barrier between calls.
__device__ __forceinline__ void syrk16_ring_tile(const uint16_t* __restrict__ xhi, const uint16_t* __restrict__ xlo,
                                                 int xrows, int ldo, int mb, int nb, int qb, int qe,
                                                 float* __restrict__ dst) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave & 1;
  const int wn = wave >> 1;
  int off[kRing16Loads];
#pragma unroll
  for (int v = 0; v < kRing16Loads; ++v) {
    const int ch = wave * kRing16Loads + v;
    const int blk = (ch >> 1) & 7;
    int row = ((ch >> 4) ? nb : mb) * kSyrkTile + blk * 16 + (lane & 15);
    row = row < xrows ? row : 0;
    off[v] = (row * ldo + (lane >> 4) * 8) * 2;
  }
  const int nch = ldo / 32;
  auto src = [&](int step, int operand, int plane) -> const uint16_t* {
    (void)operand;
    const int qq = step / nch;
    return (plane ? xlo : xhi) + (long long)(qb + qq) * xrows * ldo + (step - qq * nch) * 32;
  };
  auto sign_at = [&](int) { return 0; };
  f4 acc[4][4];
#pragma unroll
  for (int mi = 0; mi < 4; ++mi)
#pragma unroll
    for (int ni = 0; ni < 4; ++ni) acc[mi][ni] = f4{0.f, 0.f, 0.f, 0.f};
  dma_ring16<false>(src, off, (qe - qb) * nch, (const uint16_t*)nullptr, sign_at, acc);
#pragma unroll
  for (int mi = 0; mi < 4; ++mi)
#pragma unroll
    for (int ni = 0; ni < 4; ++ni) {
      const int col = wn * 64 + ni * 16 + (lane & 15);
#pragma unroll
      for (int r = 0; r < 4; ++r) dst[(wm * 64 + mi * 16 + 4 * (lane >> 4) + r) * kSyrkTile + col] = acc[mi][ni][r];
    }
}

// The MFMA core of the BF16x3 kernels with 256 x 256 tiles (eight waves):
// acc += A B^T over `steps` steps of 32 k, A and B each 256 rows of bf16 hi
// and lo planes. Wave w computes rows 128 (w & 1) .. + 128 of A against rows
// 64 (w >> 1) .. + 64 of B (8 x 4 blocks of 16 x 16, 128 FP32 accumulators
// per lane). A stage holds one step of both operands in 1 KB chunks of 16
// rows x 32 k (chunk 32 operand + 2 block + plane, 64 KB); two stages
// alternate, the loads of step k + 1 in flight during step k's MFMAs, so a
// step moves half the bytes per MFMA of the 128 x 128 ring. Waves 0-3 load
// A's chunks, waves 4-7 B's: addr(step, v) is this lane's 16-byte source of
// load v of its wave (chunk 8 wave + v) at that step. The stages are two
// separate LDS arrays, chosen statically (the loop is unrolled by two), which
// lets the compiler see that a step's LDS reads do not touch the stage the
// loads in flight write, so it does not wait for those loads before the
// reads. Called by the whole workgroup; it returns with every load and LDS
// read complete, so the stages may take new loads after the next barrier.
constexpr int kR256Threads = 512;
constexpr int kR256Loads = 8;          // load instructions per wave per stage
constexpr int kR256Stage = 64 * 512;   // uint16 elements per stage (64 KB)

template <bool ILV = false, class Addr>
__device__ __forceinline__ void ring256(const Addr& addr, int steps, f4 (&acc)[8][4]) {
  __shared__ __attribute__((aligned(16))) uint16_t st0[kR256Stage];
  __shared__ __attribute__((aligned(16))) uint16_t st1[kR256Stage];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave & 1;   // row half of A
  const int wn = wave >> 1;  // row quarter of B
  // ILV: chunk 2 block + h of an operand holds rows 8 h .. + 8 of the 16-row block, each row as
  // 8 segments of 16 bytes (logical segment 4 plane + k group, stored at segment logical ^ row),
  // so that the MFMA operand reads of 8 consecutive rows fall in distinct banks.
  const int r8 = lane & 7;
  const int ilv_off = ((lane >> 3) & 1) * 512 + r8 * 64;
  auto chunk = [&](const uint16_t* stage, int op, int blk, int plane) -> bf8 {
    if constexpr (ILV)
      return lds_bf8(stage + ((op * 32 + blk * 2) * 512 + ilv_off + ((plane * 4 + (lane >> 4)) ^ r8) * 8));
    else
      return lds_bf8(stage + ((op * 32 + blk * 2 + plane) * 512 + lane * 8));
  };
  // The wave's 8 row blocks of A in two halves of 4 (operand registers for 4 A blocks at a time).
  auto compute = [&](const uint16_t* stage) {
#pragma unroll
    for (int mh = 0; mh < 2; ++mh) {
      bf8 ah[4], al[4];
#pragma unroll
      for (int mi = 0; mi < 4; ++mi) {
        ah[mi] = chunk(stage, 0, wm * 8 + mh * 4 + mi, 0);
        al[mi] = chunk(stage, 0, wm * 8 + mh * 4 + mi, 1);
      }
#pragma unroll
      for (int ni = 0; ni < 4; ++ni) {
        const bf8 bh = chunk(stage, 1, wn * 4 + ni, 0);
        const bf8 bl = chunk(stage, 1, wn * 4 + ni, 1);
#pragma unroll
        for (int mi = 0; mi < 4; ++mi) acc[mh * 4 + mi][ni] = mma3(ah[mi], al[mi], bh, bl, acc[mh * 4 + mi][ni]);
      }
    }
  };
  auto issue = [&](int step, uint16_t* stage) {
#pragma unroll
    for (int v = 0; v < kR256Loads; ++v)
      __builtin_amdgcn_global_load_lds((const void*)addr(step, v),
                                       (lds_void_t*)(stage + (wave * kR256Loads + v) * 512), 16, 0, 0);
  };
  if (steps <= 0) return;
  issue(0, st0);
  wait_vm_lgkm0<0>();
  barrier_nofence();
  for (int k = 0; k < steps; k += 2) {
    // Past the last step the loads repeat it into the stage no later step reads.
    issue(min(k + 1, steps - 1), st1);
    __builtin_amdgcn_sched_barrier(0);  // the loads go out before the step's MFMAs
    compute(st0);
    __builtin_amdgcn_sched_barrier(0);
    wait_vm_lgkm0<0>();
    barrier_nofence();
    if (k + 1 < steps) {
      issue(min(k + 2, steps - 1), st0);
      __builtin_amdgcn_sched_barrier(0);
      compute(st1);
      __builtin_amdgcn_sched_barrier(0);
      wait_vm_lgkm0<0>();
      barrier_nofence();
    }
  }
}

// BF16x3 SYRK with 256 x 256 tiles: the four 128 x 128 quadrants of a
// 256-row tile pair in one workgroup (ring256). XILV: X interleaved (hi and
// lo per 32-column block, as the 256 x 256 half-transform writes it), loaded
// as whole 128-byte lines into the ring's interleaved chunks (7.5 ms against
// 8.7 from the hi/lo planes at nao 1500 / naux 5000 / nocc 250). Partial slots as in
// syrk16_dma_kernel: the tile's quadrants are written as the partial tiles
// of their 128-row tile pairs (the upper quadrant of a diagonal pair, and
// quadrants past the last 128-row block, are not written). Column signs +1
// (the occupied orbitals).
template <bool XILV>
__global__ __launch_bounds__(kR256Threads, 1) void syrk16_256_kernel(const uint16_t* __restrict__ xhi,
                                                                     const uint16_t* __restrict__ xlo, int naux,
                                                                     int xrows, int ldo, int nsplit, int npairs,
                                                                     int npairs128, int nb128, int run,
                                                                     float* __restrict__ partial) {
  int s, pair;
  syrk_coords(blockIdx.x, npairs, s, pair);
  int mb, nb;
  tile_of(pair, mb, nb);
  int cb, ce;
  slot_range(s, nsplit, naux, run, cb, ce);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave & 1;
  const int wn = wave >> 1;
  // Load v of this wave is chunk 8 wave + v = 32 operand + 2 block + plane (waves 0-3 operand A,
  // the rows of block mb; waves 4-7 operand B, block nb). Rows past xrows read row 0: their
  // products land in rows and columns of K past nao, never read.
  // XILV (X interleaved, hi and lo per 32-column block): load v fills the ring's interleaved
  // chunk 8 wave + v, rows 8 (chunk & 31) .. + 8, lane l the row's segment (l & 7) ^ row.
  int off[kR256Loads];
#pragma unroll
  for (int v = 0; v < kR256Loads; ++v) {
    const int ch = wave * kR256Loads + v;
    if constexpr (XILV) {
      const int r = lane >> 3;
      int row = ((ch >> 5) ? nb : mb) * 256 + (ch & 31) * 8 + r;
      row = row < xrows ? row : 0;
      off[v] = (row * 2 * ldo + ((lane & 7) ^ r) * 8) * 2;
    } else {
      const int blk = (ch >> 1) & 15;
      int row = ((ch >> 5) ? nb : mb) * 256 + blk * 16 + (lane & 15);
      row = row < xrows ? row : 0;
      off[v] = (row * ldo + (lane >> 4) * 8) * 2;
    }
  }
  const int nch = ldo / 32;
  // The partial tile this wave writes into: 128-row tile pair (2 mb + wm, 2 nb + wn / 2), columns
  // 64 (wn & 1) .. + 64 of it.
  const int qr = 2 * mb + wm, qc = 2 * nb + (wn >> 1);
  const bool writes = qr < nb128 && qc < nb128 && qr >= qc;
  for (int c = cb; c < ce; ++c) {
    int qb, qe;
    slot_aux(c, nsplit, naux, run, qb, qe);
    auto addr = [&](int step, int v) -> const char* {
      const int qq = step / nch;
      if constexpr (XILV) {
        const long long base = (long long)(qb + qq) * xrows * 2 * ldo + (step - qq * nch) * 64;
        return (const char*)(xhi + base) + (unsigned)off[v];
      } else {
        const long long base = (long long)(qb + qq) * xrows * ldo + (step - qq * nch) * 32;
        return (const char*)(((v & 1) ? xlo : xhi) + base) + (unsigned)off[v];
      }
    };
    f4 acc[8][4];
#pragma unroll
    for (int mi = 0; mi < 8; ++mi)
#pragma unroll
      for (int ni = 0; ni < 4; ++ni) acc[mi][ni] = f4{0.f, 0.f, 0.f, 0.f};
    // The previous slot's LDS reads and loads have all returned (ring256 ends on a wait for
    // both), so the stages may take this slot's loads once every wave is here.
    __syncthreads();
    ring256<XILV>(addr, (qe - qb) * nch, acc);
    if (writes) {
      // The lane's offset is opaque here, so its 32 store addresses are formed per slot rather than
      // hoisted out of the slot loop (where they would outlive the accumulators' registers).
      int at = (4 * (lane >> 4)) * kSyrkTile + (lane & 15);
      asm volatile("" : "+v"(at));
      float* dst = partial + ((long long)c * npairs128 + tidx(qr, qc)) * (kSyrkTile * kSyrkTile) + (wn & 1) * 64 + at;
#pragma unroll
      for (int mi = 0; mi < 8; ++mi)
#pragma unroll
        for (int ni = 0; ni < 4; ++ni)
#pragma unroll
          for (int r = 0; r < 4; ++r) dst[(mi * 16 + r) * kSyrkTile + ni * 16] = acc[mi][ni][r];
    }
  }
}

// BF16x3 half-transform with 256 x 256 tiles (ring256 with its interleaved
// chunk layout) from the bf16 full copy of B and C^T, both in the
// interleaved layout of xform16_dma_kernel: tile (mb, nb) of X_q into X's
// hi/lo planes, one tile per workgroup. Each load reads whole 128-byte lines
// (8 rows x 32 k, hi and lo): 15.9 ms at nao 1500 / naux 5000 / nocc 250,
// against 17.9 with separate planes (every load then used half of each line
// it touched) and 17.6 with interleaved planes loaded as 16-row half-line
// chunks. Rows of B past npad and of C^T past ldo read row 0; X rows past
// npad (up to xrows) are written as zeros.
template <bool XILV>
__global__ __launch_bounds__(kR256Threads, 1) void xform16_256_kernel(
    const uint16_t* __restrict__ b, int npad, const uint16_t* __restrict__ ct, int ldo, uint16_t* __restrict__ xhi,
    uint16_t* __restrict__ xlo, int xrows, int qbase, int nblocks_n, int nblocks_m, int nwg) {
  const int logical = xcd_remap(blockIdx.x, nwg);
  const int nb = logical % nblocks_n;
  const int mb = (logical / nblocks_n) % nblocks_m;
  const int q = qbase + logical / (nblocks_n * nblocks_m);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave & 1;
  const int wn = wave >> 1;
  // Waves 0-3 load B_q's rows of block mb, waves 4-7 C^T's rows of block nb.
  const bool is_c = wave >= 4;
  // Load v of this wave fills chunk 8 wave + v: rows 8 (chunk & 31) .. + 8 of its operand, lane l
  // the row's 16-byte segment l & 7 (the ring's interleaved chunk layout), i.e. logical segment
  // (l & 7) ^ row of the row's 128-byte line of the step (32 hi, then 32 lo).
  int off[kR256Loads];
#pragma unroll
  for (int v = 0; v < kR256Loads; ++v) {
    const int c32 = (wave * kR256Loads + v) & 31;
    const int r = lane >> 3;
    int row = (is_c ? nb : mb) * 256 + c32 * 8 + r;
    row = row < (is_c ? ldo : npad) ? row : 0;
    off[v] = (row * 2 * npad + ((lane & 7) ^ r) * 8) * 2;
  }
  const uint16_t* src = is_c ? ct : b + (long long)q * 2 * npad * npad;
  auto addr = [&](int step, int v) -> const char* { return (const char*)(src + step * 64) + (unsigned)off[v]; };
  f4 acc[8][4];
#pragma unroll
  for (int mi = 0; mi < 8; ++mi)
#pragma unroll
    for (int ni = 0; ni < 4; ++ni) acc[mi][ni] = f4{0.f, 0.f, 0.f, 0.f};
  ring256<true>(addr, npad / 32, acc);
  // XILV: X_q as [xrows][ldo / 32][64] (hi then lo per 32-column block) from xhi; else the hi
  // plane at xhi, the lo plane at xlo.
  const int ldx = XILV ? 2 * ldo : ldo;                                    // row stride
  auto col_at = [&](int col) { return XILV ? (col >> 5) * 64 + (col & 31) : col; };
  const long long lo_at = XILV ? 32 : (long long)(xlo - xhi);                // lo part from hi
  const long long xbase = (long long)q * xrows * ldx;
  if ((mb + 1) * 256 <= npad && (nb + 1) * 256 <= ldo) {
    // A tile inside X (and inside B's rows): no bounds to check. Column wn 64 + ni 16 + lane & 15
    // stays within one 32-column block for each ni.
    uint16_t* th = xhi + xbase + (long long)(mb * 256 + wm * 128 + 4 * (lane >> 4)) * ldx +
                   col_at(nb * 256 + wn * 64 + (lane & 15));
#pragma unroll
    for (int mi = 0; mi < 8; ++mi)
#pragma unroll
      for (int ni = 0; ni < 4; ++ni)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float v = acc[mi][ni][r];
          const uint16_t h = bf16_of(v);
          const long long o = (mi * 16 + r) * ldx + (XILV ? (ni >> 1) * 64 + (ni & 1) * 16 : ni * 16);
          th[o] = h;
          th[o + lo_at] = bf16_of(v - f32_of(h));
        }
  } else {
#pragma unroll
    for (int mi = 0; mi < 8; ++mi)
#pragma unroll
      for (int ni = 0; ni < 4; ++ni) {
        const int col = nb * 256 + wn * 64 + ni * 16 + (lane & 15);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int row = mb * 256 + wm * 128 + mi * 16 + 4 * (lane >> 4) + r;
          if (row < xrows && col < ldo) {
            const float v = row < npad ? acc[mi][ni][r] : 0.f;
            const uint16_t h = bf16_of(v);
            const long long o = xbase + (long long)row * ldx + col_at(col);
            xhi[o] = h;
            xhi[o + lo_at] = bf16_of(v - f32_of(h));
          }
        }
      }
  }
}

// BF16x3 half-transform over the ring from the bf16 full copy of B (b:
// [naux][npad][npad / 32][64], each 32-column block as 32 hi then the same
// 32 lo) and C^T in the same interleaved layout (ct: [ldo][npad / 32][64]):
// the 128 x 128 tile (mb, nb) of X_q into X's hi/lo planes. A stage's hi and
// lo chunks of a 16-row block come from the two halves of the same 128-byte
// lines.
__global__ __launch_bounds__(kThreads, 1) void xform16_dma_kernel(const uint16_t* __restrict__ b, int npad,
                                                                  const uint16_t* __restrict__ ct, int ldo,
                                                                  uint16_t* __restrict__ xhi, uint16_t* __restrict__ xlo,
                                                                  int xrows, int qbase, int nblocks_n, int nblocks_m,
                                                                  int nwg) {
  const int logical = xcd_remap(blockIdx.x, nwg);
  const int nb = logical % nblocks_n;
  const int mb = (logical / nblocks_n) % nblocks_m;
  const int q = qbase + logical / (nblocks_n * nblocks_m);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave & 1;
  const int wn = wave >> 1;
  int off[kRing16Loads];
#pragma unroll
  for (int v = 0; v < kRing16Loads; ++v) {
    const int ch = wave * kRing16Loads + v;
    const bool is_b = (ch >> 4) != 0;
    const int blk = (ch >> 1) & 7;
    int row = (is_b ? nb : mb) * kSyrkTile + blk * 16 + (lane & 15);
    row = row < (is_b ? ldo : npad) ? row : 0;
    off[v] = (row * 2 * npad + (lane >> 4) * 8) * 2;
  }
  const long long plane = (long long)q * 2 * npad * npad;
  auto src = [&](int step, int operand, int pl) -> const uint16_t* {
    return (operand ? ct : b + plane) + step * 64 + pl * 32;
  };
  auto no_sign = [](int) { return 0; };
  f4 acc[4][4];
#pragma unroll
  for (int mi = 0; mi < 4; ++mi)
#pragma unroll
    for (int ni = 0; ni < 4; ++ni) acc[mi][ni] = f4{0.f, 0.f, 0.f, 0.f};
  dma_ring16<false>(src, off, npad / 32, (const uint16_t*)nullptr, no_sign, acc);
  const long long xbase = (long long)q * xrows * ldo;
#pragma unroll
  for (int mi = 0; mi < 4; ++mi)
#pragma unroll
    for (int ni = 0; ni < 4; ++ni) {
      const int col = nb * kSyrkTile + wn * 64 + ni * 16 + (lane & 15);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = mb * kSyrkTile + wm * 64 + mi * 16 + 4 * (lane >> 4) + r;
        if (row < xrows && col < ldo) {
          const float v = row < npad ? acc[mi][ni][r] : 0.f;
          const uint16_t h = bf16_of(v);
          xhi[xbase + (long long)row * ldo + col] = h;
          xlo[xbase + (long long)row * ldo + col] = bf16_of(v - f32_of(h));
        }
      }
    }
}

// The full bf16 hi/lo copy of the packed FP64 tensor (hi plane [naux][npad][npad], then the lo
// plane): the element split of launch_split (hi = bf16(fp32(b)), lo = bf16(fp32(b) - hi)), tiles
// transposed through LDS as in expand_full_kernel.
__global__ __launch_bounds__(kThreads) void expand_full16_kernel(const double* __restrict__ packed, long long p,
                                                                 int naux, int ntp, int npad,
                                                                 uint16_t* __restrict__ out) {
  __shared__ uint32_t tile[kTile][kTile + 1];
  const long long jobs = (long long)naux * ntp;
  for (long long job = blockIdx.x; job < jobs; job += gridDim.x) {
    const int q = (int)(job / ntp);
    const int t = (int)(job - (long long)q * ntp);
    int tr = (int)((sqrt(8.0 * (double)t + 1.0) - 1.0) * 0.5);
    while ((tr + 1) * (tr + 2) / 2 <= t) ++tr;
    while (tr * (tr + 1) / 2 > t) --tr;
    const int tc = t - tr * (tr + 1) / 2;
    const double* src = packed + q * p + (long long)t * kTileElems;
    const long long oq = (long long)q * 2 * npad * npad;
    for (int e = threadIdx.x; e < kTileElems; e += kThreads) {
      const int i = e / kTile, j = e % kTile;
      const float x = (float)src[e];
      const uint16_t h = bf16_of(x);
      const uint16_t l = bf16_of(x - f32_of(h));
      tile[i][j] = (uint32_t)h | ((uint32_t)l << 16);
      // Row tr 32 + i, column block tc: hi at 64 tc + j, lo 32 further.
      const long long o = oq + (long long)(tr * kTile + i) * 2 * npad + tc * 2 * kTile + j;
      out[o] = h;
      out[o + kTile] = l;
    }
    if (tr != tc) {
      __syncthreads();
      for (int e = threadIdx.x; e < kTileElems; e += kThreads) {
        const int i = e / kTile, j = e % kTile;
        const uint32_t v = tile[j][i];
        const long long o = oq + (long long)(tc * kTile + i) * 2 * npad + tr * 2 * kTile + j;
        out[o] = (uint16_t)(v & 0xFFFFu);
        out[o + kTile] = (uint16_t)(v >> 16);
      }
    }
    __syncthreads();
  }
}

// Sum over the partial slots k = part, part + PARTS, ... of two neighbouring
// elements, eight loads in flight.
template <typename T, int PARTS>
__device__ __forceinline__ double2 slot_sum(const T* __restrict__ src, int part, int nslot, long long stride) {
  typedef T pair_t __attribute__((ext_vector_type(2)));
  double2 sum = make_double2(0.0, 0.0);
  int k = part;
  for (; k + 7 * PARTS < nslot; k += 8 * PARTS) {
    pair_t v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = *(const pair_t*)(src + (long long)(k + u * PARTS) * stride);
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      sum.x += (double)v[u].x;
      sum.y += (double)v[u].y;
    }
  }
  for (; k < nslot; k += PARTS) {
    const pair_t v = *(const pair_t*)(src + (long long)k * stride);
    sum.x += (double)v.x;
    sum.y += (double)v.y;
  }
  return sum;
}

// K from the partial tiles: one workgroup per (lower tile pair, STRIP rows of
// the tile). 64 threads hold a row (two elements each, coalesced) and PARTS
// thread groups share the slots, combined in LDS in a fixed order, so the
// result does not depend on the run. The lower triangle is written to
// K[bm rows][bn columns] and, through the LDS copy, to its mirror
// K[bn rows][bm columns]; elements above the diagonal of a diagonal tile are
// not read (the masked kernels leave them unwritten). Tile (bm, bn) holds K
// from row bm edge and column bn edge on, edge <= 128 rows and columns of it.
// With ANTI (the non-symmetric exchange), S = sum of `partial`'s slots and
// A = sum of `anti`'s: K[m][n] (+)= S + A, K[n][m] (+)= S - A.
//
// Bound by the latency of the slot chain when the tiles are few and the slots
// many (one tile, 304 slots: 16 workgroups walking 304 dependent loads took
// 311 us of a 362 us build at nao 100; 8 groups of 8 loads in flight take the
// chain to a few), by HBM otherwise.
constexpr int kRedThreads = 512;

//
// With COMPLEX (the k-point exchange, one result per blockIdx.y with nslot
// slots each): K[m][n] (+)= S + i A, K[n][m] (+)= S - i A, interleaved.
template <typename T, int STRIP, bool ANTI, bool COMPLEX = false>
__global__ __launch_bounds__(kRedThreads) void syrk_reduce_kernel(const T* __restrict__ partial,
                                                                  const T* __restrict__ anti, int nslot, int npairs,
                                                                  int nao, int edge, int accumulate,
                                                                  double* __restrict__ out) {
  constexpr int PARTS = kRedThreads / (STRIP * (kSyrkTile / 2));
  constexpr int NS = ANTI ? 2 : 1;
  constexpr int LD = kSyrkTile + 2;
  __shared__ __attribute__((aligned(16))) double part_sum[NS][PARTS][STRIP][LD];
  const int pair = blockIdx.x / (kSyrkTile / STRIP);
  const int strip = blockIdx.x % (kSyrkTile / STRIP);
  int bm, bn;
  tile_of(pair, bm, bn);
  const int row0 = bm * edge + strip * STRIP;
  if (strip * STRIP >= edge || row0 >= nao) return;
  const int t = threadIdx.x;
  const int col = (t & (kSyrkTile / 2 - 1)) * 2;
  const int lr = (t / (kSyrkTile / 2)) % STRIP;
  const int part = t / (STRIP * (kSyrkTile / 2));
  const int row = row0 + lr, gcol = bn * edge + col;
  const long long stride = (long long)npairs * (kSyrkTile * kSyrkTile);
  if constexpr (COMPLEX) {
    partial += blockIdx.y * nslot * stride;
    anti += blockIdx.y * nslot * stride;
    out += 2LL * blockIdx.y * nao * nao;
  }
  if (row < nao && col < edge && gcol <= row) {
    const long long at = (long long)pair * (kSyrkTile * kSyrkTile) + (strip * STRIP + lr) * kSyrkTile + col;
    *(double2*)&part_sum[0][part][lr][col] = slot_sum<T, PARTS>(partial + at, part, nslot, stride);
    if constexpr (ANTI)
      *(double2*)&part_sum[1][part][lr][col] = slot_sum<T, PARTS>(anti + at, part, nslot, stride);
  }
  __syncthreads();
  for (int e = t; e < STRIP * kSyrkTile; e += kRedThreads) {
    const int r = e / kSyrkTile, c = e % kSyrkTile;
    const int gr = row0 + r, gc = bn * edge + c;
    if (gr >= nao || c >= edge || gc > gr) continue;
    double ss = 0.0, aa = 0.0;
#pragma unroll
    for (int q = 0; q < PARTS; ++q) {
      ss += part_sum[0][q][r][c];
      if constexpr (ANTI) aa += part_sum[1][q][r][c];
    }
    const long long o = (long long)gr * nao + gc;
    if constexpr (COMPLEX) {
      if (gr == gc) aa = 0.0;
      double2* k = (double2*)out;
      const double2 old = accumulate ? k[o] : make_double2(0.0, 0.0);
      k[o] = make_double2(old.x + ss, old.y + aa);
      part_sum[0][0][r][c] = ss;
      part_sum[NS - 1][0][r][c] = aa;
    } else {
      out[o] = (ANTI && accumulate ? out[o] : 0.0) + ss + aa;
      part_sum[0][0][r][c] = ss - aa;
    }
  }
  __syncthreads();
  for (int e = t; e < STRIP * kSyrkTile; e += kRedThreads) {
    const int c = e / STRIP, r = e % STRIP;
    const int gr = row0 + r, gc = bn * edge + c;
    if (gr >= nao || c >= edge || gc >= gr) continue;
    const long long o = (long long)gc * nao + gr;
    if constexpr (COMPLEX) {
      double2* k = (double2*)out;
      const double2 old = accumulate ? k[o] : make_double2(0.0, 0.0);
      k[o] = make_double2(old.x + part_sum[0][0][r][c], old.y - part_sum[NS - 1][0][r][c]);
    } else {
      out[o] = (ANTI && accumulate ? out[o] : 0.0) + part_sum[0][0][r][c];
    }
  }
}

template <typename T, int NI>
hipError_t launch_units(const T* b, long long p, int naux, int nao, const T* cf, int ngroups, bool zero_block, T* x,
                        int ldo, int waves, hipStream_t s) {
  const int nt = n_tiles(nao);
  const int units = naux * xform_units_per_aux<T>(nao);
  const long long group_elems = (long long)nt * NI * XFrag<T>::BLOCK;
  // Units per workgroup: about eight k steps each, so that the first loads of a workgroup are a
  // small part of its life, unless that leaves fewer than 1024 workgroups.
  const int most = std::max(1, units / (waves * 1024) * ngroups);
  const int per = waves * std::max(1, std::min(8 / nt, most));
  const long long nwg = (long long)((units + per - 1) / per) * ngroups;
  if (nwg >= (1LL << 24)) return hipErrorInvalidValue;
  hipLaunchKernelGGL((xform_units_kernel<T, NI>), dim3((unsigned)nwg), dim3(64 * waves), 0, s, b, p, nt, cf,
                     group_elems, ngroups, x, x_rows(nao), ldo, units, per, nao, zero_block ? 1 : 0, (int)nwg);
  return hipGetLastError();
}

template <typename T>
hipError_t launch_units_n(int ni, const T* b, long long p, int naux, int nao, const T* cf, int ngroups,
                          bool zero_block, T* x, int ldo, int waves, hipStream_t s) {
  switch (ni) {
    case 1: return launch_units<T, 1>(b, p, naux, nao, cf, ngroups, zero_block, x, ldo, waves, s);
    case 2: return launch_units<T, 2>(b, p, naux, nao, cf, ngroups, zero_block, x, ldo, waves, s);
    case 3: return launch_units<T, 3>(b, p, naux, nao, cf, ngroups, zero_block, x, ldo, waves, s);
    case 4: return launch_units<T, 4>(b, p, naux, nao, cf, ngroups, zero_block, x, ldo, waves, s);
    case 5: return launch_units<T, 5>(b, p, naux, nao, cf, ngroups, zero_block, x, ldo, waves, s);
    case 6: return launch_units<T, 6>(b, p, naux, nao, cf, ngroups, zero_block, x, ldo, waves, s);
    case 7: return launch_units<T, 7>(b, p, naux, nao, cf, ngroups, zero_block, x, ldo, waves, s);
    default: return launch_units<T, 8>(b, p, naux, nao, cf, ngroups, zero_block, x, ldo, waves, s);
  }
}

template <int BN>
hipError_t launch_x16_t(const uint16_t* bhi, const uint16_t* blo, long long p, int naux, int nao,
                        const uint16_t* cthi, const uint16_t* ctlo, int ldo, uint16_t* xhi, uint16_t* xlo,
                        hipStream_t s) {
  const int nt = n_tiles(nao);
  const int npad = nt * kTile;
  const int xrows = x_rows(nao);
  const int nbm = (xrows + 127) / 128;
  const int nbn = (ldo + BN - 1) / BN;
  const int per = std::max(1, (1 << 24) / (nbn * nbm));
  for (int base = 0; base < naux; base += per) {
    const int count = std::min(per, naux - base);
    const int nwg = nbn * nbm * count;
    hipLaunchKernelGGL((xform_bf16x3_kernel<BN>), dim3((unsigned)nwg), dim3(kThreads), 0, s, bhi, blo, p, nt, cthi,
                       ctlo, npad, ldo, xhi, xlo, xrows, base, nbn, nbm, nwg);
    hipError_t err = hipGetLastError();
    if (err != hipSuccess) return err;
  }
  return hipSuccess;
}

}  // namespace

hipError_t launch_expand_full(const double* packed, long long p, int naux, int nao, int precision, void* out,
                              hipStream_t s) {
  const int npad = n_tiles(nao) * kTile;
  const int ntp = (int)n_tile_pairs(nao);
  const dim3 grid((unsigned)std::min<long long>((long long)naux * ntp, 1 << 20));
  if (precision == HFJK_FP64)
    hipLaunchKernelGGL(expand_full_kernel<double>, grid, dim3(kThreads), 0, s, packed, p, naux, ntp, npad,
                       (double*)out);
  else if (precision == HFJK_FP32)
    hipLaunchKernelGGL(expand_full_kernel<float>, grid, dim3(kThreads), 0, s, packed, p, naux, ntp, npad,
                       (float*)out);
  else
    hipLaunchKernelGGL(expand_full16_kernel, grid, dim3(kThreads), 0, s, packed, p, naux, ntp, npad,
                       (uint16_t*)out);
  return hipGetLastError();
}

bool x16_tiles256(int ldo, int bn16) { return ldo > kSyrkTile && (bn16 == 0 || bn16 == 256); }

hipError_t launch_half_transform_full(const void* bfull, int precision, int naux, int nao, const void* ct, int ldo,
                                      void* x, hipStream_t s, int bn16, bool x_ilv) {
  const int npad = n_tiles(nao) * kTile;
  const int xrows = x_rows(nao);
  if (x_ilv && !(precision == HFJK_BF16X3 && x16_tiles256(ldo, bn16))) return hipErrorInvalidValue;
  if (precision == HFJK_BF16X3 && x16_tiles256(ldo, bn16)) {
    // BF16x3 with more than 128 occupied columns: the 256 x 256 tiles.
    const uint16_t* bh = (const uint16_t*)bfull;
    const uint16_t* ch = (const uint16_t*)ct;
    uint16_t* xh = (uint16_t*)x;
    const long long nx16 = (long long)naux * xrows * ldo;
    const int nbn = (ldo + 255) / 256;
    const int nbm = (xrows + 255) / 256;
    const int per = std::max(1, (1 << 22) / (nbn * nbm));  // keep a launch below 2^32 work-items
    for (int base = 0; base < naux; base += per) {
      const int count = std::min(per, naux - base);
      const int nwg = nbn * nbm * count;
      if (x_ilv)
        hipLaunchKernelGGL(xform16_256_kernel<true>, dim3((unsigned)nwg), dim3(kR256Threads), 0, s, bh, npad, ch, ldo,
                           xh, xh + nx16, xrows, base, nbn, nbm, nwg);
      else
        hipLaunchKernelGGL(xform16_256_kernel<false>, dim3((unsigned)nwg), dim3(kR256Threads), 0, s, bh, npad, ch,
                           ldo, xh, xh + nx16, xrows, base, nbn, nbm, nwg);
      hipError_t err = hipGetLastError();
      if (err != hipSuccess) return err;
    }
    return hipSuccess;
  }
  const int nbn = (ldo + kSyrkTile - 1) / kSyrkTile;
  const int nbm = (xrows + kSyrkTile - 1) / kSyrkTile;
  const int per = std::max(1, (1 << 24) / (nbn * nbm));  // keep a launch below 2^32 work-items
  for (int base = 0; base < naux; base += per) {
    const int count = std::min(per, naux - base);
    const int nwg = nbn * nbm * count;
    if (precision == HFJK_FP64) {
      hipLaunchKernelGGL((xform_dma_kernel<double, 1>), dim3((unsigned)nwg), dim3(kThreads), 0, s,
                         (const double*)bfull, nao, npad, (const double*)ct, ldo, (double*)x, xrows, base, nbn, nbm,
                         nwg);
    } else if (precision == HFJK_FP32) {
      hipLaunchKernelGGL((xform_dma_kernel<float, 1>), dim3((unsigned)nwg), dim3(kThreads), 0, s,
                         (const float*)bfull, nao, npad, (const float*)ct, ldo, (float*)x, xrows, base, nbn, nbm, nwg);
    } else {
      // BF16x3: B and C^T interleaved (hi and lo per 32-column block), X as hi then lo plane.
      uint16_t* xh = (uint16_t*)x;
      const long long nx16 = (long long)naux * xrows * ldo;
      hipLaunchKernelGGL(xform16_dma_kernel, dim3((unsigned)nwg), dim3(kThreads), 0, s, (const uint16_t*)bfull, npad,
                         (const uint16_t*)ct, ldo, xh, xh + nx16, xrows, base, nbn, nbm, nwg);
    }
    hipError_t err = hipGetLastError();
    if (err != hipSuccess) return err;
  }
  return hipSuccess;
}

hipError_t launch_orbitals_bf16x3(const double* c, int nao, int nocc, void* out, hipStream_t s, bool interleaved) {
  const int npad = n_tiles(nao) * kTile;
  const int ldo = occ_ld(nocc);
  const long long n = (long long)npad * ldo;
  uint16_t* hi = (uint16_t*)out;
  if (interleaved)
    hipLaunchKernelGGL(orbitals_bf16x3_kernel<true>, dim3(grid_for(n)), dim3(kThreads), 0, s, c, nao, nocc, npad, ldo,
                       hi, hi + n);
  else
    hipLaunchKernelGGL(orbitals_bf16x3_kernel<false>, dim3(grid_for(n)), dim3(kThreads), 0, s, c, nao, nocc, npad,
                       ldo, hi, hi + n);
  return hipGetLastError();
}

int charge_groups(int nao) { return (nao + kChargeRows - 1) / kChargeRows; }

hipError_t launch_charges_from_x(const void* x, int precision, int naux, int nao, int ldo, const void* cpad,
                                 double* parts, double* gamma, int max_groups, hipStream_t s, bool x_ilv) {
  const int xrows = x_rows(nao);
  const int ng = charge_groups(nao);
  const long long plane = (long long)naux * xrows * ldo;
  const long long nitems = (long long)naux * ng;
  // At most 2^30 workgroups (each loops over its items), or max_groups when set.
  long long groups = std::min<long long>(nitems, 1LL << 30);
  if (max_groups > 0) groups = std::min<long long>(groups, max_groups);
  const dim3 grid((unsigned)groups);
  if (precision == HFJK_FP64)
    hipLaunchKernelGGL(charges_from_x_kernel<0>, grid, dim3(kThreads), 0, s, x, plane, nao, xrows, ldo, cpad, ng,
                       nitems, parts);
  else if (precision == HFJK_FP32)
    hipLaunchKernelGGL(charges_from_x_kernel<1>, grid, dim3(kThreads), 0, s, x, plane, nao, xrows, ldo, cpad, ng,
                       nitems, parts);
  else if (!x_ilv)
    hipLaunchKernelGGL(charges_from_x_kernel<2>, grid, dim3(kThreads), 0, s, x, plane, nao, xrows, ldo, cpad, ng,
                       nitems, parts);
  else
    hipLaunchKernelGGL(charges_from_x_kernel<3>, grid, dim3(kThreads), 0, s, x, plane, nao, xrows, ldo, cpad, ng,
                       nitems, parts);
  hipError_t err = hipGetLastError();
  if (err != hipSuccess) return err;
  hipLaunchKernelGGL(charge_reduce_kernel, dim3((unsigned)((naux + kThreads - 1) / kThreads)), dim3(kThreads), 0, s,
                     parts, naux, ng, gamma);
  return hipGetLastError();
}

int syrk_pairs(int nao) {
  const int nb = (x_rows(nao) + kSyrkTile - 1) / kSyrkTile;
  return nb * (nb + 1) / 2;
}

// FP64 / FP32 on the direct-LDS ring: 32-bit lane offsets within one aux function's X.
static bool syrk_dma_ok(int precision, int nao, int ldo, int kind) {
  return kind != 1 && precision != HFJK_BF16X3 && ldo <= kDmaMaxLdo && (long long)x_rows(nao) * ldo < (1LL << 31);
}

// The rows are cut into ceil(nao / 128) blocks of equal height rather than
// into 128-row blocks and a remainder: nao 288 as 3 x 96 instead of 128, 128
// and 32 gives tiles of 9 and 6 blocks per wave instead of 16, 10, 4 and 1, so
// that the workgroups end together (210 -> 182 us at naux 1356, nocc 60).
int syrk_row_block(int nao) {
  const int nblk = (nao + 15) / 16;
  const int nb = (nblk + 7) / 8;
  return (nblk + nb - 1) / nb * 16;
}

int syrk_edge(int precision, int nao, int ldo, bool is_signed, int kind) {
  return !is_signed && kind != 3 && syrk_dma_ok(precision, nao, ldo, kind) ? syrk_row_block(nao) : kSyrkTile;
}

// Blocks of the busiest wave of tile (r, c), of 16.
static int tile_blocks(int nblk, int eb, int r, int c) {
  int most = 0;
  for (int wm = 0; wm < 2; ++wm)
    for (int wn = 0; wn < 2; ++wn) {
      int count = 0;
      for (int br = wm; br < std::min(eb, nblk - eb * r); br += 2)
        for (int bc = wn; bc < std::min(eb, nblk - eb * c); bc += 2) count += r != c || bc <= br;
      most = std::max(most, count);
    }
  return most;
}

// The split count with the least modelled time. Workgroups go to two slots
// per CU, each XCD taking the splits of its residue, in launch order; a k step
// of a whole tile holds a slot for 1.7 us (32 FP64 or 64 FP32 MFMAs per wave,
// 2048 cycles, two workgroups sharing the SIMDs), a masked one for its share
// but no less than the load pipeline's 0.45 us; each workgroup adds 4 us to
// fill and drain; workgroups drift, so the end is late by a share of the
// longest one; FP64 writes and reads back a partial per split and tile.
// (A fixed target of 2048 workgroups wrote 270 MB of partials whatever the
// size, and at nao 709 / naux 2503 in FP32 left 25 of 104 splits without a
// slot.) Signed columns run one workgroup per CU on 128-row tiles and take the
// same count where their runs are the same: within 9 % of the best of 2048,
// 1024, 512 and 256 workgroups from nao 50 to 1500 (FP64 288 / 1356 / 60 569
// us for 523, the largest distance), where the fixed target took 1180 us there
// and 355 for 32 at 100.
struct SplitModel {
  int npairs, slots;
  bool partials;
  double chunk_steps;
  std::vector<double> step_us;  // of every tile, in launch order
  double step_sum = 0.0, step_max = 0.0;
};

struct SplitCandidate {
  int n8, per, used;
  double alone, least;  // least: no schedule of its jobs ends before
};

// The schedule's end; past `limit` some time that is past it too.
static double split_model_us(const SplitModel& m, const SplitCandidate& c, double limit, std::vector<double>& busy) {
  busy.assign(m.slots, 0.0);  // a heap: the earliest free slot on top
  const double work = c.alone * c.per * m.chunk_steps;
  double end = 0.0;
  for (int s = 0; s < c.used && end <= limit; ++s)
    for (double step : m.step_us) {
      const double t = busy[0] + (work * step + 4.0);
      end = std::max(end, t);
      int at = 0;
      for (int child = 1; child < m.slots; child = 2 * at + 1) {
        child += child + 1 < m.slots && busy[child + 1] < busy[child];
        if (busy[child] >= t) break;
        busy[at] = busy[child];
        at = child;
      }
      busy[at] = t;
    }
  return end;
}

static int modelled_split_count(int precision, int naux, int nao, int ldo, int run, int cus) {
  const int nblk = (nao + 15) / 16, eb = syrk_row_block(nao) / 16;
  const int nb = (nblk + 7) / 8;
  SplitModel m;
  m.npairs = nb * (nb + 1) / 2;
  m.slots = std::max(1, 2 * cus / 8);  // of one XCD
  m.partials = run == 0;
  m.chunk_steps = (double)(run == 0 ? 1 : run) * ldo / (precision == HFJK_FP64 ? 8 : 16);
  const int nslot = run == 0 ? naux : (naux + run - 1) / run;
  const double partial_us = m.npairs * 2.0 * kSyrkTile * kSyrkTile * 8.0 / 5e6;
  for (int r = 0; r < nb && m.npairs <= 1024; ++r)
    for (int c = 0; c <= r; ++c) {
      m.step_us.push_back(std::max(0.45, 1.7 * tile_blocks(nblk, eb, r, c) / 16.0));
      m.step_sum += m.step_us.back();
      m.step_max = std::max(m.step_max, m.step_us.back());
    }
  // The candidates' costs with the schedule's end bounded from below by the mean load of a slot and
  // by the longest job; schedules are formed from the least bound on, until no bound left is below
  // the best of them.
  const int top = std::min((nslot + 7) / 8, m.npairs <= 1024 ? std::max(1, 24 * m.slots / m.npairs) : 1);
  std::vector<SplitCandidate> list;
  for (int n8 = 1; n8 <= top; ++n8) {
    SplitCandidate c;
    c.n8 = n8;
    c.per = (nslot + 8 * n8 - 1) / (8 * n8);  // chunks of the fullest split
    if (n8 > 1 && c.per == (nslot + 8 * n8 - 9) / (8 * n8 - 8)) continue;
    c.used = std::min(n8, (((nslot + c.per - 1) / c.per) + 7) / 8);  // splits of one XCD that hold chunks
    c.alone = c.used * m.npairs * 2 <= m.slots ? 0.58 : 1.0;
    const double work = c.alone * c.per * m.chunk_steps;
    const double longest = work * m.step_max + 4.0;
    const double load = c.used * (work * m.step_sum + 4.0 * m.npairs) / m.slots;
    c.least = std::max(load, longest) + 0.3 * longest + (m.partials ? 8 * n8 * partial_us : 0.0);
    list.push_back(c);
  }
  std::sort(list.begin(), list.end(), [](const SplitCandidate& x, const SplitCandidate& y) { return x.least < y.least; });
  int best = 8;
  double best_us = 1e300;
  std::vector<double> busy;
  for (const SplitCandidate& c : list) {
    if (c.least * (1.0 - 1e-9) > best_us || m.step_us.empty()) break;
    const double longest = c.alone * m.step_max * c.per * m.chunk_steps + 4.0;
    const double rest = 0.3 * longest + (m.partials ? 8 * c.n8 * partial_us : 0.0);
    const double us = split_model_us(m, c, best_us - rest, busy) + rest;
    if (us < best_us || (us == best_us && 8 * c.n8 < best)) {
      best_us = us;
      best = 8 * c.n8;
    }
  }
  return best;
}

// The model takes 1 us at nao 100 and 0.3 ms at 1500, on the host, and every
// call and workspace query of a build asks it: the last answers are kept per
// thread, for as many shapes as a loop over molecules and both spins meets.
int syrk_split_count(int precision, int naux, int nao, int ldo, int run, int cus) {
  struct Shape {
    int precision, naux, nao, ldo, run, cus;
    bool operator==(const Shape& o) const {
      return precision == o.precision && naux == o.naux && nao == o.nao && ldo == o.ldo && run == o.run && cus == o.cus;
    }
  };
  constexpr int kKept = 64;
  static thread_local Shape shapes[kKept];
  static thread_local int splits[kKept], kept = 0, next = 0;
  const Shape shape{precision, naux, nao, ldo, run, cus};
  for (int i = 0; i < kept; ++i)
    if (shapes[i] == shape) return splits[i];
  const int count = modelled_split_count(precision, naux, nao, ldo, run, cus);
  shapes[next] = shape;
  splits[next] = count;
  kept = std::max(kept, next + 1);
  next = (next + 1) % kKept;
  return count;
}

double syrk_instance_us(int precision, int naux, int nao, int nocc, bool ring, double& whole_us) {
  const int nblk = (nao + 15) / 16, nb = (nblk + 7) / 8;
  const bool masked = ring && precision != HFJK_BF16X3;
  const int eb = masked ? syrk_row_block(nao) / 16 : 8;
  const double steps = (double)naux * ((nocc + 7) / 8) * (precision == HFJK_FP64 ? 1.0 : 0.5);
  double sum = 0.0, most = 0.0;
  for (int r = 0; r < nb; ++r)
    for (int c = 0; c <= r; ++c) {
      // BF16x3: about 0.8 us per 32 k of a 128 x 128 tile on its ring, padding included.
      const double us = masked ? std::max(0.45, 1.7 * tile_blocks(nblk, eb, r, c) / 16.0)
                               : precision == HFJK_BF16X3 ? 0.4 : 1.7;
      sum += us;
      most = std::max(most, us);
    }
  whole_us = most * steps;
  return sum * steps;
}

int syrk_tile() { return kSyrkTile; }

// Column tile: the tuned value when one is set, else the smallest of
// 32/64/128/256 that covers ldo.
static int pick_bn(int bn, int ldo) {
  if (bn == 32 || bn == 64 || bn == 128 || bn == 256) return bn;
  return ldo <= 32 ? 32 : ldo <= 64 ? 64 : ldo <= 128 ? 128 : 256;
}

// FP64 / FP32 half-transform from the packed B. bn caps the columns of a
// group (0 = 128, what the accumulators have room for), bm = 64 runs two
// waves per workgroup instead of four. A last group narrower than the others
// runs in a launch of its own.
template <typename T>
hipError_t launch_x_typed(const T* b, long long p, int naux, int nao, const T* cf, int nocc, int ldo, T* x, int bn,
                          int bm, hipStream_t s) {
  const ColumnGroups cg = column_groups(nocc, ldo, bn);
  const int waves = bm == 64 ? 2 : 4;
  const bool zero = cg.groups * cg.blocks + cg.tail < ldo / 16;
  hipError_t e = launch_units_n<T>(cg.blocks, b, p, naux, nao, cf, cg.groups, zero && cg.tail == 0, x, ldo, waves, s);
  if (e != hipSuccess || cg.tail == 0) return e;
  const long long done = (long long)cg.groups * cg.blocks;
  return launch_units_n<T>(cg.tail, b, p, naux, nao, cf + done * n_tiles(nao) * XFrag<T>::BLOCK, 1, zero,
                           x + done * 16, ldo, waves, s);
}

hipError_t launch_half_transform(const void* b, int precision, long long p, int naux, int nao, const void* cf,
                                 int nocc, int ldo, void* x, int bn, int bm, hipStream_t s) {
  if (precision == HFJK_FP64)
    return launch_x_typed<double>((const double*)b, p, naux, nao, (const double*)cf, nocc, ldo, (double*)x, bn, bm, s);
  return launch_x_typed<float>((const float*)b, p, naux, nao, (const float*)cf, nocc, ldo, (float*)x, bn, bm, s);
}

template <int NI = 1>
static hipError_t launch_rows_n(int ni, const double* b, long long rows, int len, int b0, int nblocks, int ngroup,
                                const double* cf, long long group_elems, double* x, int ldo, hipStream_t s) {
  if constexpr (NI < kMaxGroupBlocks) {
    if (ni != NI)
      return launch_rows_n<NI + 1>(ni, b, rows, len, b0, nblocks, ngroup, cf, group_elems, x, ldo, s);
  }
  const long long per = (rows + 63) / 64;
  if (per * nblocks >= (1LL << 24)) return hipErrorInvalidValue;
  hipLaunchKernelGGL(rows_units_kernel<NI>, dim3((unsigned)(per * nblocks)), dim3(kThreads), 0, s, b, rows, len, b0,
                     ngroup, cf, group_elems, x, ldo, (int)per);
  return hipGetLastError();
}

hipError_t launch_rows_transform(const double* b, long long rows, int len, int b0, int nblocks, int ngroup,
                                 const double* frag, int columns, double* x, int ldo, hipStream_t s) {
  const ColumnGroups cg = column_groups(columns, ldo, 0);
  const int kpad = (len + kTile - 1) / kTile * kTile;
  const long long group_elems = (long long)kpad * columns;
  for (int g = 0; g < cg.groups + (cg.tail > 0 ? 1 : 0); ++g) {
    const int ni = g < cg.groups ? cg.blocks : cg.tail;
    const hipError_t e = launch_rows_n(ni, b, rows, len, b0, nblocks, ngroup, frag + (long long)g * cg.blocks * 16 * kpad,
                                       group_elems, x + g * cg.blocks * 16, ldo, s);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

hipError_t launch_prepare_orbitals(const double* c, int nao, int nocc, int precision, void* pad, void* ct, void* frag,
                                   int bn, const double* signs_in, double* signs, hipStream_t s) {
  const int npad = n_tiles(nao) * kTile, ldo = occ_ld(nocc);
  const dim3 grid((unsigned)grid_for((long long)npad * ldo)), blk(kThreads);
  const ColumnGroups cg = column_groups(nocc, ldo, bn);
  if (precision == HFJK_FP64)
    hipLaunchKernelGGL(prepare_orbitals_kernel<double>, grid, blk, 0, s, c, nao, nocc, npad, ldo, (double*)pad,
                       (double*)ct, (double*)frag, cg, signs_in, signs);
  else
    hipLaunchKernelGGL(prepare_orbitals_kernel<float>, grid, blk, 0, s, c, nao, nocc, npad, ldo, (float*)pad,
                       (float*)ct, (float*)frag, cg, signs_in, signs);
  return hipGetLastError();
}

hipError_t launch_half_transform_bf16x3(const uint16_t* b, long long p, int naux, int nao, const void* ct, int ldo,
                                        void* x, int bn, hipStream_t s, const uint16_t* b_lo) {
  bn = pick_bn(bn, ldo);
  const uint16_t* bhi = b;
  const uint16_t* blo = b_lo != nullptr ? b_lo : b + (long long)naux * p;
  const long long nct = (long long)n_tiles(nao) * kTile * ldo;
  const uint16_t* cthi = (const uint16_t*)ct;
  const uint16_t* ctlo = cthi + nct;
  const long long nx = (long long)naux * x_rows(nao) * ldo;
  uint16_t* xhi = (uint16_t*)x;
  uint16_t* xlo = xhi + nx;
  if (bn == 32) return launch_x16_t<32>(bhi, blo, p, naux, nao, cthi, ctlo, ldo, xhi, xlo, s);
  if (bn == 64) return launch_x16_t<64>(bhi, blo, p, naux, nao, cthi, ctlo, ldo, xhi, xlo, s);
  if (bn == 128) return launch_x16_t<128>(bhi, blo, p, naux, nao, cthi, ctlo, ldo, xhi, xlo, s);
  return launch_x16_t<256>(bhi, blo, p, naux, nao, cthi, ctlo, ldo, xhi, xlo, s);
}

int syrk_run_aux(int precision, int ldo) {
  if (precision == HFJK_FP64) return 0;
  return std::max(1, kSyrkRunProducts / std::max(ldo, 1));
}

// A run is one workgroup's least work, and runs of 4096 products leave a small
// build a handful of workgroups (nao 96 / naux 336 / nocc 20: 3 runs of 128
// aux functions, 225 us). Shorter runs only add FP64 sums of partial tiles, so
// they go down to a workgroup per CU, and no further than 128 columns of X,
// eight ring steps, where filling the ring costs as much as the products.
// The XCDs take the runs of 128-row tiles in turn, so their number is a
// multiple of eight: 18 runs of 15 tiles gave some XCDs 45 workgroups for
// their 32 CUs where 16 give each 30 (FP32 600 / 2000 / nocc 30: J and K 1.07
// -> 0.95 ms, signed 1.05 -> 0.83). BF16x3's unsigned 256 x 256 tiles, fewer
// and larger, take as many runs as there are CUs per 128-row tile (a multiple
// of eight below it cost 2 to 3 % from nao 250 to 450).
// Signed columns run one workgroup per CU, so where 4096 products end the runs
// before they fit a round, runs that fill two to four rounds evenly are shorter
// in all (500 / 1750 / 60: 28 runs of 64 in two rounds, 48 of 37 too, 1.22 ->
// 0.99 ms); unsigned ones, two to a CU, fill the gaps themselves and only pay
// for the partials (288 / 1356 / 200: 0.85 -> 0.91).
int syrk_run_for(int precision, int naux, int nao, int ldo, int cus, bool is_signed) {
  const int most = syrk_run_aux(precision, ldo);
  if (most == 0) return 0;
  const int pairs = syrk_pairs(nao), xcd = std::max(1, cus / 8);
  const int least = std::min(most, (128 + ldo - 1) / ldo);
  const bool tiles256 = precision == HFJK_BF16X3 && !is_signed;
  const long long slots = 8 * std::max(1, xcd / pairs);
  const long long even = tiles256 ? ((long long)naux * pairs + cus - 1) / cus : (naux + slots - 1) / slots;
  const int run = (int)std::max<long long>(least, std::min<long long>(most, even));
  if (!is_signed || run < most) return run;
  int best = most;
  double best_us = 1e300;  // rounds of 0.85 us per 16 columns and 4 us to fill and drain, and the partials
  for (long long k = (naux + 8LL * most - 1) / (8LL * most); k * pairs <= 4 * xcd; ++k) {
    const int cut = (int)std::max<long long>(least, (naux + 8 * k - 1) / (8 * k));
    const double us = (k * pairs + xcd - 1) / xcd * (0.85 * cut * ldo / 16 + 4.0) + 8.0 * k * pairs * 0.026;
    if (us < best_us) {
      best_us = us;
      best = cut;
    }
  }
  return best;
}

int syrk_slots(int naux, int run, int nsplit) { return run == 0 ? nsplit : (naux + run - 1) / run; }

bool syrk16_tiles256(int nao, int ldo, bool is_signed, int kind, int shift) {
  return !is_signed && shift == 0 && kind != 1 && kind != 2 && ldo <= kDmaMaxLdo &&
         (long long)x_rows(nao) * ldo * 2 < (1LL << 31);
}

hipError_t launch_syrk(const void* x, int precision, int naux, int nao, int ldo, const double* signs,
                       bool is_signed, int nsplit, int run, void* partial, int kind, hipStream_t s,
                       const double* auxsign, int shift, bool x_ilv, int nocc, int xrows) {
  if (xrows <= 0) xrows = x_rows(nao);
  const int edge = syrk_edge(precision, nao, ldo, is_signed, kind);
  if (nocc <= 0 || nocc > ldo) nocc = ldo;
  const int npairs = syrk_pairs(nao);
  // Per-aux signs are applied by the signed FP64/FP32 direct-LDS kernels only; a column shift by
  // the signed direct-LDS kernels of every precision.
  const bool ring_ok = is_signed && kind != 1 && ldo <= kDmaMaxLdo && (long long)xrows * ldo < (1LL << 30);
  if (auxsign != nullptr && (!ring_ok || precision == HFJK_BF16X3)) return hipErrorInvalidValue;
  const int shift_step = precision == HFJK_FP64 ? 16 : 32;  // columns of a ring step
  if (shift != 0 && (!ring_ok || shift % shift_step != 0 || shift < 0 || shift >= ldo)) return hipErrorInvalidValue;
  const unsigned grid = (unsigned)(npairs * nsplit);
  // The direct-load kernel keeps per-lane element offsets within one aux
  // function's X in 32 bits and the sign table in LDS.
  const bool dma = syrk_dma_ok(precision, nao, ldo, kind);
  // Signed columns need the LDS sign table: the one-workgroup-per-CU ring.
  const bool two_wg = kind != 3 && !is_signed;
  if (dma && precision == HFJK_FP64 && is_signed)
    hipLaunchKernelGGL((syrk_dma_kernel<double, true, 2>), dim3(grid), dim3(kThreads), 0, s, (const double*)x, naux,
                       nao, xrows, ldo, signs, auxsign, shift, nsplit, npairs, run, (double*)partial);
  else if (dma && precision == HFJK_FP64 && two_wg)
    hipLaunchKernelGGL(syrk_ring_kernel<double>, dim3(grid), dim3(kThreads), 0, s, (const double*)x, naux, nao, xrows,
                       ldo, nocc, edge, nsplit, npairs, run, (double*)partial);
  else if (dma && precision == HFJK_FP64)
    hipLaunchKernelGGL((syrk_dma_kernel<double, false, 2>), dim3(grid), dim3(kThreads), 0, s, (const double*)x, naux,
                       nao, xrows, ldo, signs, auxsign, shift, nsplit, npairs, run, (double*)partial);
  else if (dma && is_signed)
    hipLaunchKernelGGL((syrk_dma_kernel<float, true, 2>), dim3(grid), dim3(kThreads), 0, s, (const float*)x, naux,
                       nao, xrows, ldo, signs, auxsign, shift, nsplit, npairs, run, (float*)partial);
  else if (dma && two_wg)
    hipLaunchKernelGGL(syrk_ring_kernel<float>, dim3(grid), dim3(kThreads), 0, s, (const float*)x, naux, nao, xrows,
                       ldo, nocc, edge, nsplit, npairs, run, (float*)partial);
  else if (dma)
    hipLaunchKernelGGL((syrk_dma_kernel<float, false, 2>), dim3(grid), dim3(kThreads), 0, s, (const float*)x, naux,
                       nao, xrows, ldo, signs, auxsign, shift, nsplit, npairs, run, (float*)partial);
  else if (precision == HFJK_FP64)
    hipLaunchKernelGGL(syrk_kernel<double>, dim3(grid), dim3(kThreads), 0, s, (const double*)x, naux, xrows, ldo,
                       signs, nsplit, npairs, run, (double*)partial);
  else if (precision == HFJK_FP32)
    hipLaunchKernelGGL(syrk_kernel<float>, dim3(grid), dim3(kThreads), 0, s, (const float*)x, naux, xrows, ldo, signs,
                       nsplit, npairs, run, (float*)partial);
  else {
    const long long nx = (long long)naux * xrows * ldo;
    const uint16_t* xhi = (const uint16_t*)x;
    const bool ring16 = kind != 1 && ldo <= kDmaMaxLdo && (long long)xrows * ldo * 2 < (1LL << 31);
    // Unsigned (occupied orbitals, no column shift): the 256 x 256 tiles unless the 128-row ring is
    // asked for (kind 2); their grid holds about four workgroups per CU of a 256-CU device.
    if (x_ilv && !syrk16_tiles256(nao, ldo, is_signed, kind, shift)) return hipErrorInvalidValue;
    if (ring16 && !is_signed && shift == 0 && kind != 2 && run > 0) {
      const int nb128 = (xrows + kSyrkTile - 1) / kSyrkTile;
      const int nb256 = (nb128 + 1) / 2;
      const int np256 = nb256 * (nb256 + 1) / 2;
      const int nslot = (naux + run - 1) / run;
      const int ns256 = std::max(8, std::min((nslot + 7) / 8 * 8, 1024 / np256 / 8 * 8));
      if (x_ilv)
        hipLaunchKernelGGL(syrk16_256_kernel<true>, dim3((unsigned)(np256 * ns256)), dim3(kR256Threads), 0, s, xhi,
                           xhi + nx, naux, xrows, ldo, ns256, np256, npairs, nb128, run, (float*)partial);
      else
        hipLaunchKernelGGL(syrk16_256_kernel<false>, dim3((unsigned)(np256 * ns256)), dim3(kR256Threads), 0, s, xhi,
                           xhi + nx, naux, xrows, ldo, ns256, np256, npairs, nb128, run, (float*)partial);
    } else if (ring16 && is_signed)
      hipLaunchKernelGGL(syrk16_dma_kernel<true>, dim3(grid), dim3(kThreads), 0, s, xhi, xhi + nx, naux, xrows, ldo,
                         signs, shift, nsplit, npairs, run, (float*)partial);
    else if (ring16)
      hipLaunchKernelGGL(syrk16_dma_kernel<false>, dim3(grid), dim3(kThreads), 0, s, xhi, xhi + nx, naux, xrows,
                         ldo, signs, 0, nsplit, npairs, run, (float*)partial);
    else
      hipLaunchKernelGGL(syrk_bf16x3_kernel, dim3(grid), dim3(kThreads), 0, s, xhi, xhi + nx, naux, xrows, ldo,
                         signs, nsplit, npairs, run, (float*)partial);
  }
  return hipGetLastError();
}

// Strip height: 8 rows (64-byte runs in the mirror) where that fills the
// device four times over, else 2 and 1 rows, whose workgroups split the slots
// over 4 and 8 thread groups (nao 100: 100 workgroups instead of 13).
template <typename T, bool ANTI>
static hipError_t launch_reduce_t(const T* partial, const T* anti, int nslot, int nao, int edge, bool accumulate,
                                  double* out, hipStream_t s) {
  const int npairs = syrk_pairs(nao);
  const int acc = accumulate ? 1 : 0;
  const dim3 blk(kRedThreads);
  if (npairs * (kSyrkTile / 8) >= 1024)
    hipLaunchKernelGGL((syrk_reduce_kernel<T, 8, ANTI>), dim3((unsigned)(npairs * (kSyrkTile / 8))), blk, 0, s,
                       partial, anti, nslot, npairs, nao, edge, acc, out);
  else if (npairs * (kSyrkTile / 2) >= 512)
    hipLaunchKernelGGL((syrk_reduce_kernel<T, 2, ANTI>), dim3((unsigned)(npairs * (kSyrkTile / 2))), blk, 0, s,
                       partial, anti, nslot, npairs, nao, edge, acc, out);
  else
    hipLaunchKernelGGL((syrk_reduce_kernel<T, 1, ANTI>), dim3((unsigned)(npairs * kSyrkTile)), blk, 0, s, partial,
                       anti, nslot, npairs, nao, edge, acc, out);
  return hipGetLastError();
}

hipError_t launch_syrk_reduce_complex(const double* sym, const double* anti, int nslot, int nao, int nk,
                                      bool accumulate, void* out, hipStream_t s) {
  const int npairs = syrk_pairs(nao);
  hipLaunchKernelGGL((syrk_reduce_kernel<double, 2, true, true>), dim3((unsigned)(npairs * (kSyrkTile / 2)), (unsigned)nk),
                     dim3(kRedThreads), 0, s, sym, anti, nslot, npairs, nao, kSyrkTile, accumulate ? 1 : 0,
                     (double*)out);
  return hipGetLastError();
}

hipError_t launch_syrk_reduce2(const void* sym, const void* anti, int precision, int nslot, int nao,
                               bool accumulate, double* out, hipStream_t s) {
  if (precision == HFJK_FP64)
    return launch_reduce_t<double, true>((const double*)sym, (const double*)anti, nslot, nao, kSyrkTile, accumulate, out,
                                         s);
  return launch_reduce_t<float, true>((const float*)sym, (const float*)anti, nslot, nao, kSyrkTile, accumulate, out, s);
}

hipError_t launch_syrk_reduce(const void* partial, int precision, int nslot, int nao, int edge, double* out,
                              hipStream_t s) {
  if (precision == HFJK_FP64)
    return launch_reduce_t<double, false>((const double*)partial, nullptr, nslot, nao, edge, false, out, s);
  return launch_reduce_t<float, false>((const float*)partial, nullptr, nslot, nao, edge, false, out, s);
}

// ------------------------------------------------------------------ batched (persistent)
//
// Every instance of a batch contributes items to each phase; a fixed grid of
// workgroups pulls items from per-XCD counters (batch_next) until its
// share is exhausted, so instances of very different sizes share one launch
// and balance dynamically.

namespace {

template <int BN>
__global__ __launch_bounds__(kThreads) void batch_xform16_kernel(BatchView v, const uint16_t* __restrict__ b,
                                                                  long long b_plane, const uint16_t* __restrict__ cbase,
                                                                  long long c_plane, uint16_t* __restrict__ xbase,
                                                                  long long x_plane) {
  __shared__ __attribute__((aligned(16))) Xform16Smem<BN> sm;
  const long long* pre = v.prefix + (long long)kPhXform * (v.ninst + 1);
  for (;;) {
    long long end;
    const long long item = batch_next(v.prefix, v.counters, v.ninst, kPhXform, end);
    if (item >= end) break;
    const int i = batch_find(pre, v.ninst, item);
    const BatchInst in = v.insts[i];
    const long long local = item - pre[i];
    const int nb = (int)(local % in.nbn);
    const int mb = (int)((local / in.nbn) % in.nbm);
    const int q = (int)(local / ((long long)in.nbn * in.nbm));
    const uint16_t* hq = b + in.b_off + (long long)q * in.p;
    const uint16_t* ct = cbase + in.cp_off;
    uint16_t* xh = xbase + in.x_off + (long long)q * in.xrows * in.ldo;
    xform16_tile<BN>(hq, hq + b_plane, in.nt, ct, ct + c_plane, in.nt * kTile, in.ldo, xh, xh + x_plane, in.xrows,
                     mb, nb, sm);
  }
}

// FP64 / FP32 half-transform items: in.qg units of one column group.
template <typename T>
__global__ __launch_bounds__(kThreads, 2) void batch_xform_kernel(BatchView v, const T* __restrict__ b,
                                                                  const T* __restrict__ cbase, T* __restrict__ xbase) {
  __shared__ __attribute__((aligned(16))) T lds0[kMaxGroupBlocks * XFrag<T>::BLOCK];
  __shared__ __attribute__((aligned(16))) T lds1[kMaxGroupBlocks * XFrag<T>::BLOCK];
  const long long* pre = v.prefix + (long long)kPhXform * (v.ninst + 1);
  for (;;) {
    long long end;
    const long long item = batch_next(v.prefix, v.counters, v.ninst, kPhXform, end);
    if (item >= end) break;
    const int i = batch_find(pre, v.ninst, item);
    const BatchInst in = v.insts[i];
    const int local = (int)(item - pre[i]);
    const int g = local % in.nbn;
    const int u0 = local / in.nbn * in.qg;
    const int u1 = min(u0 + in.qg, in.naux * xform_units_per_aux<T>(in.nao));
    const ColumnGroups cg = in.cg;
    const int nb = g < cg.groups ? cg.blocks : cg.tail;
    const int block0 = g * cg.blocks;
    const bool zero = g == in.nbn - 1 && block0 + nb < in.ldo / 16;
    const T* bi = b + in.b_off;
    const T* cf = cbase + in.cp_off + (long long)block0 * in.nt * XFrag<T>::BLOCK;
    T* x = xbase + in.x_off + block0 * 16;
#define HFJK_UNITS(N) \
  case N: xform_units<T, N>(bi, in.p, in.nt, cf, x, in.xrows, in.ldo, u0, u1, in.nao, zero, lds0, lds1); break;
    switch (nb) {
      HFJK_UNITS(1) HFJK_UNITS(2) HFJK_UNITS(3) HFJK_UNITS(4)
      HFJK_UNITS(5) HFJK_UNITS(6) HFJK_UNITS(7) HFJK_UNITS(8)
      default: break;
    }
#undef HFJK_UNITS
  }
}

union Xform16SmemAny {
  Xform16Smem<32> s32;
  Xform16Smem<64> s64;
  Xform16Smem<128> s128;
};

__global__ __launch_bounds__(kThreads, 2) void batch_xform16_any_kernel(BatchView v, const uint16_t* __restrict__ b,
                                                                      long long b_plane,
                                                                      const uint16_t* __restrict__ cbase,
                                                                      long long c_plane, uint16_t* __restrict__ xbase,
                                                                      long long x_plane) {
  __shared__ __attribute__((aligned(16))) Xform16SmemAny sm;
  const long long* pre = v.prefix + (long long)kPhXform * (v.ninst + 1);
  for (;;) {
    long long end;
    const long long item = batch_next(v.prefix, v.counters, v.ninst, kPhXform, end);
    if (item >= end) break;
    const int i = batch_find(pre, v.ninst, item);
    const BatchInst in = v.insts[i];
    const long long local = item - pre[i];
    const int nb = (int)(local % in.nbn);
    const int mb = (int)((local / in.nbn) % in.nbm);
    const int q0 = (int)(local / ((long long)in.nbn * in.nbm)) * in.qg;
    const int q1 = min(in.naux, q0 + in.qg);
    const uint16_t* hq = b + in.b_off;
    const uint16_t* ct = cbase + in.cp_off;
    uint16_t* xh = xbase + in.x_off;
    if (in.bn == 32)
      xform16_tiles<32, true>(hq, hq + b_plane, in.p, in.nt, ct, ct + c_plane, in.nt * kTile, in.ldo, xh,
                              xh + x_plane, in.xrows, mb, nb, q0, q1, sm.s32, in.nao, in.nocc);
    else if (in.bn == 64)
      xform16_tiles<64, true>(hq, hq + b_plane, in.p, in.nt, ct, ct + c_plane, in.nt * kTile, in.ldo, xh,
                              xh + x_plane, in.xrows, mb, nb, q0, q1, sm.s64, in.nao, in.nocc);
    else
      xform16_tiles<128, true>(hq, hq + b_plane, in.p, in.nt, ct, ct + c_plane, in.nt * kTile, in.ldo, xh,
                               xh + x_plane, in.xrows, mb, nb, q0, q1, sm.s128, in.nao, in.nocc);
  }
}

// SYRK items of the instances with 128-row tiles whose X offsets fit the
// direct-LDS ring (32-bit byte offsets within one aux function's X): one
// (tile pair, split) per item, the partial layout of batch_syrk_kernel.
template <typename T>
__global__ __launch_bounds__(kThreads, 2) void batch_syrk_ring_kernel(BatchView v, const T* __restrict__ xbase,
                                                                       T* __restrict__ kbase) {
  const long long* pre = v.prefix + (long long)kPhSyrkRing * (v.ninst + 1);
  for (;;) {
    long long end;
    // batch_next's barriers also order this item's LDS loads after the previous item's reads.
    const long long item = batch_next(v.prefix, v.counters, v.ninst, kPhSyrkRing, end);
    if (item >= end) break;
    const int i = batch_find(pre, v.ninst, item);
    const BatchInst in = v.insts[i];
    const long long local = item - pre[i];
    const int pair = (int)(local % in.npairs);
    const int s = (int)(local / in.npairs);
    int mb, nb;
    tile_of(pair, mb, nb);
    const int qb = (int)((long long)s * in.naux / in.nsplit);
    const int qe = (int)((long long)(s + 1) * in.naux / in.nsplit);
    syrk_ring_tile<T, 1>(xbase + in.x_off, in.xrows, in.ldo, in.nocc, mb, nb, in.se, qb, qe,
                         kbase + in.kp_off + ((long long)s * in.npairs + pair) * (kSyrkTile * kSyrkTile), in.nao);
  }
}

template <typename T>
__global__ __launch_bounds__(kThreads) void batch_syrk_kernel(BatchView v, const T* __restrict__ xbase,
                                                               const double* __restrict__ ws64, T* __restrict__ kbase) {
  __shared__ SyrkSmem<T> sm;
  const long long* pre = v.prefix + (long long)kPhSyrk * (v.ninst + 1);
  for (;;) {
    long long end;
    const long long item = batch_next(v.prefix, v.counters, v.ninst, kPhSyrk, end);
    if (item >= end) break;
    const int i = batch_find(pre, v.ninst, item);
    const BatchInst in = v.insts[i];
    const long long local = item - pre[i];
    const int pair = (int)(local % in.npairs);
    const int s = (int)(local / in.npairs);
    int mb, nb;
    tile_of(pair, mb, nb);
    const int qb = (int)((long long)s * in.naux / in.nsplit);
    const int qe = (int)((long long)(s + 1) * in.naux / in.nsplit);
    T* dst = kbase + in.kp_off + ((long long)s * in.npairs + pair) * ((long long)in.st * in.st);
    if (in.st == 64)
      syrk_tile<T, 64>(xbase + in.x_off, qb, qe, in.xrows, in.ldo, ws64 + in.sg_off, mb, nb, dst, sm);
    else
      syrk_tile<T, kSyrkTile>(xbase + in.x_off, qb, qe, in.xrows, in.ldo, ws64 + in.sg_off, mb, nb, dst, sm);
  }
}

__global__ __launch_bounds__(kThreads) void batch_syrk16_kernel(BatchView v, const uint16_t* __restrict__ xbase,
                                                                 long long x_plane, const double* __restrict__ ws64,
                                                                 float* __restrict__ kbase) {
  __shared__ __attribute__((aligned(16))) Syrk16Smem sm;
  const long long* pre = v.prefix + (long long)kPhSyrk * (v.ninst + 1);
  for (;;) {
    long long end;
    const long long item = batch_next(v.prefix, v.counters, v.ninst, kPhSyrk, end);
    if (item >= end) break;
    const int i = batch_find(pre, v.ninst, item);
    const BatchInst in = v.insts[i];
    const long long local = item - pre[i];
    const int pair = (int)(local % in.npairs);
    const int s = (int)(local / in.npairs);
    int mb, nb;
    tile_of(pair, mb, nb);
    const int qb = (int)((long long)s * in.naux / in.nsplit);
    const int qe = (int)((long long)(s + 1) * in.naux / in.nsplit);
    const uint16_t* xh = xbase + in.x_off;
    syrk16_tile(xh, xh + x_plane, qb, qe, in.xrows, in.ldo, ws64 + in.sg_off, mb, nb,
                kbase + in.kp_off + ((long long)s * in.npairs + pair) * (kSyrkTile * kSyrkTile), sm);
  }
}

// The BF16x3 SYRK items on the direct-LDS ring (every instance whose X offsets fit it).
__global__ __launch_bounds__(kThreads, 1) void batch_syrk16_ring_kernel(BatchView v,
                                                                         const uint16_t* __restrict__ xbase,
                                                                         long long x_plane,
                                                                         float* __restrict__ kbase) {
  const long long* pre = v.prefix + (long long)kPhSyrkRing * (v.ninst + 1);
  for (;;) {
    long long end;
    const long long item = batch_next(v.prefix, v.counters, v.ninst, kPhSyrkRing, end);
    if (item >= end) break;
    const int i = batch_find(pre, v.ninst, item);
    const BatchInst in = v.insts[i];
    const long long local = item - pre[i];
    const int pair = (int)(local % in.npairs);
    const int s = (int)(local / in.npairs);
    int mb, nb;
    tile_of(pair, mb, nb);
    const int qb = (int)((long long)s * in.naux / in.nsplit);
    const int qe = (int)((long long)(s + 1) * in.naux / in.nsplit);
    const uint16_t* xh = xbase + in.x_off;
    syrk16_ring_tile(xh, xh + x_plane, in.xrows, in.ldo, mb, nb, qb, qe,
                     kbase + in.kp_off + ((long long)s * in.npairs + pair) * (kSyrkTile * kSyrkTile));
  }
}

// K of every instance from its partial tiles: one item per (lower tile pair,
// strip of 512 elements of the tile), two neighbouring elements per thread
// and eight slots in flight (one element per thread over a serial slot chain,
// the upper triangle reading the tiles by columns: 122 us for 12 water
// clusters). The lower triangle is stored and, through LDS, its mirror.
template <typename T>
__global__ __launch_bounds__(kThreads) void batch_syrk_reduce_kernel(BatchView v, const T* __restrict__ kbase,
                                                                      double* __restrict__ kout) {
  __shared__ __attribute__((aligned(16))) double sum[2 * kThreads];
  const long long* pre = v.prefix + (long long)kPhSyrkReduce * (v.ninst + 1);
  for (long long item = blockIdx.x; item < v.items[kPhSyrkReduce]; item += gridDim.x) {
    const int i = batch_find(pre, v.ninst, item);
    const BatchInst in = v.insts[i];
    const int st = in.st;
    const int rows = 2 * kThreads / st;        // tile rows of a strip
    const int strips = st / rows;              // strips of a tile
    const long long local = item - pre[i];
    const int pair = (int)(local / strips), strip = (int)(local % strips);
    int bm, bn;
    tile_of(pair, bm, bn);
    const int edge = in.se;
    const int row0 = bm * edge + strip * rows;
    if (strip * rows >= edge || row0 >= in.nao) continue;
    const int e = 2 * threadIdx.x;
    const int row = row0 + e / st, col = bn * edge + e % st;
    if (row < in.nao && e % st < edge && col <= row)
      *(double2*)&sum[e] = slot_sum<T, 1>(kbase + in.kp_off + (long long)pair * st * st + (long long)strip * 2 * kThreads + e,
                                          0, in.nsplit, (long long)in.npairs * st * st);
    __syncthreads();
    double* k = kout + in.d_off;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int f = threadIdx.x + u * kThreads;
      const int r = row0 + f / st, c = bn * edge + f % st;
      if (r < in.nao && f % st < edge && c <= r) k[(long long)r * in.nao + c] = sum[f];
      const int mr = row0 + f % rows, mc = bn * edge + f / rows;
      if (mr < in.nao && f / rows < edge && mc < mr) k[(long long)mc * in.nao + mr] = sum[(f % rows) * st + f / rows];
    }
    __syncthreads();
  }
}

}  // namespace

namespace {
// A persistent kernel's grid: a workgroup per item up to `grid`, a multiple of 8.
dim3 persistent_grid(long long items, int grid) {
  return dim3((unsigned)std::max(8LL, std::min<long long>(grid, (items + 7) / 8 * 8)));
}
}  // namespace

hipError_t launch_batch_xform(BatchView v, int precision, int bn, const void* b, long long b_plane, const void* cbase,
                              long long c_plane, void* xbase, long long x_plane, int grid, hipStream_t s) {
  const dim3 g = persistent_grid(v.items[kPhXform], grid), blk(kThreads);
  if (precision == HFJK_FP64) {
    hipLaunchKernelGGL(batch_xform_kernel<double>, g, blk, 0, s, v, (const double*)b, (const double*)cbase,
                       (double*)xbase);
  } else if (precision == HFJK_FP32) {
    hipLaunchKernelGGL(batch_xform_kernel<float>, g, blk, 0, s, v, (const float*)b, (const float*)cbase,
                       (float*)xbase);
  } else {
    // bn = 256: one fixed tile for every instance; otherwise each instance's own tile.
    const uint16_t* bb = (const uint16_t*)b;
    const uint16_t* cb = (const uint16_t*)cbase;
    uint16_t* xb = (uint16_t*)xbase;
    if (bn == 256)
      hipLaunchKernelGGL((batch_xform16_kernel<256>), g, blk, 0, s, v, bb, b_plane, cb, c_plane, xb, x_plane);
    else
      hipLaunchKernelGGL(batch_xform16_any_kernel, g, blk, 0, s, v, bb, b_plane, cb, c_plane, xb, x_plane);
  }
  return hipGetLastError();
}

hipError_t launch_batch_syrk(BatchView v, int precision, const void* xbase, long long x_plane, const double* ws64,
                             void* kbase, int grid, hipStream_t s) {
  const dim3 blk(kThreads);
  // grid = two workgroups per CU, the FP64 / FP32 ring kernel's occupancy; workgroups that find
  // no CU free start late, find their share taken and leave.
  const dim3 ring = persistent_grid(v.items[kPhSyrkRing], grid), staged = persistent_grid(v.items[kPhSyrk], grid);
  const bool any_ring = v.items[kPhSyrkRing] > 0, any_staged = v.items[kPhSyrk] > 0;
  if (precision == HFJK_FP64) {
    if (any_staged)
      hipLaunchKernelGGL(batch_syrk_kernel<double>, staged, blk, 0, s, v, (const double*)xbase, ws64, (double*)kbase);
    if (any_ring)
      hipLaunchKernelGGL(batch_syrk_ring_kernel<double>, ring, blk, 0, s, v, (const double*)xbase, (double*)kbase);
  } else if (precision == HFJK_FP32) {
    if (any_staged)
      hipLaunchKernelGGL(batch_syrk_kernel<float>, staged, blk, 0, s, v, (const float*)xbase, ws64, (float*)kbase);
    if (any_ring)
      hipLaunchKernelGGL(batch_syrk_ring_kernel<float>, ring, blk, 0, s, v, (const float*)xbase, (float*)kbase);
  } else {
    if (any_staged)
      hipLaunchKernelGGL(batch_syrk16_kernel, staged, blk, 0, s, v, (const uint16_t*)xbase, x_plane, ws64,
                         (float*)kbase);
    if (any_ring)
      hipLaunchKernelGGL(batch_syrk16_ring_kernel, ring, blk, 0, s, v, (const uint16_t*)xbase, x_plane, (float*)kbase);
  }
  return hipGetLastError();
}

hipError_t launch_batch_syrk_reduce(BatchView v, int precision, const void* kbase, double* k,
                                    hipStream_t s) {
  const dim3 g = batch_grid(v.items[kPhSyrkReduce]), blk(kThreads);
  if (precision == HFJK_FP64)
    hipLaunchKernelGGL(batch_syrk_reduce_kernel<double>, g, blk, 0, s, v, (const double*)kbase, k);
  else
    hipLaunchKernelGGL(batch_syrk_reduce_kernel<float>, g, blk, 0, s, v, (const float*)kbase, k);
  return hipGetLastError();
}

}  // namespace hfjk
