// TaylorF2 integrand of a row from tables, shared by the block-projected time
// transform (gwl_band.hip) and the inner products (gwl_inner.hip).  A
// wavefront holds its rows' constants; products are written with explicit
// fused multiply-adds so that a row's value does not depend on which kernel
// variant or slot evaluated it.
#pragma once
#include "gwl_device.h"

namespace gwl {

// x - floor(x) in one instruction (v_fract_f64)
__device__ __forceinline__ double fract1(double x) { return __builtin_amdgcn_fract(x); }

template <typename C>
__device__ __forceinline__ C cmul_fma(C a, C b) {
  return cmk<C>(fma(a.x, b.x, -(a.y * b.y)), fma(a.x, b.y, a.y * b.x));
}

// Uniform base plus a 32-bit byte offset: the load's own addressing does the sum.
template <typename V>
__device__ __forceinline__ V load_at(const void* base, unsigned off) {
  return *reinterpret_cast<const V*>(reinterpret_cast<const char*>(base) + off);
}

// Two neighbouring complex values.
template <typename C>
__device__ __forceinline__ void load_pair(const C* p, unsigned off, C* to) {
  if constexpr (sizeof(C) == 8) {
    const float4 v = load_at<float4>(p, off);
    to[0] = cmk<C>(v.x, v.y);
    to[1] = cmk<C>(v.z, v.w);
  } else {
    to[0] = load_at<C>(p, off);
    to[1] = load_at<C>(p, off + sizeof(C));
  }
}

// The integrand is |C_r| exp(-2 pi i phi(f)) [conj(dw_r) + sum_k rho_k
// exp(-2 pi i f (dt_k - dt_r)) conj(dw_k)] with r the row's reference detector
// (its largest amplitude) and phi(f) = Psi(f) / 2pi + f dt_r - arg(C_r) / 2pi
// in float64, without whole cycles before the sin / cos; |C_r| scales the
// row's result.
template <typename T, int ND>
struct Tf2Row {
  static constexpr int NO = ND - 1;
  double c[9];  // c[4] holds c4r
  double dtr;
  double dd[NO > 0 ? NO : 1];  // dt_k - dt_r
  // C_k / C_r, and what rounding it left (a rounding here would shift the
  // whole row's sum; those of single bins average out)
  cplx<T> rho[NO > 0 ? NO : 1];
  cplx<T> rlo[NO > 0 ? NO : 1];
  int ref, kb, ke;
};

template <typename T, int ND>
__device__ __forceinline__ void tf2_row(const RowW& rw, Tf2Row<T, ND>& b) {
#pragma unroll
  for (int k = 0; k < 9; ++k) b.c[k] = rw.c[k];
  b.c[4] = rw.c4r;
  b.ref = rw.ref;
  b.dtr = rw.dt[0];
#pragma unroll
  for (int d = 1; d < ND; ++d)
    if (d == b.ref) b.dtr = rw.dt[d];
#pragma unroll
  for (int k = 0; k < ND - 1; ++k) b.dd[k] = (k < b.ref ? rw.dt[k] : rw.dt[k + 1]) - b.dtr;
  b.kb = rw.kb;
  b.ke = rw.ke;
}

// exp(-2 pi i cycles), rounded, as a rotation applied ``mean`` times on
// average after an exact phase: the rounded factor w (1 + eps) shifts the mean
// by mean eps, which corr takes out.
template <typename T>
__device__ __forceinline__ cplx<T> tf2_rotation(double cycles, double mean, double2& corr) {
  const double2 w = expm2pi(fract1(cycles));
  const cplx<T> r = cmk<cplx<T>>((T)w.x, (T)w.y);
  const double er = 1.0 - mean * (w.x * (double)r.x + w.y * (double)r.y - 1.0);
  const double ei = -mean * (w.x * (double)r.y - w.y * (double)r.x);
  corr = make_double2(corr.x * er - corr.y * ei, corr.x * ei + corr.y * er);
  return r;
}

// rho_k times the rotations' correction and, in float32, the gain of
// tf2_rotated's exponential (the shared one's is in the tables), as a sum of
// two numbers.
template <typename T, int ND>
__device__ __forceinline__ void tf2_rho(const RowW& rw, int k, double2 corr, Tf2Row<T, ND>& b) {
  constexpr double gain = sizeof(T) == 4 ? kExpm2piGain : 1.0;
  const double pr = gain * (rw.rre[k] * corr.x - rw.rim[k] * corr.y);
  const double pi = gain * (rw.rre[k] * corr.y + rw.rim[k] * corr.x);
  b.rho[k] = cmk<cplx<T>>((T)pr, (T)pi);
  b.rlo[k] = cmk<cplx<T>>((T)(pr - (double)b.rho[k].x), (T)(pi - (double)b.rho[k].y));
}

// Cycles without their whole number.  float32: the nearest one is taken off,
// not the one below, which halves the rounding of the fraction: every detector
// of an element shares it, so its errors add up over them.
template <typename T>
__device__ __forceinline__ double tf2_fraction(double x) {
  return sizeof(T) == 4 ? x - __builtin_rint(x) : fract1(x);
}

// rho_k exp(-2 pi i f dd_k)
template <typename T, int ND>
__device__ __forceinline__ cplx<T> tf2_rotated(const Tf2Row<T, ND>& b, int k, double f) {
  const cplx<T> e = expm2pi((T)tf2_fraction<T>(f * b.dd[k]));
  cplx<T> r = cmul_fma(b.rho[k], e);
  if constexpr (sizeof(T) == 4) {
    r.x = fma(b.rlo[k].x, e.x, fma(-b.rlo[k].y, e.y, r.x));
    r.y = fma(b.rlo[k].x, e.y, fma(b.rlo[k].y, e.x, r.y));
  }
  return r;
}

// phi(f) in cycles at a tabled basis point (u = f^1/3, v = f^-1/3, ln f):
// c0 v^5 + c1 v^3 + c2 v^2 + c3 v + c4r + c5 u + c6 u^2 + dt_r u^3 + (c7 + c8 u) ln f
template <typename T, int ND>
__device__ __forceinline__ double tf2_cycles(const Tf2Row<T, ND>& b, double u, double v,
                                             double lf) {
  double a = fma(b.c[0], v * v, b.c[1]);
  a = fma(a, v, b.c[2]);
  a = fma(a, v, b.c[3]);
  double s = fma(a, v, b.c[4]);
  s = fma(fma(fma(b.dtr, u, b.c[6]), u, b.c[5]), u, s);
  return fma(fma(b.c[8], u, b.c[7]), lf, s);
}

// conj(d_r) + sum_k rot_k conj(d_k), times exp(-2 pi i cycles)
template <typename T, int ND>
__device__ __forceinline__ cplx<T> tf2_product(double cycles, const cplx<T>* rot,
                                               const cplx<T> (*d)[2], int i) {
  using C = cplx<T>;
  C y = cmk<C>(d[0][i].x, -d[0][i].y);
#pragma unroll
  for (int k = 0; k < ND - 1; ++k) {
    const C dw = d[k + 1][i];
    y.x = fma(rot[k].x, dw.x, fma(rot[k].y, dw.y, y.x));
    y.y = fma(rot[k].y, dw.x, fma(-rot[k].x, dw.y, y.y));
  }
  return cmul_fma(expm2pi((T)tf2_fraction<T>(cycles)), y);
}

// Rows of one workgroup sorted by reference detector (stable), so that the
// two rows of a wavefront mostly read the detectors' tables in the same
// order: the index (0 .. 7) of the row with rank k.  Lane l < 8 holds row l's
// key.
__device__ __forceinline__ int ranked_row(int key, int lane, int k) {
  const unsigned long long below = (1ull << lane) - 1ull;
  int rank = 0;
#pragma unroll
  for (int d = 0; d <= GWL_MAX_DET; ++d) {
    const unsigned long long m = __ballot(key == d) & 0xffull;
    rank += (d < key) ? __popcll(m) : (d == key ? __popcll(m & below) : 0);
  }
  const unsigned long long at = __ballot(lane < 8 && rank == k) & 0xffull;
  return __builtin_ctzll(at | 0x100ull) & 7;
}

// The wavefront's R of the workgroup's 4 R rows from row0 on, in the order of
// their reference detectors; returns how many are live (dead slots repeat the
// first row).
template <int R>
__device__ __forceinline__ int pick_rows(const RowW* rows, long long row0, long long n, int lane,
                                         int wid, long long* pick) {
  if constexpr (R == 1) {
    pick[0] = row0 + wid;
    return pick[0] < n ? 1 : 0;
  } else {
    static_assert(R == 2, "eight rows a workgroup");
    const long long mine = row0 + lane;
    const int key = (lane < 8 && mine < n) ? rows[mine].ref : GWL_MAX_DET;
    int live = 0;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int at = __builtin_amdgcn_readfirstlane(ranked_row(key, lane, wid * R + r));
      pick[r] = row0 + at;
      if (pick[r] < n) ++live;  // dead rows rank last
    }
#pragma unroll
    for (int r = 1; r < R; ++r)
      if (r >= live) pick[r] = pick[0];
    return live;
  }
}

}  // namespace gwl
