// Time-marginalised TaylorF2 likelihood: the window bins of the transform by
// band-limited block projections on the matrix cores (gfx950).
//
// The reference evaluates d_inner_h_array = 4/T FFT_N of h conj(d) / S and
// keeps the bins inside the time prior (bilby/gw/likelihood/base.py:325-330,
// 794-820): L of N, 0.2 s of the segment.  With jd the window's centre bin and
// kappa = j - jd, |kappa| <= L / 2,
//   X[j] = sum_n x[n] exp(-2 pi i n kappa / N),  x[n] = integrand exp(-2 pi i n jd / N)
// (the data tables carry the exp(.. jd ..) factor).  The N bins are cut into
// NB blocks of B = N / NB bins.  Inside a block exp(-2 pi i t kappa / N) is a
// kernel of time-bandwidth product B L / N = L / NB <= 4, so 16 functions
// reproduce it to rounding:
//   exp(-i c x y) = sum_{p < 16} U_p(x) V_p(y),   x = t / (B/2), y = kappa / (L/2)
// with U_p the prolate spheroidal functions of bandwidth c = pi B L / (2 N)
// (D. Slepian, H. O. Pollak, Bell Syst. Tech. J. 40, 1961) and V_p their
// transforms.  The largest error over t and kappa grows with the window and a
// little with B: for NB = 128 (float32 arithmetic) 5e-11 at L = 420, 1.2e-9 at
// L = 512 (B = 128), 1.2e-10 and 2.9e-9 at B = 1024; for NB = 256 (float64) below
// 2e-15 at L = 420, 1.4e-14 at L = 512 (B = 64), 3.8e-14 at B = 512.  Then
//   C[b][p] = sum_t x[b B + t] U_p(t)              k_band: MFMA, M = 16 blocks, N = 16 p, K = bins
//   D_p[q] = sum_b C[b][p] W_NB^(b q)              k_band_finish: 16 DFTs of NB points
//   X[j] = exp(-i pi (B - 1) kappa / N) sum_p V_p(kappa) D_p[kappa mod NB]
//
// Lane l of a wavefront evaluates the integrand of bin t = 4 s + l / 16 of
// block l mod 16 of its group of 16: the value is the MFMA's A operand in the
// register it was computed in.  There is no transform of the N bins and no
// exchange between lanes; what is left per bin is the integrand itself (the
// float64 phase, one sin / cos pair, the detectors' products and rotations).
//
// Bound: instruction issue.  A step (64 bins of one row, three detectors)
// takes 35 vector instructions at 4.9 cycles, two of them sin / cos at 10, and
// two MFMAs of 34; the float32 MFMA and the vector ALU do not overlap
// (measured: 1 MFMA + 8 FMAs take the sum of both at 1, 2 and 4 wavefronts per
// SIMD).  Against a 512-point FFT of every sub-sequence in registers and LDS
// (94 instructions a step): 1501 rows of 131072 bins, two detectors 740 -> 315
// us; 4096 rows of 16384 bins, three detectors 239 -> 137 us, and 62 us to
// finish them, where the epilogue was part of the 239.  float64, 509 rows of
// 16384 bins, three detectors: 271 us (tiles of 8 rows through LDS
// transforms, k_time) -> 47, and 17 to finish them.
#include "gwl_internal.h"
#include "gwl_tf2_rows.h"

#include <algorithm>
#include <cmath>

namespace gwl {

namespace {

constexpr int kNP = 16;        // functions per block
constexpr int kBandWaves = 4;  // wavefronts per workgroup of k_band
constexpr int kChunk = 8;      // steps between exact rotation phases and float64 flushes

template <typename T> struct BandTypes;
template <> struct BandTypes<float> {
  typedef float V4 __attribute__((ext_vector_type(4)));
  static constexpr int NB = 128;
};
template <> struct BandTypes<double> {
  typedef double V4 __attribute__((ext_vector_type(4)));
  static constexpr int NB = 256;
};

// D[16][16] += A[16][4] B[4][16]: lane l holds A[l % 16][l / 16] and
// B[l / 16][l % 16]; accumulator r holds D[4 (l / 16) + r][l % 16] (float32),
// D[4 r + l / 16][l % 16] (float64).
__device__ __forceinline__ BandTypes<float>::V4 band_mfma(float a, float b,
                                                          BandTypes<float>::V4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ BandTypes<double>::V4 band_mfma(double a, double b,
                                                           BandTypes<double>::V4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// Steps of 4 bins a block, padded (with zero data) to even: a load brings two.
template <typename T>
__host__ __device__ __forceinline__ int band_steps(int N) {
  const int s = N / BandTypes<T>::NB / 4;
  return s + (s & 1);
}

// The event fields the integrand reads.
template <typename T>
struct BandEv {
  const double2* uv;  // (f^1/3, f^-1/3), order (group, step, lane)
  const double2* lf;  // ln f of two steps, order (group, pair of steps, lane)
  const cplx<T>* dw;  // [nd] d / S f^-7/6 exp(2 pi i n jd / N), pairs as lf
  const T* u;         // U_p(t) in MFMA B-operand order, pairs (pair of steps, lane)
  double df;
  size_t M;           // table elements a detector: bins, steps padded to even
  int S, B;           // steps (even) per group of 16 blocks, bins per block
};

template <typename T>
__host__ __device__ __forceinline__ const BandDev& band_dev(const EvDev& ev) {
  if constexpr (sizeof(T) == 4) return ev.band32;
  else return ev.band64;
}

template <typename T>
__device__ __forceinline__ BandEv<T> band_ev(const EvDev& ev) {
  const BandDev& bd = band_dev<T>(ev);
  BandEv<T> b;
  b.uv = bd.uv;
  b.lf = reinterpret_cast<const double2*>(bd.lf);
  b.dw = reinterpret_cast<const cplx<T>*>(bd.dw);
  b.u = reinterpret_cast<const T*>(bd.u);
  b.df = ev.df;
  b.B = ev.N / BandTypes<T>::NB;
  b.S = band_steps<T>(ev.N);
  b.M = (size_t)BandTypes<T>::NB * 4 * b.S;
  return b;
}

// Row constants in the registers of a wavefront, with the rotation of one
// step and the detectors' tables, the reference detector's first.
template <typename T, int ND>
struct BandRow : Tf2Row<T, ND> {
  static constexpr int NO = ND - 1;
  cplx<T> w[NO > 0 ? NO : 1];  // exp(-2 pi i 4 df dd): one step
  const cplx<T>* dwr;
  const cplx<T>* dwo[NO > 0 ? NO : 1];
};

template <typename T, int ND>
__device__ __forceinline__ void band_row(const BandEv<T>& ev, const RowW& rw, BandRow<T, ND>& b) {
  tf2_row<T, ND>(rw, b);
#pragma unroll
  for (int k = 0; k < ND - 1; ++k) {
    double2 corr = make_double2(1.0, 0.0);
    b.w[k] = tf2_rotation<T>((4.0 * ev.df) * b.dd[k], 0.5 * (kChunk - 1), corr);
    tf2_rho<T, ND>(rw, k, corr, b);
    b.dwo[k] = ev.dw + (size_t)(k < b.ref ? k : k + 1) * ev.M;
  }
  b.dwr = ev.dw + (size_t)b.ref * ev.M;
}

// What two steps read: the basis, the block function and the data of the
// reference detector, then the others' (one set where the rows share it).
template <typename T, int ND, int R, bool SHARED>
struct BandIn {
  double2 uv[2];
  double2 lf;
  T u[2];
  cplx<T> d[SHARED ? 1 : R][ND][2];
};

// ep: the pair's element (g S + s) / 2 * 64 + lane, sp: s / 2 * 64 + lane.
template <typename T, int ND, int R, bool SHARED>
__device__ __forceinline__ void band_load(const BandEv<T>& ev, const BandRow<T, ND>* b,
                                          unsigned ep, unsigned sp, int lane,
                                          BandIn<T, ND, R, SHARED>& in) {
  const unsigned e = 2 * ep - (unsigned)lane;
  in.uv[0] = load_at<double2>(ev.uv, e * 16u);
  in.uv[1] = load_at<double2>(ev.uv, e * 16u + 1024u);
  in.lf = load_at<double2>(ev.lf, ep * 16u);
  if constexpr (sizeof(T) == 4) {
    const float2 u = load_at<float2>(ev.u, sp * 8u);
    in.u[0] = u.x;
    in.u[1] = u.y;
  } else {
    const double2 u = load_at<double2>(ev.u, sp * 16u);
    in.u[0] = u.x;
    in.u[1] = u.y;
  }
#pragma unroll
  for (int r = 0; r < (SHARED ? 1 : R); ++r) {
    load_pair(b[r].dwr, ep * (unsigned)(2 * sizeof(cplx<T>)), in.d[r][0]);
#pragma unroll
    for (int k = 0; k < ND - 1; ++k)
      load_pair(b[r].dwo[k], ep * (unsigned)(2 * sizeof(cplx<T>)), in.d[r][k + 1]);
  }
}

// One integrand value (over |C_r|) of bin n; the rotations move on by a step.
template <typename T, int ND, bool MASK>
__device__ __forceinline__ cplx<T> band_value(const BandRow<T, ND>& b, cplx<T>* rot,
                                              const cplx<T> (*d)[2], int i, int n, double u,
                                              double v, double lf) {
  using C = cplx<T>;
  C x = tf2_product<T, ND>(tf2_cycles<T, ND>(b, u, v, lf), rot, d, i);
#pragma unroll
  for (int k = 0; k < ND - 1; ++k) rot[k] = cmul_fma(rot[k], b.w[k]);
  if constexpr (MASK) {
    const bool in = n >= b.kb && n <= b.ke;
    x = cmk<C>(in ? x.x : (T)0, in ? x.y : (T)0);
  }
  return x;
}

// C of the R rows over steps [sb, se) of groups [g0, g1): complex element (g *
// 4 + k) * 64 + lane of out[r] is the lane's accumulator k.  Loads run
// two steps ahead of the arithmetic (left to the compiler each load is issued
// at its use, which exposes the L2 latency several times a step at two
// wavefronts per SIMD).
template <typename T, int ND, int R, bool MASK, bool SHARED>
__device__ __forceinline__ void band_groups(const BandEv<T>& ev, const BandRow<T, ND>* b, int g0,
                                            int g1, int sb, int se, int lane, double* const* out,
                                            int nlive) {
  constexpr int NO = ND - 1;
  using C = cplx<T>;
  using V4 = typename BandTypes<T>::V4;
  using In = BandIn<T, ND, R, SHARED>;
  In in[2];
  const bool whole = (se - sb) % kChunk == 0;
  const int hs = ev.S >> 1;
  auto at = [&](int g, int s) { return (unsigned)(g * hs + (s >> 1)) * 64u + (unsigned)lane; };
  if (whole) band_load(ev, b, at(g0, sb), at(0, sb), lane, in[0]);
  for (int g = g0; g < g1; ++g) {
    const int n0 = ev.B * (16 * g + (lane & 15)) + (lane >> 4);
    double acc[R][8];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int k = 0; k < 8; ++k) acc[r][k] = 0.0;
    for (int s0 = sb; s0 < se; s0 += kChunk) {
      V4 re[R], im[R];
      C rot[R][NO > 0 ? NO : 1];
      const double f0 = (double)(n0 + 4 * s0) * ev.df;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        re[r] = (V4){0, 0, 0, 0};
        im[r] = (V4){0, 0, 0, 0};
#pragma unroll
        for (int k = 0; k < NO; ++k) rot[r][k] = tf2_rotated<T, ND>(b[r], k, f0);
      }
      auto pair = [&](int j, const In& v) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int r = 0; r < R; ++r) {
            const C x = band_value<T, ND, MASK>(b[r], rot[r], v.d[SHARED ? 0 : r], i,
                                                n0 + 4 * (s0 + j + i), v.uv[i].x, v.uv[i].y,
                                                i ? v.lf.y : v.lf.x);
            re[r] = band_mfma(x.x, v.u[i], re[r]);
            im[r] = band_mfma(x.y, v.u[i], im[r]);
          }
      };
      if (whole) {
        // the next chunk: of this group, of the next, or (last) this one again
        const bool more = s0 + kChunk < se;
        const int gn = more ? g : min(g + 1, g1 - 1), sn = more ? s0 + kChunk : sb;
        const unsigned ep = at(g, s0), sp = at(0, s0), epn = at(gn, sn), spn = at(0, sn);
#pragma unroll
        for (int j = 0; j < kChunk; j += 2) {
          const bool here = j + 2 < kChunk;
          band_load(ev, b, here ? ep + 32u * (j + 2) : epn, here ? sp + 32u * (j + 2) : spn, lane,
                    in[((j >> 1) + 1) & 1]);
          __builtin_amdgcn_sched_barrier(0);
          pair(j, in[(j >> 1) & 1]);
        }
      } else {
        for (int j = 0; j < min(kChunk, se - s0); j += 2) {
          band_load(ev, b, at(g, s0 + j), at(0, s0 + j), lane, in[0]);
          pair(j, in[0]);
        }
      }
      // sums of more than kChunk steps are float64
#pragma unroll
      for (int r = 0; r < R; ++r)
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          acc[r][k] += (double)re[r][k];
          acc[r][4 + k] += (double)im[r][k];
        }
    }
#pragma unroll
    for (int r = 0; r < R; ++r)
      if (r < nlive) {
        double2* o = reinterpret_cast<double2*>(out[r]) + (size_t)g * 256 + lane;
#pragma unroll
        for (int k = 0; k < 4; ++k) o[64 * k] = make_double2(acc[r][k], acc[r][4 + k]);
      }
  }
}

// Groups [ga, gb) that meet bins [kb, ke].  The others' sums are zero, and are
// neither computed nor written nor read: rows cut at the ISCO use a small part
// of the band (4096 such rows of 16384 bins, three detectors: 194 us with every
// group, 95 without; one wavefront per row with the 512-point transform 137).
// Kernels of events without the cut (CUT false) have none of this, which would
// take them 1 %.
template <typename T>
__device__ __forceinline__ void band_support(int B, int kb, int ke, int& ga, int& gb) {
  ga = kb / (16 * B);
  gb = kb <= ke ? min(BandTypes<T>::NB / 16, ke / (16 * B) + 1) : ga;
}

template <typename T, int ND, int R, bool CUT>
__device__ __forceinline__ void band_rows(const EvDev& ev, const RowW* rows, long long row0,
                                          long long n, int g0, int g1, int sb, int se, double* out,
                                          size_t row_stride, int lane, int wid) {
  long long pick[R];
  const int live = pick_rows<R>(rows, row0, n, lane, wid, pick);
  if (live == 0) return;
  const BandEv<T> be = band_ev<T>(ev);
  BandRow<T, ND> b[R];
  double* o[R];
  int nomask = 1, shared = 1, ga = g1, gb = g0;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const RowW& rw = rows[pick[r]];
    band_row<T, ND>(be, rw, b[r]);
    nomask &= rw.nomask;
    shared &= b[r].ref == b[0].ref;
    o[r] = out + (size_t)pick[r] * row_stride;
    if constexpr (CUT) {
      int sa, sz;
      band_support<T>(be.B, rw.kb, rw.ke, sa, sz);
      if (sa < sz) {
        ga = min(ga, sa);
        gb = max(gb, sz);
      }
    }
  }
  if constexpr (CUT) {
    g0 = max(g0, ga);
    g1 = min(g1, gb);
    if (g0 >= g1) return;
  }
  if (nomask && shared)
    band_groups<T, ND, R, false, true>(be, b, g0, g1, sb, se, lane, o, live);
  else if (nomask)
    band_groups<T, ND, R, false, R == 1>(be, b, g0, g1, sb, se, lane, o, live);
  else
    band_groups<T, ND, R, true, R == 1>(be, b, g0, g1, sb, se, lane, o, live);
}

// Split ``k`` of a row's work: Gg parts of the groups of 16 blocks times Gs
// parts of each block's steps (whole chunks), so that the float32 sums of a
// row do not depend on the split.
struct BandSplit {
  int gg, gs;
};

template <typename T>
__device__ __forceinline__ void band_range(int S, BandSplit sp, int k, int& g0, int& g1, int& sb,
                                           int& se) {
  constexpr int NG = BandTypes<T>::NB / 16;
  const int kg = k % sp.gg, ks = k / sp.gg;
  g0 = kg * NG / sp.gg;
  g1 = (kg + 1) * NG / sp.gg;
  const int chunks = (S + kChunk - 1) / kChunk;
  sb = (int)((long long)ks * chunks / sp.gs) * kChunk;
  se = min(S, (int)((long long)(ks + 1) * chunks / sp.gs) * kChunk);
}

// out: [n][gs][NB * 16 * 2] doubles
struct BandArgs {
  EvDev ev;
  const RowW* rows;
  long long n;
  BandSplit split;
  double* out;
};

// 2 rows per wavefront share each table load; at 2 wavefronts per SIMD the
// 256 registers hold both rows' state
template <typename T, int ND, int R, bool CUT>
__global__ __launch_bounds__(64 * kBandWaves, 2) void k_band(BandArgs a) {
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  constexpr size_t kRow = (size_t)BandTypes<T>::NB * kNP * 2;
  int g0, g1, sb, se;
  band_range<T>(band_steps<T>(a.ev.N), a.split, blockIdx.y, g0, g1, sb, se);
  const int ks = blockIdx.y / a.split.gg;
  band_rows<T, ND, R, CUT>(a.ev, a.rows, (long long)blockIdx.x * (kBandWaves * R), a.n, g0, g1, sb, se,
                      a.out + ks * kRow, kRow * a.split.gs, lane, wid);
}

// ------------------------------------------------------------------ finish
// 16-point DFT in registers: x[n] -> X[k], both in natural order.
__device__ __forceinline__ void dft16(double2* x) {
  double2 f[4][4];
#pragma unroll
  for (int a = 0; a < 4; ++a) {
    double2 t[4] = {x[a], x[a + 4], x[a + 8], x[a + 12]};
    dft4(t);
#pragma unroll
    for (int u = 0; u < 4; ++u) f[u][a] = t[u];
  }
  constexpr double c1 = 0.92387953251128675613, s1 = 0.38268343236508977173;
  constexpr double h = 0.70710678118654752440;
  const double2 w1 = make_double2(c1, -s1), w2 = make_double2(h, -h), w3 = make_double2(s1, -c1);
  f[1][1] = cmul(f[1][1], w1);
  f[1][2] = cmul(f[1][2], w2);
  f[1][3] = cmul(f[1][3], w3);
  f[2][1] = cmul(f[2][1], w2);
  f[2][2] = cmul_mi(f[2][2]);
  f[2][3] = cmul(f[2][3], make_double2(-h, -h));
  f[3][1] = cmul(f[3][1], w3);
  f[3][2] = cmul(f[3][2], make_double2(-h, -h));
  f[3][3] = cmul(f[3][3], make_double2(-c1, s1));
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    dft4(f[u]);
#pragma unroll
    for (int v = 0; v < 4; ++v) x[u + 4 * v] = f[u][v];
  }
}

constexpr int kFinThreads = 256;
// LDS address of (row, p): the pitch of 17 and the skew of one per 16 rows
// keep rows that differ by 1 or by 16 in different banks.
constexpr int kPitch = kNP + 1;
__device__ __forceinline__ int fin_at(int row, int p) { return row * kPitch + (row >> 4) + p; }

// the block sums, then the twiddles W_NB^m
template <typename T>
constexpr size_t finish_lds() {
  return ((size_t)BandTypes<T>::NB * kPitch + BandTypes<T>::NB / 16 + BandTypes<T>::NB) *
         sizeof(double2);
}

// The distance table's values at the workgroup's coordinates (two a thread,
// NaN: none).  A row reads one y interval, so the table is a spline in x
// alone: its coefficients by . ct and the knots and reciprocals between the
// row's smallest and largest coordinate (typically 200 of 800 intervals) go to
// LDS in coalesced loads.  Gathered from global memory, 14 loads a value touch
// dozens of lines each and the cache's tag rate bounds the whole kernel.
template <int NB>
__device__ __forceinline__ void fin_distance_values(const SplineDev& sp, const SplineY& yy,
                                                    const double* d, double* val, double* lds,
                                                    double2* red) {
  constexpr int kCap = NB * kPitch * 2 / 5;  // intervals that fit (5 arrays)
  const int t = threadIdx.x;
  bool in[2];
  int first[2];
  double lo = INFINITY, hi = -INFINITY;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    in[i] = yy.inside && d[i] >= sp.xmin && d[i] <= sp.xmax;
    first[i] = in[i] ? sp.ix[spline_bucket((unsigned)__double2hiint(d[i]))] : 3;
    if (in[i]) {
      lo = fmin(lo, d[i]);
      hi = fmax(hi, d[i]);
    }
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    lo = fmin(lo, __shfl_xor(lo, off, 64));
    hi = fmax(hi, __shfl_xor(hi, off, 64));
  }
  if ((t & 63) == 0) red[t >> 6] = make_double2(lo, hi);
  __syncthreads();  // and every thread is done with the block sums
#pragma unroll
  for (int w = 0; w < kFinThreads / 64; ++w) {
    lo = fmin(lo, red[w].x);
    hi = fmax(hi, red[w].y);
  }
  if (!(lo <= hi)) return;  // (uniform) no value inside the table
  // from the first interval of lo's bucket to the first of the bucket after
  // hi's: the row's intervals and a few more
  const unsigned klo = spline_bucket((unsigned)__double2hiint(lo));
  const unsigned khi = min(spline_bucket((unsigned)__double2hiint(hi)) + 1u, 65535u);
  const int l0 = sp.ix[__builtin_amdgcn_readfirstlane(klo)] - 3;         // first coefficient
  const int n = sp.ix[__builtin_amdgcn_readfirstlane(khi)] - l0 + 4;     // to the last knot + 3
  if (n > kCap) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
      if (in[i]) val[i] = spline_x(sp, yy, d[i]);
    return;
  }
  double *tx = lds, *r1 = tx + n, *r2 = r1 + n, *r3 = r2 + n, *g = r3 + n;
  for (int k = t; k < n; k += kFinThreads) {
    const int l = l0 + k;
    tx[k] = sp.tx[l];
    r1[k] = sp.rx[l];
    r2[k] = sp.rx[(sp.nx + 4) + l];
    r3[k] = sp.rx[2 * (sp.nx + 4) + l];
    if (l < sp.nx) {
      const double* c = sp.ct + (size_t)(yy.ly - 3) * sp.nx + l;
      g[k] = yy.by[0] * c[0] + yy.by[1] * c[sp.nx] + yy.by[2] * c[2 * (size_t)sp.nx] +
             yy.by[3] * c[3 * (size_t)sp.nx];
    }
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 2; ++i)
    if (in[i]) {
      const double x = d[i];
      int l = first[i] - l0;
      while (l < n - 4 && tx[l + 1] <= x) ++l;
      // spline_basis on the staged arrays
      const double d0 = x - tx[l], d1 = x - tx[l - 1], d2 = x - tx[l - 2];
      const double u1 = tx[l + 1] - x, u2 = tx[l + 2] - x, u3 = tx[l + 3] - x;
      const double a0 = u1 * r1[l], a1 = d0 * r1[l];
      const double f0 = a0 * r2[l], f1 = a1 * r2[l + 1];
      const double b0 = f0 * u1, b1 = fma(f0, d1, f1 * u2), b2 = f1 * d0;
      const double g0 = b0 * r3[l], g1 = b1 * r3[l + 1], g2 = b2 * r3[l + 2];
      val[i] = g[l - 3] * (g0 * u1) + g[l - 2] * fma(g0, d2, g1 * u2) +
               g[l - 1] * fma(g1, d1, g2 * u3) + g[l] * (g2 * d0);
    }
}

// One workgroup finishes one row: 16 DFTs of NB points (radix NB / 16 over the
// groups in the registers the sums are loaded to, then 16 through LDS), the
// 16-term contraction at each window bin, and the marginalisation
// (base.py:794-820).  4096 rows, L = 419: 62 us, 13 ns a row: 1.4 us a row and
// CU of vector issue, 0.5 of LDS and 0.7 of loads, which overlap only in part
// at three workgroups per CU (92 us with the distance table gathered from
// global memory, 68 with the sums staged through LDS first).
template <typename T, bool CUT>
__device__ __forceinline__ void band_finish_row(const EvDev& ev, const RowW& rw, const double* c,
                                                int gs, double* out, double2* x, double2* red) {
  constexpr int NB = BandTypes<T>::NB, NG = NB / 16;
  const int t = threadIdx.x;
  if (!rw.valid) {
    if (t == 0) *out = row_valid_sentinel();
    return;
  }
  const BandDev& bd = band_dev<T>(ev);
  double2* tw = x + NB * kPitch + NB / 16;
  const double norm = 4.0 / ev.T;
  const double hh = rw.hh * norm, hs = rw.hscale, jit = rw.jitter, amp = rw.amp * norm;
  const bool dist = (ev.flags & GWL_DISTANCE_MARG) != 0;
  SplineY yy;
  // (its loads first: the block sums' are waited for in order)
  if (dist) yy = spline_y(ev.sp, hh * hs * hs);
  {
    // thread (accumulator k, lane l) holds function p = l mod 16 of the blocks
    // 16 g + res, g < NG: over g
    const int p = t & 15, h = (t & 63) >> 4, k = t >> 6;
    const int res = sizeof(T) == 4 ? 4 * h + k : 4 * k + h;
    const double2* src = reinterpret_cast<const double2*>(c) + t;
    double2 y[NG];
    if constexpr (!CUT) {
#pragma unroll
      for (int g = 0; g < NG; ++g) y[g] = src[g * 256];
      for (int i = 1; i < gs; ++i) {
        src += NB * kNP;
#pragma unroll
        for (int g = 0; g < NG; ++g) y[g] = cadd(y[g], src[g * 256]);
      }
    } else {
      int ga, gb;
      band_support<T>(ev.N / NB, rw.kb, rw.ke, ga, gb);
#pragma unroll
      for (int g = 0; g < NG; ++g) {
        y[g] = make_double2(0.0, 0.0);
        if (g >= ga && g < gb)
          for (int i = 0; i < gs; ++i) y[g] = cadd(y[g], src[g * 256 + i * (NB * kNP)]);
      }
    }
    if (t < NB) tw[t] = expm2pi((double)t / (double)NB);
    __syncthreads();
    if constexpr (NG == 8) dft8(y);
    else dft16(y);
#pragma unroll
    for (int q = 1; q < NG; ++q) y[q] = cmul(y[q], tw[res * q]);
#pragma unroll
    for (int q = 0; q < NG; ++q) x[fin_at(res + 16 * q, p)] = y[q];
  }
  __syncthreads();
  // Lane l of wavefront w contracts block frequency q = 32 w + l mod 32 over
  // half of the functions (l / 32) for its up to four window bins; the halves
  // are exchanged and each lane keeps two bins.  (NB = 256: two of q, two
  // bins each.)
  constexpr int kQ = NB / 128;
  const int lane = t & 63, half = lane >> 5, wv = t >> 6;
  const int L = ev.L, p0 = half * (kNP / 4);
  int jq[4];   // the four bins, clamped to the window
  bool inq[4];
  int qa[kQ];
#pragma unroll
  for (int i = 0; i < kQ; ++i) {
    qa[i] = 32 * wv + (lane & 31) + 128 * i;
#pragma unroll
    for (int a = 0; a < 4 / kQ; ++a) {
      const int jj = ((qa[i] + L / 2) & (NB - 1)) + NB * a;
      jq[i * (4 / kQ) + a] = min(jj, L - 1);
      inq[i * (4 / kQ) + a] = jj < L;
    }
  }
  const double2* vt = bd.v + (size_t)p0 * L;
  double2 va[2][4];
#pragma unroll
  for (int p = 0; p < 2; ++p)
#pragma unroll
    for (int a = 0; a < 4; ++a) va[p][a] = vt[(size_t)p * L + jq[a]];
  if (t < NG * 16) {
    // over res: thread (p, q0) -> D_p[q0 + NG q1] at row q1 + 16 q0
    const int p = t & 15, q0 = t >> 4;
    double2 y[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) y[i] = x[fin_at(i + 16 * q0, p)];
    dft16(y);
#pragma unroll
    for (int i = 0; i < 16; ++i) x[fin_at(i + 16 * q0, p)] = y[i];
  }
  __syncthreads();
  double sr[4] = {0.0, 0.0, 0.0, 0.0}, si[4] = {0.0, 0.0, 0.0, 0.0};
  auto contract = [&](int p, const double2* v) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < kQ; ++i) {
      const double2* d = x + fin_at((qa[i] / NG) + 16 * (qa[i] & (NG - 1)), 2 * (p0 + p));
      const double2 de = d[0], od = d[1];
      // V is real for even functions, -i times the table for odd ones
#pragma unroll
      for (int b = 0; b < 4 / kQ; ++b) {
        const int a = i * (4 / kQ) + b;
        sr[a] = fma(v[a].x, de.x, fma(v[a].y, od.y, sr[a]));
        si[a] = fma(v[a].x, de.y, fma(-v[a].y, od.x, si[a]));
      }
    }
  };
#pragma unroll
  for (int p = 0; p < 2; ++p) contract(p, va[p]);
#pragma unroll
  for (int p = 0; p < 2; ++p)
#pragma unroll
    for (int a = 0; a < 4; ++a) va[p][a] = vt[(size_t)(p + 2) * L + jq[a]];
#pragma unroll
  for (int p = 0; p < 2; ++p) contract(p + 2, va[p]);
  double xr[2], xi[2], tt[2], val[2] = {-INFINITY, -INFINITY};
  const double nan = __builtin_nan("");
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    // bin i of the lower lanes, i + 2 of the upper ones
    const double mr = half ? sr[i + 2] : sr[i], mi = half ? si[i + 2] : si[i];
    const double gr = half ? sr[i] : sr[i + 2], gi = half ? si[i] : si[i + 2];
    xr[i] = mr + __shfl_xor(gr, 32, 64);
    xi[i] = mi + __shfl_xor(gi, 32, 64);
    const int jj = half ? jq[i + 2] : jq[i];
    tt[i] = (ev.start + (double)(ev.jlo + jj + 1) * ev.tstep) + jit;
    const bool in = (half ? inq[i + 2] : inq[i]) && tt[i] >= ev.tmin && tt[i] <= ev.tmax;
    const double2 w = bd.rot[jj];
    const double ar = amp * (xr[i] * w.x - xi[i] * w.y), ai = amp * (xr[i] * w.y + xi[i] * w.x);
    // under distance marginalisation xr becomes the table's coordinate
    if (!in)
      xr[i] = nan;
    else if (dist)
      xr[i] = (ev.flags & GWL_PHASE_MARG) ? cabs2d(ar, ai) * hs : ar * hs;
    else
      val[i] = epi_value(ev.flags, ev.sp, yy, hh, hs, ar, ai) + time_log_weight(ev, tt[i]);
  }
  if (dist) {
    fin_distance_values<NB>(ev.sp, yy, xr, val, reinterpret_cast<double*>(x), red);
    if (ev.tpd)
#pragma unroll
      for (int i = 0; i < 2; ++i) val[i] += time_log_weight(ev, tt[i]);
    __syncthreads();  // red is used again below
  }
  // logsumexp (NaN values count as zero weight, as lse_push counts them)
  double m = fmax(val[0], val[1]);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) m = fmax(m, __shfl_xor(m, off, 64));
  double sum = 0.0;
#pragma unroll
  for (int i = 0; i < 2; ++i) sum += val[i] > -INFINITY ? exp(val[i] - m) : 0.0;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) sum += __shfl_xor(sum, off, 64);
  if (lane == 0) red[wv] = make_double2(m, sum);
  __syncthreads();
  if (wv == 0) {  // lane w merges wavefront w's state
    const double2 st = red[lane & 3];
    double mx = fmax(st.x, __shfl_xor(st.x, 1, 64));
    mx = fmax(mx, __shfl_xor(mx, 2, 64));
    double s = st.x > -INFINITY ? st.y * exp(st.x - mx) : 0.0;
    s += __shfl_xor(s, 1, 64);
    s += __shfl_xor(s, 2, 64);
    if (t == 0) {
      const double b = time_lse_scale(ev, ev.tdelta);
      *out = (mx > -INFINITY) ? log(b * s) + mx : -INFINITY;
    }
  }
}

struct FinishArgs {
  EvDev ev;
  const RowW* rows;
  const double* c;
  int gs;
  double* out;
};

template <typename T, bool CUT>
__global__ __launch_bounds__(kFinThreads) void k_band_finish(FinishArgs a) {
  extern __shared__ double2 lds[];
  __shared__ double2 red[kFinThreads / 64];
  const long long r = blockIdx.x;
  constexpr size_t kRow = (size_t)BandTypes<T>::NB * kNP * 2;
  band_finish_row<T, CUT>(a.ev, a.rows[r], a.c + (size_t)r * a.gs * kRow, a.gs, a.out + r, lds, red);
}

// float64 rows of short segments: both in one workgroup per row.  A row's block
// sums are 64 KB, more than it reads otherwise; here they stay in the LDS that
// k_band_finish loads them to (the same values, bit for bit).  1024 bins, two
// detectors, 4096 rows: 165 us in two kernels, 121 in one (148 with tiles of
// 512-point transforms, k_time); 16384 rows: 632, 444 (432).
template <int ND, bool CUT>
__global__ __launch_bounds__(kFinThreads) void k_band_row(BandArgs a) {
  using T = double;
  extern __shared__ double2 lds[];
  __shared__ double2 red[kFinThreads / 64];
  const long long r = blockIdx.x;
  const RowW& rw = a.rows[r];
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const BandEv<T> be = band_ev<T>(a.ev);
  constexpr int per = BandTypes<T>::NB / 16 / (kFinThreads / 64);  // groups a wavefront
  int g0 = wid * per, g1 = g0 + per;
  if constexpr (CUT) {
    int ga, gb;
    band_support<T>(be.B, rw.kb, rw.ke, ga, gb);
    g0 = max(g0, ga);
    g1 = min(g1, gb);
  }
  if (rw.valid && g0 < g1) {
    BandRow<T, ND> b[1];
    band_row<T, ND>(be, rw, b[0]);
    double* const o[1] = {reinterpret_cast<double*>(lds)};
    if (rw.nomask) band_groups<T, ND, 1, false, true>(be, b, g0, g1, 0, be.S, lane, o, 1);
    else band_groups<T, ND, 1, true, true>(be, b, g0, g1, 0, be.S, lane, o, 1);
  }
  __syncthreads();
  band_finish_row<T, CUT>(a.ev, rw, reinterpret_cast<const double*>(lds), 1, a.out + r, lds, red);
}

// ------------------------------------------------------------------ multi-event
struct BandMultiArgs {
  const EvDev* evs;
  const long long* rows;
  const int* groups;
  const RowW* const* roww;
  double* const* c;
  const MultiItem* items;
  const int* n_items;
};

// Workgroup: one item of the longest-first list (8 rows of an event, one of
// its G parts of the block groups).
template <bool CUT>
__global__ __launch_bounds__(64 * kBandWaves, 2) void k_band_multi(BandMultiArgs a) {
  if ((int)blockIdx.x >= *a.n_items) return;
  const MultiItem m = a.items[blockIdx.x];
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const EvDev& ev = a.evs[m.e];
  constexpr int NB = BandTypes<float>::NB;
  constexpr size_t kRow = (size_t)NB * kNP * 2;
  int g0, g1, sb, se;
  band_range<float>(band_steps<float>(ev.N), BandSplit{a.groups[m.e], 1}, m.g, g0, g1, sb, se);
  switch (ev.nd) {
    case 1:
      band_rows<float, 1, 2, CUT>(ev, a.roww[m.e], m.row0, a.rows[m.e], g0, g1, sb, se, a.c[m.e], kRow,
                             lane, wid);
      break;
    case 2:
      band_rows<float, 2, 2, CUT>(ev, a.roww[m.e], m.row0, a.rows[m.e], g0, g1, sb, se, a.c[m.e], kRow,
                             lane, wid);
      break;
    default:
      band_rows<float, 3, 2, CUT>(ev, a.roww[m.e], m.row0, a.rows[m.e], g0, g1, sb, se, a.c[m.e], kRow,
                             lane, wid);
  }
}

struct FinishMultiArgs {
  const EvDev* evs;
  const long long* rows;
  const RowW* const* roww;
  double* const* c;
  double* const* out;
  const int* block_event;
  const long long* block_row0;
  const int* n_blocks;
};

// One workgroup per row; a block of the list covers kMultiEpiRows rows.
template <bool CUT>
__global__ __launch_bounds__(kFinThreads) void k_band_finish_multi(FinishMultiArgs a) {
  extern __shared__ double2 lds[];
  __shared__ double2 red[kFinThreads / 64];
  const int blk = blockIdx.x / kMultiEpiRows;
  if (blk >= *a.n_blocks) return;
  const int e = a.block_event[blk];
  const long long r = a.block_row0[blk] + blockIdx.x % kMultiEpiRows;
  if (r >= a.rows[e]) return;
  constexpr size_t kRow = (size_t)BandTypes<float>::NB * kNP * 2;
  band_finish_row<float, CUT>(a.evs[e], a.roww[e][r], a.c[e] + (size_t)r * kRow, 1, a.out[e] + r,
                              lds, red);
}

// ------------------------------------------------------------------ tables
// (f^1/3, f^-1/3), ln f and dw f^-7/6 exp(2 pi i n jd / N): element (g S + s)
// 64 + l is bin B (16 g + l mod 16) + 4 s + l / 16; ln f and dw interleave the
// two steps of a pair.
template <typename T>
__global__ __launch_bounds__(256) void k_band_tables(EvDev ev, int jd, double2* uv, double* lf,
                                                     cplx<T>* dw) {
  constexpr int NB = BandTypes<T>::NB;
  const int B = ev.N / NB, S = band_steps<T>(ev.N);
  const long long M = (long long)NB * 4 * S;
  const long long e = (long long)blockIdx.x * 256 + threadIdx.x;
  if (e >= M) return;
  const int l = (int)(e & 63), gs = (int)(e >> 6), g = gs / S, s = gs - g * S;
  const bool in = 4 * s < B;
  const int n = in ? B * (16 * g + (l & 15)) + 4 * s + (l >> 4) : 0;
  double2 b2 = make_double2(0.0, 0.0);
  double ln = 0.0, amp = 0.0;
  if (n > 0) {
    double b[kNB];
    tf2_basis((double)n * ev.df, b);
    b2 = make_double2(b[5], b[3]);
    ln = b[7];
    amp = b[1] * sqrt(b[3]) * (sizeof(T) == 4 ? kExpm2piGain : 1.0);
  }
  const long long e2 = (((long long)g * (S / 2) + (s >> 1)) * 64 + l) * 2 + (s & 1);
  uv[e] = b2;
  lf[e2] = ln;
  const long long ph = ((long long)n * jd) % ev.N;
  double sn, cs;
  sincospi(2.0 * (double)ph / (double)ev.N, &sn, &cs);
  const size_t i = (size_t)(n % ev.Q) * ev.P + n / ev.Q;  // the data's decimated order
  for (int d = 0; d < ev.nd; ++d) {
    const double2 w = ev.dw64[(size_t)d * ev.N + i];
    dw[(size_t)d * M + e2] = cmk<cplx<T>>((T)((w.x * cs - w.y * sn) * amp),
                                          (T)((w.x * sn + w.y * cs) * amp));
  }
}

// The block functions are set up in extended precision: the float64 transform
// takes them rounded once.
using Real = long double;
using Mat = std::vector<std::vector<Real>>;

// Eigenvectors of a symmetric n x n matrix by cyclic Jacobi rotations, in
// ascending order of the eigenvalues: vec[k][i].
void jacobi(Mat a, Mat& vec) {
  const int n = (int)a.size();
  Mat v(n, std::vector<Real>(n, 0.0L));
  for (int i = 0; i < n; ++i) v[i][i] = 1;
  for (int sweep = 0; sweep < 60; ++sweep) {
    Real off = 0, diag = 0;
    for (int i = 0; i < n; ++i)
      for (int j = 0; j < n; ++j) (i == j ? diag : off) += a[i][j] * a[i][j];
    if (off <= 1e-40L * diag) break;
    for (int p = 0; p < n; ++p)
      for (int q = p + 1; q < n; ++q) {
        if (a[p][q] == 0) continue;
        const Real th = (a[q][q] - a[p][p]) / (2 * a[p][q]);
        const Real t = (th >= 0 ? 1.0L : -1.0L) / (std::fabs(th) + std::sqrt(th * th + 1));
        const Real c = 1 / std::sqrt(t * t + 1), s = t * c;
        for (int k = 0; k < n; ++k) {
          const Real x = a[k][p], y = a[k][q];
          a[k][p] = c * x - s * y;
          a[k][q] = s * x + c * y;
        }
        for (int k = 0; k < n; ++k) {
          const Real x = a[p][k], y = a[q][k];
          a[p][k] = c * x - s * y;
          a[q][k] = s * x + c * y;
        }
        for (int k = 0; k < n; ++k) {
          const Real x = v[k][p], y = v[k][q];
          v[k][p] = c * x - s * y;
          v[k][q] = s * x + c * y;
        }
      }
  }
  std::vector<int> order(n);
  for (int i = 0; i < n; ++i) order[i] = i;
  std::sort(order.begin(), order.end(), [&](int i, int j) { return a[i][i] < a[j][j]; });
  vec.assign(n, std::vector<Real>(n));
  for (int k = 0; k < n; ++k)
    for (int i = 0; i < n; ++i) vec[k][i] = v[i][order[k]];
}

constexpr int kLeg = 48;  // Legendre terms (c <= 2 pi needs about 30)

// U_p(t) [B][16] and V_p(kappa) [8][L][2] (p even, odd; odd p: the real factor
// of -i).
// The prolate functions psi_p come from their differential operator, which is
// tridiagonal in the normalised Legendre polynomials within each parity;
// with psi_p = sum_k beta_pk P_k the transform is
// V_p(y) = sum_k beta_pk sqrt(2 (2k + 1)) (-i)^k j_k(c y).
void band_functions(int NB, int B, int L, std::vector<double>& u, std::vector<double>& v) {
  const Real c = 3.14159265358979323846264338327950288L * L / (2 * NB);
  Mat beta(kNP, std::vector<Real>(kLeg, 0.0L));
  for (int par = 0; par < 2; ++par) {
    const int n = kLeg / 2;
    Mat a(n, std::vector<Real>(n, 0.0L)), vec;
    for (int i = 0; i < n; ++i) {
      const Real k = 2 * i + par;
      a[i][i] = k * (k + 1) + c * c * (2 * k * k + 2 * k - 1) / ((2 * k - 1) * (2 * k + 3));
      if (i + 1 < n)
        a[i][i + 1] = a[i + 1][i] =
            c * c * (k + 1) * (k + 2) / ((2 * k + 3) * std::sqrt((2 * k + 1) * (2 * k + 5)));
    }
    jacobi(a, vec);
    for (int p = 0; p < kNP / 2; ++p)
      for (int i = 0; i < n; ++i) beta[2 * p + par][2 * i + par] = vec[p][i];
  }
  // (the square roots once: in the loops they were most of an event's set-up)
  Real up[kLeg], vp[kLeg];
  for (int k = 0; k < kLeg; ++k) {
    up[k] = std::sqrt(k + 0.5L);
    vp[k] = std::sqrt((Real)(2 * (2 * k + 1))) * (((k >> 1) & 1) ? -1 : 1);
  }
  u.assign((size_t)B * kNP, 0.0);
  for (int t = 0; t < B; ++t) {
    const Real x = (t - 0.5L * (B - 1)) / (0.5L * B);
    Real p0 = 1, p1 = x, sum[kNP] = {0};
    for (int k = 0; k < kLeg; ++k) {
      const Real pk = p0 * up[k];
      for (int p = k & 1; p < kNP; p += 2) sum[p] += beta[p][k] * pk;
      const Real p2 = ((2 * k + 3) * x * p1 - (k + 1) * p0) / (k + 2);
      p0 = p1;
      p1 = p2;
    }
    for (int p = 0; p < kNP; ++p) u[(size_t)t * kNP + p] = (double)sum[p];
  }
  v.assign((size_t)kNP * L, 0.0);
  for (int m = 0; m <= L / 2; ++m) {  // kappa = m and -m: V_p(-y) = (-1)^p V_p(y)
    const Real z = c * m / (0.5L * L);
    // spherical Bessel functions by downward recurrence, sum (2k + 1) j_k^2 = 1
    Real jk[kLeg] = {0};
    if (m == 0) {
      jk[0] = 1;
    } else {
      Real hi = 0, lo = 1e-300L, norm = 0, val[kLeg] = {0};
      for (int k = kLeg + 40; k >= 0; --k) {  // lo = j_k, hi = j_{k+1} (unnormalised)
        if (k < kLeg) val[k] = lo;
        norm += (2 * k + 1) * lo * lo;
        const Real down = (2 * k + 1) / z * lo - hi;
        hi = lo;
        lo = down;
      }
      const Real j0 = std::sin(z) / z;
      const Real j1 = j0 / z - std::cos(z) / z;
      Real sc = 1 / std::sqrt(norm);
      const bool by0 = std::fabs(j0) > std::fabs(j1);
      if ((by0 ? val[0] * j0 : val[1] * j1) < 0) sc = -sc;
      for (int k = 0; k < kLeg; ++k) jk[k] = val[k] * sc;
    }
    for (int p = 0; p < kNP; ++p) {
      Real s = 0;
      for (int k = p & 1; k < kLeg; k += 2)
        s += beta[p][k] * vp[k] * jk[k];
      double* vp2 = v.data() + ((size_t)(p >> 1) * L + L / 2) * 2 + (p & 1);
      if (L / 2 + m < L) vp2[2 * m] = (double)s;
      vp2[-2 * m] = (p & 1) ? -(double)s : (double)s;
    }
  }
}

template <typename T>
int init_band(EvDev& ev, BandDev& bd, char* p) {
  constexpr int NB = BandTypes<T>::NB;
  const int B = ev.N / NB, S = band_steps<T>(ev.N), L = ev.L, jd = ev.jlo + L / 2;
  const size_t M = (size_t)NB * 4 * S;
  auto take = [&](size_t nb) {
    char* q = p;
    p += (nb + 255) / 256 * 256;
    return q;
  };
  double2* uv = reinterpret_cast<double2*>(take(M * sizeof(double2)));
  double* lf = reinterpret_cast<double*>(take(M * sizeof(double)));
  cplx<T>* dw = reinterpret_cast<cplx<T>*>(take(ev.nd * M * sizeof(cplx<T>)));
  T* u = reinterpret_cast<T*>(take((size_t)S * 64 * sizeof(T)));
  double2* v = reinterpret_cast<double2*>(take((size_t)kNP * L * sizeof(double)));
  double2* rot = reinterpret_cast<double2*>(take((size_t)L * sizeof(double2)));
  std::vector<double> hu, hv;
  band_functions(NB, B, L, hu, hv);
  std::vector<T> lane_u((size_t)S * 64);
  for (int s = 0; 4 * s < B; ++s)
    for (int l = 0; l < 64; ++l)
      lane_u[((size_t)(s >> 1) * 64 + l) * 2 + (s & 1)] =
          (T)hu[(size_t)(4 * s + (l >> 4)) * kNP + (l & 15)];
  std::vector<double2> hr(L);
  for (int jj = 0; jj < L; ++jj) {
    const long double a = -3.14159265358979323846264338327950288L * (B - 1) *
                          (long double)(jj - L / 2) / (long double)ev.N;
    hr[jj] = make_double2((double)std::cos(a), (double)std::sin(a));
  }
  GWL_HIP_CHECK(hipMemcpy(u, lane_u.data(), lane_u.size() * sizeof(T), hipMemcpyHostToDevice));
  GWL_HIP_CHECK(hipMemcpy(v, hv.data(), hv.size() * sizeof(double), hipMemcpyHostToDevice));
  GWL_HIP_CHECK(hipMemcpy(rot, hr.data(), hr.size() * sizeof(double2), hipMemcpyHostToDevice));
  hipLaunchKernelGGL(k_band_tables<T>, dim3((unsigned)((M + 255) / 256)), dim3(256), 0, 0, ev, jd,
                     uv, lf, dw);
  GWL_HIP_CHECK(hipGetLastError());
  bd.uv = uv;
  bd.lf = lf;
  bd.dw = dw;
  bd.u = u;
  bd.v = v;
  bd.rot = rot;
  return GWL_OK;
}

template <typename T>
size_t band_bytes(const EvDev& ev) {
  const size_t S = band_steps<T>(ev.N), M = (size_t)BandTypes<T>::NB * 4 * S;
  const size_t b = M * 24 + ev.nd * M * sizeof(cplx<T>) + S * 64 * sizeof(T) +
                   (size_t)ev.L * (kNP * 8 + 16) + 8 * 256;
  return (b + 255) / 256 * 256;
}

// Block sums of one pass (32 KB a row in float32, 64 in float64): they stay in
// the 256 MB last-level cache between the two kernels.  Passes are full but for
// the last: of equal size they take longer (4097, 4500 and 8200 rows of 16384
// bins, three detectors: 200, 219, 379 us full, 214, 226, 399 equal).
constexpr size_t kPassBytes = (size_t)128 << 20;
constexpr long long kMinPassRows = 64;

template <typename T> constexpr size_t band_row_bytes() {
  return (size_t)BandTypes<T>::NB * kNP * 2 * sizeof(double);
}

// How a batch is cut: R rows per wavefront, then the groups, so that 24 to 48
// wavefronts per CU are queued (8 run at once, and three rounds or more even out
// the ends: 4096 rows of 16384 bins take 208, 199, 194 and 194 us with 8, 16, 32
// and 64, parts of 8, 4, 2 and one group; 24 asks for the third of these), then,
// where all groups leave the chip short of 8, the steps (each part adds a row
// of sums to read back).  A caller's tile sets both targets.
template <typename T>
BandSplit band_split(const gwl_event* e, long long n, int& R) {
  const EvDev& ev = e->dev;
  constexpr int NG = BandTypes<T>::NB / 16;
  const int chunks = (band_steps<T>(ev.N) + kChunk - 1) / kChunk;
  const int wpc = e->tile_wg_per_cu;
  const long long target = (long long)e->ctx->n_cu * (wpc > 0 ? wpc : 24);
  const long long least = (long long)e->ctx->n_cu * (wpc > 0 ? wpc : 8);
  R = sizeof(T) == 4 && n * NG >= 2 * least ? 2 : 1;
  const long long items = (n + R - 1) / R;
  BandSplit sp{1, 1};
  while (sp.gg < NG && items * sp.gg < target) sp.gg *= 2;
  while (sp.gs < 8 && 2 * sp.gs <= chunks && items * sp.gg * sp.gs < least) sp.gs *= 2;
  return sp;
}

template <typename T, int ND, bool CUT>
void launch_band_cut(const BandArgs& a, int R, hipStream_t st) {
  const unsigned nsplit = (unsigned)(a.split.gg * a.split.gs);
  const long long per = kBandWaves * R;
  const dim3 grid((unsigned)((a.n + per - 1) / per), nsplit);
  if constexpr (sizeof(T) == 4) {
    if (R == 2) {
      hipLaunchKernelGGL((k_band<T, ND, 2, CUT>), grid, dim3(64 * kBandWaves), 0, st, a);
      return;
    }
  }
  hipLaunchKernelGGL((k_band<T, ND, 1, CUT>), grid, dim3(64 * kBandWaves), 0, st, a);
}

bool cut_rows(const EvDev& ev) { return (ev.flags & GWL_TF2_END_ISCO) != 0; }

template <typename T, int ND>
void launch_band(const BandArgs& a, int R, hipStream_t st) {
  if (cut_rows(a.ev)) launch_band_cut<T, ND, true>(a, R, st);
  else launch_band_cut<T, ND, false>(a, R, st);
}

template <int ND>
void launch_band_row(const BandArgs& a, size_t lds, hipStream_t st) {
  const dim3 grid((unsigned)a.n), block(kFinThreads);
  if (cut_rows(a.ev)) hipLaunchKernelGGL((k_band_row<ND, true>), grid, block, lds, st, a);
  else hipLaunchKernelGGL((k_band_row<ND, false>), grid, block, lds, st, a);
}

// One kernel from a row per CU on, on segments where it was slower than k_time.
bool band_row_wins(const gwl_event* e, int64_t n) {
  return e->dev.N <= 2048 && n >= e->ctx->n_cu;
}

}  // namespace

namespace {

// Whole steps of four bins in every block.
template <typename T>
bool band_fits(const EvDev& ev) {
  return ev.approx == GWL_TAYLORF2 && (ev.flags & GWL_TIME_MARG) && ev.P == 512 && ev.L <= 512 &&
         ev.N % (4 * BandTypes<T>::NB) == 0;
}

// Row constants of every row, then the block sums of a pass: at least
// kMinPassRows rows, kPassBytes where the workspace allows.
template <typename T>
size_t band_ws(long long rows, long long pass) {
  return ((size_t)rows * sizeof(RowW) + 255) / 256 * 256 + (size_t)pass * band_row_bytes<T>();
}

template <typename T>
size_t band_ws_bytes_t(const gwl_event* e, int64_t rows) {
  if (!band_dev<T>(e->dev).uv) return 0;
  // steps are cut (gs <= 8) only below two rounds of whole groups
  const long long wpc = e->tile_wg_per_cu > 0 ? e->tile_wg_per_cu : 8;
  const long long few = 2 * wpc * e->ctx->n_cu / (BandTypes<T>::NB / 16) + 1;
  const long long most = std::max<long long>(rows, 8 * std::min<long long>(rows, few));
  return band_ws<T>(rows, std::min<long long>(most, kPassBytes / band_row_bytes<T>()));
}

template <typename T>
int launch_band_eval_t(gwl_event* e, const double* params, int64_t n, int ld, double* out,
                       hipStream_t st) {
  const EvDev& ev = e->dev;
  char* ws = reinterpret_cast<char*>(e->ws);
  RowW* rows = reinterpret_cast<RowW*>(ws);
  const size_t head = ((size_t)n * sizeof(RowW) + 255) / 256 * 256;
  double* c = reinterpret_cast<double*>(ws + head);
  const long long room =
      e->ws_bytes > head ? (long long)((e->ws_bytes - head) / band_row_bytes<T>()) : 0;
  if (room < 1) {
    set_error("workspace too small for the time transform");
    return GWL_E_INVALID;
  }
  const size_t lds = finish_lds<T>();
  if (lds > e->ctx->lds_per_block) {
    set_error("time transform exceeds the LDS of a workgroup");
    return GWL_E_UNSUPPORTED;
  }
  if (int rc = launch_rowconst(e, params, n, ld, rows, st)) return rc;
  if (sizeof(T) == 8 && band_row_wins(e, n)) {
    BandArgs a{};
    a.ev = ev;
    a.rows = rows;
    a.n = n;
    a.out = out;
    if (int rc = timing_begin(e, st)) return rc;
    switch (ev.nd) {
      case 1: launch_band_row<1>(a, lds, st); break;
      case 2: launch_band_row<2>(a, lds, st); break;
      case 3: launch_band_row<3>(a, lds, st); break;
      default: launch_band_row<4>(a, lds, st); break;
    }
    GWL_HIP_CHECK(hipGetLastError());
    return timing_end(e, st);
  }
  const long long tile = std::min<long long>(
      std::min<long long>(room, kPassBytes / band_row_bytes<T>()), n);
  for (long long r0 = 0; r0 < n; r0 += tile) {
    const long long m = std::min<long long>(tile, n - r0);
    BandArgs a{};
    int R = 1;
    a.ev = ev;
    a.rows = rows + r0;
    a.n = m;
    a.split = band_split<T>(e, m, R);
    while (a.split.gs > 1 && m * a.split.gs > room) a.split.gs /= 2;
    a.out = c;
    if (int rc = timing_begin(e, st)) return rc;
    switch (ev.nd) {
      case 1: launch_band<T, 1>(a, R, st); break;
      case 2: launch_band<T, 2>(a, R, st); break;
      case 3: launch_band<T, 3>(a, R, st); break;
      default: launch_band<T, 4>(a, R, st); break;
    }
    GWL_HIP_CHECK(hipGetLastError());
    if (int rc = timing_end(e, st, r0 + m == n)) return rc;
    FinishArgs f{ev, rows + r0, c, a.split.gs, out + r0};
    hipLaunchKernelGGL((cut_rows(ev) ? k_band_finish<T, true> : k_band_finish<T, false>),
                       dim3((unsigned)m), dim3(kFinThreads), lds, st, f);
    GWL_HIP_CHECK(hipGetLastError());
  }
  return GWL_OK;
}

}  // namespace

bool band_tables_wanted(const EvDev& ev) { return band_fits<float>(ev); }

size_t band_table_bytes(const EvDev& ev) {
  return band_bytes<float>(ev) + (band_fits<double>(ev) ? band_bytes<double>(ev) : 0);
}

int band_table_init(EvDev& ev, char* p) {
  if (int rc = init_band<float>(ev, ev.band32, p)) return rc;
  if (band_fits<double>(ev))
    if (int rc = init_band<double>(ev, ev.band64, p + band_bytes<float>(ev))) return rc;
  GWL_HIP_CHECK(hipDeviceSynchronize());
  return GWL_OK;
}

bool band_eligible(const gwl_event* e, bool fp64) {
  if (!(fp64 ? e->dev.band64.uv : e->dev.band32.uv)) return false;
  if (e->transform == GWL_TRANSFORM_WAVE) return true;
  return e->transform == GWL_TRANSFORM_AUTO && e->tile_rows == 0;
}

size_t band_ws_min_bytes(const gwl_event*, int64_t rows, bool fp64) {
  const long long pass = std::min<long long>(std::max<long long>(rows, 8), kMinPassRows);
  return fp64 ? band_ws<double>(rows, pass) : band_ws<float>(rows, pass);
}

size_t band_ws_bytes(const gwl_event* e, int64_t rows) {
  return std::max(band_ws_bytes_t<float>(e, rows), band_ws_bytes_t<double>(e, rows));
}

int launch_band_eval(gwl_event* e, bool fp64, const double* params, int64_t n, int ld,
                     double* out, hipStream_t st) {
  return fp64 ? launch_band_eval_t<double>(e, params, n, ld, out, st)
              : launch_band_eval_t<float>(e, params, n, ld, out, st);
}

size_t band_multi_row_bytes() { return band_row_bytes<float>(); }

size_t band_multi_lds_bytes() { return finish_lds<float>(); }

int band_multi_launch(gwl_multi* m, hipStream_t st) {
  BandMultiArgs a;
  a.evs = m->d_evs;
  a.rows = m->d_rows;
  a.groups = m->d_groups;
  a.roww = reinterpret_cast<const RowW* const*>(m->d_roww);
  a.c = reinterpret_cast<double* const*>(m->d_parts);
  a.items = m->d_items;
  a.n_items = m->d_n_items;
  // eager launches cover the current lists; a captured graph, the largest ones
  const size_t items = m->capturing ? m->max_items : (size_t)std::max(1, m->n_items);
  const size_t blocks = m->capturing ? m->max_blocks : (size_t)std::max(1, m->n_blocks);
  bool cut = false;
  for (const gwl_event* e : m->events) cut = cut || cut_rows(e->dev);
  hipLaunchKernelGGL(cut ? k_band_multi<true> : k_band_multi<false>, dim3((unsigned)items),
                     dim3(64 * kBandWaves), 0, st, a);
  GWL_HIP_CHECK(hipGetLastError());
  FinishMultiArgs f;
  f.evs = m->d_evs;
  f.rows = m->d_rows;
  f.roww = a.roww;
  f.c = a.c;
  f.out = m->d_outs;
  f.block_event = m->d_block_event;
  f.block_row0 = m->d_block_row0;
  f.n_blocks = m->d_n_blocks;
  hipLaunchKernelGGL(cut ? k_band_finish_multi<true> : k_band_finish_multi<false>,
                     dim3((unsigned)(blocks * kMultiEpiRows)), dim3(kFinThreads),
                     band_multi_lds_bytes(), st, f);
  GWL_HIP_CHECK(hipGetLastError());
  return GWL_OK;
}

}  // namespace gwl

extern "C" int gwl_band_functions_host(int32_t n_blocks, int32_t n_bins, int32_t n_window,
                                       double* u, double* v) {
  if ((n_blocks != 128 && n_blocks != 256) || n_bins < 1 || n_window < 1 || n_window > 512 || !u ||
      !v) {
    gwl::set_error("gwl_band_functions_host: invalid argument");
    return GWL_E_INVALID;
  }
  std::vector<double> hu, hv;
  gwl::band_functions(n_blocks, n_bins, n_window, hu, hv);
  std::copy(hu.begin(), hu.end(), u);
  std::copy(hv.begin(), hv.end(), v);
  return GWL_OK;
}
