// Per-row constants of the TaylorF2 time-marginalised likelihood (k_rowconst:
// phase coefficients, detector amplitudes and delays, support, and <h|h> from
// per-event prefix sums of f^-7/3 sigma^2 / S, gw/utils.py:118-138), the
// evaluation of short segments by one wavefront per row, and the
// window transform under calibration marginalisation: one wavefront per (row,
// pair of response curves), 512-point transforms of the decimated
// sub-sequences as three radix-8 passes on registers (lane l holds elements
// l + 64 s) with two LDS transposes private to the wavefront, the window bins
// accumulated in float64.
#include "gwl_internal.h"
#include "gwl_tf2_rows.h"

#include <algorithm>
#include <mutex>

namespace gwl {

constexpr int kWP = 512;      // transform length
constexpr int kWaves = 4;     // wavefronts (rows) per workgroup
constexpr int kXch = 576;     // per-wave exchange buffer, padded (float2)
constexpr int kTw3 = 7 * 64;  // pass-3 twiddles W_512^(s l), [s - 1][l]

// LDS tables of the transform: tw[m] = W_512^m and tw3[s - 1][l] =
// W_512^(s l mod 512) (so that lane l reads consecutive entries), both
// from float64 sincospi.
__device__ inline void init_wave_tables(float2* tw, float2* tw3) {
  init_twiddles<kWP, 64 * kWaves>(tw);
  for (int k = threadIdx.x; k < kTw3; k += 64 * kWaves) {
    const int s = k / 64 + 1, l = k & 63;
    const int e = (s * l) & (kWP - 1);
    double sn, cs;
    sincospi(-2.0 * (double)e / (double)kWP, &sn, &cs);
    tw3[k] = make_float2((float)cs, (float)sn);
  }
}

__device__ __forceinline__ int xpad(int e) { return e + (e >> 3); }

// Orders the LDS accesses of one wavefront (the wave executes them in order;
// this keeps the compiler from moving them across).
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

struct RowArgs {
  EvDev ev;
  const double* params;
  int ld;
  long long n;
  RowW* rows;
  double2* c64 = nullptr;  // [n][GWL_MAX_DET] float64 detector amplitudes, or null
  const int* count = nullptr;  // if set: only rows r < *count exist (n bounds it)
  int* zero = nullptr;         // cleared by the first thread
  const int* index = nullptr;  // if set: row r's parameters are row index[r]
};

// Row constants of 64 rows by two wavefronts: the first takes the TaylorF2
// part (phase coefficients, amplitude), then the support and <h|h>; the
// second the sky part (GMST, antenna patterns, delays), then the reference
// detector and the relative amplitudes.  Bound by the latency of these
// float64 chains, a few wavefronts a CU at any batch: the two halves run on
// two SIMDs at the same time and meet once, in LDS.  As odd and even lanes
// of one wavefront, which runs them one after the other, with the rest after
// both: 11.0 us for 33 rows on two detectors and 20 for 1000 on three; now 6.8
// and 14.
constexpr int kRowconstRows = 64;

struct RowShare {
  double fp[GWL_MAX_DET][kRowconstRows], fc[GWL_MAX_DET][kRowconstRows];
  double amp0[kRowconstRows], ci[kRowconstRows], c4[kRowconstRows];
};

__device__ inline void rowconst_pair(const EvDev& ev, const double* row, bool live, RowW* w,
                                     double2* c64, RowShare& sh) {
  const int l = threadIdx.x & 63;
  const bool first = threadIdx.x < 64;
  double fisco = 0.0;
  int valid = 0;
  if (live && first) {
    Tf2Part t;
    tf2_part(ev, row, t);
#pragma unroll
    for (int k = 0; k < 9; ++k) w->c[k] = t.c[k];
    sh.amp0[l] = t.amp0;
    sh.ci[l] = t.ci;
    sh.c4[l] = t.c[4];
    fisco = t.fisco;
    valid = t.valid;
  } else if (live) {
    double fp[GWL_MAX_DET], fc[GWL_MAX_DET], dt[GWL_MAX_DET], hscale, jitter;
    sky_part(ev, row, fp, fc, dt, hscale, jitter);
#pragma unroll
    for (int d = 0; d < GWL_MAX_DET; ++d) {
      const bool on = d < ev.nd;
      sh.fp[d][l] = on ? fp[d] : 0.0;
      sh.fc[d][l] = on ? fc[d] : 0.0;
      w->dt[d] = on ? dt[d] : 0.0;
    }
    w->hscale = hscale;
    w->jitter = jitter;
  }
  __syncthreads();
  if (!live) return;
  const double amp0 = sh.amp0[l], ci = sh.ci[l];
  const double ap = amp0 * (1.0 + ci * ci) / 2.0, ax = amp0 * ci;
  double cre[GWL_MAX_DET], cim[GWL_MAX_DET], cabs2[GWL_MAX_DET];
#pragma unroll
  for (int d = 0; d < GWL_MAX_DET; ++d) {
    const bool on = d < ev.nd;
    cre[d] = on ? sh.fp[d][l] * ap : 0.0;
    cim[d] = on ? -sh.fc[d][l] * ax : 0.0;
    cabs2[d] = on ? cre[d] * cre[d] + cim[d] * cim[d] : 0.0;
  }
  if (first) {
    int lo, hi, kb, ke;
    mask_range(ev, lo, hi);
    tf2_support(ev, fisco, valid, lo, hi, kb, ke);
    double hh = 0.0;
#pragma unroll
    for (int d = 0; d < GWL_MAX_DET; ++d) {
      w->cabs2[d] = cabs2[d];
      if (d < ev.nd && kb <= ke) {
        const double* ps = ev.hps + (size_t)d * (ev.N + 2);
        hh += cabs2[d] * (ps[ke + 1] - ps[kb]);
      }
    }
    w->hh = hh;
    w->kb = kb;
    w->ke = ke;
    w->valid = valid;
    w->nomask = (kb <= lo && ke >= hi) ? 1 : 0;
    w->pad = 0;
    return;
  }
  // reference detector: the largest |C_d|, so that |rho_k| <= 1
  int ref = 0;
  double cr = cre[0], ci_ = cim[0], best = cabs2[0];
#pragma unroll
  for (int d = 0; d < GWL_MAX_DET; ++d) {
    w->cre[d] = (float)cre[d];
    w->cim[d] = (float)cim[d];
    if (c64) c64[d] = make_double2(cre[d], cim[d]);
    if (d > 0 && d < ev.nd && cabs2[d] > best) {
      ref = d;
      cr = cre[d];
      ci_ = cim[d];
      best = cabs2[d];
    }
  }
  const double a2 = cr * cr + ci_ * ci_;
  w->ref = ref;
  w->amp = sqrt(a2);
  w->c4r = sh.c4[l] - (a2 > 0.0 ? atan2(ci_, cr) / kTwoPi : 0.0);
#pragma unroll
  for (int k = 0; k < GWL_MAX_DET - 1; ++k) {
    const int d = k < ref ? k : k + 1;
    const double xr = k < ref ? cre[k] : cre[k + 1], xi = k < ref ? cim[k] : cim[k + 1];
    double re = 0.0, im = 0.0;
    if (d < ev.nd && a2 > 0.0) {  // C_d conj(C_ref) / |C_ref|^2
      re = (xr * cr + xi * ci_) / a2;
      im = (xi * cr - xr * ci_) / a2;
    }
    w->rre[k] = re;
    w->rim[k] = im;
  }
}

__global__ __launch_bounds__(2 * kRowconstRows) void k_rowconst(RowArgs a) {
  __shared__ RowShare sh;
  const long long r = (long long)blockIdx.x * kRowconstRows + (threadIdx.x & 63);
  const bool live = r < (a.count ? min(a.n, (long long)*a.count) : a.n);
  if (a.zero && blockIdx.x == 0 && threadIdx.x == 0) *a.zero = 0;
  const long long at = a.index && live ? (long long)a.index[r] : r;
  rowconst_pair(a.ev, a.params + at * a.ld, live, a.rows + r,
                a.c64 ? a.c64 + r * GWL_MAX_DET : nullptr, sh);
}

// The event fields the row loop reads.
struct WaveEv {
  const double* tf2b;
  const float2* dwa32;
  double df;
  int N, Q, jlo, L, nd, pad;
};

__device__ __forceinline__ WaveEv wave_ev(const EvDev& ev) {
  WaveEv w;
  w.tf2b = ev.tf2b;
  w.dwa32 = ev.dwa32;
  w.df = ev.df;
  w.N = ev.N;
  w.Q = ev.Q;
  w.jlo = ev.jlo;
  w.L = ev.L;
  w.nd = ev.nd;
  w.pad = 0;
  return w;
}

// ------------------------------------------------------------------ short segments
// One wavefront evaluates one row from the integrand to the marginalised lnL
// (float32 integrand, float64 from there on): 512-point transforms of the Q
// sub-sequences as three radix-8 passes on registers with two exchanges
// through LDS private to the wavefront, the window sums by Horner's rule over
// descending sub-sequences (acc <- acc W_N^j + Y_n2[j mod 512]), the
// marginalisation (base.py:794-820) in the same wavefront.
//
// Bound: vector issue.  Block projections (gwl_band.hip) take half of the
// instructions a bin but finish a row in 15 to 20 ns however short the segment
// is; here that is 3 to 6.  The transform is float64 because its vector
// instructions issue at the rate of unpacked float32 ones: float32 passes were
// 9 % faster (4096 rows of 4096 bins, two detectors) and added 1e-7 to the error.
// Exchanges move the real parts, then the imaginary ones, which leaves room for
// four workgroups a CU (76 us; whole values at three 87); the integrand stays
// in float32 until all of it is there (68).
constexpr int kTw2 = 7 * 8;  // pass-2 twiddles W_64^(s k), [s - 1][k]

// tw2[s - 1][k] = W_64^(s k) (lane l uses k = l mod 8), tw3[s - 1][l] =
// W_512^(s l), and wt[l + 64 s] = W_N^j for the window bin j = l + 64 s (mod 512).
__device__ inline void init_row_tables(double2* tw2, double2* tw3, double2* wt, int N, int jlo) {
  double sn, cs;
  for (int k = threadIdx.x; k < kTw2; k += 64 * kWaves) {
    sincospi(-2.0 * (double)(((k / 8 + 1) * (k & 7)) & 63) / 64.0, &sn, &cs);
    tw2[k] = make_double2(cs, sn);
  }
  for (int k = threadIdx.x; k < kTw3; k += 64 * kWaves) {
    sincospi(-2.0 * (double)(((k / 64 + 1) * (k & 63)) & (kWP - 1)) / (double)kWP, &sn, &cs);
    tw3[k] = make_double2(cs, sn);
  }
  for (int k = threadIdx.x; k < kWP; k += 64 * kWaves) {
    const int j = jlo + ((k - jlo) & (kWP - 1));
    sincospi(-2.0 * (double)j / (double)N, &sn, &cs);
    wt[k] = make_double2(cs, sn);
  }
}

// x[s] goes to element to + s step, then lane l takes elements l + 64 s: the
// real parts, then the imaginary ones through the same buffer.
__device__ __forceinline__ void row_exchange(double2* x, double* xb, int to, int step, int lane) {
#pragma unroll
  for (int s = 0; s < 8; ++s) xb[xpad(to + s * step)] = x[s].x;
  wave_sync();
#pragma unroll
  for (int s = 0; s < 8; ++s) x[s].x = xb[xpad(lane + 64 * s)];
  wave_sync();
#pragma unroll
  for (int s = 0; s < 8; ++s) xb[xpad(to + s * step)] = x[s].y;
  wave_sync();
#pragma unroll
  for (int s = 0; s < 8; ++s) x[s].y = xb[xpad(lane + 64 * s)];
  wave_sync();
}

// A row's constants, with the detectors' rotations of one step of 64 elements
// and their tables, the reference detector's first.
template <int ND>
struct TimeRow : Tf2Row<float, ND> {
  static constexpr int NO = ND - 1;
  float2 w[NO > 0 ? NO : 1];
  const float2* dwr;
  const float2* dwo[NO > 0 ? NO : 1];
};

// Sub-sequence n2 of one row: integrand (with MASK, zero outside [kb, ke], and
// slots of 64 elements outside it are not evaluated), transform, Horner step.
template <int ND, bool MASK>
__device__ __forceinline__ void time_row_step(const WaveEv& ev, const TimeRow<ND>& b, int n2,
                                              const double2* tw2l, const double2* tw3,
                                              const double2* wt, double* xb, int lane, int base2,
                                              double* accr, double* acci) {
  constexpr int NO = ND - 1;
  const int Q = ev.Q;
  // elements of the support: kb <= Q i + n2 <= ke
  const int ilo = MASK ? (b.kb - n2 + Q - 1) / Q : 0;
  const int ihi = !MASK ? kWP - 1 : b.ke >= n2 ? (b.ke - n2) / Q : -1;
  double2 x[8];
  if (ilo <= ihi) {  // (uniform)
    const double f0 = (double)(Q * lane + n2) * ev.df;
    float2 rot[NO > 0 ? NO : 1];
#pragma unroll
    for (int k = 0; k < NO; ++k) rot[k] = tf2_rotated<float, ND>(b, k, f0);
    const size_t e0 = (size_t)n2 * kWP + lane;
    const double* tb = ev.tf2b + 3 * e0;
    float2 v[8];
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      v[s] = make_float2(0.f, 0.f);
      if (!MASK || (64 * s <= ihi && 64 * s + 63 >= ilo)) {  // (uniform)
        float2 d[ND][2];
        d[0][0] = b.dwr[e0 + 64 * s];
#pragma unroll
        for (int k = 0; k < NO; ++k) d[k + 1][0] = b.dwo[k][e0 + 64 * s];
        const double* t = tb + 3 * 64 * s;
        v[s] = tf2_product<float, ND>(tf2_cycles<float, ND>(b, t[0], t[1], t[2]), rot, d, 0);
        if constexpr (MASK) {
          const int i = lane + 64 * s;
          const bool in = i >= ilo && i <= ihi;
          v[s] = make_float2(in ? v[s].x : 0.f, in ? v[s].y : 0.f);
        }
      }
#pragma unroll
      for (int k = 0; k < NO; ++k) rot[k] = cmul_fma(rot[k], b.w[k]);
    }
#pragma unroll
    for (int s = 0; s < 8; ++s) x[s] = make_double2(v[s].x, v[s].y);
    dft8(x);
    row_exchange(x, xb, 8 * lane, 1, lane);
#pragma unroll
    for (int s = 1; s < 8; ++s) x[s] = cmul(x[s], tw2l[(s - 1) * 8]);
    dft8(x);
    row_exchange(x, xb, base2, 8, lane);
#pragma unroll
    for (int s = 1; s < 8; ++s) x[s] = cmul(x[s], tw3[(s - 1) * 64 + lane]);
    dft8(x);
  } else {
#pragma unroll
    for (int s = 0; s < 8; ++s) x[s] = make_double2(0.0, 0.0);
  }
#pragma unroll
  for (int s = 0; s < 8; ++s) {
    const double2 w = wt[lane + 64 * s];
    const double ar = accr[s], ai = acci[s];
    accr[s] = fma(ar, w.x, fma(-ai, w.y, x[s].x));
    acci[s] = fma(ar, w.y, fma(ai, w.x, x[s].y));
  }
}

// One row, after init_row_tables.
template <int ND>
__device__ __forceinline__ void time_row_eval(const EvDev& ev, const RowW& rw, double* out,
                                              const double2* tw2, const double2* tw3,
                                              const double2* wt, double* xb, int lane) {
  if (!rw.valid) {
    if (lane == 0) *out = row_valid_sentinel();
    return;
  }
  const WaveEv wv = wave_ev(ev);
  TimeRow<ND> b;
  tf2_row<float, ND>(rw, b);
#pragma unroll
  for (int k = 0; k < ND - 1; ++k) {
    // (most of a signal's weight lies in the first slots: element i is the
    // frequency i / 1024 of the sampling rate)
    double2 corr = make_double2(1.0, 0.0);
    b.w[k] = tf2_rotation<float>((64.0 * (double)ev.Q * ev.df) * b.dd[k], 1.0, corr);
    tf2_rho<float, ND>(rw, k, corr, b);
    b.dwo[k] = ev.dwa32 + (size_t)(k < b.ref ? k : k + 1) * ev.N;
  }
  b.dwr = ev.dwa32 + (size_t)b.ref * ev.N;
  const double2* tw2l = tw2 + (lane & 7);
  const int base2 = 64 * (lane >> 3) + (lane & 7);
  double accr[8], acci[8];
#pragma unroll
  for (int s = 0; s < 8; ++s) accr[s] = acci[s] = 0.0;
  if (rw.nomask)
    for (int n2 = ev.Q - 1; n2 >= 0; --n2)
      time_row_step<ND, false>(wv, b, n2, tw2l, tw3, wt, xb, lane, base2, accr, acci);
  else
    for (int n2 = ev.Q - 1; n2 >= 0; --n2)
      time_row_step<ND, true>(wv, b, n2, tw2l, tw3, wt, xb, lane, base2, accr, acci);
  const double norm = 4.0 / ev.T, amp = rw.amp * norm;
  const double hh = rw.hh * norm, hs = rw.hscale, jit = rw.jitter;
  SplineY yy;
  if (ev.flags & GWL_DISTANCE_MARG) yy = spline_y(ev.sp, hh * hs * hs);
  double m = -INFINITY, sum = 0.0;
#pragma unroll
  for (int s = 0; s < 8; ++s) {
    const int jj = (lane + 64 * s - ev.jlo) & (kWP - 1);
    if (jj < ev.L) {
      const double t = (ev.start + (double)(ev.jlo + jj + 1) * ev.tstep) + jit;
      if (t >= ev.tmin && t <= ev.tmax)
        lse_push(m, sum, epi_value(ev.flags, ev.sp, yy, hh, hs, amp * accr[s], amp * acci[s]) +
                             time_log_weight(ev, t));
    }
  }
  lse_wave(m, sum);
  if (lane == 0) *out = (m > -INFINITY) ? log(time_lse_scale(ev, ev.tdelta) * sum) + m : -INFINITY;
}

struct TimeRowArgs {
  EvDev ev;
  const RowW* rows;
  long long n;
  double* out;
};

template <int ND>
__global__ __launch_bounds__(64 * kWaves, 4) void k_time_row(TimeRowArgs a) {
  __shared__ double2 wt[kWP], tw2[kTw2], tw3[kTw3];
  __shared__ double xch[kWaves * kXch];
  init_row_tables(tw2, tw3, wt, a.ev.N, a.ev.jlo);
  __syncthreads();
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const long long r = (long long)blockIdx.x * kWaves + wid;
  if (r >= a.n) return;
  time_row_eval<ND>(a.ev, a.rows[r], a.out + r, tw2, tw3, wt, xch + wid * kXch, threadIdx.x & 63);
}

// The rows of several events that take this form: four to a workgroup of the
// list.
struct TimeRowMultiArgs {
  const EvDev* evs;
  const long long* rows;
  const RowW* const* roww;
  double* const* out;
  const int* block_event;
  const long long* block_row0;
  const int* n_blocks;
};

__global__ __launch_bounds__(64 * kWaves, 4) void k_time_row_multi(TimeRowMultiArgs a) {
  static_assert(kWaves == kMultiEpiRows, "rows per block of the list");
  __shared__ double2 wt[kWP], tw2[kTw2], tw3[kTw3];
  __shared__ double xch[kWaves * kXch];
  if ((int)blockIdx.x >= *a.n_blocks) return;
  const int e = a.block_event[blockIdx.x];
  const EvDev& ev = a.evs[e];
  init_row_tables(tw2, tw3, wt, ev.N, ev.jlo);
  __syncthreads();
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const long long r = a.block_row0[blockIdx.x] + wid;
  if (r >= a.rows[e]) return;
  double* xb = xch + wid * kXch;
  switch (ev.nd) {
    case 1: time_row_eval<1>(ev, a.roww[e][r], a.out[e] + r, tw2, tw3, wt, xb, lane); break;
    case 2: time_row_eval<2>(ev, a.roww[e][r], a.out[e] + r, tw2, tw3, wt, xb, lane); break;
    default: time_row_eval<3>(ev, a.roww[e][r], a.out[e] + r, tw2, tw3, wt, xb, lane);
  }
}

// ------------------------------------------------------------------ calibration
// Calibration and time marginalisation together (base.py:305-324, 862-877):
// for every response curve c the transform at the window of
//   sum_d cal_{c,d}(n) h_d(n) conj(d_d(n)) / S_d(n)
// and <h|h>_c = sum_d |C_d|^2 sum_n f^-7/3 sigma^2 / S_d |cal_{c,d}|^2 over
// the support (per-curve prefix sums), the time-marginalised lnL per curve,
// then the logsumexp over curves minus ln C.  One wavefront per (row, block
// of kCalCurves curves): the per-detector integrand of a sub-sequence is
// computed once and combined with each curve of the block before that
// curve's transform; the grid runs the curve blocks slowest, so a block's
// curve values stay in L2 while many rows use them.
constexpr int kCalCurves = 2;

// Per-detector h conj(d) / S at decimated element i (bin nbin), zero for
// detectors past nd (the float64 phase and float32 products of
// integrand_tf2, kept apart per detector).
template <int ND>
__device__ __forceinline__ void integrand_tf2_det(const WaveEv& ev, const RowW& rw, int i,
                                                  int nbin, float2* out) {
  const double f = (double)nbin * ev.df;
  const double* tb = ev.tf2b + 3 * (size_t)i;
  const double u = tb[0], v = tb[1], lf = tb[2];
  const double v2 = v * v, v3 = v2 * v;
  double s = rw.c[4];
  s = fma(rw.c[0], v3 * v2, s);
  s = fma(rw.c[1], v3, s);
  s = fma(rw.c[2], v2, s);
  s = fma(rw.c[3], v, s);
  s = fma(rw.c[5], u, s);
  s = fma(rw.c[6], u * u, s);
  s = fma(rw.c[7], lf, s);
  s = fma(rw.c[8], u * lf, s);
#pragma unroll
  for (int d = 0; d < ND; ++d) {
    const double cyc = fma(f, rw.dt[d], s);
    const float2 e = expm2pi((float)(cyc - floor(cyc)));
    const float2 dw = ev.dwa32[(size_t)d * ev.N + i];
    const float hr = rw.cre[d] * e.x - rw.cim[d] * e.y;
    const float hi = rw.cre[d] * e.y + rw.cim[d] * e.x;
    out[d] = make_float2(hr * dw.x + hi * dw.y, hi * dw.x - hr * dw.y);
  }
}

// The three radix-8 passes of one 512-point sub-sequence transform (inputs
// x[s] = element l + 64 s of lane l) and the window accumulation of the
// sub-sequence of wt into accr / acci (bins j = l + 64 s mod 512).
__device__ __forceinline__ void wave_transform_accumulate(const WaveEv& ev, float2* x,
                                                          const WindowTwiddle<kWP>& wt,
                                                          const float2* tw, const float2* tw3,
                                                          float2* xb, int lane, double* accr,
                                                          double* acci) {
  const int k2 = 8 * (lane & 7);
  const int base2 = 64 * (lane >> 3) + (lane & 7);
  dft8(x);
#pragma unroll
  for (int s = 0; s < 8; ++s) xb[xpad(8 * lane + s)] = x[s];
  wave_sync();
#pragma unroll
  for (int s = 0; s < 8; ++s) x[s] = xb[xpad(lane + 64 * s)];
#pragma unroll
  for (int s = 1; s < 8; ++s) x[s] = cmul(x[s], tw[(s * k2) & (kWP - 1)]);
  dft8(x);
  wave_sync();
#pragma unroll
  for (int s = 0; s < 8; ++s) xb[xpad(base2 + 8 * s)] = x[s];
  wave_sync();
#pragma unroll
  for (int s = 0; s < 8; ++s) x[s] = xb[xpad(lane + 64 * s)];
#pragma unroll
  for (int s = 1; s < 8; ++s) x[s] = cmul(x[s], tw3[(s - 1) * 64 + lane]);
  dft8(x);
  wave_sync();
  const double invN = 1.0 / (double)ev.N;
#pragma unroll
  for (int s = 0; s < 8; ++s) {
    const int jj = (lane + 64 * s - ev.jlo) & (kWP - 1);
    if (jj < ev.L) {
      const unsigned j = (unsigned)(ev.jlo + jj);
      const float2 t = expm2pi((float)((double)wt(j) * invN));
      const float2 z = cmul(t, x[s]);
      accr[s] += (double)z.x;
      acci[s] += (double)z.y;
    }
  }
}

struct CalTimeArgs {
  EvDev ev;
  const RowW* rows;
  long long n;
  long long rowblocks;  // ceil(n / kWaves)
  int nc;
  const float2* cal;    // [nc][nd][N] curve values, decimated order
  const double* calps;  // [nc][nd][N + 2] prefix sums of f^-7/3 sigma^2 / S |cal|^2
  double* lnl;          // [n][nc] time-marginalised lnL per curve
  // float64 form: the curves' float32 remainders (cal = hi + lo to 48 bits),
  // the rows' float64 detector amplitudes, W_N^m (m < N)
  const float2* cal_lo;
  const double2* c64;
  const double2* wN;
};

// The float64 integrand of each detector at decimated element i (bin nbin):
// C_d exp(-2 pi i (Psi(f) / 2 pi + f dt_d)) f^-7/6 conj(d_d / S_d) sigma.
template <int ND>
__device__ __forceinline__ void integrand_tf2_det64(const WaveEv& ev, const RowW& rw,
                                                    const double2* c64, const double2* dw64,
                                                    int i, int nbin, double2* out) {
  const double f = (double)nbin * ev.df;
  const double* tb = ev.tf2b + 3 * (size_t)i;
  const double u = tb[0], v = tb[1], lf = tb[2];
  const double v2 = v * v, v3 = v2 * v;
  double s = rw.c[4];
  s = fma(rw.c[0], v3 * v2, s);
  s = fma(rw.c[1], v3, s);
  s = fma(rw.c[2], v2, s);
  s = fma(rw.c[3], v, s);
  s = fma(rw.c[5], u, s);
  s = fma(rw.c[6], u * u, s);
  s = fma(rw.c[7], lf, s);
  s = fma(rw.c[8], u * lf, s);
  const double amp = v3 * sqrt(v);  // f^-7/6 (v = f^-1/3)
#pragma unroll
  for (int d = 0; d < ND; ++d) {
    const double cyc = fma(f, rw.dt[d], s);
    const double2 h = cmul(c64[d], expm2pi(cyc - floor(cyc)));
    const double2 w = dw64[(size_t)d * ev.N + i];
    const double wr = w.x * amp, wi = w.y * amp;
    out[d] = make_double2(h.x * wr + h.y * wi, h.y * wr - h.x * wi);
  }
}

// float64 form of wave_transform_accumulate: the three radix-8 passes in
// float64 through the wave's exchange buffer, the window accumulation with
// W_N^(n2 j mod N) from the event's float64 table.
__device__ __forceinline__ void wave_transform_accumulate64(const WaveEv& ev, double2* x,
                                                            const WindowTwiddle<kWP>& wt,
                                                            const double2* tw, const double2* tw3,
                                                            double2* xb, int lane,
                                                            const double2* wN, double* accr,
                                                            double* acci) {
  const int k2 = 8 * (lane & 7);
  const int base2 = 64 * (lane >> 3) + (lane & 7);
  dft8(x);
#pragma unroll
  for (int s = 0; s < 8; ++s) xb[xpad(8 * lane + s)] = x[s];
  wave_sync();
#pragma unroll
  for (int s = 0; s < 8; ++s) x[s] = xb[xpad(lane + 64 * s)];
#pragma unroll
  for (int s = 1; s < 8; ++s) x[s] = cmul(x[s], tw[(s * k2) & (kWP - 1)]);
  dft8(x);
  wave_sync();
#pragma unroll
  for (int s = 0; s < 8; ++s) xb[xpad(base2 + 8 * s)] = x[s];
  wave_sync();
#pragma unroll
  for (int s = 0; s < 8; ++s) x[s] = xb[xpad(lane + 64 * s)];
#pragma unroll
  for (int s = 1; s < 8; ++s) x[s] = cmul(x[s], tw3[(s - 1) * 64 + lane]);
  dft8(x);
  wave_sync();
#pragma unroll
  for (int s = 0; s < 8; ++s) {
    const int jj = (lane + 64 * s - ev.jlo) & (kWP - 1);
    if (jj < ev.L) {
      const unsigned j = (unsigned)(ev.jlo + jj);
      const double2 z = cmul(wN[wt(j)], x[s]);
      accr[s] += z.x;
      acci[s] += z.y;
    }
  }
}

template <int ND>
__global__ __launch_bounds__(64 * kWaves, 2) void k_cal_time_w(CalTimeArgs a) {
  extern __shared__ double lds_d[];
  const EvDev& ev = a.ev;
  float2* tw = reinterpret_cast<float2*>(lds_d);
  float2* tw3 = tw + kWP;
  float2* xch = tw3 + kTw3;
  const bool dist = (ev.flags & GWL_DISTANCE_MARG) != 0;
  init_wave_tables(tw, tw3);
  __syncthreads();
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const long long cb = blockIdx.x / a.rowblocks;
  const long long r = (blockIdx.x - cb * a.rowblocks) * kWaves + wid;
  if (r >= a.n) return;
  const int c0 = (int)cb * kCalCurves;
  const int ncb = min(kCalCurves, a.nc - c0);
  const RowW& rw = a.rows[r];
  if (!rw.valid) {
    if (lane < ncb) a.lnl[(size_t)r * a.nc + c0 + lane] = row_valid_sentinel();
    return;
  }
  const WaveEv wv = wave_ev(ev);
  const int Q = ev.Q;
  const int kb = rw.kb, ke = rw.ke;
  float2* xb = xch + wid * kXch;
  double accr[kCalCurves][8], acci[kCalCurves][8];
#pragma unroll
  for (int cc = 0; cc < kCalCurves; ++cc)
#pragma unroll
    for (int s = 0; s < 8; ++s) accr[cc][s] = acci[cc][s] = 0.0;
  WindowTwiddle<kWP> wt(ev.jlo, Q, 0);
  for (int n2 = 0; n2 < Q; ++n2, wt.next()) {
    const int ilo = (kb - n2 + Q - 1) / Q;
    const int ihi = ke >= n2 ? (ke - n2) / Q : -1;
    if (ilo > ihi) continue;  // nothing of the support in this sub-sequence
    float2 xd[8][ND];
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      const int i = lane + 64 * s;
      if (i >= ilo && i <= ihi) {
        integrand_tf2_det<ND>(wv, rw, n2 * kWP + i, Q * i + n2, xd[s]);
      } else {
#pragma unroll
        for (int d = 0; d < ND; ++d) xd[s][d] = make_float2(0.f, 0.f);
      }
    }
#pragma unroll
    for (int cc = 0; cc < kCalCurves; ++cc) {
      if (cc >= ncb) break;
      const float2* cal = a.cal + (size_t)(c0 + cc) * ND * ev.N + (size_t)n2 * kWP;
      float2 x[8];
#pragma unroll
      for (int s = 0; s < 8; ++s) {
        float xr = 0.f, xi = 0.f;
#pragma unroll
        for (int d = 0; d < ND; ++d) {
          const float2 k = cal[(size_t)d * ev.N + lane + 64 * s];
          xr += k.x * xd[s][d].x - k.y * xd[s][d].y;
          xi += k.x * xd[s][d].y + k.y * xd[s][d].x;
        }
        x[s] = make_float2(xr, xi);
      }
      wave_transform_accumulate(wv, x, wt, tw, tw3, xb, lane, accr[cc], acci[cc]);
    }
  }
  // epilogue per curve: time-marginalised lnL (base.py:794-820 per curve)
  const double norm = 4.0 / ev.T, xnorm = norm * kExpm2piGain;  // (the window's twiddles)
  const double hs = rw.hscale, jit = rw.jitter;
  const double b = time_lse_scale(ev, ev.tdelta);
#pragma unroll
  for (int cc = 0; cc < kCalCurves; ++cc) {
    if (cc >= ncb) break;
    const int c = c0 + cc;
    double hh = 0.0;
    if (kb <= ke) {
#pragma unroll
      for (int d = 0; d < ND; ++d) {
        const double* ps = a.calps + ((size_t)c * ND + d) * (ev.N + 2);
        hh += rw.cabs2[d] * (ps[ke + 1] - ps[kb]);
      }
    }
    hh *= norm;
    SplineY yy;
    if (dist) yy = spline_y(ev.sp, hh * hs * hs);
    double m = -INFINITY, sum = 0.0;
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      const int jj = (lane + 64 * s - ev.jlo) & (kWP - 1);
      if (jj < ev.L) {
        const int j = ev.jlo + jj;
        const double t = (ev.start + (double)(j + 1) * ev.tstep) + jit;
        if (t >= ev.tmin && t <= ev.tmax)
          lse_push(m, sum, epi_value(ev.flags, ev.sp, yy, hh, hs, xnorm * accr[cc][s],
                                     xnorm * acci[cc][s]) +
                               time_log_weight(ev, t));
      }
    }
    lse_wave(m, sum);
    if (lane == 0) a.lnl[(size_t)r * a.nc + c] = (m > -INFINITY) ? log(b * sum) + m : -INFINITY;
  }
}

// The float64 form of k_cal_time_w (base.py:305-324 in float64): the
// integrand in float64 (float64 sin / cos of the phase, float64 amplitudes
// and data), curve values hi + lo, float64 transforms and twiddles.  Tables
// in LDS: W_512^m and the pass-3 twiddles in float64, the exchange buffers.
// The float64 integrand of a curve pair needs up to 256 registers per lane:
// one workgroup per CU is asked for so that nothing spills.
template <int ND>
__global__ __launch_bounds__(64 * kWaves, 1) void k_cal_time_w64(CalTimeArgs a) {
  extern __shared__ double lds_d[];
  const EvDev& ev = a.ev;
  double2* tw = reinterpret_cast<double2*>(lds_d);
  double2* tw3 = tw + kWP;
  double2* xch = tw3 + kTw3;
  const bool dist = (ev.flags & GWL_DISTANCE_MARG) != 0;
  for (int k = threadIdx.x; k < kWP; k += 64 * kWaves) {
    double sn, cs;
    sincospi(-2.0 * (double)k / (double)kWP, &sn, &cs);
    tw[k] = make_double2(cs, sn);
  }
  for (int k = threadIdx.x; k < kTw3; k += 64 * kWaves) {
    const int e = ((k / 64 + 1) * (k & 63)) & (kWP - 1);
    double sn, cs;
    sincospi(-2.0 * (double)e / (double)kWP, &sn, &cs);
    tw3[k] = make_double2(cs, sn);
  }
  __syncthreads();
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const long long cb = blockIdx.x / a.rowblocks;
  const long long r = (blockIdx.x - cb * a.rowblocks) * kWaves + wid;
  if (r >= a.n) return;
  const int c0 = (int)cb * kCalCurves;
  const int ncb = min(kCalCurves, a.nc - c0);
  const RowW& rw = a.rows[r];
  if (!rw.valid) {
    if (lane < ncb) a.lnl[(size_t)r * a.nc + c0 + lane] = row_valid_sentinel();
    return;
  }
  double2 c64[ND];
#pragma unroll
  for (int d = 0; d < ND; ++d) c64[d] = a.c64[r * GWL_MAX_DET + d];
  const WaveEv wv = wave_ev(ev);
  const int Q = ev.Q;
  const int kb = rw.kb, ke = rw.ke;
  double2* xb = xch + wid * kXch;
  double accr[kCalCurves][8], acci[kCalCurves][8];
#pragma unroll
  for (int cc = 0; cc < kCalCurves; ++cc)
#pragma unroll
    for (int s = 0; s < 8; ++s) accr[cc][s] = acci[cc][s] = 0.0;
  WindowTwiddle<kWP> wt(ev.jlo, Q, 0);
  for (int n2 = 0; n2 < Q; ++n2, wt.next()) {
    const int ilo = (kb - n2 + Q - 1) / Q;
    const int ihi = ke >= n2 ? (ke - n2) / Q : -1;
    if (ilo > ihi) continue;
    double2 xd[8][ND];
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      const int i = lane + 64 * s;
      if (i >= ilo && i <= ihi) {
        integrand_tf2_det64<ND>(wv, rw, c64, ev.dw64, n2 * kWP + i, Q * i + n2, xd[s]);
      } else {
#pragma unroll
        for (int d = 0; d < ND; ++d) xd[s][d] = make_double2(0.0, 0.0);
      }
    }
#pragma unroll
    for (int cc = 0; cc < kCalCurves; ++cc) {
      if (cc >= ncb) break;
      const size_t off = (size_t)(c0 + cc) * ND * ev.N + (size_t)n2 * kWP;
      const float2* hi = a.cal + off;
      const float2* lo = a.cal_lo + off;
      double2 x[8];
#pragma unroll
      for (int s = 0; s < 8; ++s) {
        double xr = 0.0, xi = 0.0;
#pragma unroll
        for (int d = 0; d < ND; ++d) {
          const size_t e = (size_t)d * ev.N + lane + 64 * s;
          const float2 kh = hi[e], kl = lo[e];
          const double kr = (double)kh.x + (double)kl.x, ki = (double)kh.y + (double)kl.y;
          xr += kr * xd[s][d].x - ki * xd[s][d].y;
          xi += kr * xd[s][d].y + ki * xd[s][d].x;
        }
        x[s] = make_double2(xr, xi);
      }
      wave_transform_accumulate64(wv, x, wt, tw, tw3, xb, lane, a.wN, accr[cc], acci[cc]);
    }
  }
  const double norm = 4.0 / ev.T;
  const double hs = rw.hscale, jit = rw.jitter;
  const double b = time_lse_scale(ev, ev.tdelta);
#pragma unroll
  for (int cc = 0; cc < kCalCurves; ++cc) {
    if (cc >= ncb) break;
    const int c = c0 + cc;
    double hh = 0.0;
    if (kb <= ke) {
#pragma unroll
      for (int d = 0; d < ND; ++d) {
        const double* ps = a.calps + ((size_t)c * ND + d) * (ev.N + 2);
        hh += rw.cabs2[d] * (ps[ke + 1] - ps[kb]);
      }
    }
    hh *= norm;
    SplineY yy;
    if (dist) yy = spline_y(ev.sp, hh * hs * hs);
    double m = -INFINITY, sum = 0.0;
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      const int jj = (lane + 64 * s - ev.jlo) & (kWP - 1);
      if (jj < ev.L) {
        const int j = ev.jlo + jj;
        const double t = (ev.start + (double)(j + 1) * ev.tstep) + jit;
        if (t >= ev.tmin && t <= ev.tmax)
          lse_push(m, sum, epi_value(ev.flags, ev.sp, yy, hh, hs, norm * accr[cc][s],
                                     norm * acci[cc][s]) +
                               time_log_weight(ev, t));
      }
    }
    lse_wave(m, sum);
    if (lane == 0) a.lnl[(size_t)r * a.nc + c] = (m > -INFINITY) ? log(b * sum) + m : -INFINITY;
  }
}

// One wavefront per row, lanes over curves: logsumexp_c(lnL_c) - ln C
// (base.py:877).
__global__ __launch_bounds__(256) void k_cal_time_epi(const RowW* rows, long long n, int nc,
                                                      const double* lnl, double* out) {
  const long long r = (long long)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (r >= n) return;
  const int lane = threadIdx.x & 63;
  if (!rows[r].valid) {
    if (lane == 0) out[r] = row_valid_sentinel();
    return;
  }
  double m = -INFINITY, sum = 0.0;
  for (int c = lane; c < nc; c += 64) lse_push(m, sum, lnl[(size_t)r * nc + c]);
  lse_wave(m, sum);
  if (lane == 0) out[r] = (m > -INFINITY) ? log(sum) + m - log((double)nc) : -INFINITY;
}

// ------------------------------------------------------------------ multi-event
struct RowMultiArgs {
  const EvDev* evs;
  const double* const* params;
  const long long* rows;
  RowW* const* roww;
  int ld;
};

__global__ __launch_bounds__(2 * kRowconstRows) void k_rowconst_multi(RowMultiArgs a) {
  __shared__ RowShare sh;
  const int e = blockIdx.y;
  const long long r = (long long)blockIdx.x * kRowconstRows + (threadIdx.x & 63);
  rowconst_pair(a.evs[e], a.params[e] + r * a.ld, r < a.rows[e], a.roww[e] + r, nullptr, sh);
}

// f^1/3, f^-1/3, ln f and d / S f^-7/6 at every decimated element.
__global__ __launch_bounds__(256) void k_tf2_tables(EvDev ev, double* tb, float2* dwa) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= ev.N) return;
  const int n = ev.Q * (i & (ev.P - 1)) + (i >> ev.logP);
  double u = 0.0, v = 0.0, lf = 0.0, amp = 0.0;
  if (n > 0) {
    double b[kNB];
    tf2_basis((double)n * ev.df, b);
    u = b[5];
    v = b[3];
    lf = b[7];
    amp = b[1] * sqrt(b[3]);
  }
  tb[3 * (size_t)i + 0] = u;
  tb[3 * (size_t)i + 1] = v;
  tb[3 * (size_t)i + 2] = lf;
  for (int d = 0; d < ev.nd; ++d) {
    const double2 w = ev.dw64[(size_t)d * ev.N + i];
    dwa[(size_t)d * ev.N + i] =
        make_float2((float)(w.x * amp * kExpm2piGain), (float)(w.y * amp * kExpm2piGain));
  }
}

size_t time_wave_table_bytes(const EvDev& ev) {
  return (size_t)ev.N * (3 * sizeof(double) + ev.nd * sizeof(float2));
}

int init_time_wave_tables(EvDev& ev, char* p) {
  double* tb = reinterpret_cast<double*>(p);
  float2* dwa = reinterpret_cast<float2*>(tb + 3 * (size_t)ev.N);
  hipLaunchKernelGGL(k_tf2_tables, dim3((unsigned)((ev.N + 255) / 256)), dim3(256), 0, 0, ev, tb, dwa);
  GWL_HIP_CHECK(hipGetLastError());
  GWL_HIP_CHECK(hipDeviceSynchronize());
  ev.tf2b = tb;
  ev.dwa32 = dwa;
  return GWL_OK;
}

int time_wave_tables(gwl_event* e) {
  static std::mutex mu;  // (several calibrations of one event made at once)
  std::lock_guard<std::mutex> lock(mu);
  if (e->dev.tf2b) return GWL_OK;
  const size_t bytes = time_wave_table_bytes(e->dev);
  if (!e->wave_mem && hipMalloc(&e->wave_mem, bytes) != hipSuccess) {
    e->wave_mem = nullptr;
    set_error("hipMalloc failed for the transform tables");
    return GWL_E_NOMEM;
  }
  e->wave_bytes = bytes;
  return init_time_wave_tables(e->dev, static_cast<char*>(e->wave_mem));
}

// k_cal_time_w: the 512-entry pass-2 table, tw3, the exchange buffers
// (float64 kernel: the same tables in float64)
static size_t cal_time_lds_bytes(const EvDev& ev, bool fp64) {
  size_t b = (size_t)(kWP + kTw3 + kWaves * kXch) * (fp64 ? sizeof(double2) : sizeof(float2));
  return b;
}

int launch_rowconst(const gwl_event* e, const double* params, int64_t n, int ld, RowW* rows,
                    hipStream_t st, const int* count, int* zero, const int* index) {
  RowArgs ra{e->dev, params, ld, n, rows, nullptr, count, zero, index};
  hipLaunchKernelGGL(k_rowconst, dim3((unsigned)((n + kRowconstRows - 1) / kRowconstRows)),
                     dim3(2 * kRowconstRows), 0, st, ra);
  GWL_HIP_CHECK(hipGetLastError());
  return GWL_OK;
}

// Short segments and many rows: a wavefront per row fills the chip from about
// 16 rows per CU on, and its time goes with the bins; block projections keep
// the chip busy with few rows, and most of their time goes with the rows.
// Per launch, us, this and block projections, two detectors: 1024 bins 23 and 31
// (512 rows), 24 and 49 (1024), 36 and 91 (4096), 105 and 339 (16384); 2048 bins
// 33 and 46 (1024), 53 and 88 (4096); 4096 bins 47 and 68 (2048), 68 and 102
// (4096), 229 and 384 (16384); 8192 bins 116 and 123 (4096), 406 and 468 (16384);
// below the line 4096 bins 48 and 51 (1024), 8192 bins 85 and 78 (2048).
bool time_row_wins(const gwl_event* e, int64_t n) {
  return e->transform == GWL_TRANSFORM_AUTO && e->dev.tf2b && e->dev.N <= kTimeRowBins &&
         512 * n >= (int64_t)e->ctx->n_cu * e->dev.N;
}

int launch_time_row(gwl_event* e, const double* params, int64_t n, int ld, double* out,
                    hipStream_t st) {
  const EvDev& ev = e->dev;
  RowW* rows = reinterpret_cast<RowW*>(e->ws);
  if (roww_bytes(n) > e->ws_bytes) {
    set_error("workspace too small for the time transform");
    return GWL_E_INVALID;
  }
  if (int rc = launch_rowconst(e, params, n, ld, rows, st)) return rc;
  const TimeRowArgs a{ev, rows, (long long)n, out};
  const dim3 grid((unsigned)((n + kWaves - 1) / kWaves)), block(64 * kWaves);
  if (int rc = timing_begin(e, st)) return rc;
  switch (ev.nd) {
    case 1: hipLaunchKernelGGL(k_time_row<1>, grid, block, 0, st, a); break;
    case 2: hipLaunchKernelGGL(k_time_row<2>, grid, block, 0, st, a); break;
    case 3: hipLaunchKernelGGL(k_time_row<3>, grid, block, 0, st, a); break;
    default: hipLaunchKernelGGL(k_time_row<4>, grid, block, 0, st, a); break;
  }
  GWL_HIP_CHECK(hipGetLastError());
  return timing_end(e, st);
}

size_t roww_bytes(int64_t rows) { return (size_t)rows * sizeof(RowW); }

bool cal_time_eligible(const gwl_event* e) {
  const EvDev& ev = e->dev;
  return (ev.flags & GWL_TIME_MARG) && ev.approx == GWL_TAYLORF2 && ev.P == kWP && ev.hps &&
         ev.L <= kWP;
}

// rows: RowW, then the float64 detector amplitudes, then the per-curve lnL
static size_t cal_time_c64_offset(int64_t rows) {
  return ((size_t)rows * sizeof(RowW) + 255) / 256 * 256;
}
static size_t cal_time_lnl_offset(int64_t rows) {
  return cal_time_c64_offset(rows) + (size_t)rows * GWL_MAX_DET * sizeof(double2);
}

size_t cal_time_ws_bytes(int64_t rows, int nc) {
  return cal_time_lnl_offset(rows) + (size_t)rows * nc * sizeof(double);
}

int launch_cal_time(gwl_event* e, const double* params, int64_t n, int ld, int nc,
                    const float2* cal, const double* calps, void* ws, double* per_curve,
                    double* out, hipStream_t st, bool fp64, const float2* cal_lo,
                    const double2* wN) {
  const EvDev& ev = e->dev;
  if (fp64 && (!cal_lo || !wN)) {
    set_error("calibration time transform: float64 tables missing");
    return GWL_E_INVALID;
  }
  char* w = static_cast<char*>(ws);
  RowW* rows = reinterpret_cast<RowW*>(w);
  double2* c64 = reinterpret_cast<double2*>(w + cal_time_c64_offset(n));
  double* lnl = per_curve ? per_curve : reinterpret_cast<double*>(w + cal_time_lnl_offset(n));
  RowArgs ra{ev, params, ld, n, rows, fp64 ? c64 : nullptr};
  hipLaunchKernelGGL(k_rowconst, dim3((unsigned)((n + kRowconstRows - 1) / kRowconstRows)),
                     dim3(2 * kRowconstRows), 0, st, ra);
  GWL_HIP_CHECK(hipGetLastError());
  CalTimeArgs ca{};
  ca.ev = ev;
  ca.rows = rows;
  ca.n = n;
  ca.rowblocks = (n + kWaves - 1) / kWaves;
  ca.nc = nc;
  ca.cal = cal;
  ca.calps = calps;
  ca.lnl = lnl;
  ca.cal_lo = cal_lo;
  ca.c64 = c64;
  ca.wN = wN;
  const size_t lds = cal_time_lds_bytes(ev, fp64);
  if (lds > e->ctx->lds_per_block) {
    set_error("calibration time transform exceeds the LDS of a workgroup");
    return GWL_E_UNSUPPORTED;
  }
  const long long blocks = ca.rowblocks * ((nc + kCalCurves - 1) / kCalCurves);
  if (blocks > 0x7fffffffLL) {
    set_error("gwl_calib_eval: too many rows x curves in one call");
    return GWL_E_INVALID;
  }
  const dim3 grid((unsigned)blocks);
  if (fp64) {
    switch (ev.nd) {
      case 1: hipLaunchKernelGGL(k_cal_time_w64<1>, grid, dim3(64 * kWaves), lds, st, ca); break;
      case 2: hipLaunchKernelGGL(k_cal_time_w64<2>, grid, dim3(64 * kWaves), lds, st, ca); break;
      case 3: hipLaunchKernelGGL(k_cal_time_w64<3>, grid, dim3(64 * kWaves), lds, st, ca); break;
      default: hipLaunchKernelGGL(k_cal_time_w64<4>, grid, dim3(64 * kWaves), lds, st, ca); break;
    }
  } else {
    switch (ev.nd) {
      case 1: hipLaunchKernelGGL(k_cal_time_w<1>, grid, dim3(64 * kWaves), lds, st, ca); break;
      case 2: hipLaunchKernelGGL(k_cal_time_w<2>, grid, dim3(64 * kWaves), lds, st, ca); break;
      case 3: hipLaunchKernelGGL(k_cal_time_w<3>, grid, dim3(64 * kWaves), lds, st, ca); break;
      default: hipLaunchKernelGGL(k_cal_time_w<4>, grid, dim3(64 * kWaves), lds, st, ca); break;
    }
  }
  GWL_HIP_CHECK(hipGetLastError());
  hipLaunchKernelGGL(k_cal_time_epi, dim3((unsigned)((n + 3) / 4)), dim3(256), 0, st, rows,
                     (long long)n, nc, lnl, out);
  GWL_HIP_CHECK(hipGetLastError());
  return GWL_OK;
}

// Row constants of every event of a multi-event set.
int multi_launch_rowconst(gwl_multi* m, hipStream_t st) {
  RowMultiArgs a;
  a.evs = m->d_evs;
  a.params = m->d_params;
  a.rows = m->d_rows;
  a.roww = reinterpret_cast<RowW* const*>(m->d_roww);
  a.ld = GWL_NPARAM;
  long long maxr = 1;
  for (int64_t r : m->max_rows) maxr = std::max<long long>(maxr, r);
  hipLaunchKernelGGL(k_rowconst_multi, dim3((unsigned)((maxr + kRowconstRows - 1) / kRowconstRows),
                                              (unsigned)m->n_events),
                     dim3(2 * kRowconstRows), 0, st, a);
  GWL_HIP_CHECK(hipGetLastError());
  return GWL_OK;
}

int multi_launch_time_row(gwl_multi* m, hipStream_t st) {
  TimeRowMultiArgs a;
  a.evs = m->d_evs;
  a.rows = m->d_rows;
  a.roww = reinterpret_cast<const RowW* const*>(m->d_roww);
  a.out = m->d_outs;
  a.block_event = m->d_rblock_event;
  a.block_row0 = m->d_rblock_row0;
  a.n_blocks = m->d_n_rblocks;
  // an eager launch covers the current list, a captured graph the largest
  const size_t blocks = m->capturing ? m->max_rblocks : (size_t)m->n_rblocks;
  if (!blocks) return GWL_OK;
  hipLaunchKernelGGL(k_time_row_multi, dim3((unsigned)blocks), dim3(64 * kWaves), 0, st, a);
  GWL_HIP_CHECK(hipGetLastError());
  return GWL_OK;
}

}  // namespace gwl
