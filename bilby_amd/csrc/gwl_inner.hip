// TaylorF2 inner products without time marginalisation (gfx950): <d|h> summed
// over the band for every row (bilby/gw/utils.py:118-138), <h|h> comes with the
// row constants (prefix sums, k_rowconst).
//
// One wavefront holds two rows and walks the bins two at a time per lane
// (lane l: bins 128 q + 2 l and + 1), in units of kUnit bins whose sums go to
// their own partials, so that a row's value does not depend on the split or on
// what it is batched with.  The phase basis f^1/3, f^-1/3, ln f and d / S
// f^-7/6 are tables: evaluated in the kernel, the cube root and logarithm of
// every bin, and one sin / cos pair per detector, took three times the
// instructions.
//
// Bound: vector issue (no matrix product: the rows share no operand but the
// tables).  4095 rows, 8 s at 4096 Hz, three detectors: float32 492 -> 114 us,
// float64 over the rows past the escalation bound 416 -> 118 us (against one
// workgroup per tile of 8 or 4 rows and 1024 bins, k_reduce).
#include "gwl_internal.h"
#include "gwl_tf2_rows.h"

#include <algorithm>

namespace gwl {

namespace {

constexpr int kUnit = 1024;  // bins per partial: 8 pairs of bins a lane
constexpr int kWaves = 4;    // wavefronts per workgroup, two rows each

// bins 0 .. N (the Nyquist bin with the others), padded with zero data
__host__ __device__ __forceinline__ long long inner_bins(int N) {
  return ((long long)N + kUnit) / kUnit * kUnit;
}

template <typename T, int ND>
struct InnerRow : Tf2Row<T, ND> {
  static constexpr int NO = ND - 1;
  cplx<T> w1[NO > 0 ? NO : 1], w2[NO > 0 ? NO : 1];  // one bin, one pair (128 bins) on
  const cplx<T>* dwr;
  const cplx<T>* dwo[NO > 0 ? NO : 1];
};

template <typename T, int ND, bool SHARED>
struct InnerIn {
  double2 uv[2];
  double2 lf;
  cplx<T> d[SHARED ? 1 : 2][ND][2];
};

// pair: its index times 64 plus the lane
template <typename T, int ND, bool SHARED>
__device__ __forceinline__ void inner_load(const InnerDev& ev, const InnerRow<T, ND>* b,
                                           unsigned pair, InnerIn<T, ND, SHARED>& in) {
  in.uv[0] = load_at<double2>(ev.uv, pair * 32u);
  in.uv[1] = load_at<double2>(ev.uv, pair * 32u + 16u);
  in.lf = load_at<double2>(ev.lf, pair * 16u);
#pragma unroll
  for (int r = 0; r < (SHARED ? 1 : 2); ++r) {
    load_pair(b[r].dwr, pair * (unsigned)(2 * sizeof(cplx<T>)), in.d[r][0]);
#pragma unroll
    for (int k = 0; k < ND - 1; ++k)
      load_pair(b[r].dwo[k], pair * (unsigned)(2 * sizeof(cplx<T>)), in.d[r][k + 1]);
  }
}

// Sums of the two rows over units [u0, u1) into part[(unit n + row)].
template <typename T, int ND, bool SHARED>
__device__ __forceinline__ void inner_units(const InnerDev& ev, const InnerRow<T, ND>* b, double df,
                                            int u0, int u1, bool nomask, const long long* pick,
                                            int live, long long n, int lane, double* part) {
  constexpr int NO = ND - 1;
  using C = cplx<T>;
  constexpr int kPairs = kUnit / 128;  // per unit
  InnerIn<T, ND, SHARED> in[2];
  const unsigned last = (unsigned)(u1 * kPairs - 1);
  inner_load<T, ND, SHARED>(ev, b, (unsigned)(u0 * kPairs) * 64u + (unsigned)lane, in[0]);
  for (int u = u0; u < u1; ++u) {
    double acc[2][2] = {{0.0, 0.0}, {0.0, 0.0}};
    // (uniform) a unit outside both rows' supports sums to zero; elements
    // outside them are zeroed where the tables' own zeros do not do it
    const bool any = (b[0].kb < (u + 1) * kUnit && b[0].ke >= u * kUnit) ||
                     (b[1].kb < (u + 1) * kUnit && b[1].ke >= u * kUnit);
    if (!any)
      inner_load<T, ND, SHARED>(ev, b, min((unsigned)((u + 1) * kPairs), last) * 64u +
                                           (unsigned)lane, in[0]);
    const bool mask = !nomask && (b[0].kb > u * kUnit || b[0].ke < (u + 1) * kUnit - 1 ||
                                  b[1].kb > u * kUnit || b[1].ke < (u + 1) * kUnit - 1);
    for (int q0 = 0; any && q0 < kPairs; q0 += 4) {
      const unsigned q = (unsigned)(u * kPairs + q0);
      const int n0 = (int)(q * 128u) + 2 * lane;
      C rot[2][NO > 0 ? NO : 1];
      C s[2] = {cmk<C>((T)0, (T)0), cmk<C>((T)0, (T)0)};
#pragma unroll
      for (int r = 0; r < 2; ++r)
#pragma unroll
        for (int k = 0; k < NO; ++k)
          rot[r][k] = tf2_rotated<T, ND>(b[r], k, (double)n0 * df);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        // (the chunk has four pairs: slots alternate)
        inner_load<T, ND, SHARED>(ev, b, min(q + j + 1, last) * 64u + (unsigned)lane,
                                  in[(j + 1) & 1]);
        __builtin_amdgcn_sched_barrier(0);
        const InnerIn<T, ND, SHARED>& v = in[j & 1];
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int r = 0; r < 2; ++r) {
            C ro[NO > 0 ? NO : 1];
#pragma unroll
            for (int k = 0; k < NO; ++k) {
              ro[k] = i ? cmul_fma(rot[r][k], b[r].w1[k]) : rot[r][k];
              if (i) rot[r][k] = cmul_fma(rot[r][k], b[r].w2[k]);
            }
            C x = tf2_product<T, ND>(tf2_cycles<T, ND>(b[r], v.uv[i].x, v.uv[i].y,
                                                       i ? v.lf.y : v.lf.x),
                                     ro, v.d[SHARED ? 0 : r], i);
            if (mask) {
              const int m = n0 + 128 * j + i;
              const bool ok = m >= b[r].kb && m <= b[r].ke;
              x = cmk<C>(ok ? x.x : (T)0, ok ? x.y : (T)0);
            }
            s[r] = cadd(s[r], x);
          }
      }
      // sums of more than 8 values are float64
#pragma unroll
      for (int r = 0; r < 2; ++r) {
        acc[r][0] += (double)s[r].x;
        acc[r][1] += (double)s[r].y;
      }
    }
    // over the lanes: the halves of the wavefront keep a row each, their
    // halves a component each
    const bool up = lane & 32, im = lane & 16;
    double keep[2];
#pragma unroll
    for (int c = 0; c < 2; ++c)
      keep[c] = (up ? acc[1][c] : acc[0][c]) + __shfl_xor(up ? acc[0][c] : acc[1][c], 32, 64);
    double v = (im ? keep[1] : keep[0]) + __shfl_xor(im ? keep[0] : keep[1], 16, 64);
#pragma unroll
    for (int off = 8; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    if ((lane & 15) == 0 && (lane >> 5) < live)
      part[2 * ((long long)u * n + pick[lane >> 5]) + ((lane >> 4) & 1)] = v;
  }
}

struct InnerArgs {
  InnerDev ev;
  double df;
  int N;
  const RowW* rows;
  long long n;
  const int* count;  // if set: only rows r < *count exist (n bounds it)
  int units, split;  // units in all, parts of them in the grid
  double* part;      // [units][n][2]
};

template <typename T, int ND>
__global__ __launch_bounds__(64 * kWaves, 2) void k_inner(InnerArgs a) {
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const long long n = a.count ? min(a.n, (long long)*a.count) : a.n;
  const long long row0 = (long long)blockIdx.x * (2 * kWaves);
  if (row0 >= n) return;
  long long pick[2];
  const int live = pick_rows<2>(a.rows, row0, n, lane, wid, pick);
  if (live == 0) return;
  const size_t M = (size_t)inner_bins(a.N);
  const cplx<T>* dw = reinterpret_cast<const cplx<T>*>(
      sizeof(T) == 4 ? static_cast<const void*>(a.ev.dw32) : static_cast<const void*>(a.ev.dw64));
  InnerRow<T, ND> b[2];
  int nomask = 1;
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    const RowW& rw = a.rows[pick[r]];
    tf2_row<T, ND>(rw, b[r]);
    nomask &= rw.nomask;
#pragma unroll
    for (int k = 0; k < ND - 1; ++k) {
      double2 corr = make_double2(1.0, 0.0);
      b[r].w1[k] = tf2_rotation<T>(a.df * b[r].dd[k], 0.5, corr);
      b[r].w2[k] = tf2_rotation<T>((128.0 * a.df) * b[r].dd[k], 1.5, corr);
      tf2_rho<T, ND>(rw, k, corr, b[r]);
      b[r].dwo[k] = dw + (size_t)(k < b[r].ref ? k : k + 1) * M;
    }
    b[r].dwr = dw + (size_t)b[r].ref * M;
  }
  const int u0 = (int)((long long)blockIdx.y * a.units / a.split);
  const int u1 = (int)((long long)(blockIdx.y + 1) * a.units / a.split);
  if (b[0].ref == b[1].ref)
    inner_units<T, ND, true>(a.ev, b, a.df, u0, u1, nomask, pick, live, a.n, lane, a.part);
  else
    inner_units<T, ND, false>(a.ev, b, a.df, u0, u1, nomask, pick, live, a.n, lane, a.part);
}

__global__ __launch_bounds__(256) void k_inner_tables(EvDev ev, double2* uv, double* lf,
                                                      float2* dw32, double2* dw64) {
  const long long M = inner_bins(ev.N);
  const long long n = (long long)blockIdx.x * 256 + threadIdx.x;
  if (n >= M) return;
  double2 b2 = make_double2(0.0, 0.0);
  double ln = 0.0, amp = 0.0;
  if (n > 0 && n <= ev.N) {
    double b[kNB];
    tf2_basis((double)n * ev.df, b);
    b2 = make_double2(b[5], b[3]);
    ln = b[7];
    amp = b[1] * sqrt(b[3]);
  }
  uv[n] = b2;
  lf[n] = ln;
  for (int d = 0; d < ev.nd; ++d) {
    double2 w = make_double2(0.0, 0.0);
    if (n < ev.N) w = ev.dw64[(size_t)d * ev.N + n];
    else if (n == ev.N) w = make_double2(ev.dwN[d][0], ev.dwN[d][1]);
    w = make_double2(w.x * amp, w.y * amp);
    dw64[(size_t)d * M + n] = w;
    dw32[(size_t)d * M + n] =
        make_float2((float)(w.x * kExpm2piGain), (float)(w.y * kExpm2piGain));
  }
}

template <typename T>
int launch_inner_t(const gwl_event* e, const InnerArgs& a, hipStream_t st) {
  const dim3 grid((unsigned)((a.n + 2 * kWaves - 1) / (2 * kWaves)), (unsigned)a.split);
  switch (e->dev.nd) {
    case 1: hipLaunchKernelGGL((k_inner<T, 1>), grid, dim3(64 * kWaves), 0, st, a); break;
    case 2: hipLaunchKernelGGL((k_inner<T, 2>), grid, dim3(64 * kWaves), 0, st, a); break;
    case 3: hipLaunchKernelGGL((k_inner<T, 3>), grid, dim3(64 * kWaves), 0, st, a); break;
    default: hipLaunchKernelGGL((k_inner<T, 4>), grid, dim3(64 * kWaves), 0, st, a); break;
  }
  GWL_HIP_CHECK(hipGetLastError());
  return GWL_OK;
}

}  // namespace

int inner_units_of(const EvDev& ev) { return (int)(inner_bins(ev.N) / kUnit); }

size_t inner_table_bytes(const EvDev& ev) {
  const size_t M = (size_t)inner_bins(ev.N);
  return M * 24 + (size_t)ev.nd * M * 24;
}

int inner_table_init(EvDev& ev, char* p) {
  const size_t M = (size_t)inner_bins(ev.N);
  double2* uv = reinterpret_cast<double2*>(p);
  double2* dw64 = uv + M;
  double* lf = reinterpret_cast<double*>(dw64 + ev.nd * M);
  float2* dw32 = reinterpret_cast<float2*>(lf + M);
  hipLaunchKernelGGL(k_inner_tables, dim3((unsigned)(M / 256)), dim3(256), 0, 0, ev, uv, lf, dw32,
                     dw64);
  GWL_HIP_CHECK(hipGetLastError());
  GWL_HIP_CHECK(hipDeviceSynchronize());
  ev.inner = InnerDev{uv, reinterpret_cast<const double2*>(lf), dw32, dw64};
  return GWL_OK;
}

int launch_inner(const gwl_event* e, bool fp64, const RowW* rows, int64_t n, const int* count,
                 double* part, hipStream_t st) {
  InnerArgs a{};
  a.ev = e->dev.inner;
  a.df = e->dev.df;
  a.N = e->dev.N;
  a.rows = rows;
  a.n = n;
  a.count = count;
  a.units = inner_units_of(e->dev);
  // about 24 wavefronts per CU queued; a live count may be far below n, so
  // its rows are cut to four units at most
  const long long target = 24LL * e->ctx->n_cu, pairs = (n + 1) / 2;
  long long split = std::min<long long>(a.units, (target + pairs - 1) / pairs);
  if (count) split = std::max<long long>(split, (a.units + 3) / 4);
  a.split = (int)std::max<long long>(1, split);
  a.part = part;
  return fp64 ? launch_inner_t<double>(e, a, st) : launch_inner_t<float>(e, a, st);
}

}  // namespace gwl
