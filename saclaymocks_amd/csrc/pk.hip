// Per-mode P(k) tables on gfx950 (interpolate_pk.py).
//
// For each mode of the k-space box: k from the float32 axes with the
// reference's float32 operations (correctly rounded, as numpy's), the spline
// segment from a uniform guess table plus a short walk, a Horner cubic in
// FP64, then float32 max(P, 0) / Vcell and its square root.  And the rows of
// the missing 1D power (p1d_missing.py).
#include <math.h>

#include "fft_core.h"
#include "route.h"
#include "smk_internal.h"

using namespace smk;

namespace {

// P(k) of a piecewise-cubic spline: segment from the guess table, then a short walk
__device__ __forceinline__ double spline_eval(const smk_pk_spline& sp, double k) {
  const double g = floor((k - sp.g_lo) / sp.g_step);
  const int s = g < 0.0 ? 0 : (g >= (double)(sp.n_guess - 1) ? sp.n_guess - 1 : (int)g);
  int iv = sp.guess[s];
  while (iv + 1 < sp.n_int && sp.x[iv + 1] <= k) ++iv;
  while (iv > 0 && sp.x[iv] > k) --iv;
  const double t = k - sp.x[iv];
  const double* cc = sp.c + 4 * (int64_t)iv;
  return ((cc[0] * t + cc[1]) * t + cc[2]) * t + cc[3];
}

// the spline segment of the last point
struct Segment {
  double lo, hi;              // [lo, hi), to infinity at the ends of the spline
  double x, c0, c1, c2, c3;
  int iv;
};

__device__ __forceinline__ void find_segment(const smk_pk_spline& sp, double r_step, double k, Segment& s) {
  // mostly the next one
  int iv = s.iv + 1;
  if (!(k >= s.hi && iv < sp.n_int && (iv + 1 == sp.n_int || k < sp.x[iv + 1]))) {
    iv = sp.guess[(int)fmin(fmax((k - sp.g_lo) * r_step, 0.0), (double)(sp.n_guess - 1))];
    while (iv + 1 < sp.n_int && sp.x[iv + 1] <= k) ++iv;
    while (iv > 0 && sp.x[iv] > k) --iv;
  }
  const double* cc = sp.c + 4 * (int64_t)iv;
  s.iv = iv;
  s.x = sp.x[iv];
  s.lo = iv > 0 ? s.x : -INFINITY;
  s.hi = iv + 1 < sp.n_int ? sp.x[iv + 1] : INFINITY;
  s.c0 = cc[0];
  s.c1 = cc[1];
  s.c2 = cc[2];
  s.c3 = cc[3];
}

// The correctly rounded float32 square root, through FP64: a third-order step
// from the hardware's reciprocal square root is within 2^-51, and the root of a
// float32 is never nearer than 2^-50 to the middle of two.
__device__ __forceinline__ float sqrt_f32(float x) {
  const double d = (double)x, y = __builtin_amdgcn_rsq(d), h = d * y, e = fma(-h, y, 1.0);
  const float r = (float)fma(h, e * fma(0.375, e, 0.5), h);
  return __builtin_amdgcn_classf(x, 0x180) ? r : x;   // x if not positive and finite
}

struct TableArgs {
  smk_pk_spline sp;
  double r_step, r_lo;            // 1 / sp.g_step, -sp.g_lo / sp.g_step
  double vcell, r_vcell;          // vcell, 1 / vcell
  const float *kx, *ky, *kz;
  uint32_t ny, nzh, nch;          // nch: 64-mode pieces of a row
  float* out;
  uint64_t nrows, ngroup;         // groups of TABLE_ROWS rows
  // the grid's waves as a step over (group, piece), and its group as rows (i, j)
  uint64_t dgroup;
  uint32_t dch, di, dj;
};

// the bin of k, of bins 0 ... last of 1 / r_step (a NaN takes 0)
__device__ __forceinline__ uint32_t guess_bin(double k, double r_step, double r_lo, uint32_t last) {
  const uint32_t g = (uint32_t)fmax(fma(k, r_step, r_lo), 0.0);
  return g < last ? g : last;
}

// max(P, 0) in float32, P the cubic c at d
__device__ __forceinline__ float table_power(const double* c, double d) {
  return fmaxf((float)(((c[0] * d + c[1]) * d + c[2]) * d + c[3]), 0.0f);
}

__device__ __forceinline__ float power_global(const TableArgs& a, double k) {
  int iv = a.sp.guess[guess_bin(k, a.r_step, a.r_lo, (uint32_t)a.sp.n_guess - 1)];
  while (iv + 1 < a.sp.n_int && a.sp.x[iv + 1] <= k) ++iv;
  while (iv > 0 && a.sp.x[iv] > k) --iv;
  return table_power(a.sp.c + 4 * (int64_t)iv, k - a.sp.x[iv]);
}

constexpr int TABLE_ROWS = 4;  // rows that a wave's lanes have at a time
constexpr int SEGS = 1760;     // segments in LDS: two blocks of 1024 threads per CU
constexpr int BINS = 4096;     // bins of the guess table in LDS
// A thread per mode, the spline in global memory: tables of few modes or of
// rows that would leave many lanes of k_pk_table idle (smk_route::pk_table).
__global__ __launch_bounds__(256) void k_pk_modes(TableArgs a, uint64_t nmodes) {
  const uint64_t m = (uint64_t)blockIdx.x * 256 + threadIdx.x;
  if (m >= nmodes) return;
  const uint64_t row = m / a.nzh;
  const float kx = a.kx[row / a.ny], ky = a.ky[row % a.ny], kz = a.kz[m % a.nzh];
  const float k = sqrt_f32(add_rn(add_rn(mul_rn(kx, kx), mul_rn(ky, ky)), mul_rn(kz, kz)));
  a.out[m] = sqrt_f32((float)((double)power_global(a, (double)k) / a.vcell));
}

// A wave has 64 neighbouring modes of TABLE_ROWS rows at a time, a lane one
// column of them: k from the float32 axes as numpy's sqrt((kx*kx + ky*ky) + kz*kz),
// each operation correctly rounded.  With LDS the block keeps the segments that
// the guess table reaches (if no more than SEGS) and a guess of BINS bins; what
// they do not settle goes to the spline in global memory.
//
// A table of 40 x 2560 x 769 takes 67 us to write.  It took 375 us with a thread
// per mode: two 64-bit modulos, two FP64 square roots and two divisions each,
// and a guess table of 256 KB gathered through L1.  Now 197 with LDS and 250
// without; the instructions left (60 per mode, 7 of them conversions or
// reciprocal roots of a quarter of the rate) take about 165.  Four modes of a
// row per lane instead, with their index arithmetic: 248 and 340; eight rows:
// 205, spilling.  A spline of 1e5 nodes within reach: 1563 before, 1374.
template <bool LDS>
__global__ __launch_bounds__(LDS ? 1024 : 256) __attribute__((amdgpu_waves_per_eu(8))) void k_pk_table(TableArgs a) {
  __shared__ double x[LDS ? SEGS + 2 : 1];
  __shared__ __align__(16) double c[LDS ? 4 * (SEGS + 1) : 2];
  __shared__ uint16_t guess[LDS ? BINS : 1];   // bytes into x
  const int tid = threadIdx.x, nt = blockDim.x, lane = tid & 63;
  // the segments of the guess table's range, [s0, s0 + ns)
  int s0 = 0, ns = 0, sh = 0;
  bool lds = false;
  if (LDS) {
    s0 = a.sp.guess[0];
    ns = a.sp.guess[a.sp.n_guess - 1] - s0 + 1;
    lds = ns >= 1 && ns <= SEGS;
    if (lds) {
      while ((a.sp.n_guess - 1) >> sh >= BINS) ++sh;
      for (int q = tid; q <= (a.sp.n_guess - 1) >> sh; q += nt) {
        const int g = a.sp.guess[q << sh] - s0;
        guess[q] = (uint16_t)(8 * (g < 0 ? 0 : (g < ns ? g : ns - 1)));
      }
      // (the spline's last segment has no end; segment ns is never taken)
      for (int q = tid; q <= ns + 1; q += nt)
        x[q] = q < ns || (q == ns && s0 + ns < a.sp.n_int) ? a.sp.x[s0 + q] : (q == ns ? INFINITY : -INFINITY);
      for (int q = tid; q < 4 * ns; q += nt) c[q] = a.sp.c[4 * (int64_t)s0 + q];
    }
    __syncthreads();
  }
  // the scaling by a power of 2 is exact: bin >> sh
  const double r_bin = ldexp(a.r_step, -sh), r_bin0 = ldexp(a.r_lo, -sh);
  const uint32_t last_bin = (uint32_t)(a.sp.n_guess - 1) >> sh;
  const uint32_t w = blockIdx.x * (nt / 64) + (uint32_t)__builtin_amdgcn_readfirstlane(tid / 64);
  uint32_t ch = w % a.nch, i = w / a.nch * TABLE_ROWS / a.ny, j = w / a.nch * TABLE_ROWS % a.ny;
  for (uint64_t group = w / a.nch; group < a.ngroup;) {
    const uint64_t row = group * TABLE_ROWS;
    const uint32_t l = ch * 64 + (uint32_t)lane;
    const float kz = a.kz[l < a.nzh ? l : a.nzh - 1], cc = mul_rn(kz, kz);
    double k[TABLE_ROWS];
    float r[TABLE_ROWS];
    uint32_t iu = i, ju = j;
#pragma unroll
    for (int u = 0; u < TABLE_ROWS; ++u) {
      const float kx = a.kx[iu], ky = a.ky[ju];
      k[u] = (double)sqrt_f32(add_rn(add_rn(mul_rn(kx, kx), mul_rn(ky, ky)), cc));
      if (row + (uint64_t)u + 1 < a.nrows && ++ju == a.ny) {   // past the last row the last row again
        ju = 0;
        ++iu;
      }
    }
    bool off = false;   // past the segments in LDS, or two segments past the bin's
    if (LDS && lds) {
      uint32_t at[TABLE_ROWS];
      double x0[TABLE_ROWS];
      const char *xb = reinterpret_cast<const char*>(x), *cb = reinterpret_cast<const char*>(c);
#pragma unroll
      for (int u = 0; u < TABLE_ROWS; ++u) at[u] = guess[guess_bin(k[u], r_bin, r_bin0, last_bin)];
      // the bin's segment or the next one, mostly
#pragma unroll
      for (int u = 0; u < TABLE_ROWS; ++u) at[u] += k[u] >= *reinterpret_cast<const double*>(xb + at[u] + 8) ? 8u : 0u;
#pragma unroll
      for (int u = 0; u < TABLE_ROWS; ++u) {
        x0[u] = *reinterpret_cast<const double*>(xb + at[u]);
        const double x1 = *reinterpret_cast<const double*>(xb + at[u] + 8);
        off |= !(k[u] >= x0[u]) | !(k[u] < x1);
      }
#pragma unroll
      for (int u = 0; u < TABLE_ROWS; ++u)
        r[u] = table_power(reinterpret_cast<const double*>(cb + 4 * at[u]), k[u] - x0[u]);
    }
    if (!lds) {
      // the loads of all rows ahead of what waits for them
      int iv[TABLE_ROWS];
      double x0[TABLE_ROWS], x1[TABLE_ROWS];
#pragma unroll
      for (int u = 0; u < TABLE_ROWS; ++u)
        iv[u] = a.sp.guess[guess_bin(k[u], a.r_step, a.r_lo, (uint32_t)a.sp.n_guess - 1)];
#pragma unroll
      for (int u = 0; u < TABLE_ROWS; ++u) {
        x0[u] = a.sp.x[iv[u]];
        x1[u] = a.sp.x[iv[u] + 1];
      }
#pragma unroll
      for (int u = 0; u < TABLE_ROWS; ++u) {
        if (k[u] >= x1[u] || k[u] < x0[u]) {
          while (iv[u] + 1 < a.sp.n_int && a.sp.x[iv[u] + 1] <= k[u]) ++iv[u];
          while (iv[u] > 0 && a.sp.x[iv[u]] > k[u]) --iv[u];
          x0[u] = a.sp.x[iv[u]];
        }
      }
#pragma unroll
      for (int u = 0; u < TABLE_ROWS; ++u) r[u] = table_power(a.sp.c + 4 * (int64_t)iv[u], k[u] - x0[u]);
    } else if (off) {
#pragma unroll 1
      for (int u = 0; u < TABLE_ROWS; ++u) {
        const float v = power_global(a, u == 0 ? k[0] : (u == 1 ? k[1] : (u == 2 ? k[2] : k[3])));
        r[0] = u == 0 ? v : r[0];
        r[1] = u == 1 ? v : r[1];
        r[2] = u == 2 ? v : r[2];
        r[3] = u == 3 ? v : r[3];
      }
    }
    // the quotient through 1 / vcell, which is exact to 2^-53: rounded once where
    // it is normal, as a quotient of float32s is then no nearer than 2^-49 to the
    // middle of two; a subnormal one may be the middle itself and is divided
    float q[TABLE_ROWS];
    bool sub = false;
#pragma unroll
    for (int u = 0; u < TABLE_ROWS; ++u) {
      q[u] = (float)((double)r[u] * a.r_vcell);
      sub |= __builtin_amdgcn_classf(q[u], 0x080);
    }
    if (sub) {
#pragma unroll
      for (int u = 0; u < TABLE_ROWS; ++u) q[u] = (float)((double)r[u] / a.vcell);
    }
#pragma unroll
    for (int u = 0; u < TABLE_ROWS; ++u)
      if (l < a.nzh && row + (uint64_t)u < a.nrows) a.out[(row + (uint64_t)u) * a.nzh + l] = sqrt_f32(q[u]);
    // the next piece of this wave
    group += a.dgroup;
    i += a.di;
    j += a.dj;
    ch += a.dch;
    if (ch >= a.nch) {
      ch -= a.nch;
      ++group;
      j += TABLE_ROWS;
    }
    while (j >= a.ny) {
      j -= a.ny;
      ++i;
    }
  }
}

struct RsdArgs {
  smk_pk_spline sp;
  const double* k_par;
  const double* k_perp;
  int n_perp;
  double beta;
  int model;
  double q1, q2, kp, kv, av, bv, G;
  double dx, kny;
  double* out;
};

// k_perp * P3(k_par, k_perp) of p1d_missing.py:12-37, 49-52; lkpar = log(k_par)
template <int MODEL>
__device__ __forceinline__ double rsd_integrand(const RsdArgs& a, double kpar, double lkpar, double kperp) {
  const double k = sqrt(kpar * kpar + kperp * kperp);
  const double mu = kpar / fmax(k, 1e-15);
  const double p = fmax(spline_eval(a.sp, k), 0.0);
  double f = 1.0;
  if (MODEL == 1) {
    const double d2 = k * k * k * p * a.G * a.G / 2.0 / (M_PI * M_PI);
    // (k / k_v)^a_v mu^b_v as one exponential of logs, mu = k_par / k; the
    // reference's powers where a base is 0
    double pw;
    if (kpar > 0.0) {
      const double lk = log(k);
      pw = exp(a.av * (lk - log(a.kv)) + a.bv * (lkpar - lk));
    } else {
      pw = pow(k / a.kv, a.av) * pow(mu, a.bv);
    }
    f = exp((a.q1 * d2 + a.q2 * d2 * d2) * (1.0 - pw) - (k / a.kp) * (k / a.kp));
  } else if (MODEL == 2) {
    const double w = exp(-a.dx * a.dx * k * k / 2.0);
    f = k < a.kny ? w * w : 0.0;
  }
  const double r = 1.0 + a.beta * mu * mu;
  return kperp * r * r * f * p;
}

// The sum over [j0, j1) of a block's row of k_perp.  The trapezoid sum is taken as
// sum_j f_j (x_{j+1} - x_{j-1}) / 2 (half intervals at the ends), so each
// point is evaluated once.
template <int MODEL>
__device__ __forceinline__ double row_sum(const RsdArgs& a, double kpar, int j0, int j1) {
  const double lkpar = kpar > 0.0 ? log(kpar) : 0.0;
  const int n = a.n_perp;
  double acc = 0.0;
  for (int j = j0 + (int)threadIdx.x; j < j1; j += 256) {
    const double x = a.k_perp[j];
    const double hi = j + 1 < n ? a.k_perp[j + 1] : x;
    const double lo = j > 0 ? a.k_perp[j - 1] : x;
    acc += (hi - lo) * rsd_integrand<MODEL>(a, kpar, lkpar, x) / 2.0;
  }
  return acc;
}

// log and exp in FP64 from a table and a short polynomial (P. T. P. Tang, ACM
// TOMS 16 (1990) 378 and 15 (1989) 144): the argument is reduced to a node of
// the table and a remainder small enough for a degree of 6 and 5.  log_t: of
// normal numbers, error below 1.2 half ulps of the larger of |log x| and 1 / 2;
// exp_t: arguments of [-745, 690], relative error below 3e-16.
constexpr double LN2_HI = 0x1.62e42fefap-1, LN2_LO = 0x1.cf79abc9e3b3ap-40;   // LN2_HI: 36 bits

struct MathTables {
  // c the middles of the 128ths of [1, 2): 1 / c; log c to 36 bits after the point, and the rest
  double rcp[128], lhi[128], llo[128];
  double pw[64];              // 2^(i / 64)
};

__device__ __forceinline__ void fill_tables(MathTables& t, int tid) {
  if (tid < 128) {
    const double r = 1.0 / (1.0 + (tid + 0.5) / 128.0);
    const double l = -log(r), hi = rint(l * 0x1p36) * 0x1p-36;
    t.rcp[tid] = r;
    t.lhi[tid] = hi;
    t.llo[tid] = l - hi;
  } else if (tid < 192) {
    t.pw[tid - 128] = exp2((tid - 128) / 64.0);
  }
}

__device__ __forceinline__ double log_t(const MathTables& t, double x) {
  const uint64_t u = (uint64_t)__double_as_longlong(x);
  const double e = (double)((int)(u >> 52) - 1023);
  const int i = (int)(u >> 45) & 127;
  const double m = __longlong_as_double((long long)((u & 0x000fffffffffffffull) | 0x3ff0000000000000ull));
  const double z = fma(m, t.rcp[i], -1.0);       // |z| <= 1 / 256
  double q = fma(z, -1.0 / 6, 1.0 / 5);
  q = fma(z, q, -1.0 / 4);
  q = fma(z, q, 1.0 / 3);
  q = fma(z, q, -1.0 / 2);
  q = fma(z * z, q, fma(e, LN2_LO, t.llo[i]));
  return fma(e, LN2_HI, t.lhi[i]) + (z + q);     // the product's sum is exact
}

__device__ __forceinline__ double exp_t(const MathTables& t, double y) {
  constexpr double M = 6755399441055744.0;       // 1.5 2^52: the sum rounds to an integer
  const double s = fma(y, 64 * 1.4426950408889634, M), n = s - M;
  const double f = fma(n, -LN2_LO / 64, fma(n, -LN2_HI / 64, y));   // |f| <= ln 2 / 128
  const int k = (int)__double_as_longlong(s);
  double q = fma(f, 1.0 / 120, 1.0 / 24);
  q = fma(f, q, 1.0 / 6);
  q = fma(f, q, 0.5);
  q = fma(f * f, q, f);
  const double w = t.pw[k & 63];
  return ldexp(fma(w, q, w), k >> 6);
}

// The row's sum with fewer FP64 instructions per point (models 0 and 1): one
// reciprocal square root gives k and mu^2, the spline's segment is kept from
// one point of a lane to the next, and model 1's powers and exponentials
// are one log_t and two exp_t.  ok is cleared where an argument leaves
// their ranges or is no number: the row is then row_sum's.
//
// Bound by FP64 issue.  20000 rows of 20000 points, model 1: 344 instructions
// per point and 3.5 ms with the library's square root, divisions, log and exp,
// 110 and 1.35 ms (80% of the issue rate) here.  With the segment of every
// point looked up in the guess table 1.40; 8 waves per SIMD instead of 6 spill
// (1.55), 4 leave latencies bare (1.50).  The log's and exp's short forms in base 2
// took 6 instructions less, but their constants' rounding made the rows' error
// against exact sums four times larger; as it is, it is half of before.
template <int MODEL>
__device__ __forceinline__ double row_fast(const RsdArgs& a, const MathTables& t, double kpar, bool& ok) {
  const int n = a.n_perp;
  const double kp2 = kpar * kpar, r_step = 1.0 / a.sp.g_step;
  const double lkpar = log(kpar), lkv = log(a.kv), rkp = 1.0 / a.kp;
  const double cg = a.G * a.G / (2.0 * M_PI * M_PI);
  // the rest of 1 / k_p, whose rounding would be the same in every point
  const double rkp_lo = fma(-rkp, a.kp, 1.0) * rkp;
  Segment s;
  s.iv = -1;
  s.lo = s.hi = INFINITY;
  double acc = 0.0;
  const auto point = [&](double x, double dx) {
    const double k2 = fma(x, x, kp2);
    // 1 / k by a third-order step from the hardware's estimate
    const double y0 = __builtin_amdgcn_rsq(k2), h = k2 * y0, e = fma(-h, y0, 1.0);
    const double c = e * fma(0.375, e, 0.5);
    const double k = fma(h, c, h), rk = fma(y0, c, y0);
    if (!(k >= s.lo && k < s.hi)) find_segment(a.sp, r_step, k, s);
    const double d = k - s.x;
    const double p = fmax(fma(fma(fma(s.c0, d, s.c1), d, s.c2), d, s.c3), 0.0);
    ok = ok && k2 < 1e200;
    double g = x * p;
    if (MODEL == 1) {
      const double d2 = cg * (k * k2) * p;
      const double lk = 0.5 * log_t(t, k2);
      const double y1 = fma(a.av, lk - lkv, a.bv * (lkpar - lk));
      const double pw = exp_t(t, y1);
      const double kk = fma(k, rkp, k * rkp_lo);
      const double y2 = fma(d2 * fma(a.q2, d2, a.q1), 1.0 - pw, -(kk * kk));
      ok = ok && fabs(y1) < 690.0 && y2 < 690.0;
      g *= exp_t(t, fmax(y2, -745.0));
    }
    const double mu = kpar * rk, r = fma(a.beta * mu, mu, 1.0);
    acc = fma(dx, g * (r * r), acc);
  };
  // each wave has a quarter of the inner points, its lanes 64 points from one
  // to the next, mostly within a segment; the row's ends go to two other lanes
  const int m = n - 2, nw = (m + 3) / 4, w = (int)threadIdx.x / 64, end = (w + 1) * nw < m ? (w + 1) * nw : m;
  const double* xp = a.k_perp + 1 + w * nw + (int)(threadIdx.x & 63);
  for (int j = w * nw + (int)(threadIdx.x & 63); j < end; j += 64, xp += 64) point(xp[0], xp[1] - xp[-1]);
  if (threadIdx.x >= 254) {
    const int j = threadIdx.x == 254 ? 0 : n - 1;
    point(a.k_perp[j], a.k_perp[j > 0 ? j : 1] - a.k_perp[j > 0 ? j - 1 : 0]);
  }
  return acc * 0.5;
}

// the block's sum, in a fixed order, as the row's value
__device__ __forceinline__ void store_row(const RsdArgs& a, int i, double acc, double* red) {
  for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) a.out[i] = (((red[0] + red[1]) + red[2]) + red[3]) / 2.0 / M_PI;
}

// One block per k_par row by row_sum: rows too short or too few for what
// follows (smk_route::p1d_fast, p1d_cut_rows).
template <int MODEL>
__global__ __launch_bounds__(256) void k_p1d_rows(RsdArgs a) {
  __shared__ double red[4];
  store_row(a, blockIdx.x, row_sum<MODEL>(a, a.k_par[blockIdx.x], 0, a.n_perp), red);
}

// One block per k_par row by row_fast (models 0 and 1).
template <int MODEL>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(6))) void k_p1d_rsd_rows(RsdArgs a) {
  __shared__ double red[4];
  __shared__ MathTables t;
  const double kpar = a.k_par[blockIdx.x];
  double acc = 0.0;
  bool ok = kpar > 1e-14 && kpar < 1e100;
  if (MODEL == 1) {
    fill_tables(t, threadIdx.x);
    __syncthreads();
  }
  if (ok) acc = row_fast<MODEL>(a, t, kpar, ok);
  if (__syncthreads_or(!ok)) acc = row_sum<MODEL>(a, kpar, 0, a.n_perp);
  store_row(a, blockIdx.x, acc, red);
}

// Model 2: the integrand is 0 from k_ny on.  A block finds the range of k_perp
// within k_ny (with a margin over the rounding of k) of any of its rows, then
// sums the rows over it.  What is no number, or large enough that a product
// might overflow, counts as within.
//
// 20000 rows of 20000 points: 1.6 ms with every point evaluated, 0.21 with
// whole waves passing over the points beyond, row by row, bound by the
// 3.2 GB of k_perp that the rows read from L2; 0.09 with 8 rows to a block.
__global__ __launch_bounds__(256) void k_p1d_cut_rows(RsdArgs a, int n_par, int rows) {
  __shared__ double red[4];
  __shared__ int range[2];
  const int n = a.n_perp, i0 = blockIdx.x * rows, i1 = n_par - i0 < rows ? n_par : i0 + rows;
  if (threadIdx.x == 0) {
    range[0] = n;
    range[1] = 0;
  }
  double kp2 = INFINITY;
  bool all = !(fabs(a.beta) < 1e100);
  for (int i = i0; i < i1; ++i) {
    const double k = a.k_par[i];
    all = all || !(k * k < 1e100);
    kp2 = fmin(kp2, k * k);
  }
  const double far = a.kny * a.kny * (1.0 + 1e-12);
  __syncthreads();
  int lo = n, hi = 0;
  for (int j = threadIdx.x; j < n; j += 256) {
    const double x = a.k_perp[j], k2 = fma(x, x, kp2);
    if (all || !(k2 > far && k2 < 1e100)) {
      lo = j < lo ? j : lo;
      hi = j + 1;
    }
  }
  if (hi > 0) {
    atomicMin(&range[0], lo);
    atomicMax(&range[1], hi);
  }
  __syncthreads();
  lo = range[0] & ~255;   // whole turns of the block: the sum's order is that of the whole row
  hi = range[1];
  for (int i = i0; i < i1; ++i) {
    store_row(a, i, row_sum<2>(a, a.k_par[i], lo, hi), red);
    __syncthreads();   // red is free
  }
}

}  // namespace

extern "C" int smk_p1d_rsd_rows(const smk_pk_spline* spline, const double* k_par, int n_par, const double* k_perp,
                                int n_perp, double beta, int model, const double* prats, double dx, double kny,
                                double* out, void* stream) {
  SMK_REQUIRE(spline != nullptr && k_par != nullptr && k_perp != nullptr && out != nullptr, SMK_ERR_ARG,
              "NULL argument");
  SMK_REQUIRE(n_par >= 0 && n_perp >= 2 && model >= 0 && model <= 2, SMK_ERR_ARG, "bad grid or model");
  SMK_REQUIRE(model != 1 || prats != nullptr, SMK_ERR_ARG, "model 1 needs the Prats parameters");
  if (n_par == 0) return SMK_OK;
  RsdArgs a;
  a.sp = *spline;
  a.k_par = k_par;
  a.k_perp = k_perp;
  a.n_perp = n_perp;
  a.beta = beta;
  a.model = model;
  a.q1 = a.q2 = a.kp = a.kv = a.av = a.bv = a.G = 0.0;
  if (model == 1) {
    a.q1 = prats[0]; a.q2 = prats[1]; a.kp = prats[2]; a.kv = prats[3]; a.av = prats[4]; a.bv = prats[5];
    a.G = prats[6];
  }
  a.dx = dx;
  a.kny = kny;
  a.out = out;
  const hipStream_t st = (hipStream_t)stream;
  const int rows = model == 2 ? smk_route::p1d_cut_rows(n_par, n_perp) : 1;
  const bool fast = smk_route::p1d_fast(model, n_par, n_perp);
  void (*const whole)(RsdArgs) = model == 0   ? (fast ? k_p1d_rsd_rows<0> : k_p1d_rows<0>)
                                 : model == 1 ? (fast ? k_p1d_rsd_rows<1> : k_p1d_rows<1>)
                                              : k_p1d_rows<2>;
  if (model == 2 && rows > 0)
    hipLaunchKernelGGL(k_p1d_cut_rows, dim3((n_par + rows - 1) / rows), dim3(256), 0, st, a, n_par, rows);
  else
    hipLaunchKernelGGL(whole, dim3(n_par), dim3(256), 0, st, a);
  SMK_LAUNCH_CHECK();
  return SMK_OK;
}

extern "C" int smk_pk_table(const smk_pk_spline* spline, const float* kx, const float* ky, const float* kz, int nxs,
                            int ny, int nzh, float vcell, float* table, void* stream) {
  SMK_REQUIRE(spline != nullptr && kx != nullptr && ky != nullptr && kz != nullptr && table != nullptr, SMK_ERR_ARG,
              "NULL argument");
  SMK_REQUIRE(spline->x != nullptr && spline->c != nullptr && spline->guess != nullptr && spline->n_int >= 1 &&
                  spline->n_guess >= 1 && spline->g_step > 0.0,
              SMK_ERR_ARG, "bad spline");
  SMK_REQUIRE(nxs >= 0 && ny > 0 && nzh > 0 && vcell > 0.0f, SMK_ERR_ARG, "bad table shape");
  const uint64_t nmodes = (uint64_t)nxs * (uint64_t)ny * (uint64_t)nzh;
  if (nmodes == 0) return SMK_OK;
  SMK_REQUIRE((nmodes + 255) / 256 <= 0x7fffffffull, SMK_ERR_ARG, "table too large for one launch");
  TableArgs a;
  a.sp = *spline;
  a.r_step = 1.0 / spline->g_step;
  a.r_lo = -spline->g_lo / spline->g_step;
  a.vcell = (double)vcell;
  a.r_vcell = 1.0 / a.vcell;
  a.kx = kx;
  a.ky = ky;
  a.kz = kz;
  a.ny = (uint32_t)ny;
  a.nzh = (uint32_t)nzh;
  a.nch = (uint32_t)(((int64_t)nzh + 63) / 64);
  a.out = table;
  a.nrows = (uint64_t)nxs * (uint64_t)ny;
  a.ngroup = (a.nrows + TABLE_ROWS - 1) / TABLE_ROWS;
  const hipStream_t st = (hipStream_t)stream;
  const smk_route::PkTable route = smk_route::pk_table(nmodes, (uint64_t)nzh);
  if (route == smk_route::PK_MODES) {
    hipLaunchKernelGGL(k_pk_modes, dim3((uint32_t)((nmodes + 255) / 256)), dim3(256), 0, st, a, nmodes);
    SMK_LAUNCH_CHECK();
    return SMK_OK;
  }
  const bool lds = route == smk_route::PK_ROWS_LDS;
  // two blocks of 16 waves per CU; or as many waves as there are pieces, four to a block: fewer than 2^18 blocks
  const uint64_t blocks = lds ? 512 : (a.ngroup * a.nch + 3) / 4, waves = blocks * (lds ? 16 : 4);
  a.dgroup = waves / a.nch;
  a.dch = (uint32_t)(waves % a.nch);
  a.di = (uint32_t)(a.dgroup * TABLE_ROWS / a.ny);
  a.dj = (uint32_t)(a.dgroup * TABLE_ROWS % a.ny);
  if (lds)
    hipLaunchKernelGGL(k_pk_table<true>, dim3((uint32_t)blocks), dim3(1024), 0, st, a);
  else
    hipLaunchKernelGGL(k_pk_table<false>, dim3((uint32_t)blocks), dim3(256), 0, st, a);
  SMK_LAUNCH_CHECK();
  return SMK_OK;
}
