// Quasar draw on gfx950: the cells of the lognormal slab, columns along z.
//
// Reference: bin/draw_qso.py:186-462.  The reference builds ptot for the
// whole slab with numpy, then loops over the z planes drawing two uniforms
// per cell and a position in the cell.  Here every cell is independent:
// the uniforms come from Philox at counters fixed by the cell, so a thread
// reads its three field values (coalesced along z), forms ptot, and tests
// the two density conditions; only the rare cells that pass go on to the
// position, the angles, the RSD redshift and the footprint and redshift cut,
// and append a record through one atomic counter.  The host orders the
// records (they carry the reference's output order as a key).
#include <math.h>

#include "fft_core.h"
#include "smk_internal.h"

using namespace smk;

namespace {

constexpr uint32_t TAG_CELL = 0x71736f63u;
constexpr uint32_t TAG_X = 0x71736f78u;
constexpr uint32_t TAG_Y = 0x71736f79u;
constexpr uint32_t TAG_Z = 0x71736f7au;
constexpr double ZB1 = 1.9, ZB2 = 2.75, ZB3 = 3.6;   // constant.py:30-32
constexpr double H0_KMS = 100.0;                     // constant.py:36
constexpr double RAND_QSO_NB = 0.006;                // constant.py:10
// (1 + z_k)^-0.7 of the three bias redshifts
constexpr float INV1 = 0.47459308f;   // 2.9^-0.7
constexpr float INV2 = 0.39644059f;   // 3.75^-0.7
constexpr float INV3 = 0.34361295f;   // 4.6^-0.7

// uniform in [0, 1) with 53 bits from two Philox words
__device__ __forceinline__ double u53(uint32_t a, uint32_t b) {
  return ((double)(a >> 5) * 67108864.0 + (double)(b >> 6)) * 1.1102230246251565e-16;
}

// numpy.interp on ascending nodes, starting the search at node j; sp: NULL,
// or the segments' slopes (fp[j+1] - fp[j]) / (xp[j+1] - xp[j]) made on the
// host (the same correctly rounded operations, so the same bits, without a
// division per call)
__device__ __forceinline__ double interp_from(double x, const double* __restrict__ xp, const double* __restrict__ fp,
                                              const double* __restrict__ sp, int n, int j) {
  if (x <= xp[0]) return fp[0];
  if (x >= xp[n - 1]) return fp[n - 1];
  j = j < 0 ? 0 : (j > n - 2 ? n - 2 : j);
  while (j > 0 && xp[j] > x) --j;
  while (j < n - 2 && xp[j + 1] <= x) ++j;
  const double slope = sp ? sp[j] : (fp[j + 1] - fp[j]) / (xp[j + 1] - xp[j]);
  return slope * (x - xp[j]) + fp[j];
}

// start node for a uniform grid of nodes x0 + i * dx (a guess: interp_from
// walks to the exact node, so a reciprocal is good enough)
__device__ __forceinline__ int uniform_guess(double x, double x0, double dx) {
  const double g = floor((x - x0) * __builtin_amdgcn_rcp(dx));
  return g < 0.0 ? 0 : (g > 2.0e9 ? 2000000000 : (int)g);
}

// z(R): the comoving-distance table through its uniform guess table
__device__ __forceinline__ double z_of_r(const smk_qso_params& p, double r) {
  int b = uniform_guess(r, p.r2z_lo, p.r2z_step);
  b = b >= p.r2z_ng ? p.r2z_ng - 1 : b;
  return interp_from(r, p.r2z_chi, p.r2z_z, p.r2z_slope, p.r2z_n, p.r2z_guess[b]);
}

__device__ __forceinline__ double r_of_z(const smk_qso_params& p, double z) {
  // inverse lookup on the same nodes (z ascending, uniform in the reference's table)
  const int n = p.r2z_n;
  const double z0 = p.r2z_z[0], dz = (p.r2z_z[n - 1] - z0) / (double)(n - 1);
  return interp_from(z, p.r2z_z, p.r2z_chi, nullptr, n, uniform_guess(z, z0, dz));
}

__device__ __forceinline__ double coef_of_z(const smk_qso_params& p, double z) {
  // nodes: 0, then a regular grid from coef_z[1], then 10
  const double z1 = p.coef_z[1], dz = p.coef_z[2] - p.coef_z[1];
  return interp_from(z, p.coef_z, p.coef_c, p.coef_slope, p.coef_n, 1 + uniform_guess(z, z1, dz));
}

// a_k(z) = b(z)(1+z_k) / (b(z_k)(1+z)) with b(z) = 3.7((1+z)/3.33)^1.7
// (util.py:508-517), i.e. ((1+z)/(1+z_k))^0.7
__device__ __forceinline__ double a_of_z(double z, double zk) { return pow((1.0 + z) / (1.0 + zk), 0.7); }

// the two linear interpolations between the bias redshifts and their mix
// (draw_qso.py:247-250), with the constant divisions as products
__device__ __forceinline__ double mix(double z, double c, double e1, double e2, double e3) {
  constexpr double R12 = 1.0 / (ZB2 - ZB1), R23 = 1.0 / (ZB3 - ZB2);
  const double p12 = (e1 * (ZB2 - z) + e2 * (z - ZB1)) * R12;
  const double p23 = (e2 * (ZB3 - z) + e3 * (z - ZB2)) * R23;
  return c * (p12 - p23) + p23;
}

// mean of ptot at redshift z: exp((a_k sigma_k)^2 / 2) mixed as ptot
__device__ __forceinline__ double mean_ptot(const smk_qso_params& p, double z) {
  const double m1 = exp(0.5 * (a_of_z(z, ZB1) * p.sigma[0]) * (a_of_z(z, ZB1) * p.sigma[0]));
  const double m2 = exp(0.5 * (a_of_z(z, ZB2) * p.sigma[1]) * (a_of_z(z, ZB2) * p.sigma[1]));
  const double m3 = exp(0.5 * (a_of_z(z, ZB3) * p.sigma[2]) * (a_of_z(z, ZB3) * p.sigma[2]));
  return mix(z, coef_of_z(p, z), m1, m2, m3);
}

__device__ __forceinline__ double diffmod(double a, double b, double c) {
  double d = fmod(a - b, c);
  if (d < 0.0) d += c;   // Python's % for c > 0
  return fmin(d, c - d);
}

// the whole draw of one cell (column ix * ny + iy, cell mz of it)
__device__ __forceinline__ void draw_cell(const smk_qso_params& p, const float* __restrict__ p1,
                                          const float* __restrict__ p2, const float* __restrict__ p3,
                                          const float* __restrict__ vx, const float* __restrict__ vy,
                                          const float* __restrict__ vz, uint64_t seed,
                                          smk_qso_record* __restrict__ rec, int64_t cap,
                                          unsigned long long* __restrict__ count, uint32_t col, int mz) {
  const int ix = (int)(col / (uint32_t)p.ny), iy = (int)(col % (uint32_t)p.ny);
  const uint64_t c = (uint64_t)col * (uint64_t)p.nz + (uint64_t)mz;
  const double xc = p.x_axis[ix], yc = p.y_axis[iy], zcell = p.z_axis[mz];
  const double rc = sqrt(xc * xc + yc * yc + zcell * zcell);
  const double zc = z_of_r(p, rc / p.h);
  const U4 w = philox4x32_10_c4((uint32_t)c, (uint32_t)(c >> 32), TAG_CELL, 0u, seed);
  const double rnd1 = u53(w.x, w.y), rnd2 = u53(w.z, w.w);
  // ---- cond1 (draw_qso.py:421-429)
  if (p.randoms) {
    if (!(rnd1 > 1.0 - RAND_QSO_NB)) return;
  } else {
    // exp(p)**a_k(z), float32 as the reference's in-place float32 arrays
    // (:219-223, :236-238), evaluated as exp(a_k p) with a_k = ((1+z)/(1+z_k))^0.7
    // from one power per cell (the reference: a float32 exp, then a float32
    // power), on the hardware exp2 / log2 (a few 1e-7 relative: ptot only
    // decides the draw against a uniform)
    const float t = __builtin_amdgcn_exp2f(0.7f * __builtin_amdgcn_logf((float)(1.0 + zc)));
    const float e1 = __expf(t * INV1 * p1[c]);
    const float e2 = __expf(t * INV2 * p2[c]);
    const float e3 = __expf(t * INV3 * p3[c]);
    const double ptot = mix(zc, coef_of_z(p, zc), (double)e1, (double)e2, (double)e3);
    if (!(rnd1 < p.norm * ptot)) return;
  }
  // ---- cond2: n(z) at the cell centre, corrected for the fields' mean (:400-431)
  const double zcen = p.zfix_on ? p.zfix : zc;
  const double fi = rint((zcen - p.dn_z0) / p.dn_dz);
  double density = (fi >= 0.0 && fi < (double)p.dn_n) ? p.dn_cell[(int)fi] : 0.0;
  if (!p.randoms) density /= mean_ptot(p, zcen);
  if (!(p.density_max * rnd2 < density)) return;
  // ---- position in the cell (:433-437), angles and redshift (:438-444)
  const U4 wx = philox4x32_10_c4((uint32_t)ix, (uint32_t)mz, TAG_X, 0u, seed);
  const U4 wy = philox4x32_10_c4((uint32_t)iy, (uint32_t)mz, TAG_Y, 0u, seed);
  const U4 wz = philox4x32_10_c4((uint32_t)c, (uint32_t)(c >> 32), TAG_Z, 0u, seed);
  const double x = xc + (-0.5 * p.dx + p.dx * u53(wx.x, wx.y));
  const double y = yc + (-0.5 * p.dy + p.dy * u53(wy.x, wy.y));
  const double z = zcell + (-0.5 * p.dz + p.dz * u53(wz.x, wz.y));
  const double cr = cos(p.ra0), sr = sin(p.ra0), cd = cos(p.dec0), sd = sin(p.dec0);
  const double numra = cr * x - sd * sr * y + cd * sr * z;
  const double denra = -sr * x - sd * cr * y + cd * cr * z;
  const double numdec = cd * y + sd * z;
  const double r = sqrt(x * x + y * y + z * z);
  double ra = atan2(numra, denra);
  if (ra < 0.0) ra += 2.0 * M_PI;
  ra *= 180.0 / M_PI;
  const double dec = asin(numdec / r) * (180.0 / M_PI);
  const double red = p.zfix_on ? p.zfix : z_of_r(p, r / p.h);
  double red_rsd = red;
  if (p.rsd && !p.randoms) {
    const double vpar = (x * (double)vx[c] + y * (double)vy[c] + z * (double)vz[c]) / r;
    double rr = p.zfix_on ? r_of_z(p, red) * p.h : r;
    if (red < p.zmax + 1.0) {
      const double dg = interp_from(red, p.dg_z, p.dg_v, nullptr, p.dg_n,
                                    uniform_guess(red, p.dg_z[0], (p.dg_z[p.dg_n - 1] - p.dg_z[0]) / (p.dg_n - 1)));
      rr += vpar * (1.0 + red) * dg / (p.dgrowth0 * H0_KMS);
    }
    red_rsd = z_of_r(p, rr / p.h);
  }
  // ---- cond3 (:455-460)
  const double zsel = (p.rsd && !p.randoms) ? red_rsd : red;
  if (!(diffmod(ra, p.ra0 * (180.0 / M_PI), 360.0) < p.dra)) return;
  if (!(diffmod(dec, p.dec0 * (180.0 / M_PI), 180.0) < p.ddec)) return;
  if (!(zsel > p.zmin && zsel < p.zmax)) return;
  const unsigned long long pos = atomicAdd(count, 1ull);
  if ((int64_t)pos < cap) {
    smk_qso_record q;
    q.key = ((int64_t)mz * p.nx + ix) * p.ny + iy;
    q.x = x; q.y = y; q.z = z; q.r = r;
    q.z_qso = red; q.z_qso_rsd = red_rsd; q.ra = ra; q.dec = dec;
    rec[pos] = q;
  }
}

// every cell by draw_cell: block (column, 256-cell chunk of z), a thread per cell
__global__ __launch_bounds__(256) void k_qso_draw(smk_qso_params p, const float* __restrict__ p1,
                                                  const float* __restrict__ p2, const float* __restrict__ p3,
                                                  const float* __restrict__ vx, const float* __restrict__ vy,
                                                  const float* __restrict__ vz, uint64_t seed,
                                                  smk_qso_record* __restrict__ rec, int64_t cap,
                                                  unsigned long long* __restrict__ count) {
  const int mz = (int)(blockIdx.y * 256 + threadIdx.x);
  if (mz < p.nz) draw_cell(p, p1, p2, p3, vx, vy, vz, seed, rec, cap, count, blockIdx.x, mz);
}

// The draw with a mask of candidates.  Of the cells of a slice one in 10^4 to
// 10^2 passes the first condition, rnd1 < norm ptot; the others only need a
// bound.  Over a chunk of CHUNK cells along z the redshift, the exponents'
// factor t = (1 + z)^0.7 and the mix of the three fields' powers lie between
// values that one lane finds beforehand (k_qso_bounds), so a cell costs its
// three field values, one Philox call and three hardware exponentials
// (k_qso_filter); the cells that stay under the bound are set in a bit mask and
// take draw_cell, which decides as before (k_qso_masked).  The bound is above
// norm ptot by more than the float rounding of either side, so no cell that
// draw_cell would draw is left out.
//
// Measured on a slice of 160 x 2560 x 1536 cells: k_qso_draw 7.7 ms, bound by
// its FP64 lookups per cell; this way 1.67, of which the filter 1.55 (its VALU
// issues in 86% of the slots, 8.2e8 instructions; 4.9 TB/s, 72% of the rate of a
// kernel that only reads) and the bounds 0.05 (0.16 with one per 8 columns; found
// inside the filter's blocks 0.7, as a block waits for a few lanes' chains).
// With 10 and 100 times as many cells that pass, 10.4 and 20.5 ms against 1.97
// and 4.4; with a quasar in 5% of all cells k_qso_draw is still the slower, with
// one in 7% or more it is the faster, 47 against 65 at 15%.  draw_cell has a
// kernel of its own since in the filter's loop it took 216 registers (2 waves
// per SIMD, 9.4 ms), as a call from there 7.0.  In k_qso_masked's loop the
// compiler keeps its constants in registers, 199 of them if it may; 128 were
// faster at every density.  A bit per cell never overflows; a list of cells did, or was as
// large as a field.
constexpr int CHUNK = 128;        // cells along z of one bound: two waves
constexpr int BCOLS = 32;         // columns of one bound
constexpr int COLS = 16;          // columns per block of the filter
constexpr int ZCELLS = 1024;      // z cells per block: four per thread
constexpr int QUEUED = 1024;      // cells of a block's queue that are drawn together
constexpr uint64_t MASK_BLOCKS = 1024;   // as many as are resident

struct DrawBound {
  float tlo, thi;                 // (1 + z)^0.7 over the chunk, log2(e) folded in
  float g1, g2, g3;               // largest mix coefficients, times norm
  float pad;                      // 24 bytes
};

// the bound of the cells with x^2 + y^2 in [rxy0, rxy1] and z coordinate in [lo, hi]
__device__ __forceinline__ DrawBound draw_bounds(const smk_qso_params& p, double rxy0, double rxy1, double lo,
                                                 double hi) {
  DrawBound b;
  // distance along z: 0 if the range straddles the observer's plane
  const double near = lo > 0.0 ? lo : (hi < 0.0 ? -hi : 0.0), far = fmax(fabs(lo), fabs(hi));
  const double z0 = z_of_r(p, sqrt(rxy0 + near * near) / p.h), z1 = z_of_r(p, sqrt(rxy1 + far * far) / p.h);
  const float l2e = 1.4426950408889634f;
  b.tlo = __builtin_amdgcn_exp2f(0.7f * __builtin_amdgcn_logf((float)(1.0 + z0))) * l2e * (1.0f - 2e-5f);
  b.thi = __builtin_amdgcn_exp2f(0.7f * __builtin_amdgcn_logf((float)(1.0 + z1))) * l2e * (1.0f + 2e-5f);
  // c(z) over [z0, z1]: its ends and the nodes between them
  const double ca = coef_of_z(p, z0), cb = coef_of_z(p, z1);
  double c0 = fmin(ca, cb), c1 = fmax(ca, cb);
  int j = 1 + uniform_guess(z0, p.coef_z[1], p.coef_z[2] - p.coef_z[1]);
  j = j > p.coef_n - 1 ? p.coef_n - 1 : j;
  while (j > 0 && p.coef_z[j] > z0) --j;
  for (; j < p.coef_n && p.coef_z[j] < z1; ++j) {
    c0 = fmin(c0, p.coef_c[j]);
    c1 = fmax(c1, p.coef_c[j]);
  }
  // ptot = g1 e1 + g2 e2 + g3 e3, each g bilinear in (c, z): its largest value is at a corner
  constexpr double R12 = 1.0 / (ZB2 - ZB1), R23 = 1.0 / (ZB3 - ZB2);
  double g1 = 0.0, g2 = 0.0, g3 = 0.0;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const double z = k & 1 ? z1 : z0, c = k & 2 ? c1 : c0;
    g1 = fmax(g1, c * (ZB2 - z) * R12);
    g2 = fmax(g2, c * (z - ZB1) * R12 + (1.0 - c) * (ZB3 - z) * R23);
    g3 = fmax(g3, (1.0 - c) * (z - ZB2) * R23);
  }
  const double up = p.norm * (1.0 + 2e-3);
  b.g1 = (float)(up * g1);
  b.g2 = (float)(up * g2);
  b.g3 = (float)(up * g3);
  return b;
}

// one lane per bound: BCOLS columns, CHUNK cells of the z axis
__global__ __launch_bounds__(256) void k_qso_bounds(smk_qso_params p, DrawBound* __restrict__ bound, uint64_t n_bound,
                                                    uint32_t nch, uint32_t ncol) {
  const uint64_t q = (uint64_t)blockIdx.x * 256 + threadIdx.x;
  if (q >= n_bound) return;
  const uint32_t col0 = (uint32_t)(q / nch) * BCOLS;
  const int m0 = (int)(q % nch) * CHUNK, m1 = p.nz - m0 < CHUNK ? p.nz : m0 + CHUNK;
  double r0 = INFINITY, r1 = 0.0, lo = INFINITY, hi = -INFINITY;
  for (int k = 0; k < BCOLS; ++k) {
    const uint32_t col = col0 + (uint32_t)k < ncol ? col0 + (uint32_t)k : ncol - 1;
    const double xc = p.x_axis[col / (uint32_t)p.ny], yc = p.y_axis[col % (uint32_t)p.ny];
    r0 = fmin(r0, xc * xc + yc * yc);
    r1 = fmax(r1, xc * xc + yc * yc);
  }
#pragma unroll 8
  for (int mz = m0; mz < m1; ++mz) {
    lo = fmin(lo, p.z_axis[mz]);
    hi = fmax(hi, p.z_axis[mz]);
  }
  bound[q] = draw_bounds(p, r0, r1, lo, hi);
}

// mask: a bit per cell, 64 cells along z to a word, nw words to a column
__global__ __launch_bounds__(256) void k_qso_filter(int nz, int randoms, const float* __restrict__ p1,
                                                    const float* __restrict__ p2, const float* __restrict__ p3,
                                                    uint64_t seed, const DrawBound* __restrict__ bounds, uint32_t nch,
                                                    uint64_t* __restrict__ mask, uint32_t nw, uint32_t ncol) {
  static_assert(BCOLS % COLS == 0, "a block's columns share a bound");
  static_assert(CHUNK % 64 == 0, "a wave's cells share a bound");
  const int tid = threadIdx.x;
  const uint32_t col0 = blockIdx.x * COLS;
  const int m0 = (int)blockIdx.y * ZCELLS, m1 = nz - m0 < ZCELLS ? nz : m0 + ZCELLS;
  const DrawBound* __restrict__ bound = bounds + (uint64_t)(col0 / BCOLS) * nch;
  for (int k = 0; k < COLS && col0 + (uint32_t)k < ncol; ++k) {
    const uint64_t c0 = (uint64_t)(col0 + (uint32_t)k) * (uint64_t)nz;
    const uint32_t lo = (uint32_t)c0, hi = (uint32_t)(c0 >> 32);
    // the cells of a column share the counter's high word unless it carries
    const bool carries = lo > 0xffffffffu - (uint32_t)nz;
    // four cells per thread, the loads of all four ahead of their arithmetic
    float f[4][3];
    if (!randoms) {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int mz = m0 + tid + 256 * u < m1 ? m0 + tid + 256 * u : m1 - 1;
        f[u][0] = p1[c0 + (uint64_t)mz];
        f[u][1] = p2[c0 + (uint64_t)mz];
        f[u][2] = p3[c0 + (uint64_t)mz];
      }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int mz = m0 + tid + 256 * u;
      const int word = __builtin_amdgcn_readfirstlane(mz / 64);   // the wave's
      if (64 * word >= m1) break;
      bool maybe = true;
      if (randoms) {
        const uint64_t c = c0 + (uint64_t)mz;
        const U4 w = philox4x32_10_c4((uint32_t)c, (uint32_t)(c >> 32), TAG_CELL, 0u, seed);
        maybe = u53(w.x, w.y) > 1.0 - RAND_QSO_NB;
      } else if (!carries) {
        const DrawBound b = bound[64 * word / CHUNK];
        const U4 w = philox4x32_10_c4(lo + (uint32_t)mz, hi, TAG_CELL, 0u, seed);
        // rnd1 from below: its leading 27 bits, rounded down
        const float rnd = (float)(w.x >> 5) * (7.450580596923828e-9f * (1.0f - 2.4e-7f));
        const float e1 = __builtin_amdgcn_exp2f((f[u][0] > 0.0f ? b.thi : b.tlo) * (INV1 * f[u][0]));
        const float e2 = __builtin_amdgcn_exp2f((f[u][1] > 0.0f ? b.thi : b.tlo) * (INV2 * f[u][1]));
        const float e3 = __builtin_amdgcn_exp2f((f[u][2] > 0.0f ? b.thi : b.tlo) * (INV3 * f[u][2]));
        // (a NaN or an overflowing power fails the comparison: the cell is looked at)
        maybe = !(rnd > fmaf(b.g1, e1, fmaf(b.g2, e2, b.g3 * e3)));
      }
      const uint64_t m = __ballot(maybe && mz < m1);
      if ((tid & 63) == 0) mask[(uint64_t)(col0 + (uint32_t)k) * nw + (uint32_t)word] = m;
    }
  }
}

// draw_cell of the cells of the mask: a block takes a range of half words,
// queues their cells in LDS and draws them together
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void k_qso_masked(smk_qso_params p, const float* __restrict__ p1,
                                                    const float* __restrict__ p2, const float* __restrict__ p3,
                                                    const float* __restrict__ vx, const float* __restrict__ vy,
                                                    const float* __restrict__ vz, uint64_t seed,
                                                    smk_qso_record* __restrict__ rec, int64_t cap,
                                                    unsigned long long* __restrict__ count,
                                                    const uint32_t* __restrict__ mask, uint32_t nhalf, uint64_t total) {
  __shared__ uint32_t queue[QUEUED + 256 * 32];   // half word in the range and bit
  __shared__ int nqueue;
  const int tid = threadIdx.x;
  if (tid == 0) nqueue = 0;
  __syncthreads();
  // a range holds fewer than 2^27 half words: total / gridDim.x
  const uint64_t per = (total + gridDim.x - 1) / gridDim.x;
  const uint64_t h0 = per * blockIdx.x, h1 = h0 + per < total ? h0 + per : total;
  uint32_t next = h0 + (uint64_t)tid < h1 ? mask[h0 + (uint64_t)tid] : 0u;
  for (uint64_t hb = h0; hb < h1; hb += 256) {
    const uint64_t h = hb + (uint64_t)tid;
    uint32_t m = next;
    next = h + 256 < h1 ? mask[h + 256] : 0u;   // loaded a step ahead
    if (m != 0u) {
      int at = atomicAdd(&nqueue, __popc(m));
      for (; m != 0u; m &= m - 1u) queue[at++] = (uint32_t)(h - h0) * 32u + (uint32_t)(__ffs((int)m) - 1);
    }
    __syncthreads();
    const int n = nqueue;
    if (n > QUEUED || hb + 256 >= h1) {
      for (int q = tid; q < n; q += 256) {
        const uint64_t hh = h0 + queue[q] / 32u;
        draw_cell(p, p1, p2, p3, vx, vy, vz, seed, rec, cap, count, (uint32_t)(hh / nhalf),
                  (int)(hh % nhalf) * 32 + (int)(queue[q] % 32u));
      }
      __syncthreads();
      if (tid == 0) nqueue = 0;
    }
    __syncthreads();
  }
}

__global__ void k_clear_count(unsigned long long* c) {
  if (threadIdx.x == 0 && blockIdx.x == 0) *c = 0ull;
}

}  // namespace

// the scratch buffer: the bounds, then the mask
static uint64_t qso_bounds(const smk_qso_params& p) {
  const uint64_t ncol = (uint64_t)p.nx * (uint64_t)p.ny;
  return (ncol + BCOLS - 1) / BCOLS * (((uint64_t)p.nz + CHUNK - 1) / CHUNK);
}

extern "C" size_t smk_qso_scratch_bytes(const smk_qso_params* p) {
  if (p == nullptr || p->nx <= 0 || p->ny <= 0 || p->nz <= 0) return 0;
  return (size_t)(qso_bounds(*p) * sizeof(DrawBound) +
                  (uint64_t)p->nx * (uint64_t)p->ny * (((uint64_t)p->nz + 63) / 64) * sizeof(uint64_t));
}

extern "C" int smk_qso_draw(const smk_qso_params* p, const float* p1, const float* p2, const float* p3,
                            const float* vx, const float* vy, const float* vz, uint64_t seed,
                            smk_qso_record* records, int64_t capacity, int64_t* count, void* stream) {
  return smk_qso_draw_scratch(p, p1, p2, p3, vx, vy, vz, seed, records, capacity, count, nullptr, 0, stream);
}

extern "C" int smk_qso_draw_scratch(const smk_qso_params* p, const float* p1, const float* p2, const float* p3,
                                    const float* vx, const float* vy, const float* vz, uint64_t seed,
                                    smk_qso_record* records, int64_t capacity, int64_t* count, void* scratch,
                                    size_t scratch_bytes, void* stream) {
  SMK_REQUIRE(p != nullptr && count != nullptr, SMK_ERR_ARG, "NULL argument");
  SMK_REQUIRE(p->nx > 0 && p->ny > 0 && p->nz > 0, SMK_ERR_ARG, "empty slab");
  SMK_REQUIRE(p->randoms || (p1 != nullptr && p2 != nullptr && p3 != nullptr), SMK_ERR_ARG,
              "the three lognormal fields are needed unless randoms");
  SMK_REQUIRE(!p->rsd || p->randoms || (vx != nullptr && vy != nullptr && vz != nullptr), SMK_ERR_ARG,
              "rsd needs the three velocity boxes");
  SMK_REQUIRE(capacity >= 0 && (capacity == 0 || records != nullptr), SMK_ERR_ARG, "bad record buffer");
  SMK_REQUIRE(p->x_axis && p->y_axis && p->z_axis && p->r2z_chi && p->r2z_z && p->r2z_guess && p->coef_z &&
                  p->coef_c && p->dn_cell && (!p->rsd || (p->dg_z && p->dg_v)),
              SMK_ERR_ARG, "NULL table");
  SMK_REQUIRE(p->r2z_n >= 2 && p->r2z_ng >= 1 && p->coef_n >= 3 && p->dn_n >= 1 && (!p->rsd || p->dg_n >= 2) &&
                  p->r2z_step > 0.0 && p->dn_dz > 0.0,
              SMK_ERR_ARG, "bad table sizes");
  SMK_REQUIRE(scratch == nullptr || (scratch_bytes >= smk_qso_scratch_bytes(p) && ((uintptr_t)scratch & 7) == 0),
              SMK_ERR_ARG, "scratch too small or misaligned");
  hipStream_t s = (hipStream_t)stream;
  unsigned long long* cnt = reinterpret_cast<unsigned long long*>(count);
  hipLaunchKernelGGL(k_clear_count, dim3(1), dim3(64), 0, s, cnt);
  SMK_LAUNCH_CHECK();
  const uint64_t ncol = (uint64_t)p->nx * (uint64_t)p->ny;
  const uint32_t nzb = (uint32_t)(((int64_t)p->nz + 255) / 256);
  SMK_REQUIRE(ncol <= 0x7fffffffull && nzb <= 65535u, SMK_ERR_ARG, "slab too large for one launch");
  if (scratch == nullptr) {
    hipLaunchKernelGGL(k_qso_draw, dim3((uint32_t)ncol, nzb), dim3(256), 0, s, *p, p1, p2, p3, vx, vy, vz, seed, records,
                       capacity, cnt);
    SMK_LAUNCH_CHECK();
    return SMK_OK;
  }
  const uint64_t nb = qso_bounds(*p);
  DrawBound* bounds = static_cast<DrawBound*>(scratch);
  uint64_t* mask = reinterpret_cast<uint64_t*>(bounds + nb);
  const uint32_t nch = (uint32_t)(((int64_t)p->nz + CHUNK - 1) / CHUNK), nw = (uint32_t)(((int64_t)p->nz + 63) / 64);
  if (!p->randoms) {
    const uint64_t blocks = (nb + 255) / 256;
    hipLaunchKernelGGL(k_qso_bounds, dim3((uint32_t)blocks), dim3(256), 0, s, *p, bounds, nb, nch, (uint32_t)ncol);
    SMK_LAUNCH_CHECK();
  }
  hipLaunchKernelGGL(k_qso_filter,
                     dim3((uint32_t)((ncol + COLS - 1) / COLS), (uint32_t)(((int64_t)p->nz + ZCELLS - 1) / ZCELLS)),
                     dim3(256), 0, s, p->nz, p->randoms, p1, p2, p3, seed, bounds, nch, mask, nw, (uint32_t)ncol);
  SMK_LAUNCH_CHECK();
  const uint64_t total = 2 * ncol * nw;
  const uint64_t blocks = (total + 255) / 256 < MASK_BLOCKS ? (total + 255) / 256 : MASK_BLOCKS;
  hipLaunchKernelGGL(k_qso_masked, dim3((uint32_t)blocks), dim3(256), 0, s, *p, p1, p2, p3, vx, vy, vz, seed, records,
                     capacity, cnt, reinterpret_cast<const uint32_t*>(mask), 2 * nw, total);
  SMK_LAUNCH_CHECK();
  return SMK_OK;
}
