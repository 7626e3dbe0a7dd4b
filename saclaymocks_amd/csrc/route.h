// Which kernel a call takes, where that depends on its sizes only: plain
// functions of the host, each with the measurements that placed its lines.
#pragma once
#include <cstdint>

#include "../../include/saclaymocks_hip.h"

namespace smk_route {

// ------------------------------------------------------------ P(k) tables
// A wave of k_pk_table has 64 neighbouring modes of a row, so a row that does
// not fill its last 64 leaves lanes idle; k_pk_modes has a thread per mode
// whatever the rows.  The more of k_pk_table's lanes are in use, and the larger
// the table, the sooner k_pk_table wins.  Us, k_pk_modes against k_pk_table, by
// modes and by modes per row (lanes in use):
//          17 (27%)   29 (45%)   33 (52%)   37 (58%)   41 (64%)   100 (78%)
//   1 M    8.8, 12.7  8.4, 10.1  8.4, 9.3   8.5, 9.0   8.4, 9.0   8.4, 8.7
//   2 M    14, 22     13.5, 16   13.5, 15   13.6, 14.3 13.3, 13.6 13.2, 12.9
//   4.3 M  25, 41     24, 29     24, 26     24, 25     24, 22     24, 21
//   8 M    42, 69     41, 47     41, 41     41, 39     40, 35     40, 30
//   24 M   114, 184   113, 113   112, 101   111, 94    110, 86    111, 71
enum PkTable { PK_MODES, PK_ROWS, PK_ROWS_LDS };

// Tables from here on take k_pk_table with the spline in LDS, whose blocks
// first load 20 to 80 KB each: 3.9 million modes of 257 to a row take 19.3 us
// without, 4.3 million 20.6 with and without, 8 million 28.9 and 33.9.
constexpr uint64_t PK_LDS_MODES = 4u << 20;

constexpr PkTable pk_table(uint64_t modes, uint64_t nzh) {
  const uint64_t lanes = (nzh + 63) / 64 * 64;
  const uint64_t percent = modes < (9u << 17) ? 80 : modes < PK_LDS_MODES ? 63 : modes < (10u << 20) ? 53 : 45;
  if (100 * nzh < percent * lanes) return PK_MODES;
  return modes >= PK_LDS_MODES ? PK_ROWS_LDS : PK_ROWS;
}

// ------------------------------------------- rows of the missing 1D power
// Whether models 0 and 1 take the sum of fewer instructions (row_fast), which
// first fills its tables and finds its segments: it needs points to a row to
// pay for that, and more rows than two per CU, as with fewer the latency of a
// point decides, which it does not shorten.  Us, row_sum against row_fast, by
// points of a row:
//              model 1:  200         400         600         900         2500        20000
//   512 rows             7.1, 7.6    7.3, 8.4    8.9, 10.0   10.7, 11.8  21.9, 22.7  144, 147
//   1024 rows            7.3, 7.9    9.4, 10.4   12.0, 11.8  15.5, 14.6  33.6, 24.3  234, 149
//   2048 rows            11.0, 12.2  15.4, 15.7  19.3, 19.1  25.3, 21.9  57.2, 34.1  400, 162
//   8192 rows            34.7, 35.6  49.9, 45.3  63.5, 55.2  85.0, 66.1  197, 110    1399, 519
//              model 0:  600         1500        2500        5000        10000       20000
//   400 rows             7.2, 7.7    8.3, 9.9    11.5, 13.0  20.1, 21.9  36.4, 38.3  68.8, 63.3
//   768 rows             7.4, 8.0    9.6, 11.1   12.9, 13.7  22.5, 23.3  41.4, 40.1  78.9, 64.7
//   2048 rows            9.5, 12.2   17.2, 17.9  26.4, 22.9  45.2, 38.0  85.5, 62.5  164, 98.5
//   12000 rows           37.8, 50.5  81.4, 80.7  130, 114    248, 176    479, 254    931, 379
constexpr bool p1d_fast(int model, int n_par, int n_perp) {
  if (model == 0) return n_perp >= (n_par > 1024 ? 1500 : n_par > 512 ? 8000 : 15000);
  return model == 1 && n_par > 512 && n_perp >= (n_par > 2560 ? 350 : n_par > 1024 ? 550 : 750);
}

// Rows per block of model 2 (k_p1d_cut_rows), so that the blocks fill the card:
// 1024 blocks or more, 4096 where a row has less than a point per thread.  0:
// a few short rows, as they are, without the range of k_perp found first (100
// to 512 rows of 900 points 7.3 us against 8.0; 600 the same either way).
constexpr int p1d_cut_rows(int n_par, int n_perp) {
  if (n_par <= 512 && n_perp <= 1024) return 0;
  const int rows = n_par / (n_perp < 200 ? 4096 : 1024);
  return rows < 1 ? 1 : rows < 8 ? rows : 8;
}

// ------------------------------------------------------------- FGPA flux
// Waves that a skewer of k_fgpa_flux and k_fgpa_flux_jac gets (eight waves to a
// block).  Few skewers leave the card idle with one wave each, and a long one
// is a long chain on one wave; but eight waves share a barrier per skewer,
// which many skewers pay for.  One or two waves each also leave a part of the
// last round of blocks over the 256 CUs idle: the lower the share in use with
// the better of them, the sooner eight win.  Us with 1, 2 and 8 waves, one
// parameter set per skewer:
//             700 pixels        1400              3000             6500
//     600     7.8  7.5  7.5     9.7  7.5  7.6     18   12   9.9    35   24   16
//    1500     7.3  7.3  8.2     11.2 11.1 10.6    20.5 18.7 16.6   37   34   28
//    2000     7.8  7.7  9.9     12.6 11.6 13.0    22   20   20     40   37   38
//    3000     10.9 9.8  13.6    17.6 14.9 17.6    31   26   28     78   67   67
//    4000     11.9 12.3 17.4    18.6 18.3 22      34.5 34   36     94   101  89
//    5000     14.8 14.2 20.8    23.4 21.9 26.5    45   41   45     125  116  110
//   10000     23   23.5 38      38   38   52      103  103  114    224  227  215
//   20000     42   43   74      95   97   131     203  199  223    442  434  414
// and with parameters per pixel 6500 pixels take 59, 43, 34.5 (1500 skewers),
// 117, 106, 104 (3000) and 309, 329, 322 (10000).  Of eight waves against two,
// 2100 skewers (68% of the rounds in use) of 3000 pixels take 0.92 of the time,
// 2500 (81%) 0.98 and 2700 (88%) 1.02; of 4500 0.87, 0.93 and 0.98; 6300
// (77%) of 4500 0.93.
constexpr int64_t rounds_used(int64_t n, int64_t round) { return 100 * n / ((n + round - 1) / round * round); }

constexpr int flux_waves(int64_t n, int64_t pixels, bool per_pixel) {
  if (n <= 0) return 1;
  const int64_t mean = pixels / n;
  const int64_t one = rounds_used(n, 8 * 256), two = rounds_used(n, 4 * 256), used = one > two ? one : two;
  // eight
  if (mean >= (n <= 1200 || (n <= 1536 && per_pixel) ? 1400 : n <= 1536 ? 2000 : 6000) &&
      (n <= 4096 || one < 85 || !per_pixel))
    return 8;
  if (n <= 4096 && mean >= (used < 77 ? 2000 : used < 84 ? 3000 : used < 87 || (n > 3072 && used < 92) ? 4500 : 6000))
    return 8;
  if (n > 4096 && one < 82 && mean >= 4500) return 8;
  // two
  if (n <= 1024 || (n > 2048 && n <= 3072)) return mean >= 600 ? 2 : 1;
  if (n <= 2048) return mean >= (per_pixel ? 600 : 1400) ? 2 : 1;
  if (n <= 4096) return per_pixel && mean >= 1000 ? 2 : 1;
  return one < 85 && two > one + 5 && mean >= 1000 ? 2 : 1;
}

// ------------------------------------------- smoothing along radial lines
// Whether the smoothing over (2 dmax + 1)^3 cells of seven or more fields takes
// k_gather_radial (a tube of cells per run of pixels) or k_gather (a thread per
// pixel, each its own cells), for lines of `pixels` pixels in all and pixels
// `cells` cells apart.
//
// One cell per pixel (dmax 0) fits k_gather's L1.  A block of k_gather_radial
// does the skewers of its 256 or more pixels one after the other, each in 10 us
// or more however short it is.  With seven fields and 2e6 pixels in all dmax 1
// takes 488 us against 685 at 50 pixels per skewer and 1005 against 790 at 20;
// dmax 2 13.0 ms against 15.9 and dmax 3 21.5 against 44.1 at 2.  A batch that
// does not fill the card waits for the block with the most skewers; k_gather
// then takes as long as one pixel does, which its fields and cells decide.  Us,
// k_gather_radial against k_gather, 30000 pixels in skewers of
//                 5          20        45       100      300
//   dmax 1, 7                          58, 29   37, 24   23, 23
//           10                         61, 46   39, 39
//   dmax 2, 7     555, 267   160, 115  80, 83
//           10    587, 399
//   dmax 3, 7     887, 696
// (800000 pixels of dmax 1 in skewers of 45 218, 211; of dmax 2 in skewers of 5
// 2312, 1790).
//
// And with pixels cells apart a tube holds few of them: a
// million pixels along x or y, dmax 1, take 0.37 of k_gather's time at a half
// of a cell, 0.45 at one, 0.8 at two, 0.9 at two and a half, 1.1 at three, 1.4
// at four and 2.2 at eight (along z 0.9, 0.85, 0.85, 0.85, 0.8, 0.6, 0.8; dmax 2
// 0.8 at the most, dmax 3 0.45).
constexpr bool gather_radial(int dmax, int fields, int64_t n, int64_t pixels, double cells) {
  if (dmax < 1) return false;
  const bool fills = pixels >= 200000, ten = fields >= 10;
  const int64_t mean = dmax == 1   ? (fills ? (ten ? 40 : 60) : (ten ? 100 : 150))
                       : dmax == 2 ? (fills ? (ten ? 2 : 10) : (ten ? 10 : 30))
                                   : (fills ? 2 : (ten ? 4 : 8));
  if (pixels < mean * n) return false;
  return dmax > 1 || (cells <= 2.75 && cells >= -2.75);
}

// ------------------------------------------- the fit's transforms in pairs
// Points per thread of the pair kernels of 4096 points: with 16, two blocks fit
// a CU; with 8, one of twice the threads.
constexpr int fit_pair_points(int pairs) { return pairs > 256 ? 16 : 8; }

// -------------------------------------------------------------- box passes
// The variant (box_kernels.h) of a z pass that a plan starts with, for pencils
// of m complex points: ms against variant 0, R2C of 320 points 0.43 against 0.65
// and 384 1.94 against 2.18; C2R of 320 1.00 against 1.17, 384 8.7 against 8.9
// and 768 32.5 against 35.4; of 1280 the C2R takes us with variant 1 and 0
//   pencils   64^2      200^2     320^2     512^2       640^2
//             27  36    191  246  475  592  1190  1410  1850  2140
// and the R2C into [x][kz][y] with 1 and 0, with lines padded (p) and not
//   1p        32        242       755       2935        4920
//   0p        52        330       820       2190        3980
//   0         37        271       725       2640        4570
// (in the numpy layout, with the x and y passes, 1 and 0 not padded: 59 66,
// 708 762, 1280 1400, 3410 3700, 5385 5720).
constexpr int box_pencil(int m, bool c2r, int64_t pencils) {
  if (m == 1280) return c2r || pencils < 70000 ? 1 : 0;
  return c2r ? (m == 320 ? 1 : m == 384 || m == 768 ? 2 : 0) : (m == 320 || m == 384 ? 1 : 0);
}

// Whether an R2C of 1280 points pads its LDS lines: one that stores with the
// lanes along y reads one point of several lines, which unpadded lie in the same
// banks, but more of these fit a CU.
constexpr bool box_r2c_padded(int variant, bool trans, int64_t pencils) {
  return trans && (variant == 1 || pencils >= 200000);
}

// The variant of an x or y pass of n points that a plan starts with.  What
// decides is the lines per block that half of a CU's LDS holds (the transposed
// runs are 8 B per line) against the waves that the register tile leaves: the
// split exchange buys lines, the half tile waves.  Measured per pass, in ms
// against variant 0, at 320^3, 384^3, ... 1280 x 1280 x 512 and 2560 x 1280 x 768:
//   y, x forward   320 18 (0.051, 0.056)  384 18 (0.114, 0.128)
//                  512 17 (0.327, 0.362)  640 17 (0.482, 0.518)
//                  768 17 (0.750, 0.875)  1024 3 (1.17, 1.59)
//                  1280 6 (4.34, 4.68)    1536 3 (2.37, 3.04)
//                  2048 3 (3.48, 4.94)
//   y inverse      320 18 (0.147, 0.165)  384 18 (0.251, 0.273)
//                  640 6 (1.02, 1.11)     768 18 (1.81, 2.05)
//                  1024 3 (2.60, 2.81)    1280 6 (9.1, 10.4)
//                  1536 6 (5.41, 5.79)    2048 3 (7.9, 11.9)
//   x inverse      as forward; in the numpy layout 1280 17 (2.42, 2.55 the
//                  whole inverse), 2560 4 (4.86, 5.26)
//   x spectral     320 18 (0.153, 0.164)  384 17 (0.263, 0.288)
//                  512 16 (0.530, 0.634)  640 10 (1.12, 1.55)
//                  768 3 (1.85, 2.00)     1024 14 (2.57, 2.94)
//                  1280 12 (3.53, 4.57)   1536 3 (5.95, 7.18)
//                  2048 14 (5.68, 6.44)   2560 1 (13.2, 17.0)
//
// The split exchange pays for its barriers with longer runs, that is where the
// passes are bound by memory, not where the work box lies in the caches; and it
// leaves lanes idle where the inner extent is no multiple of its lines.  So each
// holds from a size of the work box on (MB of nx ny (nz / 2 + 1) complex
// numbers).  Us against variant 0 on both sides, boxes of n x a x c or a x n x c:
//   y forward, numpy layout  512 17: 160^2 (53 MB) 79, 75   250x300 219, 213   400^2 571, 592
//                            768 17: 160^2 (80) 108, 103    250x300 327, 315   400^2 805, 839
//                            1024 3: 128^2 (68) 89, 86      200^2 243, 242     250x300 549, 597
//                            2048 3: 64^2 (34) 62, 63       transposed 64^2 32, 27  200^2 183, 204
//   y inverse, transposed    768 18: 100^2 (31) 29, 22      250x300 127, 116   400^2 252, 249
//                            1024 3: 64^2 (17) 26, 20       256^2 (270) 178, 166  400^2 366, 366
//                            1536 6: 100^2 (63) 53, 42      200^2 155, 143     400^2 550, 583
//   x inverse, numpy layout  512 17: 160^2 (53) 125, 121    250x300 254, 260
//   x spectral               384 17: 100^2 (16) 45, 34      256^2 (101) 114, 112  400^2 264, 269
//                            768 3:  32^2 (3) 35, 32        128^2 (51) 73, 79
// With ny a multiple of 128 the points of an x line are a multiple of 1 KB apart,
// in few of the memory's channels, and longer runs pay sooner: x forward of 512
// and 768 x 256 x 256 143, 166 and 217, 257.
//
// Without an aux field the spectral pass has two line FFTs instead of three or
// four, and the variants that keep a second register tile for it lose: us of the
// pass with 16 or 14 against 0, 512^3 390, 342; 1024 x 512 x 512 939, 822; 2048 x
// 512 x 256 920, 856 (320, 384, 640, 768, 1280, 1536 and 2560 win without one too).
// Of the other lengths the general ones have variant 0 only; 4096 has others,
// which were not measured.
struct BoxDefault {
  int n, variant;
  int mb[2];   // from this size of the work box on: y, x forward; y, x inverse; both the same for the spectral pass
};

constexpr int box_strided(int kind, int nx, int ny, int nz, bool aux) {
  constexpr BoxDefault forward[] = {{320, 18, {45, 45}},  {384, 18, {95, 45}},  {512, 17, {250, 250}},
                                    {640, 17, {100, 60}}, {768, 17, {300, 300}}, {1024, 3, {250, 90}},
                                    {1280, 6, {0, 0}},    {1536, 3, {20, 20}},  {2048, 3, {160, 30}}};
  constexpr BoxDefault y_inverse[] = {{320, 18, {45, 45}}, {384, 18, {150, 150}}, {640, 6, {0, 0}},
                                      {768, 18, {450, 450}}, {1024, 3, {250, 250}}, {1280, 6, {0, 0}},
                                      {1536, 6, {460, 460}}, {2048, 3, {160, 160}}};
  constexpr BoxDefault x_inverse[] = {{320, 18, {45, 45}}, {384, 18, {60, 60}},  {512, 17, {150, 150}},
                                      {640, 17, {45, 45}}, {768, 17, {75, 75}},  {1024, 3, {90, 90}},
                                      {1280, 17, {80, 80}}, {1536, 3, {20, 20}}, {2048, 3, {60, 60}},
                                      {2560, 4, {30, 30}}};
  constexpr BoxDefault spectral[] = {{320, 18, {45, 45}}, {384, 17, {200, 200}}, {512, 16, {0, 0}}, {640, 10, {0, 0}},
                                     {768, 3, {30, 30}},  {1024, 14, {0, 0}},    {1280, 12, {0, 0}},
                                     {1536, 3, {20, 20}}, {2048, 14, {0, 0}},    {2560, 1, {0, 0}}};
  const bool x = kind == SMK_PASS_X_FWD || kind == SMK_PASS_X_INV;
  const int n = kind == SMK_PASS_Y_FWD || kind == SMK_PASS_Y_INV ? ny : nx;
  const bool aliased = x && (n == 512 || n == 768) && ny % 128 == 0;
  if (kind == SMK_PASS_X_SPECTRAL && !aux && (n == 512 || n == 1024 || n == 2048)) return 0;
  const BoxDefault* t = kind == SMK_PASS_Y_INV ? y_inverse : kind == SMK_PASS_X_INV ? x_inverse
                        : kind == SMK_PASS_X_SPECTRAL ? spectral : forward;
  const int len = kind == SMK_PASS_Y_INV ? 8 : kind == SMK_PASS_X_INV || kind == SMK_PASS_X_SPECTRAL ? 10 : 9;
  const double mb = 8e-6 * nx * ny * (nz / 2 + 1);
  for (int i = 0; i < len; ++i) {
    if (t[i].n != n) continue;
    const int from = t[i].mb[x ? 1 : 0];
    return mb >= (aliased && from > 100 ? 100 : from) ? t[i].variant : 0;
  }
  return 0;
}

}  // namespace smk_route
