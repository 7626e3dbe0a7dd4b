// Which kernel a call takes, where that depends on its sizes only: plain
// functions of the host, each with the measurements that placed its lines.
#pragma once
#include <cstdint>

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

}  // namespace smk_route
