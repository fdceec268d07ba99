// The plane-wave operator's tables as its kernels see them.
#pragma once

#include "sgw_internal.h"

namespace sgw {

struct PwDev {
  int n1, n2, n3;
  int M1, M2;           // column grid half widths; nc1 = 2M1+1, nc2 = 2M2+1
  int nc1, nc2, nslot;
  int64_t ld;
  int nproj;
  const double *vloc;          // [n3][n2][n1]
  const double *vloc_zxy;      // [n3][n1][n2]: lanes of the x stage (one per y) read rows
  const int32_t *npw;          // [ngroup]
  const int32_t *col_start;    // [ngroup][nslot]
  const int32_t *col_cnt;      // [ngroup][nslot]
  const int32_t *sorted_idx;   // [ngroup][ld]
  const int32_t *sorted_m3;    // [ngroup][ld] (reduced mod n3)
  const int32_t *slot_of;      // [ngroup][ld]
  const int32_t *m3_of;        // [ngroup][ld] (reduced mod n3)
  const int32_t *col_lo;       // [ngroup][nslot] smallest m3 of the column
  // column layout of the split z / plane transforms' T and S: ncs columns per
  // plane; packed column j of group g is grid slot col_info[g][j].x (-1:
  // none), with that column's count, start and lowest m3 in .y, .z, .w;
  // row a of the grid holds columns m2 = row_lo .. row_lo + row_cnt - 1 at
  // j = row_start[g][a] + m2 - row_lo (row_start[g][nc1]: the group's count)
  int ncs;
  const int4 *col_info;        // [ngroup][ncs]: (slot, col_cnt, col_start, col_lo)
  const int32_t *row_start;    // [ngroup][nc1 + 1]
  const int32_t *row_lo;       // [ngroup][nc1]
  const int32_t *row_cnt;      // [ngroup][nc1]
  const double *kin;           // [ngroup][ld]
  const double2 *proj;         // [ngroup][nproj][ld]
  const double *dcoef;         // [ngroup][nproj]
  const double2 *tw1, *tw2, *tw3;  // e^{+2 pi i k/n}
  double inv_nbox;
};

}  // namespace sgw
