// One application of the plane-wave operator to one vector by one workgroup,
// everything between the vector and the result in LDS.
//
// The batched kernels of operators.hip take every vector through four launches
// with the columns, the planes and the local result in memory between them:
// 20 us for a few vectors, whatever their size, and 0.14 us a vector for
// many (24^3, 6 Ha).  A sphere of a few hundred plane waves fits a CU: its columns T[z][j]
// (24 KB at 6 Ha on the 24^3 box), the rows P of the planes, the vector
// and the local result.  A block then needs barriers only, and as many
// vectors run side by side as there are CUs: 15.3 us for up to 256 vectors.
// Bound: the latency of the stages between the barriers.
//   A  columns along z, each over a lane pair; the projector overlaps on the
//      other waves
//   B  planes: y lines of the occupied rows, x lines with V(r)
//      between the two transforms (in place, a lane pair owns its column y),
//      y lines back
//   C  columns back along z into the plane waves
//   D  kinetic + local + projectors + sigma
#pragma once

#include "lanes.h"
#include "lines.h"
#include "pwdev.h"

namespace sgw {
namespace pwblock {

// threads of a block: 12 waves at 168 registers, every line over a lane pair.
// A stage costs the latency of one line's reads, transform and writes, some
// 4000 cycles whether it has one wave on a SIMD or two: whole lines on 8 waves
// take 17.5 us an application of the 24^3 cell (6 Ha) against 15.
constexpr int threads(int) { return 768; }
constexpr size_t kLds = 160 * 1024;

// LDS layout (double2 units)
struct Layout {
  int64_t x, loc, T, P, becp, info, rows, sidx, total;
};
__host__ __device__ inline int parts(int nt, int64_t ld) {
  return nt / ld >= 4 ? 4 : nt / ld >= 2 ? 2 : 1;
}
__host__ __device__ inline Layout layout(int n, int nc1, int ncs, int64_t ld, int nproj) {
  Layout l;
  l.x = 0;
  l.loc = ld;
  l.T = 2 * ld;
  l.P = l.T + (int64_t)n * ncs;
  const int64_t planes = (int64_t)n * nc1 * (n + 1);
  const int64_t sums = (parts(threads(n), ld) - 1) * ld;
  l.becp = l.P + (planes > sums ? planes : sums);
  l.info = l.becp + nproj;          // int4 per column
  l.rows = l.info + ncs;            // int4 (start, lo, cnt) per row
  l.sidx = l.rows + nc1;            // int per plane wave
  l.total = l.sidx + (ld + 3) / 4;
  return l;
}
// The operator's tables of group g into LDS (no barrier)
template <int N>
__device__ inline void load_tables(const PwDev &d, int g, double2 *s, const Layout &l) {
  constexpr int NT = threads(N);
  int4 *info = reinterpret_cast<int4 *>(s + l.info), *rows = reinterpret_cast<int4 *>(s + l.rows);
  int32_t *sidx = reinterpret_cast<int32_t *>(s + l.sidx);
  const int64_t r0 = (int64_t)g * d.nc1;
  for (int i = threadIdx.x; i < d.ncs; i += NT) info[i] = d.col_info[(int64_t)g * d.ncs + i];
  for (int i = threadIdx.x; i < d.nc1; i += NT)
    rows[i] = make_int4(d.row_start[r0 + g + i], d.row_lo[r0 + i], d.row_cnt[r0 + i], 0);
  for (int i = threadIdx.x; i < d.ld; i += NT) sidx[i] = d.sorted_idx[(int64_t)g * d.ld + i];
}

// out(e, value) for every e < ld: ((A_g + sigma) x)_e, zero past the group's
// plane waves.  x (d.ld values, zero padded) and the tables are in s and
// visible to the block; out is called by one thread per e.  The block is
// uniform here.
template <int N, typename Out>
__device__ inline void apply(const PwDev &d, int g, double2 sigma, double2 *s, const Layout &l,
                             Out out) {
  constexpr int NT = threads(N), W = NT / 64, E = lane_values(N), R = N + 1;
  static_assert(split_side(N), "sides divisible by four");
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const Line<N> ln{lane & 1};
  const int ncs = d.ncs, nc1 = d.nc1, M1 = d.M1;
  const int npw = d.npw[g];
  const int ncol = d.row_start[(int64_t)g * (nc1 + 1) + nc1];
  const double2 *x = s + l.x;
  double2 *loc = s + l.loc, *T = s + l.T, *P = s + l.P, *becp = s + l.becp;
  const int4 *info = reinterpret_cast<const int4 *>(s + l.info);
  const int4 *rows = reinterpret_cast<const int4 *>(s + l.rows);
  const int32_t *sidx = reinterpret_cast<const int32_t *>(s + l.sidx);
  const double2 *pg = d.proj + (int64_t)g * d.nproj * d.ld;
  auto freq = [](int i) { return i < N / 2 ? i : i - N; };

  // A
  const int zw = (ncol + 31) / 32;
  for (int t = wv; t < zw + d.nproj; t += W) {
    if (t < zw) {
      const int j = t * 32 + (lane >> 1);
      if (j < ncol) {
        const int4 ci = info[j];
        double2 b[E];
#pragma unroll
        for (int i = 0; i < E; ++i) {
          const int k = freq(ln.dec(i)) - ci.w;
          b[i] = keep(x[sidx[ci.z + within(k, ci.y)]], k, ci.y);
        }
        ln.template dit<+1>(b);
#pragma unroll
        for (int i = 0; i < E; ++i) T[ln.nat(i) * ncs + j] = b[i];
      }
    } else {
      const int p = t - zw;
      const double2 *pp = pg + (int64_t)p * d.ld;
      double2 acc = mk(0.0, 0.0);
#pragma unroll 4
      for (int i = lane; i < npw; i += 64) cmacc(acc, pp[i], x[i]);
      acc = mk(lanes::sum<64>(acc.x), lanes::sum<64>(acc.y));
      const double dc = d.dcoef[(int64_t)g * d.nproj + p];
      if (lane == 0) becp[p] = mk(dc * acc.x, dc * acc.y);
    }
  }
  __syncthreads();
  // B
  for (int t = tid >> 1; t < N * nc1; t += NT / 2) {
    const int zi = t / nc1, a = t - zi * nc1;
    const int4 ra = rows[a];
    const double2 *row = T + zi * ncs + ra.x;
    const int lo = ra.y, cnt = ra.z;
    double2 b[E];
#pragma unroll
    for (int i = 0; i < E; ++i) {
      const int k = freq(ln.dec(i)) - lo;
      b[i] = keep(row[within(k, cnt)], k, cnt);
    }
    ln.template dit<+1>(b);
    double2 *p = P + t * R;
#pragma unroll
    for (int i = 0; i < E; ++i) p[ln.nat(i)] = b[i];
  }
  __syncthreads();
  for (int t = tid >> 1; t < N * N; t += NT / 2) {
    const int zi = t / N, y = t - zi * N;
    double2 *p = P + zi * nc1 * R + y;
    // V(r) of the line, on its way during the first transform
    const double *v = d.vloc_zxy + zi * N * N + y;
    double2 b[E];
    double vv[E];
#pragma unroll
    for (int i = 0; i < E; ++i) vv[i] = v[ln.nat(i) * N];
#pragma unroll
    for (int i = 0; i < E; ++i) {
      const int a = freq(ln.dec(i)) + M1;
      b[i] = keep(p[within(a, nc1) * R], a, nc1);
    }
    ln.template dit<+1>(b);
#pragma unroll
    for (int i = 0; i < E; ++i) b[i] = mk(b[i].x * vv[i], b[i].y * vv[i]);
    ln.template dif<-1>(b);
#pragma unroll
    for (int i = 0; i < E; ++i) {
      const int a = freq(ln.dec(i)) + M1;
      if (a >= 0 && a < nc1) p[a * R] = b[i];
    }
  }
  __syncthreads();
  for (int t = tid >> 1; t < N * nc1; t += NT / 2) {
    const int zi = t / nc1, a = t - zi * nc1;
    const int4 ra = rows[a];
    double2 *row = T + zi * ncs + ra.x;
    const int lo = ra.y, cnt = ra.z;
    const double2 *p = P + t * R;
    double2 b[E];
#pragma unroll
    for (int i = 0; i < E; ++i) b[i] = p[ln.nat(i)];
    ln.template dif<-1>(b);
#pragma unroll
    for (int i = 0; i < E; ++i) {
      const int k = freq(ln.dec(i)) - lo;
      if (k >= 0 && k < cnt) row[k] = b[i];
    }
  }
  __syncthreads();
  // C
  for (int j = tid >> 1; j < ncol; j += NT / 2) {
    const int4 ci = info[j];
    double2 b[E];
#pragma unroll
    for (int i = 0; i < E; ++i) b[i] = T[ln.nat(i) * ncs + j];
    ln.template dif<-1>(b);
#pragma unroll
    for (int i = 0; i < E; ++i) {
      const int k = freq(ln.dec(i)) - ci.w;
      if (k >= 0 && k < ci.y)
        loc[sidx[ci.z + k]] = mk(b[i].x * d.inv_nbox, b[i].y * d.inv_nbox);
    }
  }
  // D: the projectors of a plane wave over `parts` threads
  const int ld = (int)d.ld, np = parts(NT, ld);
  const int part = tid / ld, e0 = tid - part * ld;
  auto projectors = [&](int e, int first) {
    double2 acc = mk(0.0, 0.0);
#pragma unroll 4
    for (int p = first; p < d.nproj; p += np) cmac(acc, pg[(int64_t)p * ld + e], becp[p]);
    return acc;
  };
  double2 mine = mk(0.0, 0.0);
  if (np > 1) {
    if (part < np && e0 < npw) mine = projectors(e0, part);
    if (part > 0 && part < np && e0 < npw) P[(part - 1) * ld + e0] = mine;
  }
  __syncthreads();
  for (int e = np > 1 ? (part == 0 ? e0 : ld) : tid; e < ld; e += np > 1 ? ld : NT) {
    if (e >= npw) {
      out(e, mk(0.0, 0.0));
      continue;
    }
    const double kin = d.kin[(int64_t)g * ld + e];
    const double2 xe = x[e], le = loc[e];
    double2 acc = mk(fma(kin, xe.x, le.x), fma(kin, xe.y, le.y));
    if (np > 1) {
      acc = cadd(acc, mine);
      for (int q = 1; q < np; ++q) acc = cadd(acc, P[(q - 1) * ld + e]);
    } else {
      acc = cadd(acc, projectors(e, 0));
    }
    cmac(acc, sigma, xe);
    out(e, acc);
  }
}

}  // namespace pwblock
}  // namespace sgw
