// Box FFTs between a G list and real space, one box per workgroup.
//
// A two-point function's transforms (fft6.f90) and the product of sigma_prod
// (phys/corr/src/sigma.f90:417-523) take every column r' (or row G) of a
// matrix through a 3-D FFT whose reciprocal side is a sphere of G vectors.
// As separate box passes each of them reads and writes the whole matrix (3 GB
// on the 24^3 grid), and the product took five such passes.  Here the box
// never leaves the CU: the sphere's occupied columns T[z][column] sit in LDS
// (73 KB of the box's 221 KB on the 24^3 grid with 1500 G), are transformed
// along z in place, and every wave then takes a few planes at a time through
//   x lines of the occupied y rows -> y lines -> (times g) -> y -> x
// in registers, exchanging the lines through its own LDS buffer, and puts the
// plane's columns back where they came from.  The only full-size traffic is
// the real-space operand itself, read or written once along x.
#include "spherefft.h"

#include <algorithm>
#include <cstring>

#include "ktimer.h"
#include "lines.h"

namespace sgw {
namespace {

enum { kInv = 0, kFwd = 1, kProd = 2 };
constexpr int kLdsMax = 160 * 1024;
constexpr int kPre = 2;  // list values a thread fetches ahead for its next box

constexpr int planes_per_wave(int n) { return (split_side(n) ? 32 : 64) / n; }
// dwords the index bytes of a lane's values take
constexpr int map_dwords(int n) { return (lane_values(n) + 3) / 4; }
// bytes of an index table of one line: both lanes of a pair, or one lane
constexpr int map_bytes(int n) { return 4 * map_dwords(n) * (split_side(n) ? 2 : 1); }
constexpr int kMaxCol = 255;  // column and row numbers and the empty mark are bytes

// Waves per block.  Measured on 24^3 with 1500 G (175 columns, 17 rows), one
// product of 13824 boxes: whole lines on 6 waves 1440 us, on 8 waves 2090 us
// (the twelve plane groups leave half a round idle), on 12 waves 2026 us (168
// registers, 90 of them spilled); lines over lane pairs on 12 waves 1327 us.
// Sides 18 and 27 have no lane-pair form: 18 takes blocks of two waves, four
// to a CU by registers, 27 four waves with the whole register file.
constexpr int waves_of(int n) { return n == 16 ? 4 : n == 18 ? 2 : n == 24 ? 12 : 4; }
// waves a SIMD holds at the kernels' register use
constexpr int waves_per_simd(int n) { return split_side(n) ? 3 : n == 18 ? 2 : 1; }

struct Args {
  int64_t nvec;
  int num_g, ncol, nrow;
  const int32_t *ent;    // [num_g] z * (ncol + 1) + column
  const uint32_t *map;   // [nrow] index tables of columns (ncol: empty), one of rows (nrow: empty)
  const double2 *in;
  int64_t in_sg;
  double in_scale;
  double2 *real;
  const double2 *g;
  SphereOut o;
};

// LDS bytes: T, the index tables and the waves' exchange buffers (each plane
// with one more row that stays zero)
size_t lds_bytes(int n, int ncol, int nrow) {
  size_t b = sizeof(double2) * (size_t)n * (ncol + 1);
  b += ((size_t)(nrow + 1) * map_bytes(n) + 15) / 16 * 16;
  return b + sizeof(double) * (size_t)(n + 1) * waves_of(n) * planes_per_wave(n) * (nrow + 1);
}
int blocks_per_cu(int n, size_t lds) {
  const size_t grain = 1280;  // LDS is handed out in pieces of this size
  return std::max(1, std::min((int)(kLdsMax / ((lds + grain - 1) / grain * grain)),
                              4 * waves_per_simd(n) / waves_of(n)));
}

__device__ inline unsigned map_byte(const uint32_t *m, int i) {
  return (m[i / 4] >> (8 * (i & 3))) & 0xffu;
}

// end of a stage of a wave's plane: its LDS accesses stay on their side, and
// the instruction scheduler does not move the next stage's loads up into the
// registers of this one
__device__ inline void stage() {
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_sched_barrier(0);
}

template <int N, int SIGN>
__device__ inline void z_lines(double2 *T, int ncol, int ncs, int tid, int nt) {
  constexpr int E = lane_values(N), L = split_side(N) ? 2 : 1;
  const Line<N> ln{tid & (L - 1)};
  for (int c = tid / L; c < ncol; c += nt / L) {
    double2 x[E];
#pragma unroll
    for (int i = 0; i < E; ++i) x[i] = T[ln.dec(i) * ncs + c];
    ln.template dit<SIGN>(x);
#pragma unroll
    for (int i = 0; i < E; ++i) T[ln.nat(i) * ncs + c] = x[i];
  }
}

// Bound: on 24^3 with 1500 G the product issues vector instructions in 57 % of
// its 1327 us (counters: LDS 39 %, HBM 3.7 GB at 2.8 TB/s, which is the
// operand once and the list values once); the five passes it replaces took
// 3.7 ms plus the zero fill.  The exchange moves real and imaginary parts in
// turn, which halves its buffer.  Blocks are persistent: a block's next list
// values are in flight while it transforms, and the plane's G (or, forward,
// the next plane) is loaded before the transforms that precede its use: 1327
// us against 1523 with the loads right before the product.  Holding the next
// plane's G through the whole plane spills (2437 us).
template <int N, int SIGN, int MODE>
__global__ __launch_bounds__(64 * waves_of(N), waves_per_simd(N)) void k_sphere(Args a) {
  constexpr int PL = planes_per_wave(N), W = waves_of(N), NT = 64 * W, R = N + 1;
  constexpr int E = lane_values(N), D = map_dwords(N), MB = map_bytes(N) / 4;
  constexpr int L = split_side(N) ? 2 : 1;
  extern __shared__ __align__(16) unsigned char lds_raw[];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int ncol = a.ncol, ncs = ncol + 1, nrow = a.nrow;
  double2 *T = reinterpret_cast<double2 *>(lds_raw);
  uint32_t *map = reinterpret_cast<uint32_t *>(T + N * ncs);
  double *P = reinterpret_cast<double *>(map + ((nrow + 1) * MB + 3) / 4 * 4) +
              wv * PL * (nrow + 1) * R;
  for (int i = tid; i < (nrow + 1) * MB; i += NT) map[i] = a.map[i];
  for (int i = lane; i < PL * (nrow + 1) * R; i += 64) P[i] = 0.0;

  // lane roles: x line of (plane p1, occupied row q1); y line of (plane p2, x)
  const Line<N> ln{lane & (L - 1)};
  const int ln0 = lane / L;
  const int p1 = ln0 / nrow, q1 = ln0 - p1 * nrow;
  const int p2 = ln0 / N, x2 = ln0 - p2 * N;

  // XCD k (blocks k, k + 8, ...) takes a contiguous run of boxes, so that the
  // 16-byte list values of neighbouring boxes meet in one L2 line
  const int64_t per = (a.nvec + 7) / 8;
  const int64_t first = (int64_t)(blockIdx.x & 7) * per;
  const int64_t last = first + per < a.nvec ? first + per : a.nvec;
  const int64_t step = gridDim.x >> 3;
  int64_t b = first + (blockIdx.x >> 3);
  double2 pre[kPre];
  auto fetch = [&](int64_t bb) {
#pragma unroll
    for (int k = 0; k < kPre; ++k) {
      const int e = tid + k * NT;
      pre[k] = (bb < last && e < a.num_g) ? a.in[(int64_t)e * a.in_sg + bb] : mk(0.0, 0.0);
    }
  };
  if constexpr (MODE != kFwd) fetch(b);
  // the real-space operand of this lane's y line, one plane ahead
  const double2 *src = MODE == kFwd ? a.real : a.g;
  double2 real[E];
  auto fetch_real = [&](int64_t bb, int pl) {
    if (bb >= last || pl >= N) return;
    const int c = p2 < PL && pl + p2 < N ? p2 : 0;
    const int64_t at = bb * (N * N * N) + (int64_t)(pl + c) * (N * N) + x2;
#pragma unroll
    for (int i = 0; i < E; ++i) real[i] = src[at + ln.nat(i) * N];
  };
  if constexpr (MODE == kFwd) fetch_real(b, wv * PL);
  for (; b < last; b += step) {
    __syncthreads();
    if constexpr (MODE != kFwd) {
      for (int i = tid; i < N * ncs; i += NT) T[i] = mk(0.0, 0.0);
      __syncthreads();
#pragma unroll
      for (int k = 0; k < kPre; ++k) {
        const int e = tid + k * NT;
        if (e < a.num_g) T[a.ent[e]] = mk(a.in_scale * pre[k].x, a.in_scale * pre[k].y);
      }
      for (int e = tid + kPre * NT; e < a.num_g; e += NT) {
        const double2 v = a.in[(int64_t)e * a.in_sg + b];
        T[a.ent[e]] = mk(a.in_scale * v.x, a.in_scale * v.y);
      }
      __syncthreads();
      fetch(b + step);
      z_lines<N, SIGN>(T, ncol, ncs, tid, NT);
      __syncthreads();
    }
    for (int pl = wv * PL; pl < N; pl += W * PL) {
      // lanes without a line repeat line 0 and only their stores are masked:
      // with whole stages in branches both sides' lines would stay live
      const bool on1 = p1 < PL && pl + p1 < N, on2 = p2 < PL && pl + p2 < N;
      const int c1 = on1 ? p1 : 0, r1 = on1 ? q1 : 0, c2 = on2 ? p2 : 0;
      double2 *Tz = T + (pl + c1) * ncs;
      const uint32_t *xmap = map + r1 * MB + ln.odd * D, *ymap = map + nrow * MB + ln.odd * D;
      double *l1 = P + (c1 * (nrow + 1) + r1) * R;       // this lane's x line
      double *l2 = P + c2 * (nrow + 1) * R + x2;         // this lane's y line
      double2 x[E];
      double re[E];
      uint32_t mp[D];
      if constexpr (MODE == kProd) fetch_real(b, pl);
      if constexpr (MODE != kFwd) {
#pragma unroll
        for (int i = 0; i < D; ++i) mp[i] = xmap[i];
#pragma unroll
        for (int i = 0; i < E; ++i) x[i] = Tz[map_byte(mp, i)];
        stage();
        ln.template dit<SIGN>(x);
        stage();
        // x lines to y lines, real parts then imaginary parts
        if (on1) {
#pragma unroll
          for (int i = 0; i < E; ++i) l1[ln.nat(i)] = x[i].x;
        }
        stage();
#pragma unroll
        for (int i = 0; i < D; ++i) mp[i] = ymap[i];
#pragma unroll
        for (int i = 0; i < E; ++i) re[i] = l2[map_byte(mp, i) * R];
        stage();
        if (on1) {
#pragma unroll
          for (int i = 0; i < E; ++i) l1[ln.nat(i)] = x[i].y;
        }
        stage();
#pragma unroll
        for (int i = 0; i < E; ++i) x[i] = mk(re[i], l2[map_byte(mp, i) * R]);
        stage();
        ln.template dit<SIGN>(x);
        stage();
      }
      if constexpr (MODE == kInv) {
        const int64_t at = b * (N * N * N) + (int64_t)(pl + c2) * (N * N) + x2;
        if (on2) {
#pragma unroll
          for (int i = 0; i < E; ++i) a.real[at + ln.nat(i) * N] = x[i];
        }
      } else {
#pragma unroll
        for (int i = 0; i < E; ++i) x[i] = MODE == kFwd ? real[i] : cmul(x[i], real[i]);
        stage();
        if constexpr (MODE == kFwd) {  // the wave's next plane, of this box or of the block's next
          const bool more = pl + W * PL < N;
          fetch_real(more ? b : b + step, more ? pl + W * PL : wv * PL);
        }
      }
      if constexpr (MODE != kInv) {
        constexpr int BACK = MODE == kProd ? -SIGN : SIGN;
        stage();
        ln.template dif<BACK>(x);
        stage();
#pragma unroll
        for (int i = 0; i < D; ++i) mp[i] = ymap[i];
        if (on2) {
#pragma unroll
          for (int i = 0; i < E; ++i)
            if (map_byte(mp, i) < (unsigned)nrow) l2[map_byte(mp, i) * R] = x[i].x;
        }
        stage();
#pragma unroll
        for (int i = 0; i < E; ++i) re[i] = l1[ln.nat(i)];
        stage();
        if (on2) {
#pragma unroll
          for (int i = 0; i < E; ++i)
            if (map_byte(mp, i) < (unsigned)nrow) l2[map_byte(mp, i) * R] = x[i].y;
        }
        stage();
#pragma unroll
        for (int i = 0; i < E; ++i) x[i] = mk(re[i], l1[ln.nat(i)]);
        stage();
        ln.template dif<BACK>(x);
        stage();
#pragma unroll
        for (int i = 0; i < D; ++i) mp[i] = xmap[i];
#pragma unroll
        for (int i = 0; i < E; ++i)
          if (on1 && map_byte(mp, i) < (unsigned)ncol) Tz[map_byte(mp, i)] = x[i];
        stage();
      }
    }
    if constexpr (MODE != kInv) {
      constexpr int BACK = MODE == kProd ? -SIGN : SIGN;
      __syncthreads();
      z_lines<N, BACK>(T, ncol, ncs, tid, NT);
      __syncthreads();
      for (int e = tid; e < a.num_g; e += NT) {
        const double2 t = T[a.ent[e]];
        double2 v = mk(a.o.scale * t.x, a.o.scale * t.y);
        if (a.o.has_alpha) v = cmul(a.o.alpha, v);
        if (a.o.out) a.o.out[(int64_t)e * a.o.out_sg + b] = v;
        if (a.o.sum) {
          double2 *s = a.o.sum + (int64_t)e * a.o.sum_sg + b;
          *s = cadd(*s, v);
        }
      }
    }
  }
}

template <int N, int SIGN, int MODE>
void launch_n(hipStream_t st, const SphereList &l, const Args &a) {
  auto *kern = k_sphere<N, SIGN, MODE>;
  if (l.lds() > 64 * 1024)
    SGW_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(kern),
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)l.lds()));
  const int64_t want = (a.nvec + 7) / 8 * 8;
  const unsigned grid =
      (unsigned)std::min<int64_t>(want, 256 * (int64_t)blocks_per_cu(N, l.lds()));
  kern<<<grid, 64 * waves_of(N), l.lds(), st>>>(a);
  SGW_HIP(hipGetLastError());
}

template <int MODE> void launch(hipStream_t st, const SphereList &l, int sign, const Args &a) {
  if (a.nvec <= 0) return;
  auto go = [&](auto side) {
    constexpr int N = decltype(side)::value;
    if (sign > 0) launch_n<N, 1, MODE>(st, l, a);
    else launch_n<N, -1, MODE>(st, l, a);
  };
  switch (l.n()) {
    case 16: go(std::integral_constant<int, 16>{}); break;
    case 18: go(std::integral_constant<int, 18>{}); break;
    case 24: go(std::integral_constant<int, 24>{}); break;
    case 27: go(std::integral_constant<int, 27>{}); break;
    default: throw Error{SGW_E_SHAPE, "sphere FFT: unsupported side"};
  }
}

Args args_of(const SphereList &l, int64_t nvec) {
  Args a{};
  a.nvec = nvec;
  a.num_g = l.num_g();
  a.ncol = l.ncol();
  a.nrow = l.nrow();
  a.ent = l.d_ent();
  a.map = l.d_map();
  return a;
}

}  // namespace

SphereList::SphereList(int n, const std::vector<int32_t> &nl) : n_(n), num_g_((int)nl.size()) {
  if (n != 16 && n != 18 && n != 24 && n != 27) return;
  const int n2 = n * n;
  std::vector<int> col(n2, -1), row(n, -1);
  for (int32_t p : nl) {
    col[p % n2] = 0;
    row[p % n2 / n] = 0;
  }
  for (int y = 0; y < n; ++y)
    if (row[y] == 0) row[y] = nrow_++;
  for (int c = 0; c < n2; ++c)
    if (col[c] == 0) col[c] = ncol_++;
  if (ncol_ > kMaxCol) return;
  lds_ = lds_bytes(n, ncol_, nrow_);
  fits_ = lds_ <= (size_t)kLdsMax;
  if (!fits_) return;
  h_.assign(num_g_ + (size_t)(nrow_ + 1) * map_bytes(n) / 4, 0);
  for (int g = 0; g < num_g_; ++g) h_[g] = nl[g] / n2 * (ncol_ + 1) + col[nl[g] % n2];
  // index tables: the points of one lane of a pair, then the other's
  auto put = [&](int table, int point, int value) {
    const int at = split_side(n) ? 4 * map_dwords(n) * (point & 1) + point / 2 : point;
    reinterpret_cast<uint8_t *>(h_.data() + num_g_)[table * map_bytes(n) + at] = (uint8_t)value;
  };
  for (int y = 0; y < n; ++y) {
    put(nrow_, y, row[y] >= 0 ? row[y] : nrow_);
    if (row[y] >= 0)
      for (int x = 0; x < n; ++x)
        put(row[y], x, col[y * n + x] >= 0 ? col[y * n + x] : ncol_);
  }
}

void SphereList::upload(hipStream_t st) {
  if (!fits()) return;
  d_.alloc(h_.size());
  d_.upload(h_.data(), h_.size(), st);
}

void sphere_inv(hipStream_t st, const SphereList &l, int64_t nvec, int sign, const double2 *in,
                int64_t in_sg, double in_scale, double2 *real) {
  Args a = args_of(l, nvec);
  a.in = in;
  a.in_sg = in_sg;
  a.in_scale = in_scale;
  a.real = real;
  launch<kInv>(st, l, sign, a);
}

void sphere_fwd(hipStream_t st, const SphereList &l, int64_t nvec, int sign, const double2 *real,
                const SphereOut &o) {
  Args a = args_of(l, nvec);
  a.real = const_cast<double2 *>(real);
  a.o = o;
  launch<kFwd>(st, l, sign, a);
}

void sphere_prod(hipStream_t st, const SphereList &l, int64_t nvec, int sign, const double2 *in,
                 int64_t in_sg, const double2 *g, const SphereOut &o) {
  Args a = args_of(l, nvec);
  a.in = in;
  a.in_sg = in_sg;
  a.in_scale = 1.0;
  a.g = g;
  a.o = o;
  launch<kProd>(st, l, sign, a);
}

}  // namespace sgw
