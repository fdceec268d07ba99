// Linear operators applied by the solvers: (A + sigma) x for batches of vectors.
//
//  * DenseOperator    A given as a dense column-major matrix (the reference's
//                     unit-test operator, algo/linear_solver/test/linear_solver.pf:100-113)
//  * CallbackOperator the reference's procedure argument AA(sigma, xx, Ax)
//                     (algo/linear_solver/src/select_solver.f90:77-87); runs
//                     on the host, vectors cross PCIe per call
//  * PwOperator       the plane-wave Hamiltonian of linear_op
//                     (algo/linear_solver/src/linear_op.f90:46-206):
//                     (|k+q+G|^2 + V_loc + sum_p |p> D_p <p| + sigma) x,
//                     where the projector list holds the nonlocal beta's and,
//                     with D = alpha_pv, the valence states of P_v.
#include "operators.h"
#include "ktimer.h"
#include "pwblock.h"
#include "pwdev.h"
#include "regfft.h"
#include "splitfft.h"
#include "tune.h"

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <type_traits>

// The fixed work area of PwOperator::apply_noalloc: one copy per device,
// held until the process ends.  Host code never uses this name as an address
// (on the host it is only a stand-in for the symbol); it takes the device
// address from hipGetSymbolAddress once per device (noalloc_scratch below).
static __device__ __align__(256) unsigned char scratch[SGW_NOALLOC_SCRATCH_BYTES];

namespace sgw {

namespace {

constexpr int kBlock = 256;

// ---------------------------------------------------------------------------
// dense
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kBlock) void k_dense(int64_t n, const double2 *__restrict__ a,
                                                  const double2 *__restrict__ in, int64_t sin,
                                                  double2 *__restrict__ out, int64_t sout,
                                                  int64_t ld, const double2 *__restrict__ sigma,
                                                  const int32_t *__restrict__ active) {
  const int v = blockIdx.y;
  if (active && !active[v]) return;
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i >= ld) return;
  const double2 *x = in + v * sin;
  double2 acc = mk(0, 0);
  if (i < n) {
    for (int64_t j = 0; j < n; ++j) cmac(acc, a[i + j * n], x[j]);
    cmac(acc, sigma[v], x[i]);
  }
  out[v * sout + i] = acc;
}

// ---------------------------------------------------------------------------
// plane waves
// ---------------------------------------------------------------------------
// One block per (plane z, vector v): pencil DFTs of one z-plane.
// Output S[v][slot][z]: the plane's contribution to sum_z (...) before the
// final z-transform.
__global__ __launch_bounds__(kBlock) void k_pw_plane(PwDev d, const double2 *__restrict__ in,
                                                     int64_t sin, const int32_t *__restrict__ group,
                                                     const int32_t *__restrict__ active,
                                                     double2 *__restrict__ S) {
  extern __shared__ double2 smem[];
  const int z = blockIdx.x, v = blockIdx.y;
  if (active && !active[v]) return;
  const int g = group ? group[v] : 0;
  const int n1 = d.n1, n2 = d.n2, n3 = d.n3, nc1 = d.nc1, nc2 = d.nc2, nslot = d.nslot;
  double2 *w1 = smem;                 // n1
  double2 *w2 = w1 + n1;              // n2
  double2 *pin = w2 + n2;             // nslot   (m1, m2)
  double2 *A = pin + nslot;           // nc1 * n2 (m1, y)
  double2 *B = A + nc1 * n2;          // n2 * n1  (y, x)
  for (int i = threadIdx.x; i < n1; i += kBlock) w1[i] = d.tw1[i];
  for (int i = threadIdx.x; i < n2; i += kBlock) w2[i] = d.tw2[i];
  const double2 *x = in + v * sin;
  const int32_t *cs = d.col_start + (int64_t)g * nslot, *cc = d.col_cnt + (int64_t)g * nslot;
  const int32_t *sidx = d.sorted_idx + (int64_t)g * d.ld, *sm3 = d.sorted_m3 + (int64_t)g * d.ld;
  // z inverse transform of each column at this z
  for (int c = threadIdx.x; c < nslot; c += kBlock) {
    double2 acc = mk(0, 0);
    const int st = cs[c], cnt = cc[c];
    for (int j = st; j < st + cnt; ++j) {
      int e = (sm3[j] * z) % n3;
      cmac(acc, x[sidx[j]], d.tw3[e]);
    }
    pin[c] = acc;
  }
  __syncthreads();
  // y inverse: A[m1][y] = sum_m2 pin[m1][m2] e^{+i 2pi m2 y/n2}
  for (int idx = threadIdx.x; idx < nc1 * n2; idx += kBlock) {
    const int a = idx / n2, y = idx % n2;
    double2 acc = mk(0, 0);
    for (int b = 0; b < nc2; ++b) {
      int m2 = b - d.M2;
      int e = ((m2 * y) % n2 + n2) % n2;
      cmac(acc, pin[a * nc2 + b], w2[e]);
    }
    A[idx] = acc;
  }
  __syncthreads();
  // x inverse and local potential: B[y][x] = V(x,y,z) sum_m1 A[m1][y] e^{+i 2pi m1 x/n1}
  const double *vz = d.vloc + (int64_t)z * n1 * n2;
  for (int idx = threadIdx.x; idx < n2 * n1; idx += kBlock) {
    const int y = idx / n1, xx = idx % n1;
    double2 acc = mk(0, 0);
    for (int a = 0; a < nc1; ++a) {
      int m1 = a - d.M1;
      int e = ((m1 * xx) % n1 + n1) % n1;
      cmac(acc, A[a * n2 + y], w1[e]);
    }
    const double vv = vz[idx];
    B[idx] = mk(acc.x * vv, acc.y * vv);
  }
  __syncthreads();
  // x forward: A[m1][y] = sum_x B[y][x] e^{-i 2pi m1 x/n1}
  for (int idx = threadIdx.x; idx < nc1 * n2; idx += kBlock) {
    const int a = idx / n2, y = idx % n2;
    const int m1 = a - d.M1;
    double2 acc = mk(0, 0);
    for (int xx = 0; xx < n1; ++xx) {
      int e = ((m1 * xx) % n1 + n1) % n1;
      cmac(acc, B[y * n1 + xx], cconj(w1[e]));
    }
    A[idx] = acc;
  }
  __syncthreads();
  // y forward into the sphere columns
  double2 *Sv = S + (int64_t)v * nslot * n3;
  for (int c = threadIdx.x; c < nslot; c += kBlock) {
    if (cc[c] == 0) continue;
    const int a = c / nc2, b = c % nc2;
    const int m2 = b - d.M2;
    double2 acc = mk(0, 0);
    for (int y = 0; y < n2; ++y) {
      int e = ((m2 * y) % n2 + n2) % n2;
      cmac(acc, A[a * n2 + y], cconj(w2[e]));
    }
    Sv[(int64_t)c * n3 + z] = acc;
  }
}

// The local-potential FFT pipeline runs in the element type C: double2, or
// float2 for vectors whose solve has been relaxed to FP32 (input and output
// stay FP64).  With a flag array, a kernel instance handles the vectors whose
// flag relax[v] equals `want`; without one, every vector.  The FP32 scratch
// of vector v sits in the first half of its FP64 slot.
template <typename C> __device__ inline C to_c(double2 v);
template <> __device__ inline double2 to_c<double2>(double2 v) { return v; }
template <> __device__ inline float2 to_c<float2>(double2 v) {
  return make_float2((float)v.x, (float)v.y);
}
template <typename C> __device__ inline C czero() { return CplxT<C>::make(0, 0); }
template <typename C> constexpr int kSlotScale = (int)(sizeof(double2) / sizeof(C));

__device__ inline bool precision_skip(const int32_t *__restrict__ relax, int want, int v) {
  return relax != nullptr && relax[v] != want;
}
// RL false: a kernel instance that never reads relax flags, so it compiles to
// the same code (and rounds the same) as one without them
template <bool RL>
__device__ inline bool precision_skip(const int32_t *__restrict__ relax, int want, int v) {
  return RL && precision_skip(relax, want, v);
}

// dst[c] = src[c], c < n, by one wavefront: 16 loads per lane are issued
// before the first LDS store, so a plane of up to 1024 column values costs
// one memory latency instead of one per 64 values.
template <typename C>
__device__ inline void stage_plane(const C *__restrict__ src, C *dst, int n) {
  constexpr int kB = 16;
  const int lane = threadIdx.x & 63;
  for (int c0 = 0; c0 < n; c0 += 64 * kB) {
    C t[kB];
#pragma unroll
    for (int b = 0; b < kB; ++b) {
      const int c = c0 + b * 64 + lane;
      t[b] = c < n ? src[c] : CplxT<C>::make(0, 0);
    }
#pragma unroll
    for (int b = 0; b < kB; ++b) {
      const int c = c0 + b * 64 + lane;
      if (c < n) dst[c] = t[b];
    }
  }
}

// z inverse transform of the sphere columns: T[v][z][c] = sum_m3 x(c, m3)
// e^{+2 pi i m3 z / N}.  One lane per column (m1, m2); the column's plane
// waves are consecutive in sorted order with m3 = lo .. lo + cnt - 1 (the
// sphere is convex).
template <int N, typename C>
__device__ inline void zinv_body(const PwDev &d, const double2 *__restrict__ in, int64_t sin,
                                 const int32_t *__restrict__ group,
                                 const int32_t *__restrict__ active, C *__restrict__ T,
                                 const int32_t *__restrict__ relax, int want, int v, int c);

template <int N, typename C = double2>
__global__ __launch_bounds__(64) void k_pw_zinv(PwDev d, const double2 *__restrict__ in,
                                                int64_t sin, const int32_t *__restrict__ group,
                                                const int32_t *__restrict__ active,
                                                C *__restrict__ T,
                                                const int32_t *__restrict__ relax = nullptr,
                                                int want = 0) {
  zinv_body<N, C>(d, in, sin, group, active, T, relax, want, blockIdx.y,
                  blockIdx.x * 64 + threadIdx.x);
}

template <int N, typename C>
__device__ inline void zinv_body(const PwDev &d, const double2 *__restrict__ in, int64_t sin,
                                 const int32_t *__restrict__ group,
                                 const int32_t *__restrict__ active, C *__restrict__ T,
                                 const int32_t *__restrict__ relax, int want, int v, int c) {
  if (active && !active[v]) return;
  if (precision_skip(relax, want, v)) return;
  if (c >= d.nslot) return;
  const int g = group ? group[v] : 0;
  const int cnt = d.col_cnt[(int64_t)g * d.nslot + c];
  C *Tv = T + (int64_t)v * N * d.nslot * kSlotScale<C> + c;
  if (cnt == 0) {
#pragma unroll
    for (int z = 0; z < N; ++z) Tv[(int64_t)z * d.nslot] = czero<C>();
    return;
  }
  const int st = d.col_start[(int64_t)g * d.nslot + c], lo = d.col_lo[(int64_t)g * d.nslot + c];
  const int32_t *sidx = d.sorted_idx + (int64_t)g * d.ld + st;
  const double2 *x = in + v * sin;
  C buf[N];
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const int m = i < N / 2 ? i : i - N;
    const int k = m - lo;
    buf[i] = (k >= 0 && k < cnt) ? to_c<C>(x[sidx[k]]) : czero<C>();
  }
  reg_fft<N, +1>(buf);
#pragma unroll
  for (int z = 0; z < N; ++z) Tv[(int64_t)z * d.nslot] = buf[z];
}

// z forward transform of the sphere columns back to the plane waves:
// loc[v][i] = (1/Nbox) sum_z S[v][z][c] e^{-2 pi i m3 z / N} for the plane
// waves i of column c.
template <int N, typename C = double2>
__global__ __launch_bounds__(64) void k_pw_zfwd(PwDev d, const C *__restrict__ S,
                                                const int32_t *__restrict__ group,
                                                const int32_t *__restrict__ active,
                                                double2 *__restrict__ loc,
                                                const int32_t *__restrict__ relax = nullptr,
                                                int want = 0) {
  const int v = blockIdx.y, c = blockIdx.x * 64 + threadIdx.x;
  if (active && !active[v]) return;
  if (precision_skip(relax, want, v)) return;
  if (c >= d.nslot) return;
  const int g = group ? group[v] : 0;
  const int cnt = d.col_cnt[(int64_t)g * d.nslot + c];
  if (cnt == 0) return;
  const int st = d.col_start[(int64_t)g * d.nslot + c], lo = d.col_lo[(int64_t)g * d.nslot + c];
  const int32_t *sidx = d.sorted_idx + (int64_t)g * d.ld + st;
  const C *Sv = S + (int64_t)v * N * d.nslot * kSlotScale<C> + c;
  C buf[N];
#pragma unroll
  for (int z = 0; z < N; ++z) buf[z] = Sv[(int64_t)z * d.nslot];
  reg_fft<N, -1>(buf);
  double2 *lv = loc + (int64_t)v * d.ld;
  const double sc = d.inv_nbox;
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const int m = i < N / 2 ? i : i - N;
    const int k = m - lo;
    if (k >= 0 && k < cnt) lv[sidx[k]] = mk((double)buf[i].x * sc, (double)buf[i].y * sc);
  }
}

// z transforms with each column split over a lane pair (splitfft.h): lane
// 2j + odd of the pair of column j holds N/2 of its values, so these need
// about half the registers of k_pw_zinv / k_pw_zfwd.  Columns are counted in
// the layout of d.col_info (T[v][z][j], d.ncs columns per plane).  Both lanes
// of a pair take the same early exits.  MB >= 0: the sphere's z half-width
// M3 as a compile-time constant, so values outside |m3| <= MB are literal
// zeros (inverse) or never stored (forward); -1: no such bound.
template <int N, int MB, typename C = double2, bool RL = false>
__device__ inline void zinv_split_body(const PwDev &d, const double2 *__restrict__ in,
                                       int64_t sin, const int32_t *__restrict__ group,
                                       const int32_t *__restrict__ active, C *__restrict__ T,
                                       int v, int jc, bool odd,
                                       const int32_t *__restrict__ relax = nullptr,
                                       int want = 0) {
  constexpr int H = N / 2, Q = N / 4;
  if (active && !active[v]) return;
  if (precision_skip<RL>(relax, want, v)) return;
  const int ncs = d.ncs;
  if (jc >= ncs) return;
  const int g = group ? group[v] : 0;
  const int4 ci = d.col_info[(int64_t)g * ncs + jc];  // one load for the column's tables
  if (ci.x < 0) return;  // past this group's columns
  const int cnt = ci.y;
  C *Tv = T + (int64_t)v * N * ncs * kSlotScale<C> + jc;
  const int zo = odd ? Q : 0;  // this lane's z: zo + j and H + zo + j
  if (cnt == 0) {
#pragma unroll
    for (int j = 0; j < Q; ++j) {
      Tv[(int64_t)(zo + j) * ncs] = czero<C>();
      Tv[(int64_t)(H + zo + j) * ncs] = czero<C>();
    }
    return;
  }
  const int st = ci.z, lo = ci.w;
  const int32_t *sidx = d.sorted_idx + (int64_t)g * d.ld + st;
  const double2 *x = in + v * sin;
  C b[H];
#pragma unroll
  for (int n = 0; n < H; ++n) {
    const int i = 2 * n + (odd ? 1 : 0), m = i < N / 2 ? i : i - N, k = m - lo;
    const bool band = MB < 0 || (m >= -MB && m <= MB);
    b[n] = (band && k >= 0 && k < cnt) ? to_c<C>(x[sidx[k]]) : czero<C>();
  }
  split_dit<N, +1>(b, odd);
#pragma unroll
  for (int j = 0; j < Q; ++j) {
    Tv[(int64_t)(zo + j) * ncs] = b[j];
    Tv[(int64_t)(H + zo + j) * ncs] = b[Q + j];
  }
}

template <int N, int MB, typename C = double2, bool RL = false>
__global__ __launch_bounds__(64) void k_pw_zfwd_split(PwDev d, const C *__restrict__ S,
                                                      const int32_t *__restrict__ group,
                                                      const int32_t *__restrict__ active,
                                                      double2 *__restrict__ loc,
                                                      const int32_t *__restrict__ relax = nullptr,
                                                      int want = 0) {
  constexpr int H = N / 2, Q = N / 4;
  const int v = blockIdx.y, jc = blockIdx.x * 32 + (int)(threadIdx.x >> 1);
  const bool odd = (threadIdx.x & 1) != 0;
  if (active && !active[v]) return;
  if (precision_skip<RL>(relax, want, v)) return;
  const int ncs = d.ncs;
  if (jc >= ncs) return;
  const int g = group ? group[v] : 0;
  const int4 ci = d.col_info[(int64_t)g * ncs + jc];
  if (ci.x < 0) return;  // past this group's columns
  const int cnt = ci.y;
  if (cnt == 0) return;
  const int st = ci.z, lo = ci.w;
  const int32_t *sidx = d.sorted_idx + (int64_t)g * d.ld + st;
  const C *Sv = S + (int64_t)v * N * ncs * kSlotScale<C> + jc;
  const int zo = odd ? Q : 0;
  C b[H];
#pragma unroll
  for (int j = 0; j < Q; ++j) {
    b[j] = Sv[(int64_t)(zo + j) * ncs];
    b[Q + j] = Sv[(int64_t)(H + zo + j) * ncs];
  }
  split_dif<N, -1>(b, odd);
  double2 *lv = loc + (int64_t)v * d.ld;
  const double sc = d.inv_nbox;
#pragma unroll
  for (int k = 0; k < H; ++k) {
    const int i = 2 * k + (odd ? 1 : 0), m = i < N / 2 ? i : i - N, k3 = m - lo;
    const bool band = MB < 0 || (m >= -MB && m <= MB);
    if (band && k3 >= 0 && k3 < cnt) lv[sidx[k3]] = mk((double)b[k].x * sc, (double)b[k].y * sc);
  }
}

// One wavefront per (plane z, vector v), cubic box of compile-time side N.
// The plane's pencil transforms run as register FFTs (regfft.h):
//   Z  each lane sums its sphere columns at this z (<= 2M3+1 terms),
//   Y  lane a < nc1 transforms row m1 = a - M1 over m2 -> y,
//   X  lane y < N transforms over m1 -> x, multiplies by V(x, y, z) and
//      transforms back, keeping the nc1 frequencies m1 of the sphere,
//   Y' lane a < nc1 transforms back over y -> m2 and writes the sphere
//      columns' values S[v][c][z].
// LDS holds the column values T[nc1][nc2] and one row buffer P[nc1][N] that
// the X stage overwrites column by column (each lane owns its column y).
template <int N, typename C>
__device__ inline void plane_body(const PwDev &d, const C *__restrict__ Tin,
                                  const int32_t *__restrict__ group,
                                  const int32_t *__restrict__ active, C *__restrict__ S,
                                  const int32_t *__restrict__ relax, int want, int z, int v,
                                  C *smem);

template <int N, typename C = double2>
__global__ __launch_bounds__(64) void k_pw_plane_fft(PwDev d, const C *__restrict__ Tin,
                                                     const int32_t *__restrict__ group,
                                                     const int32_t *__restrict__ active,
                                                     C *__restrict__ S,
                                                     const int32_t *__restrict__ relax = nullptr,
                                                     int want = 0) {
  extern __shared__ double2 smem_d[];
  plane_body<N, C>(d, Tin, group, active, S, relax, want, blockIdx.x, blockIdx.y,
                   reinterpret_cast<C *>(smem_d));
}

template <int N, typename C>
__device__ inline void plane_body(const PwDev &d, const C *__restrict__ Tin,
                                  const int32_t *__restrict__ group,
                                  const int32_t *__restrict__ active, C *__restrict__ S,
                                  const int32_t *__restrict__ relax, int want, int z, int v,
                                  C *smem) {
  using R = typename CplxT<C>::S;
  if (active && !active[v]) return;
  if (precision_skip(relax, want, v)) return;
  const int g = group ? group[v] : 0;
  const int nc1 = d.nc1, nc2 = d.nc2, nslot = d.nslot, M1 = d.M1, M2 = d.M2;
  const int lane = threadIdx.x;
  C *T = smem;          // nslot
  C *P = T + nslot;     // nc1 * N
  const int32_t *cc = d.col_cnt + (int64_t)g * nslot;
  const C *Tz = Tin + ((int64_t)v * N * kSlotScale<C> + z) * nslot;
  stage_plane(Tz, T, nslot);
  __syncthreads();
  C buf[N];
  if (lane < nc1) {  // Y inverse of row a
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int m = i < N / 2 ? i : i - N;
      buf[i] = (m >= -M2 && m <= M2) ? T[lane * nc2 + m + M2] : czero<C>();
    }
    reg_fft<N, +1>(buf);
#pragma unroll
    for (int i = 0; i < N; ++i) P[lane * N + i] = buf[i];
  }
  __syncthreads();
  if (lane < N) {  // X inverse, V(r), X forward of column y = lane
    const int y = lane;
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int m = i < N / 2 ? i : i - N;
      buf[i] = (m >= -M1 && m <= M1) ? P[(m + M1) * N + y] : czero<C>();
    }
    reg_fft<N, +1>(buf);
    const double *vcol = d.vloc_zxy + (int64_t)z * N * N + y;  // V(x, y, z) at vcol[x * N]
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const R vv = (R)vcol[i * N];
      buf[i] = CplxT<C>::make(buf[i].x * vv, buf[i].y * vv);
    }
    reg_fft<N, -1>(buf);
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int m = i < N / 2 ? i : i - N;
      if (m >= -M1 && m <= M1) P[(m + M1) * N + y] = buf[i];
    }
  }
  __syncthreads();
  if (lane < nc1) {  // Y forward of row a into the sphere columns
#pragma unroll
    for (int i = 0; i < N; ++i) buf[i] = P[lane * N + i];
    reg_fft<N, -1>(buf);
    C *Sz = S + ((int64_t)v * N * kSlotScale<C> + z) * nslot;
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int m = i < N / 2 ? i : i - N;
      if (m >= -M2 && m <= M2) {
        const int c = lane * nc2 + m + M2;
        if (cc[c] > 0) Sz[c] = buf[i];
      }
    }
  }
}

// FP64 plane transforms of two vectors per wavefront, planes (z, v0) and
// (z, v0 + 1): the Y stages of both planes run side by side (plane p on lanes
// [p nc1, (p + 1) nc1), which needs 2 nc1 <= 64), the X stage plane by plane on
// lanes [0, N).  The Y stages use only nc1 lanes each, so pairing the planes
// halves their share of the wavefront's time, and the loads of both planes are
// in flight together.  LDS: T[2][nslot], then P[2][nc1][N].
template <int N>
__device__ inline void plane2_body(const PwDev &d, const double2 *__restrict__ Tin,
                                   const int32_t *__restrict__ group,
                                   const int32_t *__restrict__ active, double2 *__restrict__ S,
                                   int z, int v0, int nvec, double2 *smem) {
  const int nc1 = d.nc1, nc2 = d.nc2, nslot = d.nslot, M2 = d.M2;
  const int lane = threadIdx.x;
  bool live[2];
#pragma unroll
  for (int p = 0; p < 2; ++p) live[p] = v0 + p < nvec && (!active || active[v0 + p]);
  if (!live[0] && !live[1]) return;
  double2 *T = smem, *P = smem + 2 * nslot;
#pragma unroll
  for (int p = 0; p < 2; ++p)
    if (live[p]) stage_plane(Tin + ((int64_t)(v0 + p) * N + z) * nslot, T + p * nslot, nslot);
  __syncthreads();
  // Y-stage lane mapping: plane yp, row a
  const int yp = lane < nc1 ? 0 : 1, a = lane - yp * nc1;
  const bool yrow = a < nc1 && live[yp];
  double2 buf[N];
  if (yrow) {  // Y inverse of row a
    const double2 *Tp = T + yp * nslot;
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int m = i < N / 2 ? i : i - N;
      buf[i] = (m >= -M2 && m <= M2) ? Tp[a * nc2 + m + M2] : mk(0, 0);
    }
    reg_fft<N, +1>(buf);
    double2 *Pp = P + yp * nc1 * N;
#pragma unroll
    for (int i = 0; i < N; ++i) Pp[a * N + i] = buf[i];
  }
  __syncthreads();
  if (lane < N) {  // X inverse, V(r), X forward of column y = lane, plane by plane
#pragma unroll 1
    for (int p = 0; p < 2; ++p) {
      if (!live[p]) continue;
      // Per-plane copies the compiler cannot see through: V loads, LDS
      // addresses and band masks are then formed inside the loop.  Hoisted
      // out of it they would stay live across both planes (2N loaded values,
      // N addresses, 2N mask bits) and spill.
      int y = lane, M1 = d.M1;
      __asm__ volatile("" : "+v"(y), "+s"(M1)::"memory");
      const double *vcol = d.vloc_zxy + (int64_t)z * N * N + y;  // V(x, y, z) at vcol[x * N]
      double2 *Pp = P + p * nc1 * N;
#pragma unroll
      for (int i = 0; i < N; ++i) {
        const int m = i < N / 2 ? i : i - N;
        buf[i] = (m >= -M1 && m <= M1) ? Pp[(m + M1) * N + y] : mk(0, 0);
      }
      reg_fft<N, +1>(buf);
#pragma unroll
      for (int i = 0; i < N; ++i) {
        const double vv = vcol[i * N];
        buf[i] = mk(buf[i].x * vv, buf[i].y * vv);
      }
      reg_fft<N, -1>(buf);
#pragma unroll
      for (int i = 0; i < N; ++i) {
        const int m = i < N / 2 ? i : i - N;
        if (m >= -M1 && m <= M1) Pp[(m + M1) * N + y] = buf[i];
      }
    }
  }
  __syncthreads();
  if (yrow) {  // Y forward of row a into the sphere columns
    const int v = v0 + yp;
    const double2 *Pp = P + yp * nc1 * N;
#pragma unroll
    for (int i = 0; i < N; ++i) buf[i] = Pp[a * N + i];
    reg_fft<N, -1>(buf);
    const int32_t *cc = d.col_cnt + (int64_t)(group ? group[v] : 0) * nslot;
    double2 *Sz = S + ((int64_t)v * N + z) * nslot;
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int m = i < N / 2 ? i : i - N;
      if (m >= -M2 && m <= M2) {
        const int c = a * nc2 + m + M2;
        if (cc[c] > 0) Sz[c] = buf[i];
      }
    }
  }
}

// Plane transforms of PL vectors, planes (z, v0 + p) for p < PL, by a
// block of 64 W lanes whose transforms are split over lane pairs
// (splitfft.h): every lane holds N/2 values, so the block needs about half
// the registers per lane of plane2_body and each SIMD holds two wavefronts.
// T and S are in the column layout of d.row_* ([v][z][j], d.ncs columns per
// plane; row a of the grid holds its columns m2 = lo .. hi - 1).  The split
// transforms are in rotation form (fewer per-lane selects than the select
// form, 6.5 % less time here; the two forms round differently).
//   Y  lane pair r < PL nc1: row a of plane yp (r = yp nc1 + a), m2 -> y;
//   X  the PL N (plane, column) tasks in rounds of 32 W lane pairs: column y
//      of plane p, m1 -> x, times V(x, y, z), x -> m1 (nc1 frequencies kept);
//   Y' as Y, y -> m2, into the row's columns of S.
// With PL N a multiple of 32 W (4 planes of 48 on 3 wavefronts) every lane
// pair works in every X round.  LDS holds P[PL][nc1][N + 1] (rows padded by
// one value, so that the lanes of the Y stages, one row each, fall on
// different banks); the column values T[PL][ncs] are staged into its start
// and read into registers before the Y stage overwrites them.
// MB >= 0: the sphere's half-widths M1 = M2 = MB are compile-time constants.
// Every transform input outside |m| <= MB is then a literal zero and every
// output outside it is never stored, so the compiler drops the butterflies
// that only touch those (the file is built without signed zeros and
// non-finite values, which lets x + 0 and x * 0 fold).  MB = -1: run-time
// half-widths.
template <int N, int MB, int PL, int W, typename C = double2, bool RL = false>
__device__ inline void plane_split_body(const PwDev &d, const C *__restrict__ Tin,
                                        const int32_t *__restrict__ group,
                                        const int32_t *__restrict__ active,
                                        C *__restrict__ S, int z, int v0, int nvec, C *smem,
                                        const int32_t *__restrict__ relax = nullptr,
                                        int want = 0,
                                        const int32_t *__restrict__ vlist = nullptr) {
  using R = typename CplxT<C>::S;
  constexpr int H = N / 2, Q = N / 4, NP = 32 * W;  // NP lane pairs
  constexpr int PN = N + 1;  // row stride of P: rows of N values would share LDS banks
  const int nc1 = MB >= 0 ? 2 * MB + 1 : d.nc1;
  const int ncs = d.ncs, M2 = MB >= 0 ? MB : d.M2;
  const int t = threadIdx.x, r = t >> 1;
  const bool odd = (t & 1) != 0;
  // plane p of the block belongs to vector vlist[v0 + p] (the running
  // vectors in order, then -1) or, without a list, to vector v0 + p
  int vv[PL];
  bool live[PL], any = false;
#pragma unroll
  for (int p = 0; p < PL; ++p) {
    const int i = v0 + p;
    vv[p] = i < nvec ? (vlist ? vlist[i] : i) : -1;
    live[p] = vv[p] >= 0 && (!active || active[vv[p]]) &&
              !precision_skip<RL>(relax, want, vv[p]);
    any |= live[p];
  }
  if (!any) return;
  C *P = smem, *T = smem;  // T[PL][ncs] aliases the start of P[PL][nc1][PN]
#pragma unroll
  for (int p = 0; p < PL; ++p)  // plane p staged by wavefront p mod W
    if ((t >> 6) == p % W && live[p]) {
      const int gp = group ? group[vv[p]] : 0;
      stage_plane(Tin + ((int64_t)vv[p] * N * kSlotScale<C> + z) * ncs, T + p * ncs,
                  d.row_start[(int64_t)gp * (nc1 + 1) + nc1]);
    }
  __syncthreads();
  const int yp = r / nc1, a = r - yp * nc1;
  const bool yrow = yp < PL && live[yp];
  const int vy = yrow ? (vlist ? vlist[v0 + yp] : v0 + yp) : 0;  // this lane pair's vector
  C b[H];
  if (yrow) {  // row a: columns m2 = lo .. hi - 1 of the group's layout
    const int64_t g = group ? group[vy] : 0;
    const int lo = d.row_lo[g * nc1 + a], hi = lo + d.row_cnt[g * nc1 + a];
    const C *Tp = T + yp * ncs + d.row_start[g * (nc1 + 1) + a] - lo;
#pragma unroll
    for (int n = 0; n < H; ++n) {
      const int i = 2 * n + (odd ? 1 : 0), m = i < N / 2 ? i : i - N;
      b[n] = (m >= -M2 && m <= M2 && m >= lo && m < hi) ? Tp[m] : czero<C>();
    }
  }
  __syncthreads();  // every column value is in registers before P overwrites T
  if (yrow) {  // Y inverse of row a
    split_dit<N, +1>(b, odd);
    C *Pr = P + (yp * nc1 + a) * PN + (odd ? Q : 0);
#pragma unroll
    for (int j = 0; j < Q; ++j) {
      Pr[j] = b[j];
      Pr[H + j] = b[Q + j];
    }
  }
  __syncthreads();
  // X inverse, V(r), X forward: task = (plane p, column y), round by round
#pragma unroll 1
  for (int task = r; task < PL * N; task += NP) {
    const int p = task / N;
    if (!live[p]) continue;
    // per-round copies the compiler cannot see through, so that addresses
    // and masks are formed inside the loop rather than kept live across it
    int y = task - p * N, M1 = MB >= 0 ? MB : d.M1;
    if constexpr (MB >= 0)
      __asm__ volatile("" : "+v"(y)::"memory");
    else
      __asm__ volatile("" : "+v"(y), "+s"(M1)::"memory");
    C *Pp = P + p * nc1 * PN + y;
#pragma unroll
    for (int n = 0; n < H; ++n) {
      const int i = 2 * n + (odd ? 1 : 0), m = i < N / 2 ? i : i - N;
      b[n] = (m >= -M1 && m <= M1) ? Pp[(m + M1) * PN] : czero<C>();
    }
    split_dit<N, +1>(b, odd);
    const double *vcol = d.vloc_zxy + ((int64_t)z * N + (odd ? Q : 0)) * N + y;
#pragma unroll
    for (int j = 0; j < Q; ++j) {  // x = j (+Q) and H + j (+Q)
      const R v1 = (R)vcol[j * N], v2 = (R)vcol[(H + j) * N];
      b[j] = CplxT<C>::make(b[j].x * v1, b[j].y * v1);
      b[Q + j] = CplxT<C>::make(b[Q + j].x * v2, b[Q + j].y * v2);
    }
    split_dif<N, -1>(b, odd);
#pragma unroll
    for (int k = 0; k < H; ++k) {
      const int i = 2 * k + (odd ? 1 : 0), m = i < N / 2 ? i : i - N;
      if (m >= -M1 && m <= M1) Pp[(m + M1) * PN] = b[k];
    }
  }
  __syncthreads();
  if (yrow) {  // Y forward of row a into the sphere columns
    const int v = vy;
    const C *Pr = P + (yp * nc1 + a) * PN + (odd ? Q : 0);
#pragma unroll
    for (int j = 0; j < Q; ++j) {
      b[j] = Pr[j];
      b[Q + j] = Pr[H + j];
    }
    split_dif<N, -1>(b, odd);
    const int64_t g = group ? group[v] : 0;
    const int lo = d.row_lo[g * nc1 + a], hi = lo + d.row_cnt[g * nc1 + a];
    C *Sz = S + ((int64_t)v * N * kSlotScale<C> + z) * ncs + d.row_start[g * (nc1 + 1) + a] - lo;
#pragma unroll
    for (int k = 0; k < H; ++k) {
      const int i = 2 * k + (odd ? 1 : 0), m = i < N / 2 ? i : i - N;
      if (m >= -M2 && m <= M2 && m >= lo && m < hi) Sz[m] = b[k];
    }
  }
}

// Y then X inverse transforms of one z-plane of the sphere columns Tz (in
// LDS as T) into the registers of lane y: buf[x] = value at (x, y, z).
// P (nc1 x N, LDS) is the row buffer; lanes >= N return with buf untouched.
template <int N>
__device__ inline void plane_to_real(const PwDev &d, const double2 *__restrict__ Tz, double2 *T,
                                     double2 *P, double2 (&buf)[N]) {
  const int nc1 = d.nc1, nc2 = d.nc2, nslot = d.nslot, M1 = d.M1, M2 = d.M2;
  const int lane = threadIdx.x;
  __syncthreads();
  stage_plane(Tz, T, nslot);
  __syncthreads();
  if (lane < nc1) {
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int m = i < N / 2 ? i : i - N;
      buf[i] = (m >= -M2 && m <= M2) ? T[lane * nc2 + m + M2] : mk(0, 0);
    }
    reg_fft<N, +1>(buf);
#pragma unroll
    for (int i = 0; i < N; ++i) P[lane * N + i] = buf[i];
  }
  __syncthreads();
  if (lane < N) {
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int m = i < N / 2 ? i : i - N;
      buf[i] = (m >= -M1 && m <= M1) ? P[(m + M1) * N + lane] : mk(0, 0);
    }
    reg_fft<N, +1>(buf);
  }
}

// Density response of one z-plane for one shift k (incdrhoscf):
//   D[k][z][x][y] (+)= wgt * sum_v conj(psi_v(r)) dpsi_{v,k}(r),
// dpsi from the z-transformed columns T (vector v * nshift + k of the block)
// and psi_v(r) given as Pr[v][z][x][y].  Block (z, k) owns its plane of D.
template <int N>
__global__ __launch_bounds__(64) void k_pw_plane_drho(PwDev d, const double2 *__restrict__ T,
                                                      int nbnd, int nshift,
                                                      const double2 *__restrict__ Pr, double wgt,
                                                      double2 *__restrict__ D, int accumulate) {
  extern __shared__ double2 smem[];
  const int z = blockIdx.x, k = blockIdx.y;
  const int lane = threadIdx.x;
  double2 *Ts = smem;              // nslot
  double2 *P = Ts + d.nslot;       // nc1 * N
  double2 *Dz = D + ((int64_t)k * N + z) * N * N;
  if (!accumulate && lane < N)
    for (int x = 0; x < N; ++x) Dz[(int64_t)x * N + lane] = mk(0, 0);
  double2 buf[N];
  for (int v = 0; v < nbnd; ++v) {
    const int64_t vec = (int64_t)v * nshift + k;
    plane_to_real<N>(d, T + (vec * N + z) * d.nslot, Ts, P, buf);
    if (lane < N) {
      const double2 *pz = Pr + ((int64_t)v * N + z) * N * N + lane;
#pragma unroll
      for (int x = 0; x < N; ++x) {
        const double2 p = pz[(int64_t)x * N];
        double2 *o = Dz + (int64_t)x * N + lane;
        double2 acc = *o;
        // conj(p) * dpsi
        acc.x = fma(wgt, p.x * buf[x].x + p.y * buf[x].y, acc.x);
        acc.y = fma(wgt, p.x * buf[x].y - p.y * buf[x].x, acc.y);
        *o = acc;
      }
    }
  }
}

// The same density response with the transforms split over lane pairs
// (splitfft.h), one block of 128 lanes per (z, k): lane pair r < N owns
// column y = r of the plane for all bands, so its 2 x N/2 values of D stay in
// registers instead of a read-modify-write of D per band.  Per band: the
// column values are staged in LDS, the Y stage (pairs r < nc1) writes the
// rows P[nc1][N] over them, the X stage (pairs r < N) transforms column y
// and accumulates conj(psi_v) dpsi.  MB as in plane_split_body.
template <int N, int MB>
__global__ __launch_bounds__(128, 2) void k_pw_plane_drho_split(PwDev d,
                                                             const double2 *__restrict__ T,
                                                             int nbnd, int nshift,
                                                             const double2 *__restrict__ Pr,
                                                             double wgt, double2 *__restrict__ D,
                                                             int accumulate) {
  constexpr int H = N / 2, Q = N / 4;
  extern __shared__ double2 smem[];  // P[nc1][N]; the column values staged at its start
  const int z = blockIdx.x, k = blockIdx.y;
  const int t = threadIdx.x, r = t >> 1;
  const bool odd = (t & 1) != 0;
  const int nc1 = MB >= 0 ? 2 * MB + 1 : d.nc1, nc2 = MB >= 0 ? 2 * MB + 1 : d.nc2;
  const int nslot = d.nslot, M1 = MB >= 0 ? MB : d.M1, M2 = MB >= 0 ? MB : d.M2;
  double2 *P = smem, *Ts = smem;
  const int xo = odd ? Q : 0;  // this lane's x: xo + j and H + xo + j
  double2 *Dz = D + ((int64_t)k * N + z) * N * N + r;
  double2 acc[H];
#pragma unroll
  for (int j = 0; j < H; ++j) acc[j] = mk(0, 0);
  if (accumulate && r < N) {
#pragma unroll
    for (int j = 0; j < Q; ++j) {
      acc[j] = Dz[(int64_t)(xo + j) * N];
      acc[Q + j] = Dz[(int64_t)(H + xo + j) * N];
    }
  }
  for (int v = 0; v < nbnd; ++v) {
    const int64_t vec = (int64_t)v * nshift + k;
    __syncthreads();  // the previous band's X stage is done with P
    if (t < 64) stage_plane(T + (vec * N + z) * nslot, Ts, nslot);
    __syncthreads();
    double2 b[H];
    if (r < nc1) {
      const double2 *Tr = Ts + r * nc2 + M2;
#pragma unroll
      for (int n = 0; n < H; ++n) {
        const int i = 2 * n + (odd ? 1 : 0), m = i < N / 2 ? i : i - N;
        b[n] = (m >= -M2 && m <= M2) ? Tr[m] : mk(0, 0);
      }
    }
    __syncthreads();  // every column value is in registers before P overwrites them
    if (r < nc1) {  // Y inverse of row r
      split_dit_sel<N, +1>(b, odd);
      double2 *Prow = P + r * N + xo;
#pragma unroll
      for (int j = 0; j < Q; ++j) {
        Prow[j] = b[j];
        Prow[H + j] = b[Q + j];
      }
    }
    __syncthreads();
    if (r < N) {  // X inverse of column y = r, times conj(psi_v(r)), into D
      const double2 *Pc = P + r;
#pragma unroll
      for (int n = 0; n < H; ++n) {
        const int i = 2 * n + (odd ? 1 : 0), m = i < N / 2 ? i : i - N;
        b[n] = (m >= -M1 && m <= M1) ? Pc[(m + M1) * N] : mk(0, 0);
      }
      split_dit_sel<N, +1>(b, odd);
      const double2 *pz = Pr + ((int64_t)v * N + z) * N * N + r;
#pragma unroll
      for (int j = 0; j < H; ++j) {
        const int x = (j < Q ? j : H + j - Q) + xo;
        const double2 p = pz[(int64_t)x * N];
        acc[j].x = fma(wgt, p.x * b[j].x + p.y * b[j].y, acc[j].x);
        acc[j].y = fma(wgt, p.x * b[j].y - p.y * b[j].x, acc[j].y);
      }
    }
  }
  if (r < N) {
#pragma unroll
    for (int j = 0; j < Q; ++j) {
      Dz[(int64_t)(xo + j) * N] = acc[j];
      Dz[(int64_t)(H + xo + j) * N] = acc[Q + j];
    }
  }
}

// Adjoint gradient of one z-plane over a strided set of vector pairs:
//   G[b][z][x][y] += sum_{p = b, b + nb, ...} w_p Re(conj(y_p(r)) x_p(r)),
// from the z-transformed columns Tx (x_p) and Ty (y_p) in the packed layout
// (d.col_info).  Block (z, b) owns its plane of G, which stays in registers
// over its pairs.  The lower 32 lanes of a wave transform x and the upper 32
// y, every line over a lane pair: 16 rows or columns of both to a wave, so
// one pass of ceil(N/16) waves takes all of them; a swap of the wave's halves
// then leaves the same points of x and y in one lane.
//   Bound: the latency of the two transforms and their LDS exchange, between
// two barriers a pair, at three quarters of the adds' own time.  2 048 pairs of
// the 48^3 box (half-width 4): 638 us against 2 673 with whole lines in one
// lane, x waiting in LDS and G read and written for every pair.
// MB as in plane_split_body.
constexpr int grad_waves(int n) { return (n + 15) / 16; }
template <int N, int MB>
__global__ __launch_bounds__(64 * grad_waves(N), 3) void k_pw_plane_grad(
    PwDev d, const double2 *__restrict__ Tx, const double2 *__restrict__ Ty, int np,
    const int32_t *__restrict__ group, const double *__restrict__ w, double *__restrict__ G,
    int accumulate) {
  constexpr int E = N / 2, F = N / 4, R = N + 1;
  extern __shared__ double2 smem[];
  const int z = blockIdx.x, b0 = blockIdx.y, nb = gridDim.y;
  const int lane = threadIdx.x & 63, half = lane >> 5;
  const int r = (threadIdx.x >> 6) * 16 + ((lane & 31) >> 1);
  const Line<N> ln{lane & 1};
  const int nc1 = MB >= 0 ? 2 * MB + 1 : d.nc1, M1 = MB >= 0 ? MB : d.M1;
  const int ncs = d.ncs;
  double2 *P = smem + half * nc1 * R;  // rows of x, then rows of y
  const double2 *T = half ? Ty : Tx;
  auto freq = [](int i) { return i < N / 2 ? i : i - N; };
  // G[x][y] at y = r, x = nat(i + F half)
  double *Gz = G + ((int64_t)b0 * N + z) * N * N + r;
  double acc[F];
#pragma unroll
  for (int i = 0; i < F; ++i) acc[i] = 0.0;
  auto at = [&](int i) { return (int64_t)(half ? ln.nat(i + F) : ln.nat(i)) * N; };
  if (accumulate && r < N)
#pragma unroll
    for (int i = 0; i < F; ++i) acc[i] = Gz[at(i)];
  for (int p = b0; p < np; p += nb) {
    if (r < nc1) {  // Y inverse of row r
      const int g = group ? group[p] : 0;
      const int64_t gr = (int64_t)g * nc1 + r;
      const int lo = d.row_lo[gr], cnt = d.row_cnt[gr];
      // an empty row reads the plane's first column and keeps nothing of it
      const double2 *row = T + ((int64_t)p * N + z) * ncs + (cnt > 0 ? d.row_start[gr + g] : 0);
      double2 b[E];
#pragma unroll
      for (int i = 0; i < E; ++i) {
        // off the band both points of a pair of lanes are, at compile time
        const bool band = MB < 0 || 2 * i <= MB || 2 * i + 1 >= N - MB;
        const int k = freq(ln.dec(i)) - lo;
        b[i] = band ? keep(row[within(k, cnt)], k, cnt) : mk(0, 0);
      }
      ln.template dit<+1>(b);
      double2 *Pr = P + r * R;
#pragma unroll
      for (int i = 0; i < E; ++i) Pr[ln.nat(i)] = b[i];
    }
    __syncthreads();
    if (r < N) {  // X inverse of column y = r
      double2 b[E];
#pragma unroll
      for (int i = 0; i < E; ++i) {
        const bool band = MB < 0 || 2 * i <= MB || 2 * i + 1 >= N - MB;
        const int a = freq(ln.dec(i)) + M1;
        b[i] = band ? keep(P[within(a, nc1) * R + r], a, nc1) : mk(0, 0);
      }
      ln.template dit<+1>(b);
      const double wp = w[p];
#pragma unroll
      for (int i = 0; i < F; ++i) {
        lanes::swap_halves(b[i].x, b[i + F].x);
        lanes::swap_halves(b[i].y, b[i + F].y);
        acc[i] = fma(wp, b[i + F].x * b[i].x + b[i + F].y * b[i].y, acc[i]);
      }
    }
    __syncthreads();
  }
  if (r < N)
#pragma unroll
    for (int i = 0; i < F; ++i) Gz[at(i)] = acc[i];
}

// ---------------------------------------------------------------------------
// Projector contraction per k+q group: the vectors of one group share the
// projector block proj[g] (nproj x npw), so the two complex GEMMs
//   becp = proj^H X   (nproj x nv, K = npw)   and   HX += proj (D becp)
// run per (group, chunk of kChunk plane waves, tile of kVT vectors): each
// block reads its projector chunk once for kVT vectors.
// ---------------------------------------------------------------------------
constexpr int kChunk = 64;
constexpr int kVT = 16;
constexpr int kAsmThreads = 256;  // lanes of a k_pw_assemble2 block
constexpr int kAsmBlocks = 640;   // blocks its widest shape has to fill

// columns of nvec vectors of x and of as many of y (blockIdx.z) along z
template <int N, int MB>
__global__ __launch_bounds__(64) void k_pw_zinv_pair(PwDev d, const double2 *__restrict__ x,
                                                     const double2 *__restrict__ y, int64_t sin,
                                                     const int32_t *__restrict__ group,
                                                     double2 *__restrict__ Tx,
                                                     double2 *__restrict__ Ty) {
  zinv_split_body<N, MB>(d, blockIdx.z ? y : x, sin, group, nullptr, blockIdx.z ? Ty : Tx,
                         blockIdx.y, blockIdx.x * 32 + (int)(threadIdx.x >> 1),
                         (threadIdx.x & 1) != 0);
}

// does any vector of the tile still run?  (uniform across the block)
__device__ inline bool tile_active(const int32_t *__restrict__ active,
                                   const int32_t *__restrict__ vecs, int nv) {
  // one vector to a lane: taken in turn, each costs two dependent loads (a
  // small batch's assembly 14.7 us against 13.6)
  const int lane = threadIdx.x & 63;
  return __any(lane < nv && active[vecs[lane]] != 0);
}

// becp[g][vt][p][vl] = D_p sum over the chunk partials (once per tile); one
// lane per output (p, vl), 64 outputs per block
__device__ inline void becp_reduce_body(const PwDev &d, const int32_t *__restrict__ active,
                                        const int32_t *__restrict__ gvec,
                                        const int32_t *__restrict__ gcnt, int maxper, int tiles,
                                        int nchunk, const double2 *__restrict__ part,
                                        double2 *__restrict__ becp, int bx, int g, int vt, int t);

__global__ __launch_bounds__(64) void k_pw_becp_reduce(PwDev d,
                                                       const int32_t *__restrict__ active,
                                                       const int32_t *__restrict__ gvec,
                                                       const int32_t *__restrict__ gcnt,
                                                       int maxper, int tiles, int nchunk,
                                                       const double2 *__restrict__ part,
                                                       double2 *__restrict__ becp) {
  becp_reduce_body(d, active, gvec, gcnt, maxper, tiles, nchunk, part, becp, blockIdx.x,
                   blockIdx.y, blockIdx.z, threadIdx.x);
}

__device__ inline void becp_reduce_body(const PwDev &d, const int32_t *__restrict__ active,
                                        const int32_t *__restrict__ gvec,
                                        const int32_t *__restrict__ gcnt, int maxper, int tiles,
                                        int nchunk, const double2 *__restrict__ part,
                                        double2 *__restrict__ becp, int bx, int g, int vt, int t) {
  const int cnt = gcnt[g], v0 = vt * kVT;
  if (v0 >= cnt) return;
  const int nv = min(kVT, cnt - v0), nproj = d.nproj;
  const int o = bx * 64 + t;  // t: thread of the 64 handling outputs [64 bx, 64 bx + 64)
  if (o >= nproj * kVT) return;
  if (active && !tile_active(active, gvec + g * maxper + v0, nv)) return;
  const int nck = (d.npw[g] + kChunk - 1) / kChunk;
  const int64_t stride = (int64_t)nproj * kVT;
  const double2 *pp = part + ((int64_t)g * tiles + vt) * nchunk * stride + o;
  double2 a0 = mk(0, 0), a1 = mk(0, 0), a2 = mk(0, 0), a3 = mk(0, 0);
  int c = 0;
  for (; c + 4 <= nck; c += 4) {  // four independent loads in flight
    const double2 t0 = pp[(int64_t)c * stride], t1 = pp[(int64_t)(c + 1) * stride];
    const double2 t2 = pp[(int64_t)(c + 2) * stride], t3 = pp[(int64_t)(c + 3) * stride];
    a0.x += t0.x; a0.y += t0.y;
    a1.x += t1.x; a1.y += t1.y;
    a2.x += t2.x; a2.y += t2.y;
    a3.x += t3.x; a3.y += t3.y;
  }
  for (; c < nck; ++c) {
    const double2 t = pp[(int64_t)c * stride];
    a0.x += t.x; a0.y += t.y;
  }
  const double sx = (a0.x + a1.x) + (a2.x + a3.x), sy = (a0.y + a1.y) + (a2.y + a3.y);
  const double dc = d.dcoef[(int64_t)g * nproj + o / kVT];
  becp[((int64_t)g * tiles + vt) * stride + o] = mk(sx * dc, sy * dc);
}

// part[((g*tiles + vt)*nchunk + chunk)][p][vl] = sum_{i in chunk} conj(proj_p(i)) x_v(i)
// for p0 <= p < pe: all projectors, or at most 16 of them
__device__ inline void becp_body(const PwDev &d, const double2 *__restrict__ in, int64_t sin,
                                 const int32_t *__restrict__ active,
                                 const int32_t *__restrict__ gvec,
                                 const int32_t *__restrict__ gcnt, int maxper, int tiles,
                                 int nchunk, double2 *__restrict__ part, int chunk, int g, int vt,
                                 int p0, int pe);

__global__ __launch_bounds__(256) void k_pw_becp(PwDev d, const double2 *__restrict__ in,
                                                 int64_t sin, const int32_t *__restrict__ active,
                                                 const int32_t *__restrict__ gvec,
                                                 const int32_t *__restrict__ gcnt, int maxper,
                                                 int tiles, int nchunk,
                                                 double2 *__restrict__ part) {
  becp_body(d, in, sin, active, gvec, gcnt, maxper, tiles, nchunk, part, blockIdx.x, blockIdx.y,
            blockIdx.z, 0, d.nproj);
}

__device__ inline void becp_body(const PwDev &d, const double2 *__restrict__ in, int64_t sin,
                                 const int32_t *__restrict__ active,
                                 const int32_t *__restrict__ gvec,
                                 const int32_t *__restrict__ gcnt, int maxper, int tiles,
                                 int nchunk, double2 *__restrict__ part, int chunk, int g, int vt,
                                 int p0, int pe) {
  const int cnt = gcnt[g], v0 = vt * kVT;
  const int npw = d.npw[g], i0 = chunk * kChunk;
  if (v0 >= cnt || i0 >= npw) return;
  const int nv = min(kVT, cnt - v0), lim = min(kChunk, npw - i0), nproj = d.nproj;
  if (active && !tile_active(active, gvec + g * maxper + v0, nv)) return;
  // A sum runs over the chunk's plane waves in order, whatever the tiling.  Up
  // to 16 projectors: one sum to a lane, the whole chunk staged at once (a few
  // vectors of the 32^3 box, 16 projectors: 33.9 us an application against 35.3
  // in four stages).  More: wave w takes 16 of 64 projectors, a lane 2 x 2 of
  // their 16 x 16 (projector, vector) sums, one operand read from LDS a product
  // where one sum per lane takes two; the plane waves come 16 at a time.  On
  // the 48^3 box (48 projectors, 512 slots streamed) with the z transforms
  // beside it 18.1 us a launch against 19.6 with one sum to a lane.
  // Loads are unconditional, their places clamped: under a condition each is
  // waited for by itself.
  constexpr int kIB = 16, kPB = 64;
  static_assert(kVT == 16 && kChunk % kIB == 0, "256 lanes: 4 waves of 8 x 8 lanes");
  __shared__ double2 xs[kVT][kChunk + 1];
  __shared__ double2 ps[kPB][kIB + 1];
  static_assert(kPB * (kIB + 1) >= 16 * (kChunk + 1), "16 whole rows");
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const double2 *pg = d.proj + (int64_t)g * nproj * d.ld + i0;
  double2 *pout = part + (((int64_t)g * tiles + vt) * nchunk + chunk) * nproj * kVT;
  const int npb = (nproj + kPB - 1) / kPB;
  const bool few = pe - p0 <= 16;
  double2 next[4];
  auto load = [&](int p, int i) {
    const double2 q = pg[(int64_t)min(p, pe - 1) * d.ld + min(i, lim - 1)];
    const bool in = p < pe && i < lim;
    return mk(in ? q.x : 0.0, in ? q.y : 0.0);
  };
  auto fetch = [&](int stage) {  // stage = projector block, then plane-wave block
    const int p0 = stage / (kChunk / kIB) * kPB, ib = stage % (kChunk / kIB) * kIB;
#pragma unroll
    for (int r = 0; r < 4; ++r) next[r] = load(p0 + tid / kIB + 16 * r, ib + tid % kIB);
  };
  if (few) {
#pragma unroll
    for (int r = 0; r < 4; ++r) next[r] = load(p0 + wv + 4 * r, lane);
  } else {
    fetch(0);
  }
#pragma unroll
  for (int r = 0; r < kVT / 4; ++r) {
    const int vl = wv + 4 * r;  // uniform over the wave
    const int v = gvec[g * maxper + v0 + min(vl, nv - 1)];
    const double2 val = in[v * sin + i0 + min(lane, lim - 1)];
    const bool on = vl < nv && lane < lim && (!active || active[v]);
    xs[vl][lane] = mk(on ? val.x : 0.0, on ? val.y : 0.0);
  }
  if (few) {
    double2 *rows = &ps[0][0];  // [16][kChunk + 1]
#pragma unroll
    for (int r = 0; r < 4; ++r) rows[(wv + 4 * r) * (kChunk + 1) + lane] = next[r];
    __syncthreads();
    const int p = tid / kVT, vl = tid % kVT;
    double2 acc = mk(0, 0);
    for (int i = 0; i < lim; ++i) cmacc(acc, rows[p * (kChunk + 1) + i], xs[vl][i]);
    if (p0 + p < pe) pout[(p0 + p) * kVT + vl] = acc;
    return;
  }
  const int tp = 16 * wv + (lane >> 3), tv = lane & 7;
  for (int pb = 0; pb < npb; ++pb) {
    const bool mine = pb * kPB + 16 * wv < nproj;  // uniform over the wave
    double2 acc[2][2];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b) acc[a][b] = mk(0, 0);
    for (int ib = 0; ib < kChunk; ib += kIB) {
      const int stage = pb * (kChunk / kIB) + ib / kIB;
      if (stage > 0) __syncthreads();
#pragma unroll
      for (int r = 0; r < 4; ++r) ps[tid / kIB + 16 * r][tid % kIB] = next[r];
      __syncthreads();
      if (stage + 1 < npb * (kChunk / kIB)) fetch(stage + 1);
      if (mine) {
#pragma unroll
        for (int i = 0; i < kIB; ++i) {
          const double2 pa = ps[tp][i], pb2 = ps[tp + 8][i];
          const double2 xa = xs[tv][ib + i], xb = xs[tv + 8][ib + i];
          cmacc(acc[0][0], pa, xa);
          cmacc(acc[0][1], pa, xb);
          cmacc(acc[1][0], pb2, xa);
          cmacc(acc[1][1], pb2, xb);
        }
      }
    }
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        const int p = pb * kPB + tp + 8 * a;
        if (p < nproj) pout[p * kVT + tv + 8 * b] = acc[a][b];
      }
  }
}

// out_v = kin x_v + fwfft(V invfft x_v) + proj (D becp_v) + sigma_v x_v for the
// plane waves of one chunk and the vectors of one tile; becp_v is the sum of
// the chunk partials, the local term the z forward transform of S.
// CH plane waves per block of NT lanes: thread = (plane wave i < CH, vector
// group vq < NT / CH), each thread kVT / (NT / CH) vectors.
template <int CH, int NT>
__global__ __launch_bounds__(NT) void k_pw_assemble2(
    PwDev d, const double2 *__restrict__ in, int64_t sin, double2 *__restrict__ out, int64_t sout,
    const double2 *__restrict__ sigma, const int32_t *__restrict__ active,
    const int32_t *__restrict__ gvec, const int32_t *__restrict__ gcnt, int maxper, int tiles,
    int nchunk, const double2 *__restrict__ part, const double2 *__restrict__ S,
    const double2 *__restrict__ locv) {
  extern __shared__ double2 smem[];
  const int chunk = blockIdx.x, g = blockIdx.y, vt = blockIdx.z;
  const int cnt = gcnt[g], v0 = vt * kVT;
  if (v0 >= cnt) return;
  const int nv = min(kVT, cnt - v0), nproj = d.nproj, n3 = d.n3;
  const int npw = d.npw[g], i0 = chunk * CH;
  // thread = (plane wave i of the chunk, vector quarter vq): vectors
  // vl = vq + 4k, k < 4, accumulate together so each projector value is
  // loaded once per thread
  constexpr int kVQ = NT / CH;
  constexpr int kPer = kVT / kVQ;
  static_assert(kVT % kVQ == 0, "vector groups must divide the tile");
  const int i = threadIdx.x % CH, vq = threadIdx.x / CH;
  const int64_t e = (int64_t)i0 + i;
  const bool inside = e < npw;
  // kAhead projector values are loaded together, the first before the overlaps
  // are in LDS.  One vector to a thread leaves registers for 16.  The loads are unconditional (past the last projector
  // they repeat it): under a condition each would be waited for by itself.
  // A second set in flight (16 + 16) costs a wavefront per SIMD: 18.4 us per
  // launch of the streamed 48^3 solve against 15.0.
  constexpr int kAhead = CH == 16 ? 16 : 8;
  const double2 *pg = d.proj + (int64_t)g * nproj * d.ld + (inside ? e : 0);
  double2 pv[kAhead];
  auto fetch = [&](int p0) {
#pragma unroll
    for (int q = 0; q < kAhead; ++q) pv[q] = pg[(int64_t)min(p0 + q, nproj - 1) * d.ld];
  };
  if (nproj > 0) fetch(0);
  if (active && !tile_active(active, gvec + g * maxper + v0, nv)) return;
  double2 *becp = smem;            // [nproj][kVT]
  const double2 *bsrc = part + ((int64_t)g * tiles + vt) * nproj * kVT;  // reduced D becp
  for (int o = threadIdx.x; o < nproj * kVT; o += NT) becp[o] = bsrc[o];
  const int64_t ge = (int64_t)g * d.ld + (inside ? e : 0);
  const double kin = d.kin[ge];
  int vv[kPer];
  bool on[kPer];
  bool any = false;
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const int vl = vq + kVQ * k;
    on[k] = vl < nv;
    vv[k] = on[k] ? gvec[g * maxper + v0 + vl] : 0;
    if (on[k] && active && !active[vv[k]]) on[k] = false;
    any |= on[k];
  }
  double2 xi[kPer], acc[kPer];
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    xi[k] = on[k] && inside ? in[vv[k] * sin + e] : mk(0, 0);
    acc[k] = mk(kin * xi[k].x, kin * xi[k].y);
    if (!on[k] || !inside) continue;
    if (locv) {  // z transform done by k_pw_zfwd (already scaled)
      const double2 l = locv[vv[k] * d.ld + e];
      acc[k].x += l.x;
      acc[k].y += l.y;
    } else {
      const double2 *col = S + ((int64_t)vv[k] * d.nslot + d.slot_of[ge]) * n3;
      const int mz = d.m3_of[ge];
      double2 loc = mk(0, 0);
      for (int z = 0; z < n3; ++z) cmac(loc, col[z], cconj(d.tw3[(mz * z) % n3]));
      acc[k].x = fma(loc.x, d.inv_nbox, acc[k].x);
      acc[k].y = fma(loc.y, d.inv_nbox, acc[k].y);
    }
  }
  __syncthreads();
  if (!any || e >= d.ld) return;  // no running vector in this thread's group
  if (!inside) {  // padding stays zero
#pragma unroll
    for (int k = 0; k < kPer; ++k)
      if (on[k]) out[vv[k] * sout + e] = mk(0, 0);
    return;
  }
  for (int p0 = 0; p0 < nproj; p0 += kAhead) {
#pragma unroll
    for (int q = 0; q < kAhead; ++q)
      if (p0 + q < nproj) {
#pragma unroll
        for (int k = 0; k < kPer; ++k) cmac(acc[k], pv[q], becp[(p0 + q) * kVT + vq + kVQ * k]);
      }
    if (p0 + kAhead < nproj) fetch(p0 + kAhead);
  }
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    if (!on[k]) continue;
    cmac(acc[k], sigma[vv[k]], xi[k]);
    out[vv[k] * sout + e] = acc[k];
  }
}

// f(std::integral_constant<int, M>) for the M of the list equal to m; false if none
template <int... Ms, typename F> inline bool dispatch_band(int m, F &&f) {
  bool hit = false;
  ((m == Ms ? (f(std::integral_constant<int, Ms>{}), hit = true) : false), ...);
  return hit;
}

// f(std::integral_constant<int, M>) with M = m when m is one of the sphere
// half-widths specialised for box N (the usual ones: the box is the smallest
// FFT size of at least 4M + 1, or one size up), else with M = -1
constexpr int kBandMin = 4;
constexpr int band_max(int n) {
  return n == 48 ? 11 : n == 36 ? 8 : n == 32 ? 7 : n == 24 ? 5 : -1;
}
template <int N, typename F> inline void with_band(bool enable, int m, F &&f) {
  bool hit = false;
  if (enable)
    [&]<int... I>(std::integer_sequence<int, I...>) {
      hit = dispatch_band<kBandMin + I...>(m, f);
    }(std::make_integer_sequence<int, std::max(0, band_max(N) - kBandMin + 1)>{});
  if (!hit) f(std::integral_constant<int, -1>{});
}

// Two independent stages of one FP64 application in one launch each, which
// saves a launch boundary (and the tail of the smaller stage) per pair:
//   k_pw_becp_zinv:    blocks [0, nbecp) are projector partial sums (256
//                      lanes); the rest hold four 64-lane z inverse groups;
//   k_pw_reduce_plane: blocks [0, nred) reduce the partials (64 lanes); the
//                      rest are the plane transforms (z fastest).
// The block index orders match the separate kernels' grids, and every branch
// on it is uniform within a block, so the barriers of either part are safe.
// SPLIT: the z inverse transforms split over lane pairs (32 columns per
// 64-lane group), else one lane per column.
// vlist[0 .. k) = the vectors v < nvec with active[v] != 0 (all of them
// without flags) in increasing order, vlist[k .. nvec) = -1; one block of
// 256 lanes
__device__ inline void vlist_body(int nvec, const int32_t *__restrict__ active,
                                  int32_t *__restrict__ vlist) {
  __shared__ int wsum[4];
  __shared__ int base;
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  if (t == 0) base = 0;
  __syncthreads();
  for (int v0 = 0; v0 < nvec; v0 += 256) {
    const int v = v0 + t;
    const bool on = v < nvec && (!active || active[v] != 0);
    const unsigned long long m = __ballot(on);
    if (lane == 0) wsum[w] = __popcll(m);
    __syncthreads();
    int off = base;
    for (int i = 0; i < w; ++i) off += wsum[i];
    if (on) vlist[off + __popcll(m & ((1ull << lane) - 1))] = v;
    __syncthreads();  // every lane has read base and wsum
    if (t == 0) base += wsum[0] + wsum[1] + wsum[2] + wsum[3];
    __syncthreads();
  }
  for (int i = base + t; i < nvec; i += 256) vlist[i] = -1;
}

template <int N, bool SPLIT, int MB, typename C = double2, bool RL = false>
__global__ __launch_bounds__(256) void k_pw_becp_zinv(
    PwDev d, const double2 *__restrict__ in, int64_t sin, const int32_t *__restrict__ group,
    const int32_t *__restrict__ active, const int32_t *__restrict__ gvec,
    const int32_t *__restrict__ gcnt, int maxper, int tiles, int nchunk, int ngroup, int psplit,
    double2 *__restrict__ part, C *__restrict__ T, int nvec,
    const int32_t *__restrict__ relax = nullptr, int want = 0,
    int32_t *__restrict__ vlist = nullptr) {
  // with a list to build, block 0 builds it (first, so that its serial
  // scan does not trail the launch) and the others shift down by one
  // psplit blocks take 16 projectors each of a chunk and tile, or one takes all
  const int nbecp = nchunk * ngroup * tiles * psplit, b = (int)blockIdx.x - (vlist ? 1 : 0);
  if (b < 0) {
    vlist_body(nvec, active, vlist);
    return;
  }
  if (b < nbecp) {
    const int ps = b % psplit, c = b / psplit;
    becp_body(d, in, sin, active, gvec, gcnt, maxper, tiles, nchunk, part, c % nchunk,
              (c / nchunk) % ngroup, c / (nchunk * ngroup), 16 * ps,
              psplit > 1 ? min(d.nproj, 16 * ps + 16) : d.nproj);
    return;
  }
  constexpr int kCols = SPLIT ? 32 : 64;  // columns per 64-lane group
  const int gx = ((SPLIT ? d.ncs : d.nslot) + kCols - 1) / kCols;
  const int zb = (b - nbecp) * 4 + (int)(threadIdx.x >> 6);
  if (zb >= gx * nvec) return;
  const int lane = (int)(threadIdx.x & 63);
  if constexpr (SPLIT)
    zinv_split_body<N, MB, C, RL>(d, in, sin, group, active, T, zb / gx,
                                  (zb % gx) * 32 + (lane >> 1), (lane & 1) != 0, relax, want);
  else
    zinv_body<N, C>(d, in, sin, group, active, T, RL ? relax : nullptr, want, zb / gx,
                    (zb % gx) * 64 + lane);
}

// PAIR: two vectors per plane block (plane2_body), else one (plane_body)
template <int N, bool PAIR>
__global__ __launch_bounds__(64) void k_pw_reduce_plane(
    PwDev d, const int32_t *__restrict__ group, const int32_t *__restrict__ active,
    const int32_t *__restrict__ gvec, const int32_t *__restrict__ gcnt, int maxper, int tiles,
    int nchunk, int ngroup, int nred_x, const double2 *__restrict__ part,
    double2 *__restrict__ becp, const double2 *__restrict__ T, double2 *__restrict__ S,
    int nvec) {
  extern __shared__ double2 smem_d[];
  const int nred = nred_x * ngroup * tiles, b = blockIdx.x;
  if (b < nred) {
    becp_reduce_body(d, active, gvec, gcnt, maxper, tiles, nchunk, part, becp, b % nred_x,
                     (b / nred_x) % ngroup, b / (nred_x * ngroup), threadIdx.x);
    return;
  }
  const int pb = b - nred;
  if constexpr (PAIR)
    plane2_body<N>(d, T, group, active, S, pb % N, 2 * (pb / N), nvec, smem_d);
  else
    plane_body<N, double2>(d, T, group, active, S, nullptr, 0, pb % N, pb / N, smem_d);
}

// As k_pw_reduce_plane with the split plane transforms (blocks of W
// wavefronts, PL vectors per plane block): a reduction block covers W of the
// 64-output ranges.  MB as in plane_split_body.
template <int N, int MB, int PL, int W, typename C = double2, bool RL = false>
__global__ __launch_bounds__(64 * W) void k_pw_reduce_split(
    PwDev d, const int32_t *__restrict__ group, const int32_t *__restrict__ active,
    const int32_t *__restrict__ gvec, const int32_t *__restrict__ gcnt, int maxper, int tiles,
    int nchunk, int ngroup, int nred_x, const double2 *__restrict__ part,
    double2 *__restrict__ becp, const C *__restrict__ T, C *__restrict__ S, int nvec,
    const int32_t *__restrict__ relax = nullptr, int want = 0,
    const int32_t *__restrict__ vlist = nullptr) {
  extern __shared__ double2 smem_d[];
  const int nred_w = (nred_x + W - 1) / W, nred = nred_w * ngroup * tiles, b = blockIdx.x;
  if (b < nred) {
    const int bx = W * (b % nred_w) + (int)(threadIdx.x >> 6);
    if (bx < nred_x)
      becp_reduce_body(d, active, gvec, gcnt, maxper, tiles, nchunk, part, becp, bx,
                       (b / nred_w) % ngroup, b / (nred_w * ngroup), threadIdx.x & 63);
    return;
  }
  const int pb = b - nred;
  plane_split_body<N, MB, PL, W, C, RL>(d, T, group, active, S, pb % N, PL * (pb / N), nvec,
                                        reinterpret_cast<C *>(smem_d), relax, want, vlist);
}

// The whole application of one vector per block (pwblock.h)
template <int N>
__global__ __launch_bounds__(pwblock::threads(N)) void k_pw_block(
    PwDev d, const double2 *__restrict__ in, int64_t sin, double2 *__restrict__ out, int64_t sout,
    const double2 *__restrict__ sigma, const int32_t *__restrict__ active,
    const int32_t *__restrict__ group, pwblock::Layout l) {
  extern __shared__ double2 smem_d[];
  const int v = blockIdx.x;
  if (active && !active[v]) return;
  const double2 *x = in + v * sin;
  const int g = group ? group[v] : 0;
  for (int e = threadIdx.x; e < d.ld; e += pwblock::threads(N)) smem_d[l.x + e] = x[e];
  pwblock::load_tables<N>(d, g, smem_d, l);
  __syncthreads();
  double2 *o = out + v * sout;
  pwblock::apply<N>(d, g, sigma[v], smem_d, l,
                    [&](int e, double2 r) { o[e] = r; });
}

// planes per block and wavefronts per block of the split plane kernel where
// no other shape is tried (mixed-precision batches): one plane on one
// wavefront (on the 48 box the X stage in 1.5 rounds of 32 lane pairs, 13 KB
// of LDS).  FP64 batches take the autotuned shapes at the launch (three
// planes on two wavefronts first, then this).
template <int N> struct SplitShape {
  static constexpr int PL = 1;
  static constexpr int W = 1;
};

}  // namespace

// ---------------------------------------------------------------------------
// DenseOperator
// ---------------------------------------------------------------------------
DenseOperator::DenseOperator(const double2 *h_a, int64_t n_) : a_(n_ * n_) {
  n = n_;
  ld = n_;
  a_.upload(h_a, n_ * n_);
  SGW_HIP(hipDeviceSynchronize());
}

void DenseOperator::apply(hipStream_t st, int nvec, const double2 *in, int64_t in_stride,
                          double2 *out, int64_t out_stride, const double2 *d_sigma,
                          const double2 *, const int32_t *d_active, const int32_t *,
                          const int32_t *) {
  dim3 grid((unsigned)((ld + kBlock - 1) / kBlock), nvec);
  {
    KScope ks("happly", st);
    k_dense<<<grid, kBlock, 0, st>>>(n, a_.p, in, in_stride, out, out_stride, ld, d_sigma,
                                     d_active);
  }
  SGW_HIP(hipGetLastError());
}

// ---------------------------------------------------------------------------
// CallbackOperator
// ---------------------------------------------------------------------------
void CallbackOperator::apply(hipStream_t st, int nvec, const double2 *in, int64_t in_stride,
                             double2 *out, int64_t out_stride, const double2 *,
                             const double2 *h_sigma, const int32_t *, const int32_t *h_active,
                             const int32_t *) {
  hx_.resize(n);
  hax_.resize(n);
  SGW_HIP(hipStreamSynchronize(st));
  for (int v = 0; v < nvec; ++v) {
    if (h_active && !h_active[v]) continue;
    SGW_HIP(hipMemcpy(hx_.data(), in + v * in_stride, sizeof(double2) * n, hipMemcpyDeviceToHost));
    fn_(&h_sigma[v], hx_.data(), hax_.data(), n, ctx_);
    SGW_HIP(hipMemcpy(out + v * out_stride, hax_.data(), sizeof(double2) * n,
                      hipMemcpyHostToDevice));
  }
}

// ---------------------------------------------------------------------------
// PwOperator
// ---------------------------------------------------------------------------
static std::vector<double2> twiddles(int n) {
  std::vector<double2> w(n);
  for (int k = 0; k < n; ++k) {
    double ang = 2.0 * M_PI * (double)k / n;
    w[k] = mk(std::cos(ang), std::sin(ang));
  }
  return w;
}

static inline int modn(int a, int n) { return ((a % n) + n) % n; }

// does every column (m1, m2) of every group hold a run of m3 without gaps?
static bool whole_columns(const PwDesc &desc, int M1, int M2) {
  const int nc2 = 2 * M2 + 1;
  std::vector<int32_t> lo, hi, cnt;
  for (int g = 0; g < desc.ngroup; ++g) {
    lo.assign((size_t)(2 * M1 + 1) * nc2, INT32_MAX);
    hi.assign(lo.size(), INT32_MIN);
    cnt.assign(lo.size(), 0);
    for (int i = 0; i < desc.npw[g]; ++i) {
      const int32_t *m = desc.mill + ((int64_t)g * desc.ld + i) * 3;
      const size_t c = (size_t)(m[0] + M1) * nc2 + (m[1] + M2);
      lo[c] = std::min(lo[c], m[2]);
      hi[c] = std::max(hi[c], m[2]);
      ++cnt[c];
    }
    for (size_t c = 0; c < cnt.size(); ++c)
      if (cnt[c] > 0 && hi[c] - lo[c] + 1 != cnt[c]) return false;
  }
  return true;
}

PwOperator::PwOperator(const PwDesc &desc) {
  n1_ = desc.n1; n2_ = desc.n2; n3_ = desc.n3;
  if (const char *f = std::getenv("SGW_PW_FUSE")) fuse_stages_ = std::strcmp(f, "0") != 0;
  if (const char *f = std::getenv("SGW_PW_PAIR")) pair_planes_ = std::strcmp(f, "0") != 0;
  if (const char *f = std::getenv("SGW_PW_SPLIT")) split_planes_ = std::strcmp(f, "0") != 0;
  if (const char *f = std::getenv("SGW_PW_BAND")) band_planes_ = std::strcmp(f, "0") != 0;
  SGW_REQUIRE(n1_ > 0 && n2_ > 0 && n3_ > 0 && n1_ <= 512 && n2_ <= 512 && n3_ <= 512, SGW_E_ARG,
              "pw operator: FFT box dimensions must be in [1, 512]");
  ngroup_ = desc.ngroup;
  SGW_REQUIRE(ngroup_ >= 1, SGW_E_ARG, "pw operator: need at least one group");
  ld = desc.ld;
  nproj_ = desc.nproj;
  SGW_REQUIRE(nproj_ >= 0 && nproj_ <= 4096, SGW_E_ARG, "pw operator: nproj out of range");
  npw_.assign(desc.npw, desc.npw + ngroup_);
  int M1 = 0, M2 = 0, M3 = 0;
  for (int g = 0; g < ngroup_; ++g) {
    SGW_REQUIRE(npw_[g] >= 1 && npw_[g] <= ld, SGW_E_SHAPE, "pw operator: npw must be in [1, ld]");
    for (int i = 0; i < npw_[g]; ++i) {
      const int32_t *m = desc.mill + ((int64_t)g * ld + i) * 3;
      M1 = std::max(M1, std::abs(m[0]));
      M2 = std::max(M2, std::abs(m[1]));
      M3 = std::max(M3, std::abs(m[2]));
    }
  }
  SGW_REQUIRE(2 * M1 + 1 <= n1_ && 2 * M2 + 1 <= n2_ && 2 * M3 + 1 <= n3_, SGW_E_SHAPE,
              "pw operator: the plane-wave sphere does not fit in the FFT box");
  n = npw_[0];
  box_cols_ = (int64_t)(2 * M1 + 1) * (2 * M2 + 1);
  const int M = std::max(M1, std::max(M2, M3));
  if (n1_ == n2_ && n2_ == n3_ && band_planes_ && split_planes_ && fuse_stages_ &&
      M >= kBandMin && M <= band_max(n1_) && whole_columns(desc, M1, M2)) {
    // the transforms specialised to a half-width take one for all axes, and a
    // k+q shift often leaves the three one apart; the rows this adds hold no
    // columns, and the packed layout that these transforms use has no places
    // for them.  512 vectors of the 48^3 box at half-widths (9, 8, 9): 254 us
    // against 319 without, at (7, 6, 7) 210 against 292
    M1 = M2 = M3 = M;
  }
  M1_ = M1; M2_ = M2; M3_ = M3;
  nc1_ = 2 * M1 + 1; nc2_ = 2 * M2 + 1;
  nslot_ = nc1_ * nc2_;
  // column tables
  std::vector<int32_t> col_start((size_t)ngroup_ * nslot_, 0), col_cnt((size_t)ngroup_ * nslot_, 0);
  std::vector<int32_t> sidx((size_t)ngroup_ * ld, 0), sm3((size_t)ngroup_ * ld, 0);
  std::vector<int32_t> slot_of((size_t)ngroup_ * ld, 0), m3_of((size_t)ngroup_ * ld, 0);
  std::vector<int32_t> col_lo((size_t)ngroup_ * nslot_, 0);
  for (int g = 0; g < ngroup_; ++g) {
    std::vector<std::pair<int64_t, int>> key(npw_[g]);
    std::map<int64_t, int> seen;
    for (int i = 0; i < npw_[g]; ++i) {
      const int32_t *m = desc.mill + ((int64_t)g * ld + i) * 3;
      int slot = (m[0] + M1) * nc2_ + (m[1] + M2);
      key[i] = {(int64_t)slot * 4096 + (m[2] + 2048), i};
      SGW_REQUIRE(seen.emplace(key[i].first, i).second, SGW_E_ARG,
                  "pw operator: duplicate Miller index in a sphere");
      slot_of[(size_t)g * ld + i] = slot;
      m3_of[(size_t)g * ld + i] = modn(m[2], n3_);
    }
    std::sort(key.begin(), key.end());
    for (int j = 0; j < npw_[g]; ++j) {
      int i = key[j].second;
      int slot = slot_of[(size_t)g * ld + i];
      const int m3raw = desc.mill[((int64_t)g * ld + i) * 3 + 2];
      if (col_cnt[(size_t)g * nslot_ + slot] == 0) {
        col_start[(size_t)g * nslot_ + slot] = j;
        col_lo[(size_t)g * nslot_ + slot] = m3raw;
      } else if (m3raw != col_lo[(size_t)g * nslot_ + slot] + col_cnt[(size_t)g * nslot_ + slot]) {
        columns_contiguous_ = false;  // a column with a gap in m3: no z-FFT kernels
      }
      col_cnt[(size_t)g * nslot_ + slot]++;
      sidx[(size_t)g * ld + j] = i;
      sm3[(size_t)g * ld + j] = m3_of[(size_t)g * ld + i];
    }
  }
  {
    // packed column layout: per group, row a of the grid from its first to
    // its last column with plane waves (a row of a sphere's columns is one
    // run, so the packed planes hold exactly the sphere's columns; a gap
    // would be kept, as zeros)
    const int nr = nc1_ + 1;
    std::vector<int32_t> rs((size_t)ngroup_ * nr, 0), rl((size_t)ngroup_ * nc1_, 0),
        rc((size_t)ngroup_ * nc1_, 0);
    int ncs = 1;
    for (int g = 0; g < ngroup_; ++g) {
      int j = 0;
      for (int a = 0; a < nc1_; ++a) {
        int lo = nc2_, hi = -1;
        for (int b = 0; b < nc2_; ++b)
          if (col_cnt[(size_t)g * nslot_ + a * nc2_ + b] > 0) {
            lo = std::min(lo, b);
            hi = std::max(hi, b);
          }
        rs[(size_t)g * nr + a] = j;
        if (hi >= lo) {
          rl[(size_t)g * nc1_ + a] = lo - M2_;
          rc[(size_t)g * nc1_ + a] = hi - lo + 1;
          j += hi - lo + 1;
        }
      }
      rs[(size_t)g * nr + nc1_] = j;
      ncs = std::max(ncs, j);
    }
    ncs_ = ncs;
    // (slot, count, start, lowest m3) of every packed column, (-1, 0, 0, 0)
    // past a group's columns
    auto info = [&](int g, int c) {
      const size_t i = (size_t)g * nslot_ + c;
      return make_int4(c, col_cnt[i], col_start[i], col_lo[i]);
    };
    std::vector<int4> cs((size_t)ngroup_ * ncs_, make_int4(-1, 0, 0, 0));
    for (int g = 0; g < ngroup_; ++g)
      for (int a = 0; a < nc1_; ++a)
        for (int k = 0; k < rc[(size_t)g * nc1_ + a]; ++k)
          cs[(size_t)g * ncs_ + rs[(size_t)g * nr + a] + k] =
              info(g, a * nc2_ + rl[(size_t)g * nc1_ + a] + M2_ + k);
    pk_info_.alloc(cs.size()); pk_info_.upload(cs.data(), cs.size());
    pk_row_start_.alloc(rs.size()); pk_row_start_.upload(rs.data(), rs.size());
    pk_row_lo_.alloc(rl.size()); pk_row_lo_.upload(rl.data(), rl.size());
    pk_row_cnt_.alloc(rc.size()); pk_row_cnt_.upload(rc.data(), rc.size());
    // the full grid in the same terms
    std::vector<int4> gs((size_t)ngroup_ * nslot_);
    std::vector<int32_t> grs((size_t)ngroup_ * nr), grl((size_t)ngroup_ * nc1_, -M2_),
        grc((size_t)ngroup_ * nc1_, nc2_);
    for (int g = 0; g < ngroup_; ++g) {
      for (int c = 0; c < nslot_; ++c) gs[(size_t)g * nslot_ + c] = info(g, c);
      for (int a = 0; a <= nc1_; ++a) grs[(size_t)g * nr + a] = a * nc2_;
    }
    gr_info_.alloc(gs.size()); gr_info_.upload(gs.data(), gs.size());
    gr_row_start_.alloc(grs.size()); gr_row_start_.upload(grs.data(), grs.size());
    gr_row_lo_.alloc(grl.size()); gr_row_lo_.upload(grl.data(), grl.size());
    gr_row_cnt_.alloc(grc.size()); gr_row_cnt_.upload(grc.data(), grc.size());
  }
  const int64_t nbox = (int64_t)n1_ * n2_ * n3_;
  vloc_.alloc(nbox); vloc_.upload(desc.vloc, nbox);
  {  // [z][x][y] copy for the x stage of the plane kernels
    std::vector<double> t((size_t)nbox);
    for (int z = 0; z < n3_; ++z)
      for (int y = 0; y < n2_; ++y)
        for (int x = 0; x < n1_; ++x)
          t[((size_t)z * n1_ + x) * n2_ + y] = desc.vloc[((size_t)z * n2_ + y) * n1_ + x];
    vloc_zxy_.alloc(nbox);
    vloc_zxy_.upload(t.data(), nbox);
  }
  d_npw_.alloc(ngroup_); d_npw_.upload(npw_.data(), ngroup_);
  col_start_.alloc(col_start.size()); col_start_.upload(col_start.data(), col_start.size());
  col_cnt_.alloc(col_cnt.size()); col_cnt_.upload(col_cnt.data(), col_cnt.size());
  sidx_.alloc(sidx.size()); sidx_.upload(sidx.data(), sidx.size());
  sm3_.alloc(sm3.size()); sm3_.upload(sm3.data(), sm3.size());
  slot_of_.alloc(slot_of.size()); slot_of_.upload(slot_of.data(), slot_of.size());
  m3_of_.alloc(m3_of.size()); m3_of_.upload(m3_of.data(), m3_of.size());
  col_lo_.alloc(col_lo.size()); col_lo_.upload(col_lo.data(), col_lo.size());
  kin_.alloc((size_t)ngroup_ * ld); kin_.upload(desc.kin, (size_t)ngroup_ * ld);
  if (nproj_ > 0) {
    proj_.alloc((size_t)ngroup_ * nproj_ * ld);
    proj_.upload(desc.proj, (size_t)ngroup_ * nproj_ * ld);
    dcoef_.alloc((size_t)ngroup_ * nproj_);
    dcoef_.upload(desc.dcoef, (size_t)ngroup_ * nproj_);
  }
  auto t1 = twiddles(n1_), t2 = twiddles(n2_), t3 = twiddles(n3_);
  tw_.alloc(n1_ + n2_ + n3_);
  tw_.upload(t1.data(), n1_);
  SGW_HIP(hipMemcpy(tw_.p + n1_, t2.data(), sizeof(double2) * n2_, hipMemcpyHostToDevice));
  SGW_HIP(hipMemcpy(tw_.p + n1_ + n2_, t3.data(), sizeof(double2) * n3_, hipMemcpyHostToDevice));
  // The whole operator in one block where all planes of the box fit a CU's LDS
  // at once (24^3 up to some 11 Ha).  1 vector, then 512: 28.4 and 45 us an
  // application against 32.9 and 67 (6 Ha), 29.7 and 48 against 32.1 and 64
  // (10 Ha).  Planes in two groups take 33.9 us against 33.2 (12 Ha), in three
  // 39.8 against 33.4 (20 Ha); the 32^3 box 41 to 46 against 34, the 36^3 box
  // 66 to 86 against 38.  The number of vectors has no part in the rule, so that
  // a vector's result does not depend on its batch.
  // A block reads the projectors for its vector alone, the batched kernels
  // once for 16: with more than 24 K values of them (plane waves x projectors) a
  // large batch is the slower for it.  1024 vectors, an application against
  // batched: 9 K values 94 us against 99, 19 K 115 and 114, 21 K 113 and 112; 38 K
  // 157 against 134, 45 K 144 against 131, 90 K 212 against 178 (1 vector: 56
  // against 50).
  constexpr int64_t kBlockProj = 24 * 1024;
  block_ = n1_ == 24 && n2_ == 24 && n3_ == 24 && columns_contiguous_ && fuse_stages_ &&
           split_planes_ && band_planes_ && nproj_ * ld <= kBlockProj &&
           pwblock::layout(n1_, nc1_, ncs_, ld, nproj_).total * sizeof(double2) <= pwblock::kLds;
  SGW_HIP(hipDeviceSynchronize());
}

int64_t PwOperator::group_n(int g) const { return npw_.at(g); }


void PwOperator::ensure_scratch(int nvec) {
  if (vlist_.n < (size_t)nvec) vlist_.alloc(nvec);
  size_t need = (size_t)nvec * nslot_ * n3_;
  if (S_.n < need) S_.alloc(need);
  if (T_.n < need) T_.alloc(need);
  if (loc_.n < (size_t)nvec * ld) loc_.alloc((size_t)nvec * ld);
}

void PwOperator::apply(hipStream_t st, int nvec, const double2 *in, int64_t in_stride,
                       double2 *out, int64_t out_stride, const double2 *d_sigma, const double2 *,
                       const int32_t *d_active, const int32_t *, const int32_t *d_group) {
  if (nvec <= 0) return;
  SGW_REQUIRE(d_group != nullptr || ngroup_ == 1, SGW_E_ARG,
              "pw operator: a group index per vector is required with several groups");
  SGW_REQUIRE(plan_nvec_ == nvec, SGW_E_STATE,
              "pw operator: prepare() was not called for this batch of vectors");
  ensure_scratch(nvec);
  PwWork w{T_.p,       S_.p,      loc_.p,    part_.p,      becp_.p,
           plan_vec_.p, plan_cnt_.p, plan_max_, plan_tiles_, vlist_.p};
  apply_work(st, nvec, in, in_stride, out, out_stride, d_sigma, d_active, d_group, w);
}

void PwOperator::apply_work(hipStream_t st, int nvec, const double2 *in, int64_t in_stride,
                            double2 *out, int64_t out_stride, const double2 *d_sigma,
                            const int32_t *d_active, const int32_t *d_group, const PwWork &wk) {
  KScope whole("happly", st);
  PwDev d;
  d.n1 = n1_; d.n2 = n2_; d.n3 = n3_;
  d.M1 = M1_; d.M2 = M2_; d.nc1 = nc1_; d.nc2 = nc2_; d.nslot = nslot_;
  d.ld = ld; d.nproj = nproj_;
  d.vloc = vloc_.p; d.vloc_zxy = vloc_zxy_.p; d.npw = d_npw_.p;
  d.col_start = col_start_.p; d.col_cnt = col_cnt_.p;
  d.sorted_idx = sidx_.p; d.sorted_m3 = sm3_.p; d.slot_of = slot_of_.p; d.m3_of = m3_of_.p;
  d.col_lo = col_lo_.p;
  d.ncs = nslot_; d.col_info = gr_info_.p;
  d.row_start = gr_row_start_.p; d.row_lo = gr_row_lo_.p; d.row_cnt = gr_row_cnt_.p;
  d.kin = kin_.p; d.proj = proj_.p; d.dcoef = dcoef_.p;
  d.tw1 = tw_.p; d.tw2 = tw_.p + n1_; d.tw3 = tw_.p + n1_ + n2_;
  d.inv_nbox = 1.0 / ((double)n1_ * n2_ * n3_);
  const bool cubic = n1_ == n2_ && n2_ == n3_ && columns_contiguous_;
  const size_t lds_fft = sizeof(double2) * (nslot_ + (size_t)nc1_ * n1_);
  const dim3 gcol((unsigned)((nslot_ + 63) / 64), nvec);
  if (block_ && fft_mode_ == 0) {
    d.ncs = ncs_; d.col_info = pk_info_.p;
    d.row_start = pk_row_start_.p; d.row_lo = pk_row_lo_.p; d.row_cnt = pk_row_cnt_.p;
    const pwblock::Layout l = pwblock::layout(n1_, nc1_, ncs_, ld, nproj_);
    const size_t lds = sizeof(double2) * (size_t)l.total;
    KScope ks("pw_block", st, 2);
    constexpr int NB = 24;
    SGW_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(k_pw_block<NB>),
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    k_pw_block<NB><<<nvec, pwblock::threads(NB), lds, st>>>(d, in, in_stride, out, out_stride,
                                                            d_sigma, d_active, d_group, l);
    SGW_HIP(hipGetLastError());
    return;
  }
  const double2 *locv = nullptr;
  const int nchunk = (int)((ld + kChunk - 1) / kChunk);
  const int nred_x = (nproj_ * kVT + 63) / 64;
  // FP32 (fft_mode_ 1, or 2 per vector) takes the fused split kernels where
  // the split plane kernel applies, the separate ones otherwise
  const bool split_plane_ok = split_planes_ && n1_ <= 48 && nc1_ <= 32 &&
                              sizeof(double2) * (size_t)nc1_ * (n1_ + 1) <= 64 * 1024;
  const bool fused = fuse_stages_ && cubic &&
                     (n1_ == 24 || n1_ == 32 || n1_ == 36 || n1_ == 48 || n1_ == 64) &&
                     (fft_mode_ == 0 || split_plane_ok);
  if (nproj_ > 0 && !fused) {
    // projector contraction becp = D proj^H x (a concurrent stream for it was
    // measured: no gain, the plane kernel already fills the device)
    KScope ks("pw_becp", st, 2);
    k_pw_becp<<<dim3(nchunk, ngroup_, wk.plan_tiles), 256, 0, st>>>(
        d, in, in_stride, d_active, wk.plan_vec, wk.plan_cnt, wk.plan_max, wk.plan_tiles, nchunk,
        wk.part);
    k_pw_becp_reduce<<<dim3((unsigned)nred_x, ngroup_, wk.plan_tiles), 64, 0, st>>>(
        d, d_active, wk.plan_vec, wk.plan_cnt, wk.plan_max, wk.plan_tiles, nchunk, wk.part, wk.becp);
    SGW_HIP(hipGetLastError());
  }
  auto launch_fft = [&](auto tag) {
    constexpr int NB = decltype(tag)::value;
    if (fused) {
      // no projectors: the part counts are zero and only the transforms run
      const int tiles = nproj_ > 0 ? wk.plan_tiles : 0;
      // Few chunks and tiles leave the chip idle behind each block's stages: 16
      // projectors to a block then, in one stage.  48^3 (48 projectors, 26
      // chunks of 64 plane waves): 16 vectors 7.0 us against 9.6, 64 vectors
      // 10.4 against 13.6, 128 vectors (624 blocks) 16.3 against 13.3; 36^3 (26
      // projectors, 10 chunks): 256 vectors 9.8 against 12.8.
      const int64_t nsum = (int64_t)nchunk * ngroup_ * tiles;
      const int nsplit = (nproj_ + 15) / 16;
      const int psplit = nsum * nsplit <= 512 ? std::max(nsplit, 1) : 1;
      const int64_t nbecp = nsum * psplit;
      // fft_mode_: 0 FP64, 1 FP32, 2 per vector from the relax flags.  With
      // both precisions the FP64 instances carry the projector sums and the
      // FP32 ones (tiles 0) the transforms of the relaxed vectors only.  The
      // FP64 instances read the flags only in mode 2 (template RL), so mode 0
      // runs the code it runs without an FP32 path.
      const int32_t *rl = fft_mode_ == 2 ? relax_ : nullptr;
      auto with_rl = [&](auto &&f) {
        if (rl) f(std::true_type{});
        else f(std::false_type{});
      };
      const bool run64 = fft_mode_ != 1, run32 = fft_mode_ != 0;
      const int tiles32 = run64 ? 0 : tiles;
      const int64_t nbecp32 = (int64_t)nchunk * ngroup_ * tiles32 * psplit;
      float2 *T32 = reinterpret_cast<float2 *>(wk.T), *S32 = reinterpret_cast<float2 *>(wk.S);
      // z transforms split over lane pairs: 32 columns per 64 lanes
      const bool zsplit = split_planes_;
      // T and S in the packed column layout where the split plane kernel
      // runs (it and the split z transforms are their only readers and
      // writers here); the full grid for the other plane kernels
      const bool packed = zsplit && split_plane_ok;
      // the split plane kernel's blocks take the running vectors from a list
      // (built by the z inverse launch), so that a batch with few running
      // vectors launches no blocks with dead planes among live ones
      int32_t *vl = (packed && d_active && wk.vlist) ? wk.vlist : nullptr;
      if (packed) {
        d.ncs = ncs_; d.col_info = pk_info_.p;
        d.row_start = pk_row_start_.p; d.row_lo = pk_row_lo_.p; d.row_cnt = pk_row_cnt_.p;
      }
      const int64_t gxz = zsplit ? (d.ncs + 31) / 32 : (int64_t)gcol.x;
      const int64_t nzinv = (gxz * nvec + 3) / 4;
      const int64_t nred = (int64_t)nred_x * ngroup_ * tiles;
      SGW_REQUIRE(nbecp + nzinv < INT32_MAX && nred + (int64_t)NB * nvec < INT32_MAX, SGW_E_ARG,
                  "pw operator: too many vectors for one launch");
      {
        KScope ks("pw_becp_zinv", st, 2);
        if (zsplit)
          with_band<NB>(band_planes_, M3_, [&](auto mb) {
            // the first launch's extra block (block 0) lists the running vectors
            int32_t *vl64 = run64 ? vl : nullptr, *vl32 = run64 ? nullptr : vl;
            if (run64)
              with_rl([&](auto rlt) {
                k_pw_becp_zinv<NB, true, decltype(mb)::value, double2, decltype(rlt)::value>
                    <<<(unsigned)(nbecp + nzinv + (vl64 ? 1 : 0)), 256, 0, st>>>(
                        d, in, in_stride, d_group, d_active, wk.plan_vec, wk.plan_cnt,
                        wk.plan_max, tiles, nchunk, ngroup_, psplit, wk.part, wk.T, nvec, rl, 0, vl64);
              });
            if (run32)
              k_pw_becp_zinv<NB, true, decltype(mb)::value, float2, true>
                  <<<(unsigned)(nbecp32 + nzinv + (vl32 ? 1 : 0)), 256, 0, st>>>(
                      d, in, in_stride, d_group, d_active, wk.plan_vec, wk.plan_cnt, wk.plan_max,
                      tiles32, nchunk, ngroup_, psplit, wk.part, T32, nvec, rl, 1, vl32);
          });
        else
          k_pw_becp_zinv<NB, false, -1><<<(unsigned)(nbecp + nzinv), 256, 0, st>>>(
              d, in, in_stride, d_group, d_active, wk.plan_vec, wk.plan_cnt, wk.plan_max, tiles,
              nchunk, ngroup_, psplit, wk.part, wk.T, nvec);
      }
      {
        KScope ks("pw_reduce_plane", st, 2);
        // the transforms split over lane pairs (N <= 48); else, without the
        // split, two vectors per plane block while both Y stages fit in one
        // wavefront and four such blocks still fit in a CU's LDS (N = 64
        // would spill)
        bool paired = false;
        if constexpr (NB <= 48) {
          // split transforms over lane pairs (LDS: P of the block's planes only)
          constexpr int PL = SplitShape<NB>::PL, W = SplitShape<NB>::W;
          const size_t lds_split = sizeof(double2) * PL * (size_t)nc1_ * (NB + 1);
          auto launch_split = [&](auto shape, auto mb, auto rlt) {
            constexpr int pl = decltype(shape)::value / 8, w = decltype(shape)::value % 8;
            const int64_t nred_s = (int64_t)((nred_x + w - 1) / w) * ngroup_ * tiles;
            k_pw_reduce_split<NB, decltype(mb)::value, pl, w, double2, decltype(rlt)::value>
                <<<(unsigned)(nred_s + (int64_t)NB * ((nvec + pl - 1) / pl)), 64 * w,
                   sizeof(double2) * pl * (size_t)nc1_ * (NB + 1), st>>>(
                    d, d_group, d_active, wk.plan_vec, wk.plan_cnt, wk.plan_max, tiles, nchunk,
                    ngroup_, nred_x, wk.part, wk.becp, wk.T, wk.S, nvec, rl, 0, vl);
          };
          // the relaxed vectors' FP32 plane transforms, one plane per wavefront
          auto launch_split32 = [&](auto mb) {
            const int64_t nred_s = (int64_t)nred_x * ngroup_ * tiles32;
            k_pw_reduce_split<NB, decltype(mb)::value, 1, 1, float2, true>
                <<<(unsigned)(nred_s + (int64_t)NB * nvec), 64,
                   sizeof(float2) * (size_t)nc1_ * (NB + 1), st>>>(
                    d, d_group, d_active, wk.plan_vec, wk.plan_cnt, wk.plan_max, tiles32, nchunk,
                    ngroup_, nred_x, wk.part, wk.becp, T32, S32, nvec, rl, 1, vl);
          };
          const bool band = band_planes_ && M1_ == M2_;
          static_assert(PL == 1 && W == 1,
                        "split_plane_ok is the default shape's fit test for one plane per wave");
          if (packed) {  // split_planes_, nc1_ <= 32 and lds_split <= 64 KB
            SGW_REQUIRE(lds_split <= 64 * 1024 && PL * nc1_ <= 32 * W, SGW_E_STATE,
                        "pw operator: split plane kernel does not fit");
            // compile-time sphere half-widths for the usual ones of this box;
            // the autotuner picks among three planes on two wavefronts (on
            // the 48 box: Y stage on 51 of 64 lane pairs, X stage in 2.25
            // rounds), one plane on one, one plane on two (the X stage in one
            // round) and two planes on two for this box and size class of the
            // batch (mode 2: one plane on one)
            with_band<NB>(band, M1_, [&](auto mb) {
              using I11 = std::integral_constant<int, PL * 8 + W>;
              constexpr std::false_type no_rl{};
              if (!run64) return;
              if (rl) {
                launch_split(I11{}, mb, std::true_type{});
                return;
              }
              {
                const size_t row = sizeof(double2) * (size_t)nc1_ * (NB + 1);
                const bool fit2 = nc1_ <= 32 && 2 * row <= 64 * 1024;
                const bool fit3 = fit2 && 3 * nc1_ <= 64 && 3 * row <= 64 * 1024;
                const int ncand = fit2 ? (fit3 ? 4 : 3) : 1;
                const std::string key = "plane" + std::to_string(NB) + "/M" +
                                        std::to_string(M1_) + "/b" +
                                        std::to_string((int)decltype(mb)::value) + "/n" +
                                        std::to_string(size_class(nvec));
                // shapes (planes, wavefronts): (3, 2) first where it fits (the
                // streamed 48^3 solve: 365.8k solves/s against 359.2k with
                // (1, 1)), then (1, 1), (1, 2), (2, 2)
                autotune(key, ncand, st, [&](int c) {
                  const int k = fit3 ? c : c + 1;
                  if (k == 0) launch_split(std::integral_constant<int, 3 * 8 + 2>{}, mb, no_rl);
                  else if (k == 1) launch_split(I11{}, mb, no_rl);
                  else if (k == 2)
                    launch_split(std::integral_constant<int, 1 * 8 + 2>{}, mb, no_rl);
                  else launch_split(std::integral_constant<int, 2 * 8 + 2>{}, mb, no_rl);
                });
              }
            });
            if (run32) with_band<NB>(band, M1_, [&](auto mb) { launch_split32(mb); });
            paired = true;
          } else if (pair_planes_ && 2 * nc1_ <= 64 && 2 * lds_fft <= 40 * 1024) {
            k_pw_reduce_plane<NB, true>
                <<<(unsigned)(nred + (int64_t)NB * ((nvec + 1) / 2)), 64, 2 * lds_fft, st>>>(
                    d, d_group, d_active, wk.plan_vec, wk.plan_cnt, wk.plan_max, tiles, nchunk,
                    ngroup_, nred_x, wk.part, wk.becp, wk.T, wk.S, nvec);
            paired = true;
          }
        }
        if (!paired) {
          k_pw_reduce_plane<NB, false><<<(unsigned)(nred + (int64_t)NB * nvec), 64, lds_fft, st>>>(
              d, d_group, d_active, wk.plan_vec, wk.plan_cnt, wk.plan_max, tiles, nchunk, ngroup_,
              nred_x, wk.part, wk.becp, wk.T, wk.S, nvec);
        }
      }
      {
        KScope ks("pw_zfwd", st, 2);
        if (zsplit)
          with_band<NB>(band_planes_, M3_, [&](auto mb) {
            if (run64)
              with_rl([&](auto rlt) {
                k_pw_zfwd_split<NB, decltype(mb)::value, double2, decltype(rlt)::value>
                    <<<dim3((unsigned)gxz, nvec), 64, 0, st>>>(d, wk.S, d_group, d_active,
                                                               wk.loc, rl, 0);
              });
            if (run32)
              k_pw_zfwd_split<NB, decltype(mb)::value, float2, true>
                  <<<dim3((unsigned)gxz, nvec), 64, 0, st>>>(d, S32, d_group, d_active, wk.loc,
                                                             rl, 1);
          });
        else
          k_pw_zfwd<NB><<<gcol, 64, 0, st>>>(d, wk.S, d_group, d_active, wk.loc, nullptr, 0);
      }
      locv = wk.loc;
      return;
    }
    // fft_mode_: 0 FP64, 1 FP32, 2 per vector from the relax flags
    const int32_t *rl = fft_mode_ == 2 ? relax_ : nullptr;
    float2 *T32 = reinterpret_cast<float2 *>(wk.T), *S32 = reinterpret_cast<float2 *>(wk.S);
    const bool run64 = fft_mode_ != 1, run32 = fft_mode_ != 0;
    {
      KScope ks("pw_zinv", st, 2);
      if (run64) k_pw_zinv<NB><<<gcol, 64, 0, st>>>(d, in, in_stride, d_group, d_active, wk.T, rl, 0);
      if (run32)
        k_pw_zinv<NB, float2><<<gcol, 64, 0, st>>>(d, in, in_stride, d_group, d_active, T32, rl, 1);
    }
    {
      KScope ks("pw_plane", st, 2);
      if (run64)
        k_pw_plane_fft<NB><<<dim3(NB, nvec), 64, lds_fft, st>>>(d, wk.T, d_group, d_active,
                                                                 wk.S, rl, 0);
      if (run32)
        k_pw_plane_fft<NB, float2><<<dim3(NB, nvec), 64, lds_fft / 2, st>>>(
            d, T32, d_group, d_active, S32, rl, 1);
    }
    {
      KScope ks("pw_zfwd", st, 2);
      if (run64) k_pw_zfwd<NB><<<gcol, 64, 0, st>>>(d, wk.S, d_group, d_active, wk.loc, rl, 0);
      if (run32)
        k_pw_zfwd<NB, float2><<<gcol, 64, 0, st>>>(d, S32, d_group, d_active, wk.loc, rl, 1);
    }
    locv = wk.loc;
  };
  if (cubic && n1_ == 24) {
    launch_fft(std::integral_constant<int, 24>{});
  } else if (cubic && n1_ == 32) {
    launch_fft(std::integral_constant<int, 32>{});
  } else if (cubic && n1_ == 36) {
    launch_fft(std::integral_constant<int, 36>{});
  } else if (cubic && n1_ == 48) {
    launch_fft(std::integral_constant<int, 48>{});
  } else if (cubic && n1_ == 64) {
    launch_fft(std::integral_constant<int, 64>{});
  } else {
    size_t lds_plane =
        sizeof(double2) * (n1_ + n2_ + nslot_ + (size_t)nc1_ * n2_ + (size_t)n2_ * n1_);
    SGW_REQUIRE(lds_plane <= 64 * 1024, SGW_E_ARG, "pw operator: FFT plane does not fit in LDS");
    KScope ks("pw_plane", st, 2);
    k_pw_plane<<<dim3(n3_, nvec), kBlock, lds_plane, st>>>(d, in, in_stride, d_group, d_active,
                                                          wk.S);
  }
  SGW_HIP(hipGetLastError());
  {
    const size_t lds_asm = sizeof(double2) * (size_t)nproj_ * kVT;
    KScope ks("pw_assemble", st, 2);
    // 64 plane waves x 4 vector groups, 32 x 8 or 16 x 16 to a block.  Wide
    // blocks read a projector value once for four vectors; narrow ones fill the
    // chip for a small batch and have fewer products in a row.  The widest with
    // kAsmBlocks blocks is the default: 48^3 (48 projectors, 26 chunks of 64) 512
    // vectors 21.0 / 23.9 / 28.8 us, 256 vectors 16.0 / 15.2 / 17.7, 64 vectors
    // 14.4 / 10.9 / 9.6 (8.7 with 16 values together), 16 vectors 12.6 / 9.1 / 7.8;
    // 36^3 (26 projectors, 10 chunks) 512 vectors 12.6 / 10.8 / 11.2, 256 vectors
    // 11.4 / 9.2 / 8.8.  The autotuner tries the others for each size class of
    // the batch (not when the output overwrites the input, which a second
    // launch would read)
    constexpr int NT = kAsmThreads;
    auto launch_asm = [&](auto chunk) {
      constexpr int CH = decltype(chunk)::value;
      k_pw_assemble2<CH, NT><<<dim3((unsigned)((ld + CH - 1) / CH), ngroup_, wk.plan_tiles), NT,
                               lds_asm, st>>>(d, in, in_stride, out, out_stride, d_sigma, d_active,
                                              wk.plan_vec, wk.plan_cnt, wk.plan_max,
                                              wk.plan_tiles, nchunk, wk.becp, wk.S, locv);
    };
    const int64_t per = (int64_t)ngroup_ * wk.plan_tiles;
    const int first = (ld + 63) / 64 * per >= kAsmBlocks   ? 0
                      : (ld + 31) / 32 * per >= kAsmBlocks ? 1
                                                           : 2;
    const bool disjoint = out + (int64_t)(nvec - 1) * out_stride + ld <= in ||
                          in + (int64_t)(nvec - 1) * in_stride + ld <= out;
    const std::string key = "assemble/n" + std::to_string(size_class(nvec)) + "/g" +
                            std::to_string(ngroup_) + "/p" + std::to_string(nproj_);
    autotune(
        key, disjoint ? 3 : 1, st,
        [&](int c) {
          if (c == 0) launch_asm(std::integral_constant<int, 64>{});
          else if (c == 1) launch_asm(std::integral_constant<int, 32>{});
          else launch_asm(std::integral_constant<int, 16>{});
        },
        first);
  }
  SGW_HIP(hipGetLastError());
}

void PwOperator::drho_accumulate(hipStream_t st, int group, int nbnd, int nshift,
                                 const double2 *dpsi, int64_t stride, const double2 *Pr,
                                 double wgt, double2 *D, bool accumulate) {
  const int nv = nbnd * nshift;
  if (nv <= 0) return;
  SGW_REQUIRE(group >= 0 && group < ngroup_, SGW_E_ARG, "pw operator: group index out of range");
  const bool cubic = n1_ == n2_ && n2_ == n3_ && columns_contiguous_;
  SGW_REQUIRE(cubic && (n1_ == 24 || n1_ == 32 || n1_ == 36 || n1_ == 48), SGW_E_ARG,
              "pw operator: the density response needs a cubic 24/32/36/48 box");
  const size_t lds = sizeof(double2) * (nslot_ + (size_t)nc1_ * n1_);
  SGW_REQUIRE(nshift < 65536, SGW_E_ARG, "pw operator: too many shifts");
  ensure_scratch(nv);
  std::vector<int32_t> hg(nv, group);
  DevBuf<int32_t> dg(nv);
  dg.upload(hg.data(), nv, st);
  PwDev d;
  d.n1 = n1_; d.n2 = n2_; d.n3 = n3_;
  d.M1 = M1_; d.M2 = M2_; d.nc1 = nc1_; d.nc2 = nc2_; d.nslot = nslot_;
  d.ld = ld; d.nproj = nproj_;
  d.vloc = vloc_.p; d.vloc_zxy = vloc_zxy_.p; d.npw = d_npw_.p;
  d.col_start = col_start_.p; d.col_cnt = col_cnt_.p;
  d.sorted_idx = sidx_.p; d.sorted_m3 = sm3_.p; d.slot_of = slot_of_.p; d.m3_of = m3_of_.p;
  d.col_lo = col_lo_.p;
  d.ncs = nslot_; d.col_info = gr_info_.p;
  d.row_start = gr_row_start_.p; d.row_lo = gr_row_lo_.p; d.row_cnt = gr_row_cnt_.p;
  d.kin = kin_.p; d.proj = proj_.p; d.dcoef = dcoef_.p;
  d.tw1 = tw_.p; d.tw2 = tw_.p + n1_; d.tw3 = tw_.p + n1_ + n2_;
  d.inv_nbox = 1.0 / ((double)n1_ * n2_ * n3_);
  const dim3 gcol((unsigned)((nslot_ + 63) / 64), nv);
  auto run = [&](auto tag) {
    constexpr int NB = decltype(tag)::value;
    k_pw_zinv<NB><<<gcol, 64, 0, st>>>(d, dpsi, stride, dg.p, nullptr, T_.p);
    if (split_planes_ && nc1_ <= 64) {
      // transforms split over lane pairs, D of a column in registers
      with_band<NB>(band_planes_ && M1_ == M2_, M1_, [&](auto mb) {
        k_pw_plane_drho_split<NB, decltype(mb)::value>
            <<<dim3(NB, nshift), 128, sizeof(double2) * (size_t)nc1_ * NB, st>>>(
                d, T_.p, nbnd, nshift, Pr, wgt, D, accumulate ? 1 : 0);
      });
    } else {
      k_pw_plane_drho<NB><<<dim3(NB, nshift), 64, lds, st>>>(d, T_.p, nbnd, nshift, Pr, wgt, D,
                                                             accumulate ? 1 : 0);
    }
  };
  switch (n1_) {
    case 24: run(std::integral_constant<int, 24>{}); break;
    case 32: run(std::integral_constant<int, 32>{}); break;
    case 36: run(std::integral_constant<int, 36>{}); break;
    default: run(std::integral_constant<int, 48>{}); break;
  }
  SGW_HIP(hipGetLastError());
  SGW_HIP(hipStreamSynchronize(st));  // dg is released on return
}

void PwOperator::grad_accumulate(hipStream_t st, int np, const double2 *x, const double2 *y,
                                 int64_t stride, const int32_t *d_group, const double *d_w,
                                 int nb, double *G, bool accumulate) {
  if (np <= 0) return;
  SGW_REQUIRE(d_group != nullptr || ngroup_ == 1, SGW_E_ARG,
              "pw operator: a group index per vector is required with several groups");
  const bool cubic = n1_ == n2_ && n2_ == n3_ && columns_contiguous_;
  SGW_REQUIRE(cubic && (n1_ == 24 || n1_ == 32 || n1_ == 36 || n1_ == 48), SGW_E_ARG,
              "pw operator: the V_loc gradient needs a cubic 24/32/36/48 box");
  SGW_REQUIRE(sizeof(double2) * (nslot_ + (size_t)nc1_ * n1_ + (size_t)n1_ * n1_) <= 64 * 1024,
              SGW_E_ARG, "pw operator: gradient plane does not fit in LDS");
  // the limit is that of a plane kept in LDS beside its rows; the kernel keeps
  // rows only, 18 to 55 KB at the largest spheres within it
  const size_t lds = sizeof(double2) * 2 * (size_t)nc1_ * (n1_ + 1);
  SGW_REQUIRE(nb >= 1 && nb < 65536, SGW_E_ARG, "pw operator: bad gradient partial count");
  ensure_scratch(np);
  PwDev d;
  d.n1 = n1_; d.n2 = n2_; d.n3 = n3_;
  d.M1 = M1_; d.M2 = M2_; d.nc1 = nc1_; d.nc2 = nc2_; d.nslot = nslot_;
  d.ld = ld; d.nproj = nproj_;
  d.vloc = vloc_.p; d.vloc_zxy = vloc_zxy_.p; d.npw = d_npw_.p;
  d.col_start = col_start_.p; d.col_cnt = col_cnt_.p;
  d.sorted_idx = sidx_.p; d.sorted_m3 = sm3_.p; d.slot_of = slot_of_.p; d.m3_of = m3_of_.p;
  d.col_lo = col_lo_.p;
  d.ncs = ncs_; d.col_info = pk_info_.p;
  d.row_start = pk_row_start_.p; d.row_lo = pk_row_lo_.p; d.row_cnt = pk_row_cnt_.p;
  d.kin = kin_.p; d.proj = proj_.p; d.dcoef = dcoef_.p;
  d.tw1 = tw_.p; d.tw2 = tw_.p + n1_; d.tw3 = tw_.p + n1_ + n2_;
  d.inv_nbox = 1.0 / ((double)n1_ * n2_ * n3_);
  const dim3 gcol((unsigned)((ncs_ + 31) / 32), np, 2);
  auto run = [&](auto tag) {
    constexpr int NB = decltype(tag)::value;
    with_band<NB>(band_planes_ && M1_ == M2_ && M1_ == M3_, M1_, [&](auto mb) {
      constexpr int MB = decltype(mb)::value;
      k_pw_zinv_pair<NB, MB><<<gcol, 64, 0, st>>>(d, x, y, stride, d_group, T_.p, S_.p);
      k_pw_plane_grad<NB, MB><<<dim3(NB, nb), 64 * grad_waves(NB), lds, st>>>(
          d, T_.p, S_.p, np, d_group, d_w, G, accumulate ? 1 : 0);
    });
  };
  switch (n1_) {
    case 24: run(std::integral_constant<int, 24>{}); break;
    case 32: run(std::integral_constant<int, 32>{}); break;
    case 36: run(std::integral_constant<int, 36>{}); break;
    default: run(std::integral_constant<int, 48>{}); break;
  }
  SGW_HIP(hipGetLastError());
}

void PwOperator::prepare(const int32_t *h_group, int nvec) {
  std::vector<int32_t> key(h_group ? h_group : nullptr, h_group ? h_group + nvec : nullptr);
  if (!h_group) key.assign(nvec, 0);
  if (plan_nvec_ == nvec && key == plan_key_) return;
  std::vector<std::vector<int32_t>> lists(ngroup_);
  for (int v = 0; v < nvec; ++v) {
    SGW_REQUIRE(key[v] >= 0 && key[v] < ngroup_, SGW_E_ARG, "pw operator: group index out of range");
    lists[key[v]].push_back(v);
  }
  int maxper = 1;
  for (auto &l : lists) maxper = std::max<int>(maxper, (int)l.size());
  std::vector<int32_t> vec((size_t)ngroup_ * maxper, 0), cnt(ngroup_);
  for (int g = 0; g < ngroup_; ++g) {
    cnt[g] = (int32_t)lists[g].size();
    std::copy(lists[g].begin(), lists[g].end(), vec.begin() + (size_t)g * maxper);
  }
  plan_vec_.alloc(vec.size());
  plan_vec_.upload(vec.data(), vec.size());
  plan_cnt_.alloc(cnt.size());
  plan_cnt_.upload(cnt.data(), cnt.size());
  plan_max_ = maxper;
  plan_tiles_ = (maxper + kVT - 1) / kVT;
  const int nchunk = (int)((ld + kChunk - 1) / kChunk);
  const size_t need = (size_t)ngroup_ * plan_tiles_ * nchunk * std::max(nproj_, 1) * kVT;
  if (part_.n < need) part_.alloc(need);
  const size_t needb = (size_t)ngroup_ * plan_tiles_ * std::max(nproj_, 1) * kVT;
  if (becp_.n < needb) becp_.alloc(needb);
  if (nproj_ == 0) becp_.zero();
  ensure_scratch(nvec);
  SGW_HIP(hipDeviceSynchronize());
  plan_key_ = std::move(key);
  plan_nvec_ = nvec;
}


// ---------------------------------------------------------------------------
// application without device allocation
// ---------------------------------------------------------------------------
namespace {

constexpr int kNoAllocMaxDevices = 64;
constexpr int kNoAllocMaxVec = 1024;
constexpr int kNoAllocMaxGroups = 256;
constexpr int kNoAllocMaxPlan = 16384;  // ngroup x (largest group's vector count)

std::mutex g_noalloc_mu;
void *g_noalloc_ptr[kNoAllocMaxDevices] = {};

// device address of `scratch` on the current device (looked up once per device)
unsigned char *noalloc_scratch() {
  int dev = 0;
  SGW_HIP(hipGetDevice(&dev));
  SGW_REQUIRE(dev >= 0 && dev < kNoAllocMaxDevices, SGW_E_ARG,
              "pw operator no-alloc: device index beyond the supported range");
  std::lock_guard<std::mutex> lock(g_noalloc_mu);
  if (!g_noalloc_ptr[dev]) {
    void *p = nullptr;
    SGW_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    SGW_REQUIRE(p != nullptr, SGW_E_STATE, "pw operator no-alloc: scratch symbol has no address");
    g_noalloc_ptr[dev] = p;
  }
  return static_cast<unsigned char *>(g_noalloc_ptr[dev]);
}

size_t align256(size_t b) { return (b + 255) & ~(size_t)255; }

}  // namespace

void PwOperator::apply_noalloc(hipStream_t st, int nvec, const int32_t *d_group,
                               const double2 *d_sigma, const double2 *in, int64_t ldx,
                               double2 *out) {
  SGW_REQUIRE(nvec >= 1 && nvec <= kNoAllocMaxVec, SGW_E_ARG,
              "pw operator no-alloc: nvec must be in [1, 1024]");
  SGW_REQUIRE(in && out && d_sigma, SGW_E_ARG, "pw operator no-alloc: null argument");
  SGW_REQUIRE(ldx >= ld, SGW_E_SHAPE, "pw operator no-alloc: ldx < operator ld");
  SGW_REQUIRE(d_group != nullptr || ngroup_ == 1, SGW_E_ARG,
              "pw operator no-alloc: a group index per vector is required with several groups");
  SGW_REQUIRE(ngroup_ <= kNoAllocMaxGroups, SGW_E_ARG,
              "pw operator no-alloc: more than 256 k+q groups");
  unsigned char *base = noalloc_scratch();
  // group of every vector; the wait also orders this call after earlier
  // work on the stream, which may still read the scratch array
  int32_t grp[kNoAllocMaxVec];
  if (d_group)
    SGW_HIP(hipMemcpyAsync(grp, d_group, sizeof(int32_t) * nvec, hipMemcpyDeviceToHost, st));
  SGW_HIP(hipStreamSynchronize(st));
  if (!d_group) std::fill(grp, grp + nvec, 0);
  // vectors of each group, in increasing order: plan[g * maxper + j]
  int32_t cnt[kNoAllocMaxGroups] = {};
  for (int v = 0; v < nvec; ++v) {
    SGW_REQUIRE(grp[v] >= 0 && grp[v] < ngroup_, SGW_E_ARG,
                "pw operator no-alloc: group index out of range");
    ++cnt[grp[v]];
  }
  int maxper = 1;
  for (int g = 0; g < ngroup_; ++g) maxper = std::max<int>(maxper, cnt[g]);
  SGW_REQUIRE((int64_t)ngroup_ * maxper + ngroup_ <= kNoAllocMaxPlan, SGW_E_SHAPE,
              "pw operator no-alloc: vector lists exceed 16384 entries (groups x largest group)");
  int32_t plan[kNoAllocMaxPlan];
  std::fill(plan, plan + (size_t)ngroup_ * maxper, 0);
  int32_t fill[kNoAllocMaxGroups] = {};
  for (int v = 0; v < nvec; ++v) plan[(size_t)grp[v] * maxper + fill[grp[v]]++] = v;
  std::copy(cnt, cnt + ngroup_, plan + (size_t)ngroup_ * maxper);
  // carve the work buffers
  const int tiles = (maxper + kVT - 1) / kVT;
  const int nchunk = (int)((ld + kChunk - 1) / kChunk);
  const size_t np = std::max(nproj_, 1);
  const size_t b_plan = align256(sizeof(int32_t) * ((size_t)ngroup_ * maxper + ngroup_));
  const size_t b_part = align256(sizeof(double2) * (size_t)ngroup_ * tiles * nchunk * np * kVT);
  const size_t b_becp = align256(sizeof(double2) * (size_t)ngroup_ * tiles * np * kVT);
  const size_t b_box = align256(sizeof(double2) * (size_t)nvec * box_cols_ * n3_);
  const size_t b_loc = align256(sizeof(double2) * (size_t)nvec * ld);
  const size_t b_vlist = align256(sizeof(int32_t) * (size_t)nvec);
  const size_t total = b_plan + b_part + b_becp + 2 * b_box + b_loc + b_vlist;
  SGW_REQUIRE(total <= (size_t)SGW_NOALLOC_SCRATCH_BYTES, SGW_E_SHAPE,
              "pw operator no-alloc: this batch needs " + std::to_string(total) +
                  " bytes of work space, more than the fixed " +
                  std::to_string((size_t)SGW_NOALLOC_SCRATCH_BYTES) +
                  "-byte scratch array; use fewer vectors per call");
  unsigned char *p = base;
  int32_t *d_plan = reinterpret_cast<int32_t *>(p);
  p += b_plan;
  PwWork w{};
  w.part = reinterpret_cast<double2 *>(p);
  p += b_part;
  w.becp = reinterpret_cast<double2 *>(p);
  p += b_becp;
  w.T = reinterpret_cast<double2 *>(p);
  p += b_box;
  w.S = reinterpret_cast<double2 *>(p);
  p += b_box;
  w.loc = reinterpret_cast<double2 *>(p);
  p += b_loc;
  w.vlist = reinterpret_cast<int32_t *>(p);
  w.plan_vec = d_plan;
  w.plan_cnt = d_plan + (size_t)ngroup_ * maxper;
  w.plan_max = maxper;
  w.plan_tiles = tiles;
  SGW_HIP(hipMemcpyAsync(d_plan, plan, sizeof(int32_t) * ((size_t)ngroup_ * maxper + ngroup_),
                         hipMemcpyHostToDevice, st));
  if (nproj_ == 0) SGW_HIP(hipMemsetAsync(w.becp, 0, b_becp, st));
  // the host lists above live on this stack frame: the copy must be done
  SGW_HIP(hipStreamSynchronize(st));
  apply_work(st, nvec, in, ldx, out, ldx, d_sigma, nullptr, d_group, w);
}

}  // namespace sgw
