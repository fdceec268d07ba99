// The reference form of the correlation self-energy on the device:
//  * analytic continuation of W (algo/analytic/src/analytic.f90:50-348) with
//    the Godby-Needs plasmon-pole model (godby_needs.f90) and the N-point
//    Pade approximant of Vidberg and Serene (pade.f90:41-147), one thread per
//    (G, G') element, and the robust Pade approximant (pade_robust.f90), one
//    group of 16 or 32 lanes per element;
//  * sigma_prod (phys/corr/src/sigma.f90:417-523): W(G, G') -> W(r, r') by
//    invfft6, the product G(r, r') W(r, r'), fwfft6 back, times alpha, and
//    optionally added into Sigma (sigma.f90:741).
#include <algorithm>
#include <cmath>
#include <vector>

#include "aaa.h"
#include "boxfft.h"
#include "fft6.h"
#include "ktimer.h"
#include "lanes.h"
#include "sgw_internal.h"

namespace sgw {
namespace {

constexpr int kEB = 256;
constexpr int kMaxPade = 64;  // frequencies of the symmetrised mesh
constexpr double kEps8 = 1e-8, kEps24 = 1e-24;

unsigned blocks(int64_t count) { return (unsigned)((count + kEB - 1) / kEB); }

__device__ inline double cabs2(double2 a) { return a.x * a.x + a.y * a.y; }

// principal square root
__device__ inline double2 csqrt_p(double2 z) {
  const double r = sqrt(cabs2(z));
  const double re = sqrt(0.5 * (r + z.x));
  const double im = copysign(sqrt(0.5 * fmax(r - z.x, 0.0)), z.y);
  return mk(re, im);
}

__device__ inline double2 protect(double2 x) {
  return sqrt(cabs2(x)) > kEps24 ? x : mk(kEps24, 0.0);
}

// godby_needs_coeffs (godby_needs.f90): W0 = W(0), W1 = W(i omega_p) of every
// element become the pole strength and frequency, in place
__global__ void k_gn_coeffs(int64_t ne, double omega_p, double2 *__restrict__ w0,
                            double2 *__restrict__ w1) {
  const int64_t e = (int64_t)blockIdx.x * kEB + threadIdx.x;
  if (e >= ne) return;
  const double2 a = w0[e], b = w1[e];
  double2 work = csub(a, b);
  bool zero = fabs(work.x) < kEps8;
  if (!zero) {
    work = cdiv(b, work);
    zero = work.x < kEps8;
  }
  if (!zero) {
    const double2 c2 = csqrt_p(work);
    const double2 p = mk(c2.x * omega_p, c2.y * omega_p);
    const double2 h = cmul(mk(0.5 * a.x, 0.5 * a.y), p);
    w1[e] = p;
    w0[e] = h;
  } else {
    w0[e] = mk(0.0, 0.0);
    w1[e] = mk(0.0, 0.0);
  }
}

struct Mesh {
  double2 z[kMaxPade];
  int src[kMaxPade];  // input slice of each symmetrised point
};

// pade_coeff (Vidberg-Serene recursion) per element; u_i = w[src[i]][e],
// coefficients a_p written to slice p.  The rows g(p, .) of the recursion
// are kept one at a time in g[].
__global__ void k_pade_coeffs(int64_t ne, int N, Mesh m, double2 *__restrict__ w) {
  const int64_t e = (int64_t)blockIdx.x * kEB + threadIdx.x;
  if (e >= ne) return;
  double2 g[kMaxPade];
  for (int i = 0; i < N; ++i) g[i] = protect(w[(int64_t)m.src[i] * ne + e]);
  w[e] = g[0];
  for (int p = 1; p < N; ++p) {
    const double2 gpp = g[p - 1];
    for (int i = p; i < N; ++i) {
      const double2 t1 = cdiv(gpp, g[i]);
      const double2 t2 = cdiv(g[i], g[i]);
      g[i] = protect(cdiv(csub(t1, t2), csub(m.z[i], m.z[p - 1])));
    }
    w[(int64_t)p * ne + e] = g[p];
  }
}

// ---------------------------------------------------------------------------
// Robust Pade approximation (pade_robust.f90:164-535, the SVD algorithm of
// P. Gonnet, S. Guettel and L. N. Trefethen, SIAM Rev. 55 (2013) 101-117)
// of every element from its values on a circle of N points.  One group of G
// lanes per element; lane l holds row l of the group's matrix, which lives in
// LDS column by column (column stride G).  The matrices have at most
// N/2 - 1 rows, so up to 35 points a quarter wavefront (G = 16) carries an
// element, above that half a wavefront; the group reductions give the same
// bits either way.  Numerical rank from one-sided Jacobi singular values (the
// reference calls ZGESDD); null vectors from Householder QR in the form of
// ZGEQRF + ZUNGQR (the reference's qr wrapper, lapack.f90:150-225).
//
// Bound: the chains of dependent FP64 instructions of the Jacobi pairs (HBM
// moves 2 x 16 N bytes per element).  400 x 400 elements of six poles, N = 32:
// 52.4 ms with half a wavefront per element, LDS-permute sums and full Jacobi;
// 14.5 ms with vector sums, quarter wavefronts and Jacobi left once the rank
// is certain; 12.1 ms with a pair's columns kept in registers; 2.4 ms with the
// pivoted QR deciding first (96 % of these elements; the other 4 % take half
// of the time that is left).

constexpr int kPrBlock = 128;                           // most threads per block
constexpr int kPrLdsMax = 65536;                        // LDS bytes per block
constexpr int kPrSweeps = 40;                           // Jacobi sweep limit
constexpr double kPrTol = 1e-14;                        // eps14, the default tolerance
constexpr double kSqrtEps = 1.4901161193847656e-08;     // sqrt(epsilon(1.0_dp))
constexpr double kDblEps = 2.220446049250313e-16;
constexpr int kPrSmallMax = 35;                         // most points with G = 16
// Open ranks are settled on the spot up to kPrHere elements or kPrHerePoints
// points, else through a list: an open element holds up those that share its
// wavefront, which the long Jacobi of many points makes dear; the list and the
// second launch cost 10 to 30 us.  On the spot against the list: 1 element of
// 20 points 26 us against 45, 40 000 of 20 points 256 against 281; 400 of 32
// points 590 against 771, 1 600 670 against 770, 40 000 1 947 against 1 283; 1 600
// of 36 points 1 107 against 1 057, 10 000 2 549 against 1 732.
constexpr int64_t kPrHere = 1024;
constexpr int kPrHerePoints = 20;

// LDS per element: Taylor coefficients (2 G), b (G), tau (G), the matrix
// (G x nmax), whose place the samples take before it and a after it (at least
// N: nmax = N / 2 - 2 >= 3)
template <int G> __host__ __device__ inline int pr_group_lds(int nmax) {
  return 4 * G + G * nmax;
}

__device__ inline double cabsd(double2 a) { return hypot(a.x, a.y); }

// row l of (C D)^T: A(l, i) = C(i, l) d_l = c(m+1+i-l) d_l for i < n, l <= n,
// C = rows m+1..m+n of the Toeplitz matrix of c (pade_robust.f90:347-352)
template <int G> __device__ void pr_build(double2 *A, const double2 *cc, int m, int n, int l, double d) {
  __syncwarp();
  for (int i = 0; i < n; ++i) {
    const int k = m + 1 + i - l;
    const double2 v = (l <= n && k >= 0) ? cc[k] : mk(0.0, 0.0);
    A[i * G + l] = mk(v.x * d, v.y * d);
  }
  __syncwarp();
}

// Whether the columns of A, part way through Jacobi, already fix the number of
// singular values above tol, and that number.  Columns of norm above 3 tol
// with all cosines below 1/(2 k) (k of them) have a smallest singular value
// of at least their smallest norm times sqrt(1/2), which is above 2 tol; the
// others together, below tol/2 in Frobenius norm, move no singular value by
// more than that.  The rotations still to come keep the singular values up to
// their rounding, a few 1e-16 of the matrix, against tol = 1e-14 ||c||, so
// they cannot carry one across tol.
template <int G> __device__ bool pr_decided(const double2 *A, int rows, int cols, int l,
                                            double tol, int &rho) {
  double rest = 0.0;
  uint32_t big = 0;
  for (int i = 0; i < cols; ++i) {
    const double2 a = l < rows ? A[i * G + l] : mk(0.0, 0.0);
    const double s = lanes::sum<G>(cabs2(a));
    if (s > 9.0 * tol * tol) big |= 1u << i;
    else rest += s;
  }
  if (!(rest < 0.25 * tol * tol)) return false;
  const int k = __popc(big);
  const double lim = 0.25 / ((double)k * k);
  for (uint32_t m = big; m; m &= m - 1) {
    const int p = __ffs(m) - 1;
    const double2 ap = l < rows ? A[p * G + l] : mk(0.0, 0.0);
    const double al = lanes::sum<G>(cabs2(ap));
    for (uint32_t m2 = m & (m - 1); m2; m2 &= m2 - 1) {
      const int q = __ffs(m2) - 1;
      const double2 aq = l < rows ? A[q * G + l] : mk(0.0, 0.0);
      double2 g = mk(0.0, 0.0);
      cmacc(g, ap, aq);
      g = mk(lanes::sum<G>(g.x), lanes::sum<G>(g.y));
      if (!(cabs2(g) < lim * al * lanes::sum<G>(cabs2(aq)))) return false;
    }
  }
  rho = k;
  return true;
}

// number of singular values of A (rows x cols, rows <= G) above tol:
// one-sided (Hestenes) Jacobi orthogonalises the columns, whose norms are
// then the singular values.  Each lane touches only its own row of A.  It
// stops once the number is certain; where a singular value comes near tol it
// runs to convergence.
template <int G> __device__ int pr_rank(double2 *A, int rows, int cols, int l, double tol) {
  const double ctol = sqrt((double)rows) * kDblEps;
  for (int sweep = 0; sweep < kPrSweeps; ++sweep) {
    int rot = 0;
    for (int p = 0; p + 1 < cols; ++p) {
      // column p stays in registers over its pairs; the next column is read,
      // and its norm summed, ahead of the pair that needs them
      double2 ap = l < rows ? A[p * G + l] : mk(0.0, 0.0);
      double2 aq = l < rows ? A[(p + 1) * G + l] : mk(0.0, 0.0);
      double al = lanes::sum<G>(cabs2(ap)), be = lanes::sum<G>(cabs2(aq));
      bool turned = false;
      for (int q = p + 1; q < cols; ++q) {
        double2 gm = mk(0.0, 0.0);
        cmacc(gm, ap, aq);                                   // conj(a_p) a_q
        gm = mk(lanes::sum<G>(gm.x), lanes::sum<G>(gm.y));
        const double g2 = cabs2(gm);
        const double2 an = q + 1 < cols && l < rows ? A[(q + 1) * G + l] : mk(0.0, 0.0);
        const double bn = lanes::sum<G>(cabs2(an));
        // far from the threshold its roots are not needed
        const double c2 = ctol * ctol * al * be;
        const double g = g2 < 0.5 * c2 ? 0.0 : hypot(gm.x, gm.y);
        if (g2 > 2.0 * c2 || g > ctol * sqrt(al) * sqrt(be)) {  // uniform over the group
          ++rot;
          turned = true;
          // a_q~ = a_q conj(g)/|g| makes a_p^H a_q~ = |g| real; then the real
          // rotation with t^2 + 2 zeta t - 1 = 0, |t| <= 1
          const double zeta = (be - al) / (2.0 * g);
          const double az = fabs(zeta);
          const double t =
              az > 1e150 ? 0.5 / zeta : copysign(1.0, zeta) / (az + sqrt(1.0 + zeta * zeta));
          const double cs = 1.0 / sqrt(1.0 + t * t), sn = cs * t;
          const double2 ph = mk(gm.x / g, -gm.y / g);
          const double2 aqt = cmul(aq, ph);
          if (l < rows) A[q * G + l] = mk(sn * ap.x + cs * aqt.x, sn * ap.y + cs * aqt.y);
          ap = mk(cs * ap.x - sn * aqt.x, cs * ap.y - sn * aqt.y);
          al = lanes::sum<G>(cabs2(ap));
        }
        aq = an;
        be = bn;
      }
      if (turned && l < rows) A[p * G + l] = ap;
    }
    if (rot == 0) break;
    int sure;
    if (pr_decided<G>(A, rows, cols, l, tol, sure)) return sure;
  }
  int rho = 0;
  for (int i = 0; i < cols; ++i) {
    const double2 a = l < rows ? A[i * G + l] : mk(0.0, 0.0);
    if (sqrt(lanes::sum<G>(cabs2(a))) > tol) ++rho;
  }
  return rho;
}

// The number of singular values of A above tol where a column-pivoted QR
// settles it, else -1 (Jacobi decides then; A is overwritten).  After k steps
// sigma_{k+1} is at most the Frobenius norm of what is left, required below
// tol / 2, and sigma_k at least 3 r_kk / sqrt(4^k + 6 k - 1) (Faddeev,
// Kublanovskaya and Faddeeva; the columns are pivoted), required above 2 tol.
// The margins cover the rounding of either algorithm, a few 1e-16 ||A||
// against tol = 1e-14 ||c||.
template <int G> __device__ int pr_rank_qr(double2 *A, int rows, int cols, int l, double tol) {
  // lane j keeps the squared norm of column j (-1: taken)
  double nj = -1.0, rest = 0.0;
  for (int j = 0; j < cols; ++j) {
    const double s = lanes::sum<G>(l < rows ? cabs2(A[j * G + l]) : 0.0);
    if (l == j) nj = s;
    rest += s;
  }
  double rkk = 0.0;
  int k = 0;
  while (k < cols && !(rest < 0.25 * tol * tol)) {
    const double big = lanes::max<G>(nj);
    const int p = lanes::min<G>(nj == big ? l : G - 1);
    if (!(big > 0.0) || k >= 26) return -1;  // nothing left, NaN, or no use for the bound
    if (l == p) nj = -1.0;
    rkk = sqrt(big);
    const double inv = 1.0 / rkk;
    double2 qv = l < rows ? A[p * G + l] : mk(0.0, 0.0);
    qv = mk(qv.x * inv, qv.y * inv);
    ++k;
    rest = 0.0;
    const uint64_t left = __ballot(nj >= 0.0) >> ((threadIdx.x & 63) / G * G);
    for (uint32_t m = (uint32_t)left & (uint32_t)((1ull << G) - 1); m; m &= m - 1) {
      const int j = __ffs(m) - 1;
      double2 a = l < rows ? A[j * G + l] : mk(0.0, 0.0), g = mk(0.0, 0.0);
      cmacc(g, qv, a);
      g = mk(lanes::sum<G>(g.x), lanes::sum<G>(g.y));
      a = csub(a, cmul(qv, g));
      if (l < rows) A[j * G + l] = a;
      const double s = lanes::sum<G>(cabs2(a));
      if (l == j) nj = s;
      rest += s;
    }
  }
  if (k == 0) return 0;
  // sqrt(4^k + 6 k - 1) < 2^k (1 + 6 k / 4^k)
  const double f = (double)(1u << k);
  return 3.0 * rkk > 2.0 * tol * f * (1.0 + 6.0 * k / (f * f)) ? k : -1;
}

// Householder QR of A (rows x cols, rows = cols + 1 <= 31) in place, in the
// conventions of ZGEQR2/ZLARFG: H_k = I - tau_k v_k v_k^H with v_k(k) = 1,
// beta = -sign(Re alpha) ||(alpha, x)||; R on and above the diagonal, v_k
// below it, tau_k in tau[k]
template <int G> __device__ void pr_qr(double2 *A, double2 *tau, int rows, int cols, int l) {
  for (int k = 0; k < cols; ++k) {
    __syncwarp();
    const double2 alpha = A[k * G + k];
    const bool below = l > k && l < rows;
    const double2 x = below ? A[k * G + l] : mk(0.0, 0.0);
    const double xn2 = lanes::sum<G>(cabs2(x));
    double2 tk = mk(0.0, 0.0);
    if (!(xn2 == 0.0 && alpha.y == 0.0)) {
      const double beta = -copysign(sqrt(alpha.x * alpha.x + alpha.y * alpha.y + xn2), alpha.x);
      tk = mk((beta - alpha.x) / beta, -alpha.y / beta);
      const double2 sc = cdiv(mk(1.0, 0.0), mk(alpha.x - beta, alpha.y));
      const double2 v = l == k ? mk(1.0, 0.0) : (below ? cmul(x, sc) : mk(0.0, 0.0));
      if (below) A[k * G + l] = v;
      if (l == k) A[k * G + k] = mk(beta, 0.0);
      // H_k^H = I - conj(tau_k) v v^H on the columns right of k
      const double2 ct = cconj(tk);
      for (int j = k + 1; j < cols; ++j) {
        const bool act = l >= k && l < rows;
        const double2 a = act ? A[j * G + l] : mk(0.0, 0.0);
        double2 s = mk(0.0, 0.0);
        cmacc(s, v, a);
        s = mk(lanes::sum<G>(s.x), lanes::sum<G>(s.y));
        if (act) A[j * G + l] = csub(a, cmul(ct, cmul(v, s)));
      }
    }
    if (l == 0) tau[k] = tk;
  }
  __syncwarp();
}

// row l of Q e_{rows-1}, Q = H_0 H_1 ... H_{cols-1} (the last column of the
// full Q of ZUNGQR)
template <int G> __device__ double2 pr_qlast(const double2 *A, const double2 *tau, int rows, int cols, int l) {
  double2 y = l == rows - 1 ? mk(1.0, 0.0) : mk(0.0, 0.0);
  for (int k = cols - 1; k >= 0; --k) {
    const double2 v = l == k ? mk(1.0, 0.0)
                             : ((l > k && l < rows) ? A[k * G + l] : mk(0.0, 0.0));
    double2 s = mk(0.0, 0.0);
    cmacc(s, v, y);
    s = mk(lanes::sum<G>(s.x), lanes::sum<G>(s.y));
    y = csub(y, cmul(tau[k], cmul(v, s)));
  }
  return y;
}

// pade_coeff_robust (pade_robust.f90:89-160) per element: w[f * ne + e] holds
// the values on the circle z_f = R e^{2 pi i f / N} and receives
// [m, n, a_0..a_m, b_0..b_n, 0, ...] (the reference leaves whatever was there
// beyond the coefficients; pade_eval_robust never reads it)
//
// Ranks by pr_rank_qr and, where that leaves one open, by Jacobi on the spot
// (kHere), or the element goes, untouched, to the list `open` (kList; open[0]
// their number), which a second launch works off by Jacobi (kJacobi); with
// `open` null that takes every element.
enum { kHere, kList, kJacobi };
template <int G, int RANK>
__global__ __launch_bounds__(kPrBlock) void k_pade_robust_coeffs(
    int64_t ne, int N, double radius, int nmax, double2 *__restrict__ w,
    int32_t *__restrict__ open) {
  extern __shared__ double2 pr_lds[];
  __shared__ double2 tw[kMaxPade];
  for (int t = threadIdx.x; t < N; t += blockDim.x) {
    double s, c;
    sincospi(-2.0 * t / N, &s, &c);
    tw[t] = mk(c, s);
  }
  __syncthreads();
  const int grp = threadIdx.x / G, l = threadIdx.x % G;
  const int64_t at = (int64_t)blockIdx.x * (blockDim.x / G) + grp;
  if (at >= (RANK == kJacobi && open ? open[0] : ne)) return;
  const int64_t e = RANK == kJacobi && open ? open[1 + at] : at;
  double2 *cc = pr_lds + (size_t)grp * pr_group_lds<G>(nmax);
  double2 *bv = cc + 2 * G;
  double2 *tau = bv + G;
  double2 *A = tau + G;
  double2 *fa = A;  // f before the matrix, a after it
  for (int j = l; j < N; j += G) fa[j] = w[(int64_t)j * ne + e];
  __syncwarp();

  int m = N / 2 - 2, n = m;            // the (n, n) start, pade_coeff_robust :146-147
  const int nd = m + n + 1;
  // pade_derivative (:445-535): c_k = FFT(f)_k / N / R^k, k < nd (<= N)
  double2 ck[2];
  double nrm = 0.0;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int k = l + h * G;
    double2 acc = mk(0.0, 0.0);
    if (k < nd) {
      for (int j = 0, t = 0; j < N; ++j) {  // t = j k mod N
        cmac(acc, fa[j], tw[t]);
        t += k;
        t -= t >= N ? N : 0;
      }
      acc = mk(acc.x * (1.0 / N), acc.y * (1.0 / N));
      if (fabs(radius - 1.0) > kPrTol) {
        double r = 1.0;
        for (int i = 0; i < k; ++i) r = r / radius;
        acc = mk(acc.x * r, acc.y * r);
      }
    }
    ck[h] = acc;
    nrm += cabs2(acc);
  }
  {
    const double tol = kPrTol * sqrt(lanes::sum<G>(nrm));   // near-zero coefficients dropped
    double im = 0.0;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if (cabsd(ck[h]) < tol) ck[h] = mk(0.0, 0.0);
      im = fmax(im, fabs(ck[h].y));
    }
    if (lanes::max<G>(im) < tol) {                           // real functions made real
      ck[0].y = 0.0;
      ck[1].y = 0.0;
    }
  }
  cc[l] = ck[0];
  cc[l + G] = ck[1];
  const double abs_tol = kPrTol * sqrt(lanes::sum<G>(cabs2(ck[0]) + cabs2(ck[1])));   // :276
  double cmax = 0.0, cmax_m = 0.0;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int k = l + h * G;
    cmax = fmax(cmax, cabsd(ck[h]));
    if (k <= m) cmax_m = fmax(cmax_m, cabsd(ck[h]));
  }
  cmax = lanes::max<G>(cmax);
  cmax_m = lanes::max<G>(cmax_m);
  __syncwarp();

  double2 a = mk(0.0, 0.0), b = mk(0.0, 0.0);      // row l of a and of b
  const bool zero = cmax_m <= kPrTol * cmax;
  if (zero) {                                       // zero function, returned as is (:287-306)
    m = 0;
    n = 0;
    b = l == 0 ? mk(1.0, 0.0) : b;
  } else {
    // diagonal hopping (:318-363): while rank(C) < n, shrink m and n
    while (n > 0) {
      pr_build<G>(A, cc, m, n, l, 1.0);
      int rho = RANK == kJacobi ? pr_rank<G>(A, n + 1, n, l, abs_tol)
                                : pr_rank_qr<G>(A, n + 1, n, l, abs_tol);
      if (RANK == kList && rho < 0) {
        if (l == 0) open[1 + atomicAdd(open, 1)] = (int32_t)e;
        return;
      }
      if (RANK == kHere && rho < 0) {
        pr_build<G>(A, cc, m, n, l, 1.0);
        rho = pr_rank<G>(A, n + 1, n, l, abs_tol);
      }
      if (rho == n) break;
      m -= n - rho;
      n = rho;
    }
    if (n == 0) {                                   // (:329-343)
      a = l <= m ? cc[l] : a;
      b = l == 0 ? mk(1.0, 0.0) : b;
    } else {
      // null vector of C (a unit vector, up to phase the one of ZGESDD) gives
      // the weights D = |v| + sqrt(eps); then b = D q_{n+1} of the QR of
      // (C D)^T, normalised (:366-386)
      pr_build<G>(A, cc, m, n, l, 1.0);
      pr_qr<G>(A, tau, n + 1, n, l);
      double2 y = pr_qlast<G>(A, tau, n + 1, n, l);
      const double d = l <= n ? cabsd(y) + kSqrtEps : 0.0;
      pr_build<G>(A, cc, m, n, l, d);
      pr_qr<G>(A, tau, n + 1, n, l);
      y = pr_qlast<G>(A, tau, n + 1, n, l);
      b = mk(d * y.x, d * y.y);
      const double bn = sqrt(lanes::sum<G>(cabs2(b)));
      b = mk(b.x / bn, b.y / bn);
      bv[l] = b;
      __syncwarp();
      // a = Z(0:m, 0:n) b, Z(i, j) = c(i - j) for i >= j (:389)
      if (l <= m)
        for (int j = 0; j <= min(l, n); ++j) cmac(a, cc[l - j], bv[j]);
      // leading zeros of b (and a) dropped (:392-408)
      int lam = lanes::min<G>((l <= n && cabsd(b) > kPrTol) ? l : G);
      if (lam == G) lam = 0;
      if (lam > 0) {
        fa[l] = a;
        __syncwarp();
        a = l + lam <= m ? fa[l + lam] : mk(0.0, 0.0);
        b = l + lam <= n ? bv[l + lam] : mk(0.0, 0.0);
        m -= lam;
        n -= lam;
        __syncwarp();
      }
      // trailing zeros of b dropped (:411-420)
      const int last = lanes::max<G>((l <= n && cabsd(b) > kPrTol) ? l : -1);
      if (last != n) {
        n = last;
        if (l > n) b = mk(0.0, 0.0);
      }
    }
  }
  // trailing zeros of a dropped (:425-434), then a and b over b_0 (:437-438)
  const int last_a = zero ? m : lanes::max<G>((l <= m && cabsd(a) > abs_tol) ? l : -1);
  if (last_a != m) {
    m = last_a;
    if (l > m) a = mk(0.0, 0.0);
  }
  bv[l] = b;
  __syncwarp();
  const double2 b0 = bv[0];
  a = cdiv(a, b0);
  b = cdiv(b, b0);
  __syncwarp();
  fa[l] = a;
  bv[l] = b;
  __syncwarp();
  // slices: 0 -> m, 1 -> n, 2..2+m -> a, 3+m..3+m+n -> b, the rest 0
  for (int s = l; s < N; s += G) {
    double2 v = mk(0.0, 0.0);
    if (s == 0) v = mk((double)m, 0.0);
    else if (s == 1) v = mk((double)n, 0.0);
    else if (s - 2 <= m) v = fa[s - 2];
    else if (s - 3 - m <= n) v = bv[s - 3 - m];
    w[(int64_t)s * ne + e] = v;
  }
}

// count words of device memory that are given back in the order of the stream's
// work, without a wait; p is null where there is none
struct StreamList {
  StreamList(hipStream_t st, int64_t count) : st_(st) {
    if (count > 0 && hipMallocAsync(reinterpret_cast<void **>(&p), sizeof(int32_t) * count, st) !=
                         hipSuccess) {
      (void)hipGetLastError();
      p = nullptr;
    }
  }
  ~StreamList() {
    if (p) (void)hipFreeAsync(p, st_);
  }
  StreamList(const StreamList &) = delete;
  StreamList &operator=(const StreamList &) = delete;
  int32_t *p = nullptr;

 private:
  hipStream_t st_;
};

// analytic_eval (analytic.f90:276-345): out(r, c) for r < num_g, c < num_g_p
// from the coefficients of element (gmap[r], gmap_p[c]); out zeroed before
__global__ void k_analytic_eval(int model, int N, Mesh m, double2 freq, int num_gc,
                                const double2 *__restrict__ coeff, int num_g, int num_g_p,
                                const int32_t *__restrict__ gmap,
                                const int32_t *__restrict__ gmap_p, int64_t nr,
                                double2 *__restrict__ out) {
  const int64_t e = (int64_t)blockIdx.x * kEB + threadIdx.x;
  if (e >= (int64_t)num_g * num_g_p) return;
  const int r = (int)(e % num_g), c = (int)(e / num_g);
  const int64_t ne = (int64_t)num_gc * num_gc;
  const int er = gmap[r], ec = gmap_p[c];
  if (er < 0 || er >= num_gc || ec < 0 || ec >= num_gc) {  // no such element
    out[(int64_t)c * nr + r] = mk(NAN, NAN);
    return;
  }
  const int64_t el = (int64_t)ec * num_gc + er;
  double2 res = mk(0.0, 0.0);
  if (model == 1) {  // godby_needs_model
    const double2 c1 = coeff[el], c2 = coeff[ne + el];
    if (sqrt(cabs2(c1)) > kEps8) {
      const double2 one = mk(1.0, 0.0);
      res = cmul(c1, cadd(cdiv(one, cadd(c2, freq)), cdiv(one, csub(c2, freq))));
    }
  } else if (model == SGW_AAA_APPROX) {  // aaa_approx_eval (analytic.f90:351-386)
    const int mmax = N / 3;
    int mm = 0;
    for (int c = 0; c < mmax; ++c)
      if (sqrt(cabs2(coeff[(int64_t)(2 * mmax + c) * ne + el])) > 1e-12) ++mm;
    // aaa_evaluate (aaa.f90:71-90): the barycentric form, or a support
    // point's value within 1e-14 of it
    double2 num = mk(0.0, 0.0), den = mk(0.0, 0.0);
    double dmin = INFINITY;
    int imin = 0;
    for (int c = 0; c < mm; ++c) {
      const double2 pc = coeff[(int64_t)c * ne + el];
      const double2 vc = coeff[(int64_t)(mmax + c) * ne + el];
      const double2 wc = coeff[(int64_t)(2 * mmax + c) * ne + el];
      double2 dz = csub(freq, pc);
      const double dist = sqrt(cabs2(dz));
      if (dist <= 1e-14) dz = mk(1e-14, 0.0);
      const double2 cc = cdiv(mk(1.0, 0.0), dz);
      num = cadd(num, cmul(cc, cmul(wc, vc)));
      den = cadd(den, cmul(cc, wc));
      if (dist < dmin) {
        dmin = dist;
        imin = c;
      }
    }
    res = (mm > 0 && dmin < 1e-14) ? coeff[(int64_t)(mmax + imin) * ne + el] : cdiv(num, den);
  } else if (model == SGW_AAA_POLE) {  // aaa_pole_eval (analytic.f90:430-459)
    const int half = N / 2;
    int npole = 0;
    for (int i = half; i < N; ++i)
      if (sqrt(cabs2(coeff[(int64_t)i * ne + el])) > 0.0) ++npole;
    for (int i = 0; i < npole && half + i < N; ++i)
      res = cadd(res, cdiv(coeff[(int64_t)(half + i) * ne + el],
                           csub(freq, coeff[(int64_t)i * ne + el])));
  } else if (model == SGW_PADE_ROBUST) {  // pade_eval_robust (pade_robust.f90:37-86)
    const int m = (int)lround(sqrt(cabs2(coeff[el])));
    const int n = (int)lround(sqrt(cabs2(coeff[ne + el])));
    if (4 + m + n > N) {  // degrees that do not fit the slices
      res = mk(NAN, NAN);
    } else {
      double2 num = mk(0.0, 0.0), den = mk(0.0, 0.0);
      for (int i = 2 + m; i >= 2; --i) num = cadd(coeff[(int64_t)i * ne + el], cmul(num, freq));
      for (int i = 3 + m + n; i >= 3 + m; --i)
        den = cadd(coeff[(int64_t)i * ne + el], cmul(den, freq));
      res = cdiv(num, den);
    }
  } else {  // pade_eval
    double2 a0 = mk(0.0, 0.0), a1 = coeff[el], b0 = mk(1.0, 0.0), b1 = mk(1.0, 0.0);
    for (int i = 1; i < N; ++i) {
      const double2 t = cmul(csub(freq, m.z[i - 1]), coeff[(int64_t)i * ne + el]);
      const double2 a2 = cadd(a1, cmul(t, a0)), b2 = cadd(b1, cmul(t, b0));
      a0 = a1; a1 = a2; b0 = b1; b1 = b2;
    }
    res = cdiv(a1, b1);
  }
  out[(int64_t)c * nr + r] = res;
}

__global__ void k_fill0(int64_t count, double2 *__restrict__ d) {
  const int64_t e = (int64_t)blockIdx.x * kEB + threadIdx.x;
  if (e < count) d[e] = mk(0.0, 0.0);
}

template <typename F> int guarded(F &&fn) {
  try {
    return fn();
  } catch (const Error &e) {
    set_error(e.msg);
    return e.code;
  } catch (const std::exception &e) {
    set_error(e.what());
    return SGW_E_STATE;
  }
}

// sigma_prod of one W (block w(ldw, *)): invfft6 (sigma.f90:487), the product
// with G(r, r') (:499) and fwfft6 (:510) into `o`.  S: num_g x nr_p scratch;
// full: an nr x nr_p matrix, used only where the r side is not a sphere list
// the box kernel holds.  There the first xy pass builds its planes from the
// rows S[g][r'], the z passes of both transforms and the product are one
// kernel, and the last xy pass keeps only the rows' positions.
void product(hipStream_t st, const Fft6Args &a, const Fft6Lists &l, const double2 *w, int64_t ldw,
             double2 *S, double2 *full, const double2 *green, const SphereOut &o) {
  const int64_t nr = (int64_t)a.n * a.n * a.n, nr_p = (int64_t)a.n_p * a.n_p * a.n_p;
  invfft6_rows(st, a, l, w, ldw, S);
  if (l.r.fits()) {
    SphereOut cols;
    cols.scale = 1.0 / (double)nr;
    cols.out = S;
    cols.out_sg = nr_p;
    sphere_prod(st, l.r, nr_p, -1, S, nr_p, green, cols);
  } else {
    // the plane lists: the G vectors of each z plane of the box
    const int n = a.n, num_g = a.num_g;
    std::vector<int32_t> start(n + 1, 0), gl(num_g), pos(num_g);
    for (int g = 0; g < num_g; ++g) ++start[l.nl[g] / (n * n) + 1];
    for (int z = 0; z < n; ++z) start[z + 1] += start[z];
    std::vector<int32_t> fill(start.begin(), start.end() - 1);
    for (int g = 0; g < num_g; ++g) {
      const int k = fill[l.nl[g] / (n * n)]++;
      gl[k] = g;
      pos[k] = l.nl[g] % (n * n);
    }
    DevBuf<int32_t> d_start(n + 1), d_gl(num_g), d_pos(num_g);
    d_start.upload(start.data(), n + 1, st);
    d_gl.upload(gl.data(), num_g, st);
    d_pos.upload(pos.data(), num_g, st);
    box_xy_scatter(st, n, nr_p, S, d_start.p, d_gl.p, d_pos.p, full, -1);
    box_z_product(st, n, nr_p, full, green);
    box_xy_gather(st, n, nr_p, full, d_start.p, d_gl.p, d_pos.p, 1.0 / (double)nr, S, +1);
    SGW_HIP(hipStreamSynchronize(st));  // the plane lists are freed here
  }
  fwfft6_rows(st, a, l, S, o);                                            // :519-521
}

Mesh make_mesh(int N, const sgw_complex *h_z, const int32_t *h_src) {
  SGW_REQUIRE(N >= 1 && N <= kMaxPade, SGW_E_SHAPE, "analytic: 1 <= frequencies <= 64");
  Mesh m{};
  for (int i = 0; i < N; ++i) {
    m.z[i] = make_double2(h_z[i].re, h_z[i].im);
    m.src[i] = h_src ? h_src[i] : i;
  }
  return m;
}

// the arguments of an evaluation; returns the mesh the model needs
Mesh eval_check(int32_t model, int32_t num_gc, int32_t nfreq, const sgw_complex *h_z,
                const sgw_complex *d_coeff, int32_t n, int32_t n_p, int32_t num_g,
                int32_t num_g_p, const int32_t *d_gmap, const int32_t *d_gmap_p) {
  (void)num_gc;
  const bool self_contained =
      model == SGW_PADE_ROBUST || model == SGW_AAA_APPROX || model == SGW_AAA_POLE;
  SGW_REQUIRE(d_coeff && d_gmap && d_gmap_p && (h_z || self_contained), SGW_E_ARG,
              "analytic_eval: null argument");
  SGW_REQUIRE(model >= SGW_GODBY_NEEDS && model <= SGW_AAA_POLE, SGW_E_ARG,
              "analytic_eval: model must be SGW_GODBY_NEEDS, SGW_PADE_APPROX, SGW_PADE_ROBUST, "
              "SGW_AAA_APPROX or SGW_AAA_POLE");
  SGW_REQUIRE(model != SGW_AAA_APPROX || (nfreq >= 3 && nfreq <= kMaxPade), SGW_E_SHAPE,
              "analytic_eval: AAA coefficients need 3..64 slices");
  SGW_REQUIRE(model != SGW_AAA_POLE || (nfreq >= 2 && nfreq <= kMaxPade), SGW_E_SHAPE,
              "analytic_eval: AAA pole coefficients need 2..64 slices");
  SGW_REQUIRE(model != SGW_PADE_ROBUST || (nfreq >= 4 && nfreq <= kMaxPade), SGW_E_SHAPE,
              "analytic_eval: robust Pade coefficients need 4..64 slices");
  SGW_REQUIRE(model != SGW_GODBY_NEEDS || nfreq == 2, SGW_E_SHAPE,
              "analytic_eval: Godby-Needs uses 2 coefficients");
  const int64_t nr = (int64_t)n * n * n, nr_p = (int64_t)n_p * n_p * n_p;
  SGW_REQUIRE(num_g >= 1 && num_g <= nr && num_g_p >= 1 && num_g_p <= nr_p, SGW_E_SHAPE,
              "analytic_eval: need num_g <= n^3 and num_g_p <= n_p^3");
  return self_contained ? Mesh{} : make_mesh(nfreq, h_z, nullptr);
}

}  // namespace
}  // namespace sgw

using namespace sgw;

extern "C" int sgw_analytic_coeff(int32_t model, double thres, int32_t num_g, int32_t nfreq,
                                  const sgw_complex *h_z, const int32_t *h_src,
                                  sgw_complex *d_w, void *stream) {
  return guarded([&] {
    SGW_REQUIRE(d_w && h_z && num_g >= 1, SGW_E_ARG, "analytic_coeff: null argument");
    hipStream_t st = (hipStream_t)stream;
    const int64_t ne = (int64_t)num_g * num_g;
    double2 *w = reinterpret_cast<double2 *>(d_w);
    KScope ks("analytic_coeff", st);
    if (model == SGW_GODBY_NEEDS) {
      SGW_REQUIRE(nfreq == 2, SGW_E_SHAPE, "godby_needs_coeffs: must provide exactly 2 frequencies");
      const double omega_p = h_z[1].im;
      SGW_REQUIRE(omega_p >= 0.0, SGW_E_ARG, "godby_needs_coeffs: plasmon frequency must be positive");
      k_gn_coeffs<<<blocks(ne), kEB, 0, st>>>(ne, omega_p, w, w + ne);
    } else if (model == SGW_PADE_APPROX) {
      const Mesh m = make_mesh(nfreq, h_z, h_src);
      for (int i = 0; i < nfreq; ++i)
        SGW_REQUIRE(m.src[i] >= 0 && m.src[i] < nfreq, SGW_E_ARG,
                    "pade_coeff: source slice out of range");
      k_pade_coeffs<<<blocks(ne), kEB, 0, st>>>(ne, nfreq, m, w);
    } else if (model == SGW_PADE_ROBUST) {
      // pade_coeff_robust (pade_robust.f90:89-160): the solver frequencies
      // themselves, on a circle, first point (R, 0)
      SGW_REQUIRE(h_src == nullptr, SGW_E_ARG, "pade_coeff_robust: no symmetrised mesh (h_src = NULL)");
      SGW_REQUIRE(nfreq >= 10, SGW_E_SHAPE, "pade_coeff_robust: use at least 10 frequencies to form the circle");
      SGW_REQUIRE(nfreq <= kMaxPade, SGW_E_SHAPE, "pade_coeff_robust: at most 64 frequencies");
      const double radius = h_z[0].re;
      for (int i = 0; i < nfreq; ++i)
        SGW_REQUIRE(std::fabs(std::hypot(h_z[i].re, h_z[i].im) - radius) <= 1e-12, SGW_E_ARG,
                    "pade_coeff_robust: frequencies must span circle in the complex plane");
      SGW_REQUIRE(radius > 0.0, SGW_E_ARG, "pade_robust: radius in the complex plane must be > 0");
      const int nmax = nfreq / 2 - 2;
      // The list of open elements belongs to the stream and is given back in its
      // order, so that the call returns behind its launches.  A stream under
      // capture takes every element through Jacobi; without memory for the list
      // open ranks are settled on the spot.
      hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
      if (hipStreamIsCapturing(st, &cap) != hipSuccess) {
        (void)hipGetLastError();
        cap = hipStreamCaptureStatusActive;
      }
      const bool capture = cap != hipStreamCaptureStatusNone;
      const bool here = ne <= kPrHere || nfreq <= kPrHerePoints || ne >= (1ll << 31) - 1;
      StreamList open(st, capture || here ? 0 : ne + 1);
      auto go = [&](auto group) {
        constexpr int G = decltype(group)::value;
        const int bytes = (int)sizeof(double2) * pr_group_lds<G>(nmax);   // <= 18432
        const int per = std::min(kPrBlock / G, kPrLdsMax / bytes);
        const unsigned grid = (unsigned)((ne + per - 1) / per);
        auto launch = [&](auto rank) {
          k_pade_robust_coeffs<G, decltype(rank)::value>
              <<<grid, G * per, (size_t)per * bytes, st>>>(ne, nfreq, radius, nmax, w, open.p);
          SGW_HIP(hipGetLastError());
        };
        using std::integral_constant;
        if (open.p) {
          SGW_HIP(hipMemsetAsync(open.p, 0, sizeof(int32_t), st));
          launch(integral_constant<int, kList>{});
          // as many groups as elements might be open: those past the list's end
          // leave at once
          launch(integral_constant<int, kJacobi>{});
        } else if (capture) {
          launch(integral_constant<int, kJacobi>{});
        } else {
          launch(integral_constant<int, kHere>{});
        }
      };
      if (nfreq <= kPrSmallMax) go(std::integral_constant<int, 16>{});
      else go(std::integral_constant<int, 32>{});
    } else if (model == SGW_AAA_APPROX || model == SGW_AAA_POLE) {
      // aaa_generate per element on the symmetrised mesh (analytic.f90:162-199)
      const Mesh m = make_mesh(nfreq, h_z, h_src);
      for (int i = 0; i < nfreq; ++i)
        SGW_REQUIRE(m.src[i] >= 0 && m.src[i] < nfreq, SGW_E_ARG, "aaa: source slice out of range");
      SGW_REQUIRE(thres >= 0.0, SGW_E_ARG, "aaa: threshold must be >= 0");
      aaa_coeffs(model, thres, ne, nfreq, m.z, m.src, w, st);
    } else {
      throw Error{SGW_E_ARG, "analytic_coeff: model must be SGW_GODBY_NEEDS, SGW_PADE_APPROX, "
                             "SGW_PADE_ROBUST, SGW_AAA_APPROX or SGW_AAA_POLE"};
    }
    SGW_HIP(hipGetLastError());
    return 0;
  });
}

extern "C" int sgw_analytic_eval(int32_t model, int32_t num_gc, int32_t nfreq,
                                 const sgw_complex *h_z, const sgw_complex *d_coeff,
                                 sgw_complex freq, int32_t n, int32_t n_p, int32_t num_g,
                                 int32_t num_g_p, const int32_t *d_gmap,
                                 const int32_t *d_gmap_p, sgw_complex *d_out, void *stream) {
  return guarded([&] {
    SGW_REQUIRE(d_out != nullptr, SGW_E_ARG, "analytic_eval: null argument");
    const Mesh m = eval_check(model, num_gc, nfreq, h_z, d_coeff, n, n_p, num_g, num_g_p, d_gmap,
                              d_gmap_p);
    const int64_t nr = (int64_t)n * n * n, nr_p = (int64_t)n_p * n_p * n_p;
    hipStream_t st = (hipStream_t)stream;
    double2 *out = reinterpret_cast<double2 *>(d_out);
    KScope ks("analytic_eval", st);
    k_fill0<<<blocks(nr * nr_p), kEB, 0, st>>>(nr * nr_p, out);
    k_analytic_eval<<<blocks((int64_t)num_g * num_g_p), kEB, 0, st>>>(
        model, nfreq, m, make_double2(freq.re, freq.im), num_gc,
        reinterpret_cast<const double2 *>(d_coeff), num_g, num_g_p, d_gmap, d_gmap_p, nr, out);
    SGW_HIP(hipGetLastError());
    return 0;
  });
}

extern "C" int sgw_sigma_prod(int32_t n, int32_t n_p, int32_t num_g, const int32_t *d_nl,
                              int32_t num_g_p, const int32_t *d_nl_p, double omega,
                              sgw_complex alpha, const sgw_complex *d_green, sgw_complex *d_array,
                              sgw_complex *d_sigma, int64_t ld_sigma, void *stream) {
  return guarded([&] {
    SGW_REQUIRE(d_green && d_array, SGW_E_ARG, "sigma_prod: null argument");
    SGW_REQUIRE(!d_sigma || ld_sigma >= num_g, SGW_E_SHAPE, "sigma_prod: ld_sigma < num_g");
    Fft6Args a{n, n_p, num_g, num_g_p, d_nl, d_nl_p, omega, 1,
               reinterpret_cast<double2 *>(d_array)};
    fft6_check(a, "sigma_prod");
    hipStream_t st = (hipStream_t)stream;
    const int64_t nr = (int64_t)n * n * n, nr_p = (int64_t)n_p * n_p * n_p;
    const Fft6Lists lists(st, a, "sigma_prod");
    DevBuf<double2> S((size_t)num_g * nr_p);
    {
      KScope ks("sigma_prod", st);
      SphereOut o;
      o.has_alpha = true;
      o.alpha = make_double2(alpha.re, alpha.im);
      o.out = a.f;
      o.out_sg = nr;
      o.sum = reinterpret_cast<double2 *>(d_sigma);                       // :741
      o.sum_sg = ld_sigma;
      product(st, a, lists, a.f, nr, S.p, a.f, reinterpret_cast<const double2 *>(d_green), o);
    }
    SGW_HIP(hipGetLastError());
    SGW_HIP(hipStreamSynchronize(st));  // scratch freed on return
    return 0;
  });
}

extern "C" int64_t sgw_sigma_correlation_workspace(int32_t n, int32_t n_p, int32_t num_g,
                                                   int32_t num_g_p) {
  if (n < 1 || n_p < 1 || num_g < 1 || num_g_p < 1) return 0;
  const int64_t nr_p = (int64_t)n_p * n_p * n_p;
  return (int64_t)sizeof(double2) * ((int64_t)num_g * nr_p + (int64_t)num_g * num_g_p);
}

extern "C" int sgw_sigma_correlation(
    int32_t model, int32_t num_gc, int32_t nfreq, const sgw_complex *h_z,
    const sgw_complex *d_coeff, int32_t nterm, const sgw_complex *h_freq,
    const sgw_complex *h_alpha, const int64_t *h_green, const int32_t *h_sigma, int32_t n,
    int32_t n_p, int32_t num_g, const int32_t *d_nl, int32_t num_g_p, const int32_t *d_nl_p,
    double omega, const int32_t *d_gmap, const int32_t *d_gmap_p, const sgw_complex *d_green,
    sgw_complex *d_sigma, void *d_work, int64_t work_bytes, void *stream) {
  return guarded([&] {
    const Mesh m = eval_check(model, num_gc, nfreq, h_z, d_coeff, n, n_p, num_g, num_g_p, d_gmap,
                              d_gmap_p);
    SGW_REQUIRE(nterm >= 0 && (nterm == 0 || (h_freq && h_alpha && h_green && h_sigma)) &&
                    d_green && d_sigma,
                SGW_E_ARG, "sigma_correlation: null argument or negative count");
    const int64_t need = sgw_sigma_correlation_workspace(n, n_p, num_g, num_g_p);
    SGW_REQUIRE(!d_work || work_bytes >= need, SGW_E_SHAPE,
                "sigma_correlation: workspace too small");
    // the check's matrix pointer; the box kernels need no full matrix
    Fft6Args a{n, n_p, num_g, num_g_p, d_nl, d_nl_p, omega, 1,
               reinterpret_cast<double2 *>(d_sigma)};
    fft6_check(a, "sigma_correlation");
    for (int t = 0; t < nterm; ++t)
      SGW_REQUIRE(h_green[t] >= 0 && h_sigma[t] >= 0, SGW_E_ARG,
                  "sigma_correlation: negative slice");
    hipStream_t st = (hipStream_t)stream;
    const int64_t nr = (int64_t)n * n * n, nr_p = (int64_t)n_p * n_p * n_p;
    const Fft6Lists lists(st, a, "sigma_correlation");
    DevBuf<double2> own, full;
    if (!d_work) own.alloc((size_t)need / sizeof(double2));
    if (!lists.r.fits()) full.alloc((size_t)(nr * nr_p));
    double2 *S = d_work ? static_cast<double2 *>(d_work) : own.p, *W = S + num_g * nr_p;
    for (int t = 0; t < nterm; ++t) {
      {
        KScope ks("analytic_eval", st);
        k_analytic_eval<<<blocks((int64_t)num_g * num_g_p), kEB, 0, st>>>(
            model, nfreq, m, make_double2(h_freq[t].re, h_freq[t].im), num_gc,
            reinterpret_cast<const double2 *>(d_coeff), num_g, num_g_p, d_gmap, d_gmap_p, num_g,
            W);
      }
      KScope ks("sigma_prod", st);
      SphereOut o;
      o.has_alpha = true;
      o.alpha = make_double2(h_alpha[t].re, h_alpha[t].im);
      o.sum = reinterpret_cast<double2 *>(d_sigma) + (int64_t)h_sigma[t] * num_g * num_g_p;
      o.sum_sg = num_g;
      product(st, a, lists, W, num_g, S, full.p,
              reinterpret_cast<const double2 *>(d_green) + h_green[t], o);
    }
    SGW_HIP(hipGetLastError());
    SGW_HIP(hipStreamSynchronize(st));  // the lists are freed on return
    return 0;
  });
}
