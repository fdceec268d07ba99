// AAA continuation of W on the device: aaa_generate of the vendored AAA
// library (vendor/analytic/src/aaa.f90:53-302; Nakatsukasa, Sete and
// Trefethen, SIAM J. Sci. Comput. 40 (2018) A1494) for every (G, G')
// element, and the pole-residue form of analytic.f90:389-427.
//
// Half a wavefront per element, lane l on mesh points l and l + 32 (at most 64
// points).  Per greedy step the Loewner submatrix (rows: the points that are not
// support points, columns: the support points in mesh order) sits in LDS
// column by column; its last right singular vector comes from one-sided
// (Hestenes) Jacobi with the rotations accumulated in V (the reference calls
// ZGESDD and takes the conjugated last row of V^H, which is that vector up
// to a phase; the phase cancels in the barycentric form).  Poles: the m - 1
// zeros of the barycentric denominator sum_j w_j / (z - z_j), i.e. the
// finite eigenvalues of the reference's arrowhead pencil (ZGGEV there),
// found together by Aberth-Ehrlich iteration, one lane per zero.
#include <algorithm>
#include <climits>
#include <cmath>

#include "aaa.h"
#include "lanes.h"
#include "sgw_internal.h"

namespace sgw {
namespace {

constexpr int kAaaMax = 64;                             // mesh points
constexpr double kEps6 = 1e-6, kEps14 = 1e-14;
constexpr double kDblEpsA = 2.220446049250313e-16;
constexpr int kSweeps = 40, kAberthIters = 500;

constexpr int kGrp = 32;                                // lanes per element
constexpr size_t kLdsCu = 160 * 1024;                   // LDS bytes of a CU

// sums and extrema over the mesh points or matrix rows of an element, H to a
// lane; the order is that of a 64-lane butterfly (lane l and l + 32 first)
template <int H> __device__ inline double wsum(const double (&v)[H]) {
  return lanes::sum<kGrp>(H == 2 ? v[0] + v[H - 1] : v[0]);
}
template <int H> __device__ inline double wmax(const double (&v)[H]) {
  return lanes::max<kGrp>(H == 2 ? fmax(v[0], v[H - 1]) : v[0]);
}
template <int H> __device__ inline double2 wsum2(const double2 (&v)[H]) {
  double re[H], im[H];
#pragma unroll
  for (int h = 0; h < H; ++h) {
    re[h] = v[h].x;
    im[h] = v[h].y;
  }
  return mk(wsum<H>(re), wsum<H>(im));
}
// this group's half of a wavefront ballot
__device__ inline uint32_t gballot(bool c) {
  return (uint32_t)(__ballot(c) >> (threadIdx.x & 32));
}
// the form is spelled out: a weight vector is fixed up to a phase, which comes
// from the rotations of rounding-level pairs, so that the last bit of a norm
// shows in the coefficients
__device__ inline double cabs2a(double2 a) { return fma(a.x, a.x, a.y * a.y); }
__device__ inline double cabsa(double2 a) { return hypot(a.x, a.y); }

__device__ inline uint64_t below(int l) { return l == 0 ? 0ull : (~0ull >> (64 - l)); }

// 1 / (x - y), eps14 for |x - y| <= eps14 (construct_Cauchy_matrix, aaa.f90:308-327)
__device__ inline double2 cauchy(double2 x, double2 y) {
  double2 d = csub(x, y);
  if (cabsa(d) <= kEps14) d = mk(kEps14, 0.0);
  return cdiv(mk(1.0, 0.0), d);
}

// aaa_evaluate (aaa.f90:71-90) at x from m support points in LDS
__device__ double2 aaa_eval_at(double2 x, int m, const double2 *pos, const double2 *val,
                               const double2 *wgt) {
  double2 num = mk(0.0, 0.0), den = mk(0.0, 0.0);
  double dmin = INFINITY;
  int imin = 0;
  for (int c = 0; c < m; ++c) {
    const double2 cc = cauchy(x, pos[c]);
    num = cadd(num, cmul(cc, cmul(wgt[c], val[c])));
    den = cadd(den, cmul(cc, wgt[c]));
    const double dist = cabsa(csub(x, pos[c]));
    if (dist < dmin) {
      dmin = dist;
      imin = c;
    }
  }
  return dmin < kEps14 ? val[imin] : cdiv(num, den);
}

struct AaaMesh {
  double2 z[kAaaMax];
  int src[kAaaMax];
};

// LDS per element (double2 units): A (M x mcap), V (mcap x mcap), pos, val,
// wgt, lam (mcap each)
__host__ __device__ inline int aaa_lds(int M, int mcap) { return (M + mcap + 4) * mcap; }

// model 4: slices [pos (mmax), val (mmax), wgt (mmax), 0...], mmax = max_point;
// model 5: [poles, 0..., residues, 0...] in halves of N / 2.
// status[0] = 1: a model-5 element needed more than mcap support points, or has
// NaN samples;
// status[1] = 1: more relevant poles than N / 2 (pole_correction's error)
//
// Bound: the dependent FP64 chains of the Jacobi pairs.  H mesh points and
// matrix rows to a lane; two elements share a wavefront, and the group sums
// are vector instructions (lanes.h), so the rows of a pair wait for no LDS
// permute.  400 x 400 elements, 35 points, at most 11 support points: 16.3 ms,
// against 42.4 with one wavefront per element and LDS-permute sums.  Zeros
// are written out where a value or zero is chosen: a named one makes the choice
// one of addresses, for which the compiler copies the whole mesh to private
// memory (1 312 bytes a lane, 18.2 ms).
template <int H>
__global__ __launch_bounds__(64) void k_aaa_coeffs(int64_t ne, int M, AaaMesh mesh, double thres,
                                                  int model, int max_point, int mcap,
                                                  double2 *__restrict__ w,
                                                  int32_t *__restrict__ status) {
  extern __shared__ double2 aaa_smem[];
  const int64_t e = (int64_t)blockIdx.x * (blockDim.x / kGrp) + threadIdx.x / kGrp;
  const int l = threadIdx.x % kGrp;
  if (e >= ne) return;
  double2 *A = aaa_smem + (size_t)(threadIdx.x / kGrp) * aaa_lds(M, mcap);
  double2 *V = A + M * mcap;
  double2 *pos = V + mcap * mcap;
  double2 *val = pos + mcap;
  double2 *wgt = val + mcap;
  double2 *lam = wgt + mcap;
  const uint64_t all = M == 64 ? ~0ull : (1ull << M) - 1;
  double2 zl[H], fl[H], fit[H];
  bool pt[H], sup[H];
  double d[H];
#pragma unroll
  for (int h = 0; h < H; ++h) {
    const int i = l + kGrp * h;
    pt[h] = i < M;
    sup[h] = false;
    zl[h] = pt[h] ? mesh.z[i] : mk(0.0, 0.0);
    fl[h] = pt[h] ? w[(int64_t)mesh.src[i] * ne + e] : mk(0.0, 0.0);
    d[h] = pt[h] ? cabsa(fl[h]) : 0.0;
  }
  // setup_work_type (:119-148)
  const double thres_abs = thres * wmax<H>(d);
  const double2 sumf = wsum2<H>(fl);
#pragma unroll
  for (int h = 0; h < H; ++h) fit[h] = mk(sumf.x / M, sumf.y / M);
  int m = 0;
  bool lost = false;
  const int mp = max_point;
  for (;;) {
    // update_support_point (:178-187): the first point of largest |f - fit|
#pragma unroll
    for (int h = 0; h < H; ++h) d[h] = pt[h] ? cabsa(csub(fl[h], fit[h])) : -1.0;
    const double dmax = wmax<H>(d);
    int first = INT_MAX;
#pragma unroll
    for (int h = H - 1; h >= 0; --h)
      if (d[h] == dmax) first = l + kGrp * h;
    const int j = lanes::min<kGrp>(first);
    uint64_t smask = 0;
#pragma unroll
    for (int h = 0; h < H; ++h) {
      if (l + kGrp * h == j) {
        fit[h] = fl[h];
        sup[h] = true;
      }
      smask |= (uint64_t)gballot(sup[h]) << (kGrp * h);
    }
    ++m;
    smask &= all;
    const uint64_t rmask = ~smask & all;
    const int nrows = M - m;
    // a NaN among the samples leaves no point of largest error (none, or one
    // past the mesh, or a support point again)
    lost = __popcll(smask) != m;
    if (lost) {
      if (l == 0 && model == 5) status[0] = 1;
      break;
    }
    if (m > mcap) {  // the device keeps at most mcap support points
      if (l == 0) status[0] = 1;
      break;
    }
    __syncwarp();
#pragma unroll
    for (int h = 0; h < H; ++h)
      if (sup[h]) {
        const int c = __popcll(smask & below(l + kGrp * h));
        pos[c] = zl[h];
        val[c] = fl[h];
      }
    __syncwarp();
    // determine_weight (:205-225): the Loewner submatrix, rows = the other
    // points in mesh order, columns = the support points in mesh order
#pragma unroll
    for (int h = 0; h < H; ++h) {
      const int r = __popcll(rmask & below(l + kGrp * h));
      if (pt[h] && !sup[h])
        for (int c = 0; c < m; ++c)
          A[c * M + r] = cdiv(csub(fl[h], val[c]), csub(zl[h], pos[c]));
    }
    if (l < m)
      for (int c = 0; c < m; ++c) V[c * mcap + l] = mk(l == c ? 1.0 : 0.0, 0.0);
    __syncwarp();
    auto column = [&](int c, double2 (&a)[H]) {
#pragma unroll
      for (int h = 0; h < H; ++h) a[h] = l + kGrp * h < nrows ? A[c * M + l + kGrp * h] : mk(0.0, 0.0);
    };
    auto norm2 = [&](const double2 (&a)[H]) {
      double s[H];
#pragma unroll
      for (int h = 0; h < H; ++h) s[h] = cabs2a(a[h]);
      return wsum<H>(s);
    };
    int cmin = m - 1;  // an empty submatrix: V = I, the weight is e_m
    if (nrows > 0) {
      const double ctol = sqrt((double)nrows) * kDblEpsA;
      for (int sweep = 0; sweep < kSweeps; ++sweep) {
        int rot = 0;
        for (int p = 0; p + 1 < m; ++p) {
          // column p stays in registers over its pairs
          double2 ap[H], aq[H];
          column(p, ap);
          double2 vp = l < m ? V[p * mcap + l] : mk(0.0, 0.0);
          double al = norm2(ap);
          bool turned = false;
          for (int q = p + 1; q < m; ++q) {
            column(q, aq);
            const double be = norm2(aq);
            double2 gh[H];
#pragma unroll
            for (int h = 0; h < H; ++h) {
              gh[h] = mk(0.0, 0.0);
              cmacc(gh[h], ap[h], aq[h]);
            }
            const double2 gm = wsum2<H>(gh);
            // far from the threshold its roots are not needed
            const double g2 = cabs2a(gm), c2 = ctol * ctol * al * be;
            if (g2 < 0.5 * c2) continue;
            const double g = hypot(gm.x, gm.y);
            if (!(g2 > 2.0 * c2) && !(g > ctol * sqrt(al) * sqrt(be))) continue;
            ++rot;
            turned = true;
            const double zeta = (be - al) / (2.0 * g);
            const double az = fabs(zeta);
            const double t =
                az > 1e150 ? 0.5 / zeta : copysign(1.0, zeta) / (az + sqrt(1.0 + zeta * zeta));
            const double cs = 1.0 / sqrt(1.0 + t * t), sn = cs * t;
            const double2 ph = mk(gm.x / g, -gm.y / g);
#pragma unroll
            for (int h = 0; h < H; ++h) {
              const double2 aqt = cmul(aq[h], ph);
              if (l + kGrp * h < nrows)
                A[q * M + l + kGrp * h] =
                    mk(sn * ap[h].x + cs * aqt.x, sn * ap[h].y + cs * aqt.y);
              ap[h] = mk(cs * ap[h].x - sn * aqt.x, cs * ap[h].y - sn * aqt.y);
            }
            if (l < m) {
              const double2 vqt = cmul(V[q * mcap + l], ph);
              V[q * mcap + l] = mk(sn * vp.x + cs * vqt.x, sn * vp.y + cs * vqt.y);
              vp = mk(cs * vp.x - sn * vqt.x, cs * vp.y - sn * vqt.y);
            }
            al = norm2(ap);
          }
          if (turned) {
#pragma unroll
            for (int h = 0; h < H; ++h)
              if (l + kGrp * h < nrows) A[p * M + l + kGrp * h] = ap[h];
            if (l < m) V[p * mcap + l] = vp;
          }
        }
        if (rot == 0) break;
      }
      // the right singular vector of the smallest singular value
      double smin = INFINITY;
      for (int c = 0; c < m; ++c) {
        double2 a[H];
        column(c, a);
        const double s = norm2(a);
        if (s <= smin) {  // the last of equal ones, as ZGESDD's descending order
          smin = s;
          cmin = c;
        }
      }
    }
    __syncwarp();
    if (l < m) wgt[l] = V[cmin * mcap + l];
    __syncwarp();
    // update_fit (:228-258)
#pragma unroll
    for (int h = 0; h < H; ++h)
      if (pt[h] && !sup[h]) {
        double2 num = mk(0.0, 0.0), den = mk(0.0, 0.0);
        for (int c = 0; c < m; ++c) {
          const double2 cc = cauchy(zl[h], pos[c]);
          num = cadd(num, cmul(cc, cmul(wgt[c], val[c])));
          den = cadd(den, cmul(cc, wgt[c]));
        }
        fit[h] = cdiv(num, den);
      }
    // converged (:276-282) or max_step_reached (:285-292)
#pragma unroll
    for (int h = 0; h < H; ++h)
      d[h] = pt[h] ? (cabsa(csub(fit[h], fl[h])) <= thres_abs ? 0.0 : 1.0) : 0.0;
    if (wmax<H>(d) == 0.0 || m >= mp) break;
  }
  __syncwarp();
  if (lost || m > mcap) {  // the coefficients are left as NaN
    for (int s = l; s < M; s += kGrp) w[(int64_t)s * ne + e] = mk(NAN, NAN);
    return;
  }
  if (model == 4) {
    const int mmax = max_point;
    for (int s = l; s < M; s += kGrp) {
      double2 v = mk(0.0, 0.0);
      if (s < m) v = pos[s];
      else if (s >= mmax && s < mmax + m) v = val[s - mmax];
      else if (s >= 2 * mmax && s < 2 * mmax + m) v = wgt[s - 2 * mmax];
      w[(int64_t)s * ne + e] = v;
    }
    return;
  }
  // model 5: poles (zeros of the denominator) by Aberth-Ehrlich, then the
  // residues of calculate_residual (:458-500) and pole_correction's filter
  const int nr = m - 1;
  const double2 mine[1] = {l < m ? pos[l] : mk(0.0, 0.0)};
  double2 cen = wsum2<1>(mine);
  cen = mk(cen.x / m, cen.y / m);
  double rad = lanes::max<kGrp>(l < m ? cabsa(csub(pos[l], cen)) : 0.0);
  if (!(rad > 0.0)) rad = 1.0;
  double2 lk = mk(0.0, 0.0);
  if (l < nr) {
    double s, c;
    sincospi(2.0 * l / nr + 0.23, &s, &c);
    lk = mk(cen.x + 1.5 * rad * c, cen.y + 1.5 * rad * s);
  }
  bool done = l >= nr;
  double prev = INFINITY;
  for (int it = 0; it < kAberthIters; ++it) {
    __syncwarp();
    if (l < nr) lam[l] = lk;
    __syncwarp();
    if (!done) {
      double2 sd = mk(0.0, 0.0), sd1 = mk(0.0, 0.0), sq = mk(0.0, 0.0);
      for (int c = 0; c < m; ++c) {
        const double2 inv = cdiv(mk(1.0, 0.0), csub(lk, pos[c]));
        const double2 t = cmul(wgt[c], inv);
        sd = cadd(sd, t);
        sd1 = cadd(sd1, cmul(t, inv));
        sq = cadd(sq, inv);
      }
      // p'/p = q'/q + D'/D with D = p / q, q = prod (z - z_j)
      const double2 ratio = csub(sq, cdiv(sd1, sd));
      const double2 nk = cdiv(mk(1.0, 0.0), ratio);
      double2 ak = mk(0.0, 0.0);
      for (int jj = 0; jj < nr; ++jj)
        if (jj != l) ak = cadd(ak, cdiv(mk(1.0, 0.0), csub(lk, lam[jj])));
      const double2 dl = cdiv(nk, csub(mk(1.0, 0.0), cmul(nk, ak)));
      const bool fin = isfinite(dl.x) && isfinite(dl.y);
      if (fin) lk = csub(lk, dl);
      // converged, or the corrections stopped shrinking at the rounding level
      const double a = fin ? cabsa(dl) : 0.0, al = cabsa(lk);
      done = a <= 1e-14 * al || (a >= prev && a <= 1e-10 * al);
      prev = a;
    }
    if (gballot(!done) == 0u) break;
  }
  // finite zeros only (the pencil's infinite eigenvalues are not zeros of
  // the denominator; a zero run off to infinity means sum w_j = 0)
  const bool finite_pole = l < nr && cabsa(lk) < 1e12 * (rad + cabsa(cen));
  double2 res = mk(0.0, 0.0);
  if (finite_pole) {
    const double2 sh[4] = {mk(kEps6, 0.0), mk(0.0, kEps6), mk(-kEps6, 0.0), mk(0.0, -kEps6)};
#pragma unroll
    for (int k = 0; k < 4; ++k)
      res = cadd(res, cmul(aaa_eval_at(cadd(lk, sh[k]), m, pos, val, wgt), sh[k]));
    res = mk(res.x / 4.0, res.y / 4.0);
  }
  const bool keep = finite_pole && cabsa(res) > thres;
  const uint32_t kmask = gballot(keep);
  const int cnt = __popc(kmask), half = M / 2;
  if (cnt > half) {
    if (l == 0) status[1] = 1;
    for (int s = l; s < M; s += kGrp) w[(int64_t)s * ne + e] = mk(NAN, NAN);
    return;
  }
  __syncwarp();
  if (keep) {
    const int k = __popc(kmask & (uint32_t)below(l));
    pos[k] = lk;   // the support points are no longer needed
    val[k] = res;
  }
  __syncwarp();
  for (int s = l; s < M; s += kGrp) {
    double2 v = mk(0.0, 0.0);
    if (s < cnt) v = pos[s];
    else if (s >= half && s < half + cnt) v = val[s - half];
    w[(int64_t)s * ne + e] = v;
  }
}

}  // namespace

void aaa_coeffs(int model, double thres, int64_t ne, int nfreq, const double2 *z,
                const int32_t *src, double2 *d_w, hipStream_t st) {
  SGW_REQUIRE(model == 4 || model == 5, SGW_E_ARG, "aaa: model 4 or 5");
  SGW_REQUIRE(nfreq >= 3 && nfreq <= kAaaMax, SGW_E_SHAPE, "aaa: 3 <= frequencies <= 64");
  AaaMesh mesh{};
  for (int i = 0; i < nfreq; ++i) {
    mesh.z[i] = z[i];
    mesh.src[i] = src ? src[i] : i;
  }
  // model 4: mmax = N / 3 support points at most (analytic.f90:174-175);
  // model 5: max_point = N, of which the device keeps N / 2 (beyond that the
  // Loewner submatrix has more columns than rows and its null vector is not
  // unique)
  const int max_point = model == 4 ? nfreq / 3 : nfreq;
  const int mcap = model == 4 ? nfreq / 3 : nfreq / 2;
  // Two elements share a wavefront while a CU's LDS holds more of them than its
  // SIMDs hold wavefronts (16); where it holds fewer, each has a wavefront of its
  // own, and a CU takes an odd number of them too.  A wavefront each against two
  // together: model 4 at 32 points (22 to a CU) 20.0 ms against 19.3, at 36
  // points (16) 38.7 against 42.2, at 64 (5) 113 against 187; model 5 at 24 points
  // (21) 37.4 against 35.8, at 36 (10) 180 against 240, at 64 (3) 633 against 1 415.
  const size_t one = sizeof(double2) * (size_t)aaa_lds(nfreq, mcap);  // <= 51200
  const int per = kLdsCu / one > 16 ? 2 : 1;
  const size_t lds = per * one;
  DevBuf<int32_t> status(2);
  SGW_HIP(hipMemsetAsync(status.p, 0, 2 * sizeof(int32_t), st));
  auto *kern = nfreq <= kGrp ? k_aaa_coeffs<1> : k_aaa_coeffs<2>;
  kern<<<(unsigned)((ne + per - 1) / per), kGrp * per, lds, st>>>(
      ne, nfreq, mesh, thres, model, max_point, mcap, d_w, status.p);
  SGW_HIP(hipGetLastError());
  int32_t h[2] = {0, 0};
  SGW_HIP(hipMemcpyAsync(h, status.p, sizeof(h), hipMemcpyDeviceToHost, st));
  SGW_HIP(hipStreamSynchronize(st));
  SGW_REQUIRE(h[0] == 0, SGW_E_STATE,
              "aaa: an element needs more than N/2 support points, or has NaN samples (its "
              "coefficients are NaN)");
  SGW_REQUIRE(h[1] == 0, SGW_E_STATE,
              "aaa: two many relevant poles, try reducing the coulomb threshold or increasing "
              "the number of frequencies (the element's coefficients are NaN)");
}

}  // namespace sgw
