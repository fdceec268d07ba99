// 3-D FFTs of cubic boxes whose reciprocal-space side is a short list of box
// positions (a G sphere), one box per workgroup from list to real space and
// back without an intermediate in memory.
#pragma once

#include <vector>

#include "sgw_internal.h"

namespace sgw {

// The list's occupied (x, y) columns and y rows, on the host and, after
// upload(), on the device.  Valid while the object lives.
class SphereList {
 public:
  SphereList() = default;
  // nl[g], g < num_g: box index x + n (y + n z) of every list element
  SphereList(int n, const std::vector<int32_t> &nl);
  // whether the kernels run for this side and list (their LDS holds the
  // columns and one wave's share of the planes); the caller has another path
  bool fits() const { return fits_; }
  void upload(hipStream_t st);

  int n() const { return n_; }
  int num_g() const { return num_g_; }
  int ncol() const { return ncol_; }
  int nrow() const { return nrow_; }
  size_t lds() const { return lds_; }
  const int32_t *d_ent() const { return d_.p; }
  const uint32_t *d_map() const { return reinterpret_cast<const uint32_t *>(d_.p + num_g_); }

 private:
  int n_ = 0, num_g_ = 0, ncol_ = 0, nrow_ = 0;
  bool fits_ = false;
  size_t lds_ = 0;
  std::vector<int32_t> h_;   // ent[num_g], then the index tables
  DevBuf<int32_t> d_;
};

// real[b][n^3] = FFT_sign of the box that holds in_scale * in[g * in_sg + b]
// at the list's positions and zeros elsewhere, b < nvec
void sphere_inv(hipStream_t st, const SphereList &l, int64_t nvec, int sign, const double2 *in,
                int64_t in_sg, double in_scale, double2 *real);
// v = out_scale * FFT_sign(real[b])[list], then with alpha: v = alpha v;
// out[g * out_sg + b] = v (out may be null), sum[g * sum_sg + b] += v (may be null)
struct SphereOut {
  double scale = 1.0;
  double2 *out = nullptr;
  int64_t out_sg = 0;
  bool has_alpha = false;
  double2 alpha{1.0, 0.0};
  double2 *sum = nullptr;
  int64_t sum_sg = 0;
};
void sphere_fwd(hipStream_t st, const SphereList &l, int64_t nvec, int sign, const double2 *real,
                const SphereOut &o);
// out = list values of FFT_{-sign}(g[b] * FFT_sign(box of in)); out may be in
void sphere_prod(hipStream_t st, const SphereList &l, int64_t nvec, int sign, const double2 *in,
                 int64_t in_sg, const double2 *g, const SphereOut &o);

}  // namespace sgw
