// 6-D Fourier transforms of two-point functions (fft6.f90), callable from
// other translation units of the library.
#pragma once

#include "sgw_internal.h"
#include "spherefft.h"

namespace sgw {

struct Fft6Args {
  int n, n_p, num_g, num_g_p;
  const int32_t *nl, *nl_p;  // device box-index maps of the two G lists
  double omega;              // cell volume
  int nmat;
  double2 *f;                // nmat matrices f(nr, nr_p), Fortran layout
};

void fft6_check(const Fft6Args &a, const char *who);

// The two G lists on the host and, where the box kernels of spherefft.h take
// them, as sphere lists on the device.  Reads the maps back from the device
// (synchronises `st`) and rejects indices outside the boxes.
struct Fft6Lists {
  Fft6Lists(hipStream_t st, const Fft6Args &a, const char *who);
  std::vector<int32_t> nl, nl_p;
  SphereList r, r_p;
};

// Scratch of one matrix: S[g][r'] (num_g x n_p^3).  One matrix at a time on
// `st`; the parts below work on matrix f(ldf, *) with its block at the top
// left.  rows: the r' side, S[g] = box FFT of the rows of f, and back.
void invfft6_rows(hipStream_t st, const Fft6Args &a, const Fft6Lists &l, const double2 *f,
                  int64_t ldf, double2 *s);
void fwfft6_rows(hipStream_t st, const Fft6Args &a, const Fft6Lists &l, double2 *s,
                 SphereOut out);

}  // namespace sgw
