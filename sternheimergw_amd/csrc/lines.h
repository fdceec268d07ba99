// One line of a box FFT as a lane, or a lane pair, holds it.
#pragma once

#include "regfft.h"
#include "sgw_internal.h"
#include "splitfft.h"

namespace sgw {

// Sides divisible by four split every line over a lane pair (splitfft.h): half
// the registers per lane, so twice the waves hide the LDS exchanges between
// the stages.  Other sides keep a line in one lane.
constexpr bool split_side(int n) { return n % 4 == 0; }
// values of a line in one lane
constexpr int lane_values(int n) { return split_side(n) ? n / 2 : n; }

// Values outside a run of cnt are read at its nearest end (or its first place,
// if it is empty) and replaced by zero: loads under a condition are waited
// for one by one.
__device__ inline int within(int k, int cnt) { return max(0, min(k, cnt - 1)); }
__device__ inline double2 keep(double2 v, int k, int cnt) {
  const bool in = k >= 0 && k < cnt;
  return mk(in ? v.x : 0.0, in ? v.y : 0.0);
}

// A line's values in this lane: value i is point dec(i) of a transform's
// decimated side and point nat(i) of its natural side; dit goes from the
// first to the second, dif back.
template <int N> struct Line {
  static constexpr bool S = split_side(N);
  static constexpr int E = lane_values(N), H = N / 2, Q = N / 4;
  int odd;
  __device__ int dec(int i) const { return S ? 2 * i + odd : i; }
  __device__ int nat(int i) const { return S ? (i < Q ? i : H + i - Q) + Q * odd : i; }
  template <int SIGN> __device__ void dit(double2 (&x)[E]) const {
    if constexpr (S) split_dit<N, SIGN>(x, odd);
    else reg_fft<N, SIGN>(x);
  }
  template <int SIGN> __device__ void dif(double2 (&x)[E]) const {
    if constexpr (S) split_dif<N, SIGN>(x, odd);
    else reg_fft<N, SIGN>(x);
  }
};

}  // namespace sgw
