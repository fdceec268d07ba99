// Reductions over groups of W = 16, 32 or 64 consecutive lanes in the order of
// the butterfly v += v[lane ^ o], o = W/2 .. 1: every lane gets the same bits,
// and a group of W whose upper half holds zeros gets those of a group of W/2.
// All steps are vector instructions (row swaps, row rotations, quad
// permutations) instead of the LDS permutes of __shfl_xor, whose latency the
// short dependent chains of the per-element solvers cannot hide.  The lanes
// of a group execute these together.
#pragma once

#include <hip/hip_runtime.h>

namespace sgw {

namespace lanes {

template <int CTRL> __device__ inline int dpp(int v) {
  return __builtin_amdgcn_mov_dpp(v, CTRL, 0xF, 0xF, false);
}
template <int CTRL> __device__ inline double dpp(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = dpp<CTRL>((int)b), hi = dpp<CTRL>((int)(b >> 32));
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}
// the two operands of the butterfly step o for this lane, the same two in the
// same places on both lanes of a pair
struct Pair {
  double a, b;
};
struct PairI {
  int a, b;
};
template <int O> __device__ inline PairI step(int v) {
  if constexpr (O == 32) {
    const auto r = __builtin_amdgcn_permlane32_swap((unsigned)v, (unsigned)v, false, false);
    return {(int)r[0], (int)r[1]};
  } else if constexpr (O == 16) {
    const auto r = __builtin_amdgcn_permlane16_swap((unsigned)v, (unsigned)v, false, false);
    return {(int)r[0], (int)r[1]};
  } else {
    // after the steps above o, values repeat with period 2 o in a row of 16,
    // so a rotation by o reads lane ^ o
    constexpr int ctrl = O == 8 ? 0x128 : O == 4 ? 0x124 : O == 2 ? 0x4E : 0xB1;
    return {v, dpp<ctrl>(v)};
  }
}
template <int O> __device__ inline Pair step(double v) {
  const long long b = __double_as_longlong(v);
  const PairI lo = step<O>((int)b), hi = step<O>((int)(b >> 32));
  return {__longlong_as_double(((long long)hi.a << 32) | (unsigned int)lo.a),
          __longlong_as_double(((long long)hi.b << 32) | (unsigned int)lo.b)};
}

// a of the upper 32 lanes and b of the lower 32 change places
__device__ inline void swap_halves(double &a, double &b) {
  const long long x = __double_as_longlong(a), y = __double_as_longlong(b);
  const auto lo = __builtin_amdgcn_permlane32_swap((unsigned)x, (unsigned)y, false, false);
  const auto hi = __builtin_amdgcn_permlane32_swap((unsigned)(x >> 32), (unsigned)(y >> 32), false,
                                                   false);
  a = __longlong_as_double(((long long)hi[0] << 32) | (unsigned int)lo[0]);
  b = __longlong_as_double(((long long)hi[1] << 32) | (unsigned int)lo[1]);
}

template <int O, typename T, typename F> __device__ inline T fold(T v, F f) {
  if constexpr (O == 0) {
    return v;
  } else {
    const auto p = step<O>(v);
    return fold<O / 2>(f(p.a, p.b), f);
  }
}

template <int W> __device__ inline double sum(double v) {
  return fold<W / 2>(v, [](double a, double b) { return a + b; });
}
template <int W> __device__ inline double max(double v) {
  return fold<W / 2>(v, [](double a, double b) { return fmax(a, b); });
}
template <int W> __device__ inline int max(int v) {
  return fold<W / 2>(v, [](int a, int b) { return a > b ? a : b; });
}
template <int W> __device__ inline int min(int v) {
  return fold<W / 2>(v, [](int a, int b) { return a < b ? a : b; });
}

}  // namespace lanes
}  // namespace sgw
