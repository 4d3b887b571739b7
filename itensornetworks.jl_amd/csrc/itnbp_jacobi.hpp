// Device functions of the Jacobi eigenvalue and singular value kernels.
#pragma once
#include <hip/hip_runtime.h>

// Round-robin pairing: step st of a cyclic sweep over n (even) indices.
__device__ inline void rr_pair(int n, int st, int i, int& p, int& q) {
  // positions 0..n-1; position 0 fixed, others rotate
  // (pos - 1 + st) < 2 (n - 1): one conditional subtraction instead of a modulo
  auto at = [&](int pos) {
    if (pos == 0) return 0;
    const int x = pos - 1 + st;
    return 1 + (x >= n - 1 ? x - (n - 1) : x);
  };
  p = at(i);
  q = at(n - 1 - i);
  if (p > q) {
    int t = p;
    p = q;
    q = t;
  }
}

// 1 / sqrt(x) to a rounding error or two: the hardware estimate (~2^-23) and one
// step of third order
__device__ inline double rsqrt_d(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  const double e = fma(-x * y, y, 1.0);
  return fma(y * e, fma(e, 0.375, 0.5), y);
}

// The Jacobi rotation of a column pair with squared norms al, be and inner
// product ga != 0: tan 2 theta = 2 ga / (be - al), |theta| <= pi / 4; new columns
// c p - s q and s p + c q.  Two reciprocal roots in place of the textbook form's
// three divisions and two roots (launches of 28 SVDs of 64 x 64: 640 -> 504 us, of
// 10 of 128 x 128: 2.63 -> 2.05 ms).  al, be, ga of order 1 or below (the caller
// scales), so the squares stay in range.
__device__ inline void jacobi_rotation(double al, double be, double ga, double& c, double& s) {
  const double d = be - al, g2 = 2 * ga;
  const double ri = rsqrt_d(fma(d, d, g2 * g2));
  const double c2 = fma(0.5 * fabs(d), ri, 0.5);
  const double ci = rsqrt_d(c2);
  c = c2 * ci;
  const double t = 0.5 * g2 * ri * ci;
  s = d >= 0 ? t : -t;
}
