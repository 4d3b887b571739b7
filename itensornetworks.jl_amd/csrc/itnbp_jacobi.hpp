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

// Symmetric n x n (n <= 32, row stride LD) eigendecomposition in LDS by 256 threads:
// A (entries of order 1 or below, zero past n up to an even n) is overwritten by
// diag(l), V (orthogonal on entry) times the rotations by the eigenvectors as
// columns.  Cyclic two-sided Jacobi with the round-robin pairs of rr_pair: a step
// derives the rotations in the first ne / 2 lanes, then thread (i, j) rotates the
// 2 x 2 block of row pair i and column pair j and two pairs of V.  Stops when the
// off-diagonal mass is below tol2 of the diagonal's or no longer decreases.  rc, rs:
// 16 doubles each, red: 8.
template <int LD>
__device__ inline void block_jacobi_eigh(double* A, double* V, int n, double tol2, double* rc, double* rs,
                                         double* red) {
  const int tid = threadIdx.x, ne = n + (n & 1), np = ne / 2;
  const int pi = tid >> 4, pj = tid & 15;
  double prev = INFINITY;
  for (int sweep = 0; sweep < 40 && n > 1; ++sweep) {
    double off = 0, dg = 0;
#pragma unroll
    for (int h = 0; h < 4; ++h) {
      const int i = (tid >> 5) + 8 * h, j = tid & 31;
      const double a = i < n && j < n ? A[i * LD + j] : 0.0;
      if (i != j)
        off += a * a;
      else
        dg += a * a;
    }
    for (int m = 32; m > 0; m >>= 1) {
      off += __shfl_xor(off, m);
      dg += __shfl_xor(dg, m);
    }
    if ((tid & 63) == 0) {
      red[tid >> 6] = off;
      red[4 + (tid >> 6)] = dg;
    }
    __syncthreads();
    off = (red[0] + red[1]) + (red[2] + red[3]);
    dg = (red[4] + red[5]) + (red[6] + red[7]);
    if (off <= tol2 * dg || off == 0.0 || off >= prev) break;
    prev = off;
    for (int st = 0; st < ne - 1; ++st) {
      if (tid < np) {
        int p, q;
        rr_pair(ne, st, tid, p, q);
        double c = 1, s = 0;
        const double apq = A[p * LD + q];  // the padding index of an odd n couples to nothing
        if (fabs(apq) > 1e-150) jacobi_rotation(A[p * LD + p], A[q * LD + q], apq, c, s);
        rc[tid] = c;
        rs[tid] = s;
      }
      __syncthreads();
      if (pj < np) {
        int p2, q2;
        rr_pair(ne, st, pj, p2, q2);
        const double c2 = rc[pj], s2 = rs[pj];
        double vp[2], vq[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          vp[h] = V[(pi + 16 * h) * LD + p2];
          vq[h] = V[(pi + 16 * h) * LD + q2];
        }
        if (pi < np) {
          int p1, q1;
          rr_pair(ne, st, pi, p1, q1);
          const double c1 = rc[pi], s1 = rs[pi];
          const double app = A[p1 * LD + p2], apq = A[p1 * LD + q2], aqp = A[q1 * LD + p2], aqq = A[q1 * LD + q2];
          const double bpp = c1 * app - s1 * aqp, bpq = c1 * apq - s1 * aqq;
          const double bqp = s1 * app + c1 * aqp, bqq = s1 * apq + c1 * aqq;
          A[p1 * LD + p2] = c2 * bpp - s2 * bpq;
          A[p1 * LD + q2] = s2 * bpp + c2 * bpq;
          A[q1 * LD + p2] = c2 * bqp - s2 * bqq;
          A[q1 * LD + q2] = s2 * bqp + c2 * bqq;
        }
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          V[(pi + 16 * h) * LD + p2] = c2 * vp[h] - s2 * vq[h];
          V[(pi + 16 * h) * LD + q2] = s2 * vp[h] + c2 * vq[h];
        }
      }
      __syncthreads();
    }
  }
  __syncthreads();
}
