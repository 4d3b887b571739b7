// Declarations and device functions shared by the gate-application kernels:
// the LDS kernel (k_apply.hip) and the split pipeline (k_apply_big.hip).
#pragma once
#include <hip/hip_runtime.h>

#include "itnbp_internal.hpp"

typedef double f64x4 __attribute__((ext_vector_type(4)));

constexpr int AP_XY = 8192;   // max E * n (external size x d chi_b) per side
// tall-skinny QR (E >= 4 n, n <= 16): the stacked R factors (4n x n) and the
// heads and betas of their reflectors, per side, after the side's reflectors
constexpr int AP_QRX = 4 * 16 * 16 + 4 * 16;
constexpr int AP_SIDE = AP_XY + AP_QRX;  // global scratch per side of a gate
constexpr int AP_TH = 32;     // max rows/cols of Theta (r d)
constexpr int AP_ENV = 8;     // max external bond dimension
constexpr int AP_MAXEXT = 3;  // max external bonds per side (degree 4)
constexpr int AP_SITE_D = 16; // max physical dimension of a one-site gate
// the split pipeline (k_apply_big.hip) for bonds past the LDS kernel's limits
constexpr int AP_ENV_BIG = 32;    // max external bond dimension
constexpr int AP_N_BIG = 64;      // max d chi_b
constexpr int AP_TH_BIG = 128;    // max rows/cols of Theta
constexpr int AP_KEEP_BIG = 64;   // max kept rank (the growth cap of itnbp_apply_gates)

struct ApplyItem {
  int u, v;      // vertices
  int ju, jv;    // bond axis at u, v
  long long gate;  // offset of the (d_u d_v)^2 gate
  int slot;
  int chib_in;     // bond dimension before the call (the layout may be grown past it)
};

struct ApplyParams {
  int maxdim;         // <= 0: none (still capped by the bond dimension)
  double cutoff;      // < 0: none
  int normalize;
  double eig_cutoff;  // map_eigvals cutoff (10 eps)
  int max_keep;       // stride of the singular value output
  // per-phase timestamps (wall clock; 16 slots per gate, slot 8 the SVD's
  // sweep count), or null; ITNBP_APPLY_PHASES=1
  unsigned long long* ts = nullptr;
};

__device__ inline double wave_sum_d(double v) {
  for (int m = 32; m > 0; m >>= 1) v += __shfl_xor(v, m);
  return v;
}

__device__ inline double block_sum_d(double v, double* red) {
  v = wave_sum_d(v);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  double s = 0;
  for (int i = 0; i < (int)(blockDim.x >> 6); ++i) s += red[i];
  __syncthreads();
  return s;
}

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

// One-sided Jacobi SVD of A (M x N, column-major, M >= N) in place:
// A <- U diag(s), V (N x N column-major) accumulated unless V is null.  A pair is rotated while
// |<a_p, a_q>| > tol |a_p| |a_q| with tol = 8 eps sqrt(M), the rounding error
// of the inner product itself, and while both columns are above the rounding
// level of A (|a|^2 > eps^2 ||A||_F^2): a column at that level is zero to
// working precision, and rotating it against its rounding noise would keep
// the sweeps going.  The pairs of a step are disjoint and each group of G
// threads reads and writes only its own rows of its pair, so a step needs one
// barrier (before the next step's pairing).  Returns the number of sweeps.
__device__ inline int jacobi_svd(double* A, int M, int N, double* V, double* rot, double* red) {
  const int tid = threadIdx.x;
  if (V)
    for (int i = tid; i < N * N; i += blockDim.x) V[i] = (i % N == i / N) ? 1.0 : 0.0;
  double fro = 0;
  for (int i = tid; i < M * N; i += blockDim.x) fro += A[i] * A[i];
  fro = block_sum_d(fro, red);
  if (N == 1) return 0;
  const int ne = N + (N & 1);
  const double tol = 8 * 2.220446049250313e-16 * sqrt((double)M);
  const double floor2 = 2.220446049250313e-16 * 2.220446049250313e-16 * fro;
  int sweep = 0;
  for (; sweep < 60; ++sweep) {
    int rotated = 0;
    for (int st = 0; st < ne - 1; ++st) {
      // each pair handled by a group of G threads
      // (the largest power of two <= 64 with G npair <= blockDim.x: every pair
      // has a group for N <= 2 blockDim.x)
      const int npair = ne / 2;
      int G = 64;
      while (G > 1 && G * npair > (int)blockDim.x) G >>= 1;
      const int pi = tid / G, gl = tid % G;
      double alpha = 0, beta = 0, gamma = 0;
      int p = 0, q = 0;
      const bool active = pi < npair;
      if (active) {
        rr_pair(ne, st, pi, p, q);
        if (q < N) {
          for (int i = gl; i < M; i += G) {
            const double ap = A[i + (long long)M * p], aq = A[i + (long long)M * q];
            alpha += ap * ap;
            beta += aq * aq;
            gamma += ap * aq;
          }
        }
      }
      for (int m = G / 2; m > 0; m >>= 1) {
        alpha += __shfl_xor(alpha, m);
        beta += __shfl_xor(beta, m);
        gamma += __shfl_xor(gamma, m);
      }
      double c = 1, s = 0;
      if (active && q < N && alpha > floor2 && beta > floor2 && fabs(gamma) > tol * sqrt(alpha * beta)) {
        const double zeta = (beta - alpha) / (2 * gamma);
        const double t = (zeta >= 0 ? 1.0 : -1.0) / (fabs(zeta) + sqrt(1 + zeta * zeta));
        c = 1 / sqrt(1 + t * t);
        s = c * t;
        rotated = 1;
      }
      if (active && q < N && s != 0.0) {
        for (int i = gl; i < M; i += G) {
          const double ap = A[i + (long long)M * p], aq = A[i + (long long)M * q];
          A[i + (long long)M * p] = c * ap - s * aq;
          A[i + (long long)M * q] = s * ap + c * aq;
        }
        if (V)
          for (int i = gl; i < N; i += G) {
            const double vp = V[i + N * p], vq = V[i + N * q];
            V[i + N * p] = c * vp - s * vq;
            V[i + N * q] = s * vp + c * vq;
          }
      }
      __syncthreads();
    }
    // a barrier that also tells every thread whether any pair rotated (no
    // shared flag to reset, so no thread can see the next sweep's reset)
    if (!__syncthreads_or(rotated)) break;
  }
  return sweep + 1;
}

// ---- the split pipeline (k_apply_big.hip) -----------------------------------
// device workspace of nb gates (host items) of one launch sequence, in bytes
size_t apply_big_bytes(const itnbp_net* net, const ApplyItem* items, int nb);
// launches the gates: outputs per slot as the LDS kernel's; work holds
// apply_big_bytes bytes
int apply_big_run(itnbp_net* net, const ApplyItem* items, int nb, const double* d_gates, const ApplyParams& prm,
                  void* work, double* truncerr, double* svals, int* kept, int* status);
