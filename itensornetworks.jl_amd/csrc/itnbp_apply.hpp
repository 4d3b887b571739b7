// Declarations and device functions shared by the gate-application kernels:
// the LDS kernels (k_apply.hip) and the split pipeline (k_apply_big.hip).
#pragma once
#include <hip/hip_runtime.h>

#include <vector>

#include "itnbp_internal.hpp"
#include "itnbp_jacobi.hpp"

typedef double f64x4 __attribute__((ext_vector_type(4)));

constexpr int AP_XY = 8192;   // max E * n (external size x d chi_b) per side
// global scratch per side of a gate within the LDS limits: X of an explicit side, R,
// Tq, the environments' M^{-1/2} and P, flags
constexpr int AP_SIDE = AP_XY + 1024 + 1024 + 2 * 3 * 8 * 8 + 1;
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
  // per-phase timestamps (wall clock; 16 slots per gate), or null;
  // ITNBP_APPLY_PHASES=1
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

// ---- QR of a tall side by Gram matrices ---------------------------------------
// LDS of one elimination, n <= 16 NT
template <int NT>
struct CholLds {
  static constexpr int LD = 16 * NT + 1;
  double *U, *Mi, *rows, *piv;
  __device__ explicit CholLds(double* sm) {
    U = sm;
    Mi = U + 16 * NT * LD;
    rows = Mi + 16 * NT * LD;
    piv = rows + 64 * NT;
  }
  static constexpr size_t bytes() { return sizeof(double) * (2 * 16 * NT * LD + 64 * NT + 16 * NT); }
};

// [G | 1] reduced by Gaussian elimination without exchanges, G (n x n) symmetric:
// thread (ti, tj) = (tid % 16, tid / 16) of 256 holds elements (ti + 16 a, tj + 16 b)
// of both halves in registers; only the pivot row goes through LDS, one barrier
// per column.  With G = L D L^T: U[k][j >= k] = (D L^T)[k][j], Mi = L^{-1}, piv =
// diag D.  A column whose pivot is at most thr is skipped, its piv 0.
template <int NT>
__device__ void chol_eliminate(double (&g)[NT][NT], int n, double thr, const CholLds<NT>& L) {
  constexpr int NP = 16 * NT, LD = CholLds<NT>::LD;
  const int tid = threadIdx.x, ti = tid & 15, tj = tid >> 4;
  double m[NT][NT];
#pragma unroll
  for (int a = 0; a < NT; ++a)
#pragma unroll
    for (int b = 0; b < NT; ++b) m[a][b] = ti + 16 * a == tj + 16 * b ? 1.0 : 0.0;
  // rows: [parity][G row (NP) | M row (NP)]
  if (ti == 0)
#pragma unroll
    for (int b = 0; b < NT; ++b) {
      L.rows[tj + 16 * b] = g[0][b];
      L.rows[NP + tj + 16 * b] = m[0][b];
    }
  __syncthreads();
  for (int k = 0; k < n; ++k) {
    const double* rg = L.rows + (k & 1) * 2 * NP;
    double* nx = L.rows + ((k & 1) ^ 1) * 2 * NP;
    const double p = rg[k];
    const bool ok = p > thr;
    const double inv = ok ? 1 / p : 0.0;
    if (tid < NP) {
      L.U[k * LD + tid] = rg[tid];
      L.Mi[k * LD + tid] = rg[NP + tid];
      if (tid == 0) L.piv[k] = ok ? p : 0.0;
    }
    double gj[NT], mj[NT];
#pragma unroll
    for (int b = 0; b < NT; ++b) {
      gj[b] = rg[tj + 16 * b];
      mj[b] = rg[NP + tj + 16 * b];
    }
#pragma unroll
    for (int a = 0; a < NT; ++a) {
      const int i = ti + 16 * a;
      if (i <= k || i >= n) continue;
      const double f = rg[i] * inv;
#pragma unroll
      for (int b = 0; b < NT; ++b) {
        g[a][b] -= f * gj[b];
        m[a][b] -= f * mj[b];
      }
      if (i == k + 1)
#pragma unroll
        for (int b = 0; b < NT; ++b) {
          nx[tj + 16 * b] = g[a][b];
          nx[NP + tj + 16 * b] = m[a][b];
        }
    }
    __syncthreads();
  }
}

// One pass of the QR of a tall side, X = Q R from the Gram matrices G_p of X_p
// (X_0 = X, X_{p+1} = X_p R_p^{-1}): on return U holds R_p and Mi its inverse
// transposed.  Returns whether the pass was the last.
//
// Well-conditioned sides: two passes (CholeskyQR2), Q = X R_0^{-1} R_1^{-1} never
// formed, orthogonal to ~eps cond(X); taken while the pivots of G_0 span at most
// 1e-10 (R's diagonal 1e-5).  Past that the side turns explicit: each X_{p+1} is
// stored, and the first passes factor G_p + s 1, s = 4 n eps tr G_p, which is
// positive definite for every X and leaves X_{p+1} a condition number of at most
// ~sqrt(eps) times X_p's (shifted CholeskyQR, Fukaya, Kannan, Nakatsukasa,
// Yamamoto, Yanagisawa 2020); the pass after a well-conditioned G_p is the last.
// From pass 2 columns with a pivot at most n eps max diag are dropped (zero columns
// of Q and rows of R: directions below ~1e-20 of X).  X = Q R and Q^T Q = 1 then
// hold to a few eps for every cond(X), rank-deficient X among them, as with
// Householder reflectors.
template <int NT, int PASS>
__device__ bool chol_pass(double (&a)[NT][NT], int n, bool& expl, const CholLds<NT>& L) {
  constexpr double EPS = 2.220446049250313e-16;
  constexpr int LD = CholLds<NT>::LD;
  const int tid = threadIdx.x, ti = tid & 15, tj = tid >> 4;
  double keep[NT][NT];
  bool bad = false;
#pragma unroll
  for (int i = 0; i < NT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      keep[i][j] = a[i][j];
      bad = bad || !isfinite(a[i][j]);
      const int q = ti + 16 * i;
      if (q == tj + 16 * j && q < n) L.piv[q] = a[i][j];
    }
  if (__syncthreads_or(bad)) {
    // a NaN or Inf in psi or an environment: carried to Theta, which reports it
    for (int i = tid; i < n * LD; i += 256) {
      L.U[i] = NAN;
      L.Mi[i] = 0.0;
    }
    __syncthreads();
    return PASS > 0;
  }
  double tr = 0, mx = 0;
  for (int k = 0; k < n; ++k) {
    tr += L.piv[k];
    mx = fmax(mx, L.piv[k]);
  }
  __syncthreads();
  chol_eliminate<NT>(a, n, PASS < 2 ? 0.0 : n * EPS * mx, L);
  double pmin = INFINITY, pmax = 0;
  for (int k = 0; k < n; ++k) {
    if (PASS < 2 || L.piv[k] > 0) pmin = fmin(pmin, L.piv[k]);
    pmax = fmax(pmax, L.piv[k]);
  }
  bool fin = PASS == 3 || (PASS > 0 && (!expl || (pmin > 0.5 && pmax < 2.0)));
  if (PASS < 2 && !fin && !(pmin > 1e-10 * pmax)) {
    expl = true;
    const double s = 4 * n * EPS * tr;
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        const int q = ti + 16 * i;
        a[i][j] = keep[i][j] + (q == tj + 16 * j && q < n ? s : 0.0);
      }
    __syncthreads();
    chol_eliminate<NT>(a, n, 0.0, L);
  }
  for (int i = tid; i < n * n; i += 256) {
    const int k = i / n, j = i - k * n;
    const double p = L.piv[k], sc = p > 0 ? 1 / sqrt(p) : 0.0;
    L.U[k * LD + j] = j < k ? 0.0 : L.U[k * LD + j] * sc;
    L.Mi[k * LD + j] = j > k ? 0.0 : L.Mi[k * LD + j] * sc;
  }
  __syncthreads();
  return fin;
}

// ---- SVD of Theta -----------------------------------------------------------
// sum over the 8 or 16 lanes of a (half) DPP row, the same bits in every lane
template <int CTRL>
__device__ inline double dpp_mov_d(double x) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(x), CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(x), CTRL, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}
__device__ inline double row8_sum(double v) {
  v += dpp_mov_d<0xB1>(v);   // quad_perm 1 0 3 2
  v += dpp_mov_d<0x4E>(v);   // quad_perm 2 3 0 1
  v += dpp_mov_d<0x141>(v);  // row_half_mirror
  return v;
}
__device__ inline double row16_sum(double v) {
  v = row8_sum(v);
  v += dpp_mov_d<0x140>(v);  // row_mirror
  return v;
}

// LDS of gate_svd<NP>: X (NP x (NP + 16)) and the vectors behind it
template <int NP>
struct SvdLds {
  static constexpr int LD = NP + 16;
  double *X, *vbuf, *wmv, *svec;
  int *wmi, *perm, *order, *skeep;
  __device__ explicit SvdLds(double* sm) {
    X = sm;
    vbuf = X + NP * LD;
    wmv = vbuf + 2 * NP;
    svec = wmv + 16;
    wmi = reinterpret_cast<int*>(svec + NP);
    perm = wmi + 16;
    order = perm + NP;
    skeep = order + NP;
  }
  static constexpr size_t bytes() {
    return sizeof(double) * ((size_t)NP * LD + 2 * NP + 16 + NP) + sizeof(int) * (16 + 2 * NP + 4);
  }
};

// SVD and truncation of Theta (M x N, N <= M <= NP) by a workgroup of 8 NP
// threads; thread (c, h) = (tid / 8, tid % 8) passes rows h + 8 i of column c in a
// (zero outside).  Theta P = Q R by a Householder QR with column pivoting (the
// column in registers, the reflector through LDS), then one-sided Jacobi on X =
// R^T in LDS (16 lanes per column pair, one barrier per step; rounding floor and
// stopping rule of jacobi_svd), X <- U_x diag(s): V_Theta = P U_x.  A pair is rotated
// while |<a_p, a_q>| > eps sqrt(N) |a_p| |a_q|: what is left turns the kept vectors towards
// each other by as much over their values' relative gap.  With 8 eps sqrt(N) left the site
// tensors of an 8x8 chi = 16 round were 1.1e-12 to 3.0e-12 off in six runs, now 0.9e-12
// to 1.7e-12, in the same time: the last sweeps converge quadratically, so the
// threshold costs a sweep more in some matrices only (round 8.84 -> 8.87 ms).
// The pivoting grades the columns and halves the sweeps.  Theta is scaled by a
// power of two to order 1 first (exact).  On return L.X holds U_x in the kept
// columns, L.perm the pivots, L.svec the singular values, L.order their descending order;
// the truncation (maxdim, cutoff, the bond's layout lay) and the outputs of slot
// are done.  Returns the kept rank, -1 if the gate is refused.  A step is bound by
// its dependent chain (loads, reduction, rotation, barrier) up to NP = 64 and by
// LDS bandwidth at 128.
template <int NP>
__device__ int gate_svd(double (&a)[NP / 8], int M, int N, const SvdLds<NP>& L, const ApplyParams& prm, int lay,
                        int slot, double* truncerr, double* svals, int* kept, int* status) {
  constexpr int LD = SvdLds<NP>::LD, RW = NP / 8, NW = NP / 8, RB = NP / 32;
  constexpr double EPS = 2.220446049250313e-16;
  double* X = L.X;
  const int tid = threadIdx.x, c = tid >> 3, h = tid & 7;
  double mx = 0;
  bool bad = false;
#pragma unroll
  for (int i = 0; i < RW; ++i) {
    bad = bad || !isfinite(a[i]);
    mx = fmax(mx, fabs(a[i]));
  }
  for (int m = 32; m > 0; m >>= 1) mx = fmax(mx, __shfl_xor(mx, m));
  if ((tid & 63) == 0) L.wmv[tid >> 6] = mx;
  for (int i = tid; i < NP * LD; i += 8 * NP) X[i] = 0.0;
  if (__syncthreads_or(bad)) {  // a NaN or Inf in psi or an environment
    if (tid == 0) {
      truncerr[slot] = NAN;
      if (svals)
        for (int i = 0; i < prm.max_keep; ++i) svals[(long long)slot * prm.max_keep + i] = 0.0;
      if (kept) kept[slot] = prm.maxdim > 0 && prm.maxdim < N ? prm.maxdim : N;
      status[slot] = 2;
    }
    return -1;
  }
  mx = L.wmv[0];
#pragma unroll
  for (int q = 1; q < NW; ++q) mx = fmax(mx, L.wmv[q]);
  const int ex = mx > 0 ? ilogb(mx) : 0;
#pragma unroll
  for (int i = 0; i < RW; ++i) a[i] = ldexp(a[i], -ex);
  __syncthreads();
  bool done = c >= N;
  for (int j = 0; j < N; ++j) {
    // the remaining column of largest norm over rows >= j (ties: the smaller index)
    double part = 0;
#pragma unroll
    for (int i = 0; i < RW; ++i)
      if (h + 8 * i >= j) part += a[i] * a[i];
    double best = done ? -1.0 : row8_sum(part);
    int bi = c;
    for (int m = 8; m < 64; m <<= 1) {
      const double ob = __shfl_xor(best, m);
      const int oi = __shfl_xor(bi, m);
      if (ob > best || (ob == best && oi < bi)) {
        best = ob;
        bi = oi;
      }
    }
    if ((tid & 63) == 0) {
      L.wmv[tid >> 6] = best;
      L.wmi[tid >> 6] = bi;
    }
    __syncthreads();
    best = L.wmv[0];
    bi = L.wmi[0];
#pragma unroll
    for (int q = 1; q < NW; ++q) {
      const double ob = L.wmv[q];
      const int oi = L.wmi[q];
      if (ob > best || (ob == best && oi < bi)) {
        best = ob;
        bi = oi;
      }
    }
    double* v = L.vbuf + (j & 1) * NP;
    if (c == bi) {
#pragma unroll
      for (int i = 0; i < RW; ++i) {
        const int row = h + 8 * i;
        v[row] = a[i];
        if (row < j) X[j + LD * row] = a[i];  // X[j][row] = R[row][j]
      }
      if (h == 0) L.perm[j] = c;
      done = true;
    }
    __syncthreads();
    const double xjj = v[j];
    const double nrm = sqrt(best);
    const double alpha = xjj >= 0 ? -nrm : nrm;
    const double v0 = xjj - alpha;
    const double vv = best - xjj * xjj + v0 * v0;
    const double beta = (nrm == 0.0 || vv == 0.0) ? 0.0 : 2.0 / vv;
    if (tid == 0) X[j + LD * j] = beta != 0.0 ? alpha : xjj;
    double dot = 0;
#pragma unroll
    for (int i = 0; i < RW; ++i) {
      const int row = h + 8 * i;
      if (row >= j) dot += (row == j ? v0 : v[row]) * a[i];
    }
    dot = row8_sum(dot);
    if (!done) {
      const double f = beta * dot;
#pragma unroll
      for (int i = 0; i < RW; ++i) {
        const int row = h + 8 * i;
        if (row >= j) a[i] -= f * (row == j ? v0 : v[row]);
      }
    }
  }
  __syncthreads();
  // one-sided Jacobi on X (N x N, zero-padded rows)
  const int pi = tid >> 4, gl = tid & 15;
  double fro = 0;
#pragma unroll
  for (int q = 0; q < 2; ++q) {  // group pi: columns pi, pi + NP / 2
    const double* x = X + (pi + q * (NP / 2)) * LD;
#pragma unroll
    for (int m = 0; m < RB; ++m) {
      const double2 t = *reinterpret_cast<const double2*>(x + 2 * gl + 32 * m);
      fro += t.x * t.x + t.y * t.y;
    }
  }
  fro = block_sum_d(fro, L.wmv);
  const int ne = N + (N & 1), npair = ne / 2;
  const double tol = EPS * sqrt((double)N);
  const double tol2 = tol * tol, floor2 = EPS * EPS * fro;
  for (int sweep = 0; sweep < 60 && N > 1; ++sweep) {
    int rotated = 0;
    for (int st = 0; st < ne - 1; ++st) {
      if (pi < npair) {
        int p, q;
        rr_pair(ne, st, pi, p, q);
        if (q < N) {
          double* xp = X + p * LD + 2 * gl;
          double* xq = X + q * LD + 2 * gl;
          double2 ap[RB], aq[RB];
          double al = 0, be = 0, ga = 0;
#pragma unroll
          for (int m = 0; m < RB; ++m) {
            ap[m] = *reinterpret_cast<const double2*>(xp + 32 * m);
            aq[m] = *reinterpret_cast<const double2*>(xq + 32 * m);
            al += ap[m].x * ap[m].x + ap[m].y * ap[m].y;
            be += aq[m].x * aq[m].x + aq[m].y * aq[m].y;
            ga += ap[m].x * aq[m].x + ap[m].y * aq[m].y;
          }
          al = row16_sum(al);
          be = row16_sum(be);
          ga = row16_sum(ga);
          // |ga| > tol |p| |q|
          if (al > floor2 && be > floor2 && ga * ga > tol2 * al * be) {
            double cs, sn;
            jacobi_rotation(al, be, ga, cs, sn);
            rotated = 1;
#pragma unroll
            for (int m = 0; m < RB; ++m) {
              double2 np_, nq_;
              np_.x = cs * ap[m].x - sn * aq[m].x;
              np_.y = cs * ap[m].y - sn * aq[m].y;
              nq_.x = sn * ap[m].x + cs * aq[m].x;
              nq_.y = sn * ap[m].y + cs * aq[m].y;
              *reinterpret_cast<double2*>(xp + 32 * m) = np_;
              *reinterpret_cast<double2*>(xq + 32 * m) = nq_;
            }
          }
        }
      }
      __syncthreads();
    }
    if (!__syncthreads_or(rotated)) break;
  }
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int col = pi + q * (NP / 2);
    double s = 0;
#pragma unroll
    for (int m = 0; m < RB; ++m) {
      const double2 t = *reinterpret_cast<const double2*>(X + col * LD + 2 * gl + 32 * m);
      s += t.x * t.x + t.y * t.y;
    }
    s = row16_sum(s);
    if (gl == 0) L.svec[col] = sqrt(s);
  }
  __syncthreads();
  if (tid < N) {  // descending order, ties by index
    const double s = L.svec[tid];
    int r = 0;
    for (int m = 0; m < N; ++m)
      if (L.svec[m] > s || (L.svec[m] == s && m < tid)) ++r;
    L.order[r] = tid;
  }
  __syncthreads();
  if (tid == 0) {
    double tot = 0;
    for (int i = 0; i < N; ++i) tot += L.svec[i] * L.svec[i];
    int keep = N;
    if (prm.maxdim > 0 && keep > prm.maxdim) keep = prm.maxdim;
    double disc = 0;
    for (int i = keep; i < N; ++i) disc += L.svec[L.order[i]] * L.svec[L.order[i]];
    if (prm.cutoff >= 0 && tot > 0) {
      while (keep > 1 && (disc + L.svec[L.order[keep - 1]] * L.svec[L.order[keep - 1]]) / tot <= prm.cutoff) {
        disc += L.svec[L.order[keep - 1]] * L.svec[L.order[keep - 1]];
        --keep;
      }
    }
    int st = 0;
    if (keep > lay) st = 1;  // more than the bond's layout holds
    if (!isfinite(ldexp(tot, 2 * ex))) st = 2;  // the weight leaves the range
    truncerr[slot] = st == 2 ? NAN : (tot > 0 ? disc / tot : 0.0);
    if (svals)
      for (int i = 0; i < prm.max_keep; ++i)
        svals[(long long)slot * prm.max_keep + i] = i < keep ? ldexp(L.svec[L.order[i]], ex) : 0.0;
    if (kept) kept[slot] = keep;
    status[slot] = st;
    *L.skeep = st ? -1 : keep;
  }
  __syncthreads();
  const int keep = *L.skeep;
  if (keep < 0) return -1;
  // the kept columns of X over their singular values; the values back at Theta's
  // scale.  A column at the rounding level was not rotated against the others, so its
  // direction is noise with a part in theirs: zero, which Theta has along it
  for (int i = tid; i < N * keep; i += 8 * NP) {
    const int row = i % N, o = L.order[i / N];
    const double s = L.svec[o];
    X[row + LD * o] = s * s > floor2 ? X[row + LD * o] / s : 0.0;
  }
  __syncthreads();
  if (tid < N) L.svec[tid] = ldexp(L.svec[tid], ex);
  __syncthreads();
  return keep;
}

// ---- the split pipeline (k_apply_big.hip) -----------------------------------
// The launch sequences of nb gates (host items): the end of each, as many gates as its
// device workspace may take of budget bytes (at least one; a sequence's grids have two
// rows per gate, and a gate takes 0.7 MiB, so 16 GiB stay within 65535 rows).  bytes: the
// largest workspace.  One pass over the gates.
std::vector<int> apply_big_chunks(const itnbp_net* net, const ApplyItem* items, int nb, size_t budget, size_t& bytes);
// launches the gates: outputs per slot as the LDS kernel's; work holds
// the bytes of apply_big_chunks.  The uploaded table is added to tables, which the caller keeps
// until it has waited for the stream
int apply_big_run(itnbp_net* net, const ApplyItem* items, int nb, const double* d_gates, const ApplyParams& prm,
                  void* work, double* truncerr, double* svals, int* kept, int* status,
                  std::vector<std::vector<char>>& tables);
