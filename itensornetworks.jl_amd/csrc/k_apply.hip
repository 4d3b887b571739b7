// BP-gauged two-site gate application (simple update) on the device.
//
// Semantics: ITensors.apply(o, psi; envs, maxdim, cutoff, normalize) with a
// product environment (src/apply.jl:97-146) -> simple_update_bp (src/apply.jl:33-95):
//   1. every environment message M (chi x chi, Hermitian) -> sqrt(M) and M^{-1/2}
//      by a Hermitian eigendecomposition with the eigenvalue truncation
//      cutoff = 10 eps (map_eigvals, src/apply.jl:9-25);
//   2. psi_u~ = psi_u with sqrt(M) on every external bond, reshaped to
//      X_u (external bonds) x (s_u, b_uv), QR X_u = Q_u R_u (src/apply.jl:74-75);
//   3. Theta = gate * (R_u R_v) over b_uv (src/apply.jl:78), SVD, truncation to
//      maxdim / cutoff with truncerr = discarded weight (src/apply.jl:81-89);
//   4. psi_u' = (Q_u with M^{-1/2} on the external bonds) U sqrt(S), likewise
//      psi_v' with sqrt(S) V^T (src/apply.jl:90-93); optional normalisation
//      (src/apply.jl:134-137).
// The bonds of one call are disjoint.  Within the LDS limits (external bonds <= 8,
// a side of at most 8192 elements, Theta <= 32 x 32) a call is two launches: one
// workgroup per side up to R, one per bond from Theta on; larger bonds run the
// split pipeline (k_apply_big.hip).  Small dense linear algebra: two-sided Jacobi
// in registers for the environment eigenproblems (one wave each), QR by Gram
// matrices on the matrix cores (chol_pass), one-sided (Hestenes) Jacobi SVD in LDS
// (gate_svd).  120 gates of a chi = 8 colour class: 910 us in one launch with
// Householder QR and the SVD on one wave -> 77 + 225 us.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <string>
#include <vector>

#include "itnbp_apply.hpp"
#include "itnbp_ops.hpp"

namespace {

// thread 0 of the workgroup records the end of phase ph (0: start)
__device__ inline void phase_mark(const ApplyParams& prm, int gate, int ph) {
  if (prm.ts && threadIdx.x == 0) prm.ts[gate * 16 + ph] = wall_clock64();
}

// sqrt(M), M^{-1/2} and the projector P on the kept eigenvectors of a symmetrised
// chi x chi message (column-major in global), chi <= 8, by one wave: lane i ne + j
// (ne = chi rounded up to even) holds A[i][j] and V[i][j] in registers.  Cyclic
// two-sided Jacobi with round-robin pairs (rr_pair's schedule), every lane deriving
// the rotations of its row pair and column pair from the pre-step matrix through
// shuffles, so a step needs no LDS and no barrier; stops when the off-diagonal mass
// is below 1e-30 of the diagonal's or stops decreasing (at most 40 sweeps).  Then
// the eigenvalue truncation of map_eigvals (cutoff = 10 eps, src/apply.jl:9-25),
// recomputed identically by every lane.  M is scaled by an even power of two to
// order 1 for jacobi_rotation.  S, Si and P row-major, ld chi; returns whether
// eigenvalues were dropped (P != 1).
__device__ bool env_roots_wave(const double* M, int chi, double cutoff, double* S, double* Si, double* P) {
  const int l = threadIdx.x & 63;
  const int ne = chi + (chi & 1);
  const bool live = l < ne * ne;
  const int i = live ? l / ne : 0, j = live ? l % ne : 0;
  const bool in = live && i < chi && j < chi;
  double a = in ? 0.5 * (M[i + chi * j] + M[j + chi * i]) : 0.0;
  double v = (live && i == j) ? 1.0 : 0.0;
  double mx = fabs(a);
  for (int m = 32; m > 0; m >>= 1) mx = fmax(mx, __shfl_xor(mx, m));
  const int ex = mx > 0 && isfinite(mx) ? ilogb(mx) & ~1 : 0;
  a = ldexp(a, -ex);
  if (chi > 1) {
    auto rot = [&](int p, int q, double& c, double& sn) {
      const double app = __shfl(a, p * ne + p), aqq = __shfl(a, q * ne + q), apq = __shfl(a, p * ne + q);
      c = 1.0;
      sn = 0.0;
      if (q < chi && fabs(apq) > 1e-150) jacobi_rotation(app, aqq, apq, c, sn);
    };
    double prev = INFINITY;
    for (int sweep = 0; sweep < 40; ++sweep) {
      double off = (in && i != j) ? a * a : 0.0, diag = (in && i == j) ? a * a : 0.0;
      for (int m = 32; m > 0; m >>= 1) {
        off += __shfl_xor(off, m);
        diag += __shfl_xor(diag, m);
      }
      // converged, or the off-diagonal mass no longer decreases (rounding level)
      if (off <= 1e-30 * diag || off == 0.0 || off >= prev) break;
      prev = off;
      for (int st = 0; st < ne - 1; ++st) {
        // partner of index x in step st of the round-robin schedule (rr_pair)
        // (x - 1 - st) lies in (-(ne - 1), ne - 1) and (pp - 1 + st) in [0, 2 (ne - 1)):
        // conditional corrections instead of modulos
        auto partner = [&](int x) {
          int t = x - 1 - st;
          if (t < 0) t += ne - 1;
          const int pos = x == 0 ? 0 : 1 + t;
          const int pp = ne - 1 - pos;
          int u = pp - 1 + st;
          if (u >= ne - 1) u -= ne - 1;
          return pp == 0 ? 0 : 1 + u;
        };
        const int ri = partner(i), cj = partner(j);
        double cr, sr, cc, sc;
        rot(i < ri ? i : ri, i < ri ? ri : i, cr, sr);
        rot(j < cj ? j : cj, j < cj ? cj : j, cc, sc);
        const double ao = __shfl(a, ri * ne + j);  // rows: A <- J^T A
        const double ar = i < ri ? cr * a - sr * ao : sr * ao + cr * a;
        const double aro = __shfl(ar, i * ne + cj), vo = __shfl(v, i * ne + cj);  // columns: A J, V J
        a = j < cj ? cc * ar - sc * aro : sc * aro + cc * ar;
        v = j < cj ? cc * v - sc * vo : sc * vo + cc * v;
      }
    }
  }
  double w[AP_ENV];
#pragma unroll
  for (int m = 0; m < AP_ENV; ++m) w[m] = __shfl(a, (m < ne ? m : 0) * ne + (m < ne ? m : 0));
  // truncation: rank |lambda| descending (ties by index); drop from the small
  // end while the dropped weight / total <= cutoff (keep >= 1).  Fully
  // unrolled over AP_ENV, with no run-time index into w, so that w stays in
  // registers.
  int rank[AP_ENV];
  double tot = 0;
#pragma unroll
  for (int m = 0; m < AP_ENV; ++m) {
    int r = 0;
#pragma unroll
    for (int m2 = 0; m2 < AP_ENV; ++m2)
      if (m2 < chi && (fabs(w[m2]) > fabs(w[m]) || (fabs(w[m2]) == fabs(w[m]) && m2 < m))) ++r;
    rank[m] = r;
    if (m < chi) tot += fabs(w[m]);
  }
  // the value of rank r, and the dropped prefix from the small end
  auto by_rank = [&](int r) {
    double x = 0;
#pragma unroll
    for (int m = 0; m < AP_ENV; ++m)
      if (m < chi && rank[m] == r) x = fabs(w[m]);
    return x;
  };
  int keep = chi;
  double disc = 0;
  while (keep > 1 && tot > 0 && (disc + by_rank(keep - 1)) / tot <= cutoff) {
    disc += by_rank(keep - 1);
    --keep;
  }
  unsigned kmask = 0;
#pragma unroll
  for (int m = 0; m < AP_ENV; ++m)
    if (m < chi && rank[m] < keep) kmask |= 1u << m;
  // S[r][c] = sum_m V[r][m] V[c][m] sqrt(l_m) over the kept m (lane (r, c) = (i, j))
  double sv = 0, siv = 0, pv = 0;
  for (int m = 0; m < AP_ENV; ++m) {
    const int mm = m < ne ? m : 0;
    const double vr = __shfl(v, i * ne + mm), vc = __shfl(v, j * ne + mm);
    if (m < chi && ((kmask >> m) & 1u)) {
      const double sq = sqrt(w[m]);  // NaN for a kept negative eigenvalue
      sv += vr * vc * sq;
      siv += vr * vc / sq;
      pv += vr * vc;
    }
  }
  if (in) {
    S[i * chi + j] = ldexp(sv, ex / 2);
    Si[i * chi + j] = ldexp(siv, -ex / 2);
    P[i * chi + j] = pv;
  }
  return keep < chi;
}

struct SideGeom {
  int d, k, j, chib, E, n, r;
  int dims[ITNBP_MAXR];
  int ext[AP_MAXEXT];  // external axes in order
  int next;
  long long psi_off;
  FastDiv fE, fd, fdim[ITNBP_MAXR];
  // external axis pa: stride of its index in e, its dimension, and their product
  FastDiv fst[AP_MAXEXT], fchi[AP_MAXEXT];
};

__device__ SideGeom side_geom(const VDesc& V, int j) {
  SideGeom g;
  g.d = V.dims[0];
  g.k = V.k;
  g.j = j;
  g.chib = V.dims[j];
  g.E = 1;
  g.next = 0;
  for (int a = 0; a <= V.k; ++a) g.dims[a] = V.dims[a];
  for (int a = 1; a <= V.k; ++a)
    if (a != j) {
      g.ext[g.next++] = a;
      g.E *= V.dims[a];
    }
  g.n = g.d * g.chib;
  g.r = g.E < g.n ? g.E : g.n;
  g.psi_off = V.psi_off;
  g.fE = fast_div(g.E);
  g.fd = fast_div(g.d);
  for (int a = 0; a < ITNBP_MAXR; ++a) g.fdim[a] = fast_div(a <= V.k ? V.dims[a] : 1);
  int st = 1;
  for (int pa = 0; pa < AP_MAXEXT; ++pa) {
    const int chi = pa < g.next ? V.dims[g.ext[pa]] : 1;
    g.fst[pa] = fast_div(st);
    g.fchi[pa] = fast_div(chi);
    st *= chi;
  }
  return g;
}

// natural offset of psi element (s, external multi-index e, bond b)
__device__ inline int nat_off(const SideGeom& g, int s, int e, int b) {
  int off = 0, stride = g.d, rem = e;
  for (int a = 1; a <= g.k; ++a) {
    int x;
    if (a == g.j) {
      x = b;
    } else {
      const int q = (int)g.fdim[a].div(rem);
      x = rem - q * g.dims[a];
      rem = q;
    }
    off += stride * x;
    stride *= g.dims[a];
  }
  return s + off;
}

// ---- gates within the LDS limits ------------------------------------------------
// Two launches over the gates of a call: k_gate_side, one workgroup per side, and
// k_gate_pair, one per bond.  Side s of a gate leaves in work (AP_SIDE doubles):
constexpr int AP_W_R = AP_XY;             // R, r x n
constexpr int AP_W_TQ = AP_W_R + 1024;    // Tq, n x n: Q = X Tq
constexpr int AP_W_SI = AP_W_TQ + 1024;   // M^{-1/2} per external bond, then P
constexpr int AP_W_FLAG = AP_W_SI + 2 * AP_MAXEXT * AP_ENV * AP_ENV;  // bits 0 .. 2: P != 1 on that bond; 3: explicit
static_assert(AP_W_FLAG + 1 == AP_SIDE, "layout of a side's workspace");
// work[0 .. AP_XY): the last X_p of an explicit side (chol_pass), E x n

// One side's matrix: rows e over the external bonds, columns c = s + d b.
struct ApSide {
  int d, chib, lay, lo, E, n, r, next;  // lay: the bond's layout (>= chib); lo: product of the bonds before it
  int chi[AP_MAXEXT], est[AP_MAXEXT];   // external bonds: dimension, stride in e
  long long psi_off;
  FastDiv fd, flo, flay, fE, fper[AP_MAXEXT], fest[AP_MAXEXT];
};

__device__ void ap_side(const VDesc& V, int j, int chib, ApSide& g) {
  g.d = V.dims[0];
  g.chib = chib;
  g.lay = V.dims[j];
  g.lo = 1;
  g.E = 1;
  g.next = 0;
  for (int a = 1; a <= V.k; ++a) {
    if (a == j) continue;
    if (a < j) g.lo *= V.dims[a];
    g.chi[g.next] = V.dims[a];
    g.est[g.next] = g.E;
    g.fest[g.next++] = fast_div(g.E);
    g.E *= V.dims[a];
  }
  for (int pa = 0; pa < g.next; ++pa) g.fper[pa] = fast_div(g.E / g.chi[pa]);
  g.n = g.d * chib;
  g.r = g.E < g.n ? g.E : g.n;
  g.psi_off = V.psi_off;
  g.fd = fast_div(g.d);
  g.flo = fast_div(g.lo);
  g.flay = fast_div(g.lay);
  g.fE = fast_div(g.E);
}

// pitch of a column of E rows in LDS: 2 mod 32 doubles, so that the operand
// fragments of v_mfma_f64_16x16x4f64 (16 columns x 4 rows, 4 columns x 16 rows) meet
// no bank twice per access
__host__ __device__ inline int ap_pitch(int E) { return (E + 29) / 32 * 32 + 2; }

// element (c, e) of the side behind entry i of the site tensor, in its memory
// order; false for the layout's columns past chib
__device__ inline bool ap_locate(const ApSide& g, int i, int& c, int& e, int& b) {
  const int t = (int)g.fd.div(i), u = (int)g.flo.div(t), h = (int)g.flay.div(u);
  b = u - h * g.lay;
  c = i - t * g.d + g.d * b;
  e = t - u * g.lo + g.lo * h;
  return b < g.chib;
}

__device__ void ap_load(const ApSide& g, const double* __restrict__ src, double* X, int P) {
  const int D = g.E * g.d * g.lay;
#pragma unroll 8
  for (int i = threadIdx.x; i < D; i += 256) {
    const double x = src[i];
    int c, e, b;
    if (ap_locate(g, i, c, e, b)) X[c * P + e] = x;
  }
}

// Mode product on external bond pa of the first n columns, in place: a wave owns 16
// fibres, loads their chi <= 8 entries as B operands (B[k = b][fibre]), K stays in
// registers as A operand (A[b'][b]); four groups of fibres in flight per iteration.
__device__ void ap_mode(const ApSide& g, int pa, double* X, int P, int n, const double* K) {
  const int l = threadIdx.x & 63, li = l & 15, lk = l >> 4, wv = threadIdx.x >> 6;
  const int chi = g.chi[pa], st = g.est[pa], per = (int)g.fper[pa].d, nfib = per * n;
  const double a0 = (lk < chi && li < chi) ? K[lk * chi + li] : 0.0;
  const double a1 = (4 + lk < chi && li < chi) ? K[(4 + lk) * chi + li] : 0.0;
  for (int f0 = 64 * wv; f0 < nfib; f0 += 256) {
    double x0[4], x1[4];
    int base[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int f = f0 + 16 * q + li;
      if (f < nfib) {
        const int c = (int)g.fper[pa].div(f), t = f - c * per, hi = (int)g.fest[pa].div(t);
        base[q] = c * P + (t - hi * st) + st * chi * hi;
      } else
        base[q] = -1;
      x0[q] = base[q] >= 0 && lk < chi ? X[base[q] + st * lk] : 0.0;
      x1[q] = base[q] >= 0 && 4 + lk < chi ? X[base[q] + st * (4 + lk)] : 0.0;
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      f64x4 acc = {0, 0, 0, 0};
      acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, x0[q], acc, 0, 0, 0);
      if (chi > 4) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, x1[q], acc, 0, 0, 0);
      if (base[q] >= 0 && lk < chi) X[base[q] + st * lk] = acc[0];
      if (base[q] >= 0 && 4 + lk < chi) X[base[q] + st * (4 + lk)] = acc[1];
    }
  }
  __syncthreads();
}

// Gram matrix of X (NEXT: of X Tn, Tn[c][k] = Mi[k][c], which STORE writes over X) by
// the workgroup; the element (ti + 16 a, tj + 16 b) of chol_eliminate's thread to
// g.  sum: NT (NT + 1) / 2 tiles of 256.
template <int NT, bool NEXT>
__device__ void ap_gram(const ApSide& g, double* X, int P, const CholLds<NT>& L, bool store, double* sum,
                        double (&out)[NT][NT]) {
  constexpr int LD = CholLds<NT>::LD, NTILE = NT * (NT + 1) / 2;
  const int tid = threadIdx.x, l = tid & 63, wv = tid >> 6, li = l & 15, lk = l >> 4;
  const int E = g.E, n = g.n;
  f64x4 acc[NTILE];
#pragma unroll
  for (int t = 0; t < NTILE; ++t) acc[t] = f64x4{0, 0, 0, 0};
  double tn[NT][4 * NT];
  if constexpr (NEXT) {
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int q = 0; q < 4 * NT; ++q) {
        const int c = 4 * q + lk, k = 16 * t + li;
        tn[t][q] = c < n && k < n ? L.Mi[k * LD + c] : 0.0;
      }
  }
  for (int r0 = 16 * wv; r0 < E; r0 += 64) {
    f64x4 x1[NT];
    if constexpr (NEXT) {
#pragma unroll
      for (int t = 0; t < NT; ++t) x1[t] = f64x4{0, 0, 0, 0};
#pragma unroll
      for (int q = 0; q < 4 * NT; ++q) {
        const double a = r0 + li < E && 4 * q + lk < n ? X[(4 * q + lk) * P + r0 + li] : 0.0;
#pragma unroll
        for (int t = 0; t < NT; ++t) x1[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, tn[t][q], x1[t], 0, 0, 0);
      }
      if (store)  // a wave reads and writes its own rows
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
          for (int v = 0; v < 4; ++v)
            if (16 * t + li < n && r0 + 4 * v + lk < E) X[(16 * t + li) * P + r0 + 4 * v + lk] = x1[t][v];
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      double op[NT];
#pragma unroll
      for (int t = 0; t < NT; ++t)
        op[t] = NEXT ? x1[t][v]
                     : (16 * t + li < n && r0 + 4 * v + lk < E ? X[(16 * t + li) * P + r0 + 4 * v + lk] : 0.0);
      int k = 0;
#pragma unroll
      for (int a = 0; a < NT; ++a)
#pragma unroll
        for (int b = a; b < NT; ++b, ++k)
          acc[k] = __builtin_amdgcn_mfma_f64_16x16x4f64(op[a], op[b], acc[k], 0, 0, 0);
    }
  }
  for (int q = 0; q < 4; ++q) {  // the four waves' tiles, summed in wave order
    __syncthreads();
    if (wv == q)
#pragma unroll
      for (int k = 0; k < NTILE; ++k)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          double* p = sum + k * 256 + v * 64 + l;
          *p = (q == 0 ? 0.0 : *p) + acc[k][v];
        }
  }
  __syncthreads();
  const int ti = tid & 15, tj = tid >> 4;
#pragma unroll
  for (int a = 0; a < NT; ++a)
#pragma unroll
    for (int b = 0; b < NT; ++b) {
      // tile (a, b), a <= b, row i, column j: value i / 4 of lane 16 (i % 4) + j
      const int ta = a < b ? a : b, tb = a < b ? b : a, i = a <= b ? ti : tj, j = a <= b ? tj : ti;
      out[a][b] = sum[(ta * NT - ta * (ta - 1) / 2 + tb - ta) * 256 + (i >> 2) * 64 + (i & 3) * 16 + j];
    }
}

// One pass of the side's QR: R <- R_p R, the next T or (true) the final Tq.
template <int NT, int PASS>
__device__ bool ap_qr_pass(const ApSide& g, double* X, int P, const CholLds<NT>& L, double* T, double* R,
                           double* Tq, bool& expl) {
  constexpr int LD = CholLds<NT>::LD;
  const int tid = threadIdx.x, n = g.n;
  double a[NT][NT];
  ap_gram<NT, (PASS > 0)>(g, X, P, L, expl, L.U, a);  // U is free here, Mi holds the last T
  const bool fin = chol_pass<NT, PASS>(a, n, expl, L);
  double t[NT * NT];
#pragma unroll
  for (int q = 0; q < NT * NT; ++q) {
    const int i = tid + 256 * q, k = i % n, c = i / n;
    t[q] = 0;
    if (i >= n * n) continue;
    if (PASS == 0)
      t[q] = L.U[k * LD + c];
    else
      for (int j = k; j < n; ++j) t[q] += L.U[k * LD + j] * R[j + n * c];
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < NT * NT; ++q)
    if (tid + 256 * q < n * n) R[tid + 256 * q] = t[q];
  if (fin)
    for (int i = tid; i < n * n; i += 256) {
      const int c = i % n, k = i / n;
      double x = 0;
      if (expl)
        x = L.Mi[k * LD + c];
      else
        for (int j = 0; j <= k; ++j) x += T[c + n * j] * L.Mi[k * LD + j];
      Tq[i] = x;
    }
  else if (PASS == 0)
    for (int i = tid; i < n * n; i += 256) T[i] = L.Mi[(i / n) * LD + i % n];
  __syncthreads();
  return fin;
}

// Everything of a gate that concerns one side before Theta: the environments' roots
// (one wave each), X = psi with sqrt(M) on the external bonds, X = Q R by Gram
// matrices (chol_pass), all in LDS.  A wide side (E <= n) has R = X, Q = 1.
//
// Bound: latency of one workgroup's chain.  At chi = 8 (E = 512, n = 16): load and
// roots 32 us, mode products 10, QR 19.  With Householder reflectors the products
// and the QR took 140 to 150 us per side: every column a pass over X with
// barriers, against two passes over X on the matrix cores in all.
template <int NT>
__global__ __launch_bounds__(256) void k_gate_side(const ApplyItem* __restrict__ items,
                                                   const VDesc* __restrict__ vds, const double* __restrict__ psi,
                                                   const double* __restrict__ msg, ApplyParams prm, int xsize,
                                                   double* __restrict__ work) {
  constexpr int RS = AP_ENV * AP_ENV;
  extern __shared__ __align__(16) double sm[];
  double* X = sm;
  double* S = X + xsize;  // sqrt(M) per external bond
  const CholLds<NT> L(S + AP_MAXEXT * RS);
  double* T = S + AP_MAXEXT * RS + CholLds<NT>::bytes() / sizeof(double);
  double* R = T + 256 * NT * NT;
  __shared__ ApSide g;
  __shared__ int flags;
  const int side = blockIdx.x & 1, gate = blockIdx.x >> 1, tid = threadIdx.x, wv = tid >> 6;
  const ApplyItem& it = items[gate];
  const VDesc& V = vds[side == 0 ? it.u : it.v];
  double* wk = work + (long long)blockIdx.x * AP_SIDE;
  if (side == 0) phase_mark(prm, gate, 0);
  if (tid == 0) {
    ap_side(V, side == 0 ? it.ju : it.jv, it.chib_in, g);
    flags = 0;
  }
  __syncthreads();
  const int P = ap_pitch(g.E);
  ap_load(g, psi + g.psi_off, X, P);
  if (wv < g.next) {
    // external bond wv is axis wv + 1, or wv + 2 past the gate's bond
    const int j = side == 0 ? it.ju : it.jv, a = wv + 1 < j ? wv + 1 : wv + 2;
    double* Si = wk + AP_W_SI + wv * 2 * RS;
    const bool cut = env_roots_wave(msg + V.in_msg[a], g.chi[wv], prm.eig_cutoff, S + wv * RS, Si, Si + RS);
    if (cut && (tid & 63) == 0) atomicOr(&flags, 1 << wv);
  }
  __syncthreads();
  if (side == 0) phase_mark(prm, gate, 1);
  for (int pa = 0; pa < g.next; ++pa) ap_mode(g, pa, X, P, g.n, S + pa * RS);
  if (side == 0) phase_mark(prm, gate, 2);
  double* Rg = wk + AP_W_R;
  bool expl = false;
  if (g.E <= g.n) {
    for (int i = tid; i < g.E * g.n; i += 256) {
      const int c = (int)g.fE.div(i);
      Rg[i] = X[c * P + i - c * g.E];
    }
  } else {
    double* Tq = wk + AP_W_TQ;
    if (!ap_qr_pass<NT, 0>(g, X, P, L, T, R, Tq, expl) && !ap_qr_pass<NT, 1>(g, X, P, L, T, R, Tq, expl) &&
        !ap_qr_pass<NT, 2>(g, X, P, L, T, R, Tq, expl))
      ap_qr_pass<NT, 3>(g, X, P, L, T, R, Tq, expl);
    for (int i = tid; i < g.n * g.n; i += 256) Rg[i] = R[i];
    if (expl)
      for (int i = tid; i < g.E * g.n; i += 256) {
        const int c = (int)g.fE.div(i);
        wk[i] = X[c * P + i - c * g.E];
      }
  }
  if (tid == 0) reinterpret_cast<int*>(wk + AP_W_FLAG)[0] = flags | (expl ? 8 : 0);
  if (side == 0) phase_mark(prm, gate, 3);
}

// psi' of one side in X (first d keep columns) from W: psi or Q through LDS, the
// projectors or M^{-1/2}, then X <- X W per 16 rows on the matrix cores
template <int NT>
__device__ void ap_rebuild(const ApSide& g, const double* wk, const double* psi, const double* W, int cols,
                           double* X, int P) {
  const int tid = threadIdx.x, l = tid & 63, wv = tid >> 6, li = l & 15, lk = l >> 4;
  const int flags = reinterpret_cast<const int*>(wk + AP_W_FLAG)[0], E = g.E, n = g.n;
  const bool expl = flags & 8;
  if (expl) {
    for (int i = tid; i < E * n; i += 256) {
      const int c = (int)g.fE.div(i);
      X[c * P + i - c * E] = wk[i];
    }
  } else
    ap_load(g, psi + g.psi_off, X, P);
  __syncthreads();
  for (int pa = 0; pa < g.next; ++pa)
    if (expl || (flags >> pa & 1))
      ap_mode(g, pa, X, P, n, wk + AP_W_SI + (2 * pa + (expl ? 0 : 1)) * AP_ENV * AP_ENV);
  for (int r0 = 16 * wv; r0 < E; r0 += 64) {
    double av[4 * NT];
#pragma unroll
    for (int q = 0; q < 4 * NT; ++q)
      av[q] = r0 + li < E && 4 * q + lk < n ? X[(4 * q + lk) * P + r0 + li] : 0.0;
    for (int t = 0; 16 * t < cols; ++t) {
      f64x4 acc = {0, 0, 0, 0};
      const int col = 16 * t + li;
#pragma unroll
      for (int q = 0; q < 4 * NT; ++q) {
        const double b = col < cols && 4 * q + lk < n ? W[4 * q + lk + n * col] : 0.0;
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(av[q], b, acc, 0, 0, 0);
      }
#pragma unroll
      for (int v = 0; v < 4; ++v)
        if (col < cols && r0 + 4 * v + lk < E) X[col * P + r0 + 4 * v + lk] = acc[v];
    }
  }
  __syncthreads();
}

// Theta, its SVD (gate_svd) and both sides of the bond rebuilt, one workgroup per
// gate: psi' = (psi P) Tq F, where M^{-1/2} is never applied (X = psi sqrt(M), and
// sqrt(M) M^{-1/2} = P, which is 1 unless eigenvalues were dropped); an explicit side
// takes M^{-1/2} Q F, a wide one M^{-1/2} F.  Every write to psi comes after the SVD,
// so a refused gate leaves its bond alone.
//
// Bound: latency, most of it the SVD's chain of Jacobi steps.  At chi = 8: Theta 15
// us, SVD 135 (261 on one wave), factors 5, rebuilds 22 and 17 (86 and 72 by back
// substitution and VALU products).
template <int NT>
__global__ __launch_bounds__(256) void k_gate_pair(const ApplyItem* __restrict__ items,
                                                   const VDesc* __restrict__ vds, double* __restrict__ psi,
                                                   const double* __restrict__ gates, ApplyParams prm, int wsize,
                                                   const double* __restrict__ work, double* __restrict__ truncerr,
                                                   double* __restrict__ svals, int* __restrict__ kept,
                                                   int* __restrict__ status) {
  constexpr int LD = SvdLds<AP_TH>::LD;
  extern __shared__ __align__(16) double sm[];
  double* Wl = sm;                // W of both sides, wsize each
  double* body = sm + 2 * wsize;  // the SVD's buffers, then a side's columns
  const SvdLds<AP_TH> L(body);
  double* Ru = body + SvdLds<AP_TH>::bytes() / sizeof(double);  // R_u, then Theta
  double* Rv = Ru + 1024;                                       // R_v, then V
  double* F = Rv + 1024;                                        // Theta V / sqrt(S)
  __shared__ ApSide gs[2];
  __shared__ double red[4], sgn[AP_TH];
  const int gate = blockIdx.x, tid = threadIdx.x, l = tid & 63, wv = tid >> 6, li = l & 15, lk = l >> 4;
  const ApplyItem& it = items[gate];
  const double* wk = work + (long long)gate * 2 * AP_SIDE;
  phase_mark(prm, gate, 4);
  if (tid == 0 || tid == 64)
    ap_side(vds[tid == 0 ? it.u : it.v], tid == 0 ? it.ju : it.jv, it.chib_in, gs[tid >> 6]);
  __syncthreads();
  const ApSide& gu = gs[0];
  const ApSide& gv = gs[1];
  for (int i = tid; i < gu.r * gu.n; i += 256) Ru[i] = wk[AP_W_R + i];
  for (int i = tid; i < gv.r * gv.n; i += 256) Rv[i] = wk[AP_SIDE + AP_W_R + i];
  __syncthreads();
  // Theta[(ru, su'), (rv, sv')] = sum G[(su',sv'),(su,sv)] Ru[ru, su + du b] Rv[rv, sv + dv b],
  // in the taller orientation: thread (c, h) = (tid / 8, tid % 8) has rows h + 8 i of column c
  const int du = gu.d, dv = gv.d, chib = gu.chib, dd = du * dv;
  const int Mr = gu.r * du, Nc = gv.r * dv;
  const double* G = gates + it.gate;
  const bool tr = Mr < Nc;
  const int M = tr ? Nc : Mr, N = tr ? Mr : Nc;
  double th[AP_TH / 8], x[AP_TH / 8];
#pragma unroll
  for (int i = 0; i < AP_TH / 8; ++i) {
    const int m = (tid & 7) + 8 * i, c = tid >> 3;
    double acc = 0;
    if (m < M && c < N) {
      const int row = tr ? c : m, col = tr ? m : c;
      const int sup = row / gu.r, a = row - sup * gu.r, svp = col / gv.r, b = col - svp * gv.r;
      for (int su = 0; su < du; ++su)
        for (int sv = 0; sv < dv; ++sv) {
          const double gval = G[(sup + du * svp) + dd * (su + du * sv)];
          if (gval == 0.0) continue;
          double rr = 0;
          for (int k = 0; k < chib; ++k) rr += Ru[a + gu.r * (su + du * k)] * Rv[b + gv.r * (sv + dv * k)];
          acc += gval * rr;
        }
    }
    th[i] = x[i] = acc;
  }
  phase_mark(prm, gate, 5);
  const int keep = gate_svd<AP_TH>(x, M, N, L, prm, gu.lay, it.slot, truncerr, svals, kept, status);
  phase_mark(prm, gate, 6);
  if (keep < 0) return;
  double* Th = Ru;
  double* Vt = Rv;
#pragma unroll
  for (int i = 0; i < AP_TH / 8; ++i) {
    const int m = (tid & 7) + 8 * i, c = tid >> 3;
    if (m < M && c < N) Th[m + M * c] = th[i];
  }
  for (int i = tid; i < N * keep; i += 256) {
    const int row = i % N, k = i / N;
    Vt[L.perm[row] + N * k] = L.X[row + LD * L.order[k]];
  }
  __syncthreads();
  // U sqrt(S) = Theta V / sqrt(S): 16 x 16 tiles, one per wave
  {
    const int r0 = 16 * (wv & 1), c0 = 16 * (wv >> 1);
    if (r0 < M && c0 < keep) {
      f64x4 acc = {0, 0, 0, 0};
      for (int k0 = 0; k0 < N; k0 += 4) {
        const int k = k0 + lk;
        const double a = (r0 + li < M && k < N) ? Th[r0 + li + M * k] : 0.0;
        const double b = (c0 + li < keep && k < N) ? Vt[k + N * (c0 + li)] : 0.0;
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, acc, 0, 0, 0);
      }
      if (c0 + li < keep) {
        const double s = L.svec[L.order[c0 + li]], sc = s > 0 ? 1 / sqrt(s) : 0.0;
#pragma unroll
        for (int v = 0; v < 4; ++v)
          if (r0 + 4 * v + lk < M) F[r0 + 4 * v + lk + M * (c0 + li)] = acc[v] * sc;
      }
    }
  }
  __syncthreads();  // the products above read V unscaled
  for (int i = tid; i < N * keep; i += 256) Vt[i] *= sqrt(L.svec[L.order[i / N]]);
  __syncthreads();
  // W = Tq F (n x d keep; F as r x d keep); a wide side's W = F (E x d keep)
  for (int sd = 0; sd < 2; ++sd) {
    const ApSide& g = gs[sd];
    const double* Fs = (sd == 0) == tr ? Vt : F;
    const double* Tq = wk + sd * AP_SIDE + AP_W_TQ;
    double* W = Wl + sd * wsize;
    const int n = g.n, cols = g.d * keep;
    if (g.E <= n) {
      for (int i = tid; i < g.E * cols; i += 256) W[i] = Fs[i];
    } else {
      for (int i = tid; i < n * cols; i += 256) {
        const int q = i % n, c = i / n;
        double t = 0;
#pragma unroll 4
        for (int k = 0; k < n; ++k) t += Tq[q + n * k] * Fs[k + n * c];
        W[i] = t;
      }
    }
  }
  __syncthreads();
  phase_mark(prm, gate, 7);
  double* X = body;
  for (int sd = 0; sd < 2; ++sd) {
    const ApSide& g = gs[sd];
    const int P = ap_pitch(g.E), cols = g.d * keep, E = g.E;
    const double* W = Wl + sd * wsize;
    if (E <= g.n) {
      for (int i = tid; i < E * cols; i += 256) {
        const int c = (int)g.fE.div(i);
        X[c * P + i - c * E] = W[i];
      }
      __syncthreads();
      for (int pa = 0; pa < g.next; ++pa)
        ap_mode(g, pa, X, P, cols, wk + sd * AP_SIDE + AP_W_SI + 2 * pa * AP_ENV * AP_ENV);
    } else
      ap_rebuild<NT>(g, wk + sd * AP_SIDE, psi, W, cols, X, P);
    // the largest |entry| of every new-bond slice of the first site becomes positive
    // (ties: the smallest offset in the site tensor), the same sign on both; one wave
    // per slice
    if (sd == 0) {
      for (int j = wv; j < keep; j += 4) {
        double best = -1, val = 0;
        int boff = 0x7fffffff;
        for (int i = l; i < E * g.d; i += 64) {
          const int s = (int)g.fE.div(i), e = i - s * E, hi = (int)g.flo.div(e);
          const double y = X[(s + g.d * j) * P + e];
          const int off = s + g.d * (e - hi * g.lo + g.lo * (j + g.lay * hi));
          if (fabs(y) > best || (fabs(y) == best && off < boff)) {
            best = fabs(y);
            boff = off;
            val = y;
          }
        }
        for (int m = 32; m > 0; m >>= 1) {
          const double ob = __shfl_xor(best, m), ov = __shfl_xor(val, m);
          const int oo = __shfl_xor(boff, m);
          if (ob > best || (ob == best && oo < boff)) {
            best = ob;
            boff = oo;
            val = ov;
          }
        }
        if (l == 0) sgn[j] = val < 0 ? -1.0 : 1.0;
      }
    }
    double nrm2 = 0;
    for (int i = tid; i < E * cols; i += 256) {
      const int c = (int)g.fE.div(i);
      const double y = X[c * P + i - c * E];
      nrm2 += y * y;
    }
    nrm2 = block_sum_d(nrm2, red);
    const double sc = (prm.normalize && nrm2 > 0) ? 1.0 / sqrt(nrm2) : 1.0;
    double* dst = psi + g.psi_off;
    const int D = E * g.d * g.lay;
    for (int i = tid; i < D; i += 256) {
      int c, e, b;
      ap_locate(g, i, c, e, b);
      dst[i] = b < keep ? X[c * P + e] * sgn[b] * sc : 0.0;
    }
    __syncthreads();
    phase_mark(prm, gate, 8 + sd);
  }
}

// One-site gates (apply.jl:110-116): psi_v[s', b] = sum_s O[s', s] psi_v[s, b]
// in place, then psi_v /= ||psi_v|| if normalize (:113-115).  One workgroup per
// gate; the vertices of one launch are distinct.  ops: d x d column-major per
// gate at op_off[i].
__global__ __launch_bounds__(256) void k_apply_site(const int* __restrict__ verts, const VDesc* __restrict__ vds,
                                                    double* __restrict__ psi, const double* __restrict__ ops,
                                                    const long long* __restrict__ op_off, int normalize,
                                                    double* __restrict__ norms) {
  __shared__ double O[AP_SITE_D * AP_SITE_D];
  __shared__ double red[4];
  const VDesc V = vds[verts[blockIdx.x]];
  const int d = V.dims[0];
  const int cols = V.D / d;
  double* t = psi + V.psi_off;
  for (int i = threadIdx.x; i < d * d; i += blockDim.x) O[i] = ops[op_off[blockIdx.x] + i];
  __syncthreads();
  double nrm2 = 0;
  for (int c = threadIdx.x; c < cols; c += blockDim.x) {
    double x[AP_SITE_D], y[AP_SITE_D];
    for (int s = 0; s < d; ++s) x[s] = t[(long long)c * d + s];
    for (int sp = 0; sp < d; ++sp) {
      double acc = 0;
      for (int s = 0; s < d; ++s) acc += O[sp + d * s] * x[s];
      y[sp] = acc;
      nrm2 += acc * acc;
    }
    for (int s = 0; s < d; ++s) t[(long long)c * d + s] = y[s];
  }
  const double tot = block_sum_d(nrm2, red);
  if (threadIdx.x == 0) norms[blockIdx.x] = sqrt(tot);
  if (!normalize || !(tot > 0)) return;
  const double sc = 1.0 / sqrt(tot);
  for (long long i = threadIdx.x; i < V.D; i += blockDim.x) t[i] *= sc;
}

// per-side sizes of a bond for the kernel limits: E (external size), n = d chi_b
// (the bond as it is), cols = d chi (the bond's layout during the call)
struct SideSize {
  long long E, n, cols;
};
SideSize side_size(const itnbp_net* net, int x, int e, const std::vector<int>& chi) {
  SideSize z{1, (long long)net->phys[x] * net->chi[e], (long long)net->phys[x] * chi[e]};
  for (int a = net->inc_ptr[x]; a < net->inc_ptr[x + 1]; ++a)
    if (net->inc_edge[a] != e) z.E *= chi[net->inc_edge[a]];
  return z;
}

// Checks the call and fills the launch items; goff receives the number of gate
// matrix elements.
// Rank bound of Theta for the bond e (apply.jl:74-81): each side's QR keeps
// r = min(E, d chi_e) rows, and Theta is (r_u d_u) x (r_v d_v).
long long theta_rank_bound(const itnbp_net* net, int e) {
  long long rank_bound = 1;
  for (int side = 0; side < 2; ++side) {
    const int x = net->edges[2 * e + side];
    long long E = 1;
    for (int a = net->inc_ptr[x]; a < net->inc_ptr[x + 1]; ++a)
      if (net->inc_edge[a] != e) E *= net->chi[net->inc_edge[a]];
    const long long r = std::min(E, (long long)net->phys[x] * net->chi[e]) * net->phys[x];
    rank_bound = side == 0 ? r : std::min(rank_bound, r);
  }
  return rank_bound;
}

// Checks the call against the kernel's limits with bond dimensions chi (the
// network's, or those it will have after growing) and fills the launch items;
// goff receives the number of gate matrix elements.  With fixed_bonds the
// kept rank must fit the bond as it is.
//
// With big non-null, a bond past the LDS kernel's limits that fits those of
// the split pipeline is marked (*big)[i] = 1 instead of refused.
int prepare_apply(itnbp_net* net, int n, const int* edge_ids, int maxdim, double cutoff, double* svals,
                  int max_keep, const std::vector<int>& chi, bool fixed_bonds, std::vector<ApplyItem>& items,
                  long long& goff, std::vector<char>* big = nullptr) {
  itnbp_ctx* ctx = net->ctx;
  if (net->dtype != ITNBP_F64) return itnbp_fail(ctx, ITNBP_ERR_UNSUPPORTED, "apply needs FP64 site tensors");
  if (svals && max_keep <= 0) return itnbp_fail(ctx, ITNBP_ERR_ARG, "max_keep must be > 0 with svals");
  items.assign(n, ApplyItem{});
  if (big) big->assign(n, 0);
  std::vector<char> used(net->nv, 0);
  goff = 0;
  for (int i = 0; i < n; ++i) {
    const int e = edge_ids[i];
    if (e < 0 || e >= net->ne) return itnbp_fail(ctx, ITNBP_ERR_ARG, "edge id out of range");
    const int u = net->edges[2 * e], v = net->edges[2 * e + 1];
    if (used[u] || used[v]) return itnbp_fail(ctx, ITNBP_ERR_ARG, "the bonds of one apply call must be disjoint");
    used[u] = used[v] = 1;
    // without a cutoff the kept rank is min(rank bound of Theta, maxdim), known
    // before the launch: a bond that cannot change must hold it
    const long long rank_bound = theta_rank_bound(net, e);
    const long long keep_bound = maxdim > 0 ? std::min<long long>(rank_bound, maxdim) : rank_bound;
    if (fixed_bonds && cutoff < 0 && keep_bound > chi[e])
      return itnbp_fail(ctx, ITNBP_ERR_UNSUPPORTED,
                        "apply: the truncation would keep more values than the bond dimension; pass maxdim <= chi");
    // product environment: every message into u but from v (and into v but from u) must be set
    const char* lds_why = nullptr;  // the first LDS limit the bond exceeds
    for (int side = 0; side < 2; ++side) {
      const int x = side == 0 ? u : v;
      const VDesc& V = net->vdesc[x];
      if (V.k > AP_MAXEXT + 1) return itnbp_fail(ctx, ITNBP_ERR_UNSUPPORTED, "apply supports degree <= 4");
      int chi_ext = 1;
      for (int a = net->inc_ptr[x]; a < net->inc_ptr[x + 1]; ++a) {
        const int f = net->inc_edge[a];
        if (f == e) continue;
        if (!net->msg_set[msg_id_into(net, f, x)])
          return itnbp_fail(ctx, ITNBP_ERR_STATE, "environment message not set");
        chi_ext = std::max(chi_ext, chi[f]);
      }
      const SideSize z = side_size(net, x, e, chi);
      const long long d = net->phys[x], r = std::min(z.E, z.n);
      if (lds_why) continue;
      if (chi_ext > AP_ENV) lds_why = "apply supports external bond dimensions <= 8";
      else if (z.E * z.n > AP_XY || z.E * z.cols > AP_XY) lds_why = "apply: site tensor too large for the LDS kernel";
      else if (r * d > AP_TH) lds_why = "apply: Theta larger than 32x32";
      else if (r * z.n > 1024) lds_why = "apply: R factor larger than 1024";
    }
    if (lds_why) {
      // the split pipeline: external bonds <= 32, d chi_b <= 64, Theta <= 128 x 128
      bool fits = big != nullptr;
      for (int side = 0; side < 2 && fits; ++side) {
        const int x = side == 0 ? u : v;
        const SideSize z = side_size(net, x, e, chi);
        for (int a = net->inc_ptr[x]; a < net->inc_ptr[x + 1]; ++a)
          if (net->inc_edge[a] != e && chi[net->inc_edge[a]] > AP_ENV_BIG) fits = false;
        fits = fits && z.n <= AP_N_BIG && std::min(z.E, z.n) * net->phys[x] <= AP_TH_BIG &&
               chi[e] <= AP_KEEP_BIG && z.E * std::max(z.n, z.cols) < (1LL << 30);
      }
      if (!fits) {
        if (!big) return itnbp_fail(ctx, ITNBP_ERR_UNSUPPORTED, lds_why);
        return itnbp_fail(ctx, ITNBP_ERR_UNSUPPORTED,
                          "apply supports external bond dimensions <= 32, d chi <= 64 on the bond and Theta <= "
                          "128 x 128");
      }
      (*big)[i] = 1;
    }
    items[i].u = u;
    items[i].v = v;
    items[i].ju = axis_of(net, u, e);
    items[i].jv = axis_of(net, v, e);
    items[i].gate = goff;
    items[i].slot = i;
    items[i].chib_in = net->chi[e];
    goff += (long long)net->phys[u] * net->phys[v] * net->phys[u] * net->phys[v];
  }
  return ITNBP_OK;
}

// Device memory of one apply call: launch items, gate matrices, the per-gate
// workspace of the LDS kernels (2 AP_SIDE doubles per gate) and the per-gate outputs.
struct ApplyBufs {
  ApplyItem* items;
  double* gates;
  double* work;
  double* te;
  double* sv;
  int* kept;
  int* st;
};

// bytes of each part, in the order of ApplyBufs, every part 256-byte aligned
void apply_buf_sizes(int n, long long goff, int mk, size_t (&sz)[7]) {
  auto al = [](size_t b) { return (b + 255) & ~(size_t)255; };
  sz[0] = al(n * sizeof(ApplyItem));
  sz[1] = al((size_t)goff * 8);
  sz[2] = al((size_t)n * 2 * AP_SIDE * 8);
  sz[3] = al((size_t)n * 8);
  sz[4] = al((size_t)n * mk * 8);
  sz[5] = al((size_t)n * 4);
  sz[6] = al((size_t)n * 4);
}

ApplyBufs carve_apply_bufs(char* base, int n, long long goff, int mk) {
  size_t sz[7];
  apply_buf_sizes(n, goff, mk, sz);
  ApplyBufs b;
  b.items = (ApplyItem*)base;
  base += sz[0];
  b.gates = (double*)base;
  base += sz[1];
  b.work = (double*)base;
  base += sz[2];
  b.te = (double*)base;
  base += sz[3];
  b.sv = (double*)base;
  base += sz[4];
  b.kept = (int*)base;
  base += sz[5];
  b.st = (int*)base;
  return b;
}

// Upload, the launches, read-back; every device buffer but the split
// pipeline's workspace comes from b.  Gates marked in big run on the split
// pipeline after the others, in chunks whose workspace fits the device's free
// memory (at most 16 GiB).  The network keeps a workspace of up to
// APPLY_BIG_KEEP bytes for its next call (a round is a call per colour class); a
// larger one is freed at the end of the call, so that a network does not hold
// gigabytes.  The line bounds what every network may hold; what it costs past it: a
// chi = 16 round with the workspace freed per class, and kept, 8x8 (32 gates a class)
// 5.5 and 4.3 ms, 12x12 6.6 and 5.7, 16x16 (past the line) 8.9 and 8.4, 24x24 19.8 and
// 19.7.
constexpr size_t APPLY_BIG_KEEP = 256ULL << 20;
int run_apply(itnbp_net* net, int n, const std::vector<ApplyItem>& items_in, const double* gates, long long goff,
              int maxdim, double cutoff, int normalize, double* truncerr, double* svals, int mk, int* kept,
              const ApplyBufs& b, const std::vector<char>* big = nullptr) {
  itnbp_ctx* ctx = net->ctx;
  // the LDS kernels' gates first, then the split pipeline's (every
  // output is indexed by the gate's slot, so the order is free)
  std::vector<ApplyItem> items;
  items.reserve(n);
  for (int i = 0; i < n; ++i)
    if (!big || !(*big)[i]) items.push_back(items_in[i]);
  const int nl = (int)items.size();
  for (int i = 0; i < n; ++i)
    if (big && (*big)[i]) items.push_back(items_in[i]);
  const int nb = n - nl;
  // one upload of the launch items and the gates, laid out as in b (the gates
  // follow the items at their aligned offset)
  size_t sz[7];
  apply_buf_sizes(n, goff, mk, sz);
  std::vector<char> up(sz[0] + (size_t)goff * 8);
  std::memcpy(up.data(), items.data(), n * sizeof(ApplyItem));
  std::memcpy(up.data() + sz[0], gates, (size_t)goff * 8);
  // host memory of the call's copies (up, the split pipeline's tables): every way out
  // waits for the stream before it goes
  std::vector<std::vector<char>> tables;
  struct Wait {
    hipStream_t s;
    bool on = true;
    ~Wait() {
      if (on) (void)hipStreamSynchronize(s);
    }
  } wait{ctx->stream};
  if ((char*)b.gates != (char*)b.items + sz[0])
    return itnbp_fail(ctx, ITNBP_ERR_HIP, "apply: workspace layout");
  if (hipMemcpyAsync(b.items, up.data(), up.size(), hipMemcpyHostToDevice, ctx->stream) != hipSuccess)
    return itnbp_fail(ctx, ITNBP_ERR_HIP, "apply: upload failed");
  ApplyParams prm;
  prm.maxdim = maxdim;
  prm.cutoff = cutoff;
  prm.normalize = normalize;
  prm.eig_cutoff = 10 * 2.220446049250313e-16;
  prm.max_keep = mk;
  // LDS of the two launches: a side's columns, both W, and the elimination of the
  // largest tall side (NT tiles of 16 columns)
  long long nt = 1, xside = 0, xpair = 0, wsize = 0;
  for (int i = 0; i < nl; ++i)
    for (int sd = 0; sd < 2; ++sd) {
      const VDesc& V = net->vdesc[sd == 0 ? items[i].u : items[i].v];
      const int j = sd == 0 ? items[i].ju : items[i].jv;
      const long long d = V.dims[0], lay = V.dims[j], E = V.D / (d * lay), nn = d * items[i].chib_in;
      const long long cols = d * std::min<long long>(lay, AP_TH);  // Theta's limit: kept rank <= 32
      if (E > nn) nt = std::max(nt, (nn + 15) / 16);
      xside = std::max(xside, ap_pitch((int)E) * nn);
      xpair = std::max(xpair, ap_pitch((int)E) * std::max(nn, cols));
      wsize = std::max(wsize, std::min(std::min(E, nn) * cols, 1024LL));  // r d <= 32, kept rank <= 32
    }
  const size_t lds_side = sizeof(double) * (xside + AP_MAXEXT * AP_ENV * AP_ENV + 2 * 256 * nt * nt) +
                          (nt == 1 ? CholLds<1>::bytes() : CholLds<2>::bytes());
  const size_t lds_pair =
      sizeof(double) * 2 * wsize + std::max<size_t>(sizeof(double) * xpair, SvdLds<AP_TH>::bytes() + 3 * 1024 * sizeof(double));
  const auto k_side = nt == 1 ? k_gate_side<1> : k_gate_side<2>;
  const auto k_pair = nt == 1 ? k_gate_pair<1> : k_gate_pair<2>;
  if (nl > 0) {
    hipError_t ea = hipFuncSetAttribute((const void*)k_side, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_side);
    if (ea == hipSuccess)
      ea = hipFuncSetAttribute((const void*)k_pair, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_pair);
    if (ea != hipSuccess)
      return itnbp_fail(ctx, ITNBP_ERR_HIP, std::string("apply: LDS attribute: ") + hipGetErrorString(ea));
  }
  DevBuf tsb;
  std::unique_ptr<DevBuf, void (*)(DevBuf*)> ts_guard(&tsb, [](DevBuf* x) { free_buf(*x); });
  if (getenv("ITNBP_APPLY_PHASES")) {
    ITNBP_RETCHK(ensure_buf(ctx, tsb, (size_t)n * 16 * sizeof(unsigned long long)));
    ITNBP_HIPCHK(ctx, hipMemsetAsync(tsb.p, 0, (size_t)n * 16 * sizeof(unsigned long long), ctx->stream));
    prm.ts = (unsigned long long*)tsb.p;
  }
  // the split pipeline's workspace first, so that a failed allocation leaves
  // every tensor of the call untouched
  std::vector<int> chunk_end;  // ends of the launch sequences, from item nl on
  if (nb > 0) {
    size_t fr = 0, tot = 0;
    if (hipMemGetInfo(&fr, &tot) != hipSuccess) fr = 0;
    const size_t budget = std::min<size_t>(fr / 2 + net->apply_big.bytes, 16ULL << 30);
    size_t most = 0;
    chunk_end = apply_big_chunks(net, items.data() + nl, nb, budget, most);
    ITNBP_RETCHK(ensure_buf(ctx, net->apply_big, most));
  }
  const int pm0 = prof_mark(ctx);
  if (nl > 0) {
    hipLaunchKernelGGL(k_side, dim3(2 * nl), dim3(256), lds_side, ctx->stream, (const ApplyItem*)b.items,
                       net->d_vdesc, (const double*)net->d_psi, (const double*)net->d_msg[net->cur], prm, (int)xside,
                       b.work);
    hipLaunchKernelGGL(k_pair, dim3(nl), dim3(256), lds_pair, ctx->stream, (const ApplyItem*)b.items, net->d_vdesc,
                       (double*)net->d_psi, (const double*)b.gates, prm, (int)wsize, (const double*)b.work, b.te,
                       svals ? b.sv : nullptr, b.kept, b.st);
  }
  hipError_t ek = hipGetLastError();
  prof_add(ctx, "apply_gates", pm0, prof_mark(ctx));
  if (ek == hipSuccess && nb > 0) {
    int c0 = 0;
    for (int c1 : chunk_end) {
      const int rc = apply_big_run(net, items.data() + nl + c0, c1 - c0, b.gates, prm, net->apply_big.p, b.te,
                                   svals ? b.sv : nullptr, b.kept, b.st, tables);
      if (rc != ITNBP_OK) return rc;
      c0 = c1;
    }
  }
  if (prm.ts && ek == hipSuccess) {
    // mean duration of every phase over the LDS kernels' gates that ran to the end, in us
    std::vector<unsigned long long> ts((size_t)n * 16);
    int khz = 0;
    ek = hipMemcpyAsync(ts.data(), prm.ts, ts.size() * 8, hipMemcpyDeviceToHost, ctx->stream);
    if (ek == hipSuccess) ek = hipStreamSynchronize(ctx->stream);
    if (ek == hipSuccess) ek = hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, ctx->device);
    // intervals [p, p + 1], 3 the gap between the launches
    double mean[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
    int cnt = 0;
    for (int i = 0; i < nl && ek == hipSuccess && khz > 0; ++i) {
      const unsigned long long* t = &ts[(size_t)i * 16];
      if (!t[9]) continue;
      ++cnt;
      for (int p = 0; p < 9; ++p) mean[p] += (double)(t[p + 1] - t[p]) * 1e3 / khz;
    }
    const double c = cnt;
    if (cnt > 0)
      fprintf(stderr,
              "apply phases (us, mean over %d gates): side u: load and roots %.1f, mode products %.1f, qr %.1f; "
              "pair: theta %.1f, svd %.1f, factors %.1f, rebuild_u %.1f, rebuild_v %.1f\n",
              cnt, mean[0] / c, mean[1] / c, mean[2] / c, mean[4] / c, mean[5] / c, mean[6] / c, mean[7] / c,
              mean[8] / c);
  }
  std::vector<int> st(n);
  std::vector<int> kp(n);
  // one read-back of the outputs (truncation errors, singular values, kept
  // ranks, status: consecutive in b)
  std::vector<char> dn(sz[3] + sz[4] + sz[5] + (size_t)n * 4);
  if (ek == hipSuccess && ((char*)b.sv != (char*)b.te + sz[3] || (char*)b.kept != (char*)b.sv + sz[4] ||
                           (char*)b.st != (char*)b.kept + sz[5]))
    return itnbp_fail(ctx, ITNBP_ERR_HIP, "apply: workspace layout");
  if (ek == hipSuccess) ek = hipMemcpyAsync(dn.data(), b.te, dn.size(), hipMemcpyDeviceToHost, ctx->stream);
  if (ek == hipSuccess) ek = hipStreamSynchronize(ctx->stream);
  wait.on = ek != hipSuccess;
  if (net->apply_big.bytes > APPLY_BIG_KEEP) free_buf(net->apply_big);
  if (ek != hipSuccess) return itnbp_fail(ctx, ITNBP_ERR_HIP, std::string("apply: ") + hipGetErrorString(ek));
  std::memcpy(truncerr, dn.data(), (size_t)n * 8);
  if (svals) std::memcpy(svals, dn.data() + sz[3], (size_t)n * mk * 8);
  std::memcpy(kp.data(), dn.data() + sz[3] + sz[4], (size_t)n * 4);
  std::memcpy(st.data(), dn.data() + sz[3] + sz[4] + sz[5], (size_t)n * 4);
  // a gate the kernel refused (its bond untouched) reports kept = -1
  for (int i = 0; i < n; ++i)
    if (st[i]) kp[i] = -1;
  if (kept) std::copy(kp.begin(), kp.end(), kept);
  invalidate_fast_state(net);
  for (int i = 0; i < n; ++i)
    if (st[i] == 2)
      return itnbp_fail(ctx, ITNBP_ERR_NONFINITE,
                        "apply: non-finite two-site tensor (that bond's tensors are unchanged; the other gates of "
                        "the call were applied)");
  for (int i = 0; i < n; ++i)
    if (st[i])
      return itnbp_fail(ctx, ITNBP_ERR_UNSUPPORTED,
                        "apply: the truncation keeps more values than the bond dimension (that bond's tensors "
                        "are unchanged; the other gates of the call were applied); pass maxdim <= chi");
  for (int i = 0; i < n; ++i)
    if (!std::isfinite(truncerr[i])) return itnbp_fail(ctx, ITNBP_ERR_NONFINITE, "apply: non-finite result");
  return ITNBP_OK;
}

// ---- workspace of itnbp_apply_gates_noalloc --------------------------------
// At most NOALLOC_MAX_GATES gates per call, gate matrices of at most
// NOALLOC_MAX_GATE_ELEMS elements ((d_u d_v)^2 with d <= 4) and at most
// NOALLOC_MAX_KEEP singular values per gate: 21.0 MiB in all, held by every
// GPU the library runs on until the process ends.
constexpr int NOALLOC_MAX_GATES = 128;
constexpr int NOALLOC_MAX_GATE_ELEMS = 256;
constexpr int NOALLOC_MAX_KEEP = 32;

constexpr size_t noalloc_bytes() {
  return ((NOALLOC_MAX_GATES * sizeof(ApplyItem) + 255) & ~(size_t)255) +
         (size_t)NOALLOC_MAX_GATES * NOALLOC_MAX_GATE_ELEMS * 8 + (size_t)NOALLOC_MAX_GATES * 2 * AP_SIDE * 8 +
         (size_t)NOALLOC_MAX_GATES * 8 + (size_t)NOALLOC_MAX_GATES * NOALLOC_MAX_KEEP * 8 +
         2 * (size_t)NOALLOC_MAX_GATES * 4 + 8 * 256;
}

// The array's name is a host-side stand-in: host code uses only the device
// address that hipGetSymbolAddress returns for the current device.
static __device__ __align__(256) unsigned char scratch[noalloc_bytes()];

constexpr int NOALLOC_MAX_DEVICES = 64;
std::mutex g_noalloc_mu;
void* g_noalloc_ptr[NOALLOC_MAX_DEVICES] = {};
int g_noalloc_rc[NOALLOC_MAX_DEVICES] = {};
bool g_noalloc_done[NOALLOC_MAX_DEVICES] = {};

}  // namespace

// Resolves the workspace address on `device` (current) once per device; called
// by itnbp_create.  Returns ITNBP_OK or ITNBP_ERR_HIP (then the no-allocation
// entry point refuses every call on that device).
int apply_noalloc_init(int device) {
  if (device < 0 || device >= NOALLOC_MAX_DEVICES) return ITNBP_ERR_ARG;
  std::lock_guard<std::mutex> lk(g_noalloc_mu);
  if (!g_noalloc_done[device]) {
    void* ptr = nullptr;
    const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess) {
      (void)hipGetLastError();
      ptr = nullptr;
    }
    g_noalloc_ptr[device] = ptr;
    g_noalloc_rc[device] = e == hipSuccess ? ITNBP_OK : ITNBP_ERR_HIP;
    g_noalloc_done[device] = true;
  }
  return g_noalloc_rc[device];
}

extern "C" int itnbp_apply_gates(itnbp_net* net, int n, const int* edge_ids, const double* gates,
                                 int maxdim, double cutoff, int normalize, double* truncerr,
                                 double* svals, int max_keep, int* kept) {
  if (!net || n < 0 || (n > 0 && (!edge_ids || !gates || !truncerr))) return ITNBP_ERR_ARG;
  if (n == 0) return ITNBP_OK;
  itnbp_ctx* ctx = net->ctx;
  return itnbp_guarded(ctx, [&]() -> int {
    // The new bond has the kept dimension (apply.jl:81-93).  A bond whose kept
    // rank may exceed its dimension first grows (zero-padded) to the largest
    // rank the truncation can keep, min(rank bound of Theta, maxdim); the kernel
    // writes the kept columns followed by zeros; then every bond of the call is
    // cut to its kept rank, which drops only zeros.
    for (int i = 0; i < n; ++i)
      if (edge_ids[i] < 0 || edge_ids[i] >= net->ne) return itnbp_fail(ctx, ITNBP_ERR_ARG, "edge id out of range");
    const std::vector<int> chi0 = net->chi;
    std::vector<int> target(n), chi_grow = net->chi;
    for (int i = 0; i < n; ++i) {
      const int e = edge_ids[i];
      const long long rb = theta_rank_bound(net, e);
      target[i] = (int)std::min<long long>(maxdim > 0 ? std::min<long long>(rb, maxdim) : rb, 64);
      chi_grow[e] = std::max(chi_grow[e], target[i]);
    }
    std::vector<ApplyItem> items;
    std::vector<char> big;
    long long goff = 0;
    ITNBP_RETCHK(
        prepare_apply(net, n, edge_ids, maxdim, cutoff, svals, max_keep, chi_grow, false, items, goff, &big));
    ITNBP_RETCHK(net_resize_bonds(net, chi_grow));
    const int mk = svals ? max_keep : 1;
    size_t sz[7];
    apply_buf_sizes(n, goff, mk, sz);
    size_t total = 0;
    for (size_t b : sz) total += b;
    // the net keeps the workspace between calls (a gate round is several calls)
    ITNBP_RETCHK(ensure_buf(ctx, net->apply_ws, total));
    std::vector<int> kp(n, -1);
    const int rc = run_apply(net, n, items, gates, goff, maxdim, cutoff, normalize, truncerr, svals, mk, kp.data(),
                             carve_apply_bufs((char*)net->apply_ws.p, n, goff, mk), &big);
    std::vector<int> chi_cut = net->chi;
    if (rc != ITNBP_OK) {
      // the gates that ran keep their new bonds; a refused gate's bond (its
      // tensors untouched, grown with zeros) returns to its old dimension
      for (int i = 0; i < n; ++i)
        chi_cut[edge_ids[i]] = kp[i] < 0 ? chi0[edge_ids[i]] : std::max(1, std::min(kp[i], target[i]));
      if (kept) std::copy(kp.begin(), kp.end(), kept);
      (void)net_resize_bonds(net, chi_cut);
      return rc;
    }
    for (int i = 0; i < n; ++i) {
      kp[i] = std::max(1, std::min(kp[i], target[i]));
      chi_cut[edge_ids[i]] = kp[i];
      if (svals)
        for (int j = kp[i]; j < mk; ++j) svals[(size_t)i * mk + j] = 0.0;
    }
    if (kept) std::copy(kp.begin(), kp.end(), kept);
    return net_resize_bonds(net, chi_cut);
  });
}

extern "C" int itnbp_apply_site_gates(itnbp_net* net, int n, const int* verts, const double* ops, int normalize,
                                      double* norms) {
  if (!net || n < 0 || (n > 0 && (!verts || !ops))) return ITNBP_ERR_ARG;
  if (n == 0) return ITNBP_OK;
  itnbp_ctx* ctx = net->ctx;
  return itnbp_guarded(ctx, [&]() -> int {
    if (net->dtype != ITNBP_F64) return itnbp_fail(ctx, ITNBP_ERR_UNSUPPORTED, "apply needs FP64 site tensors");
    std::vector<char> used(net->nv, 0);
    std::vector<long long> off(n);
    long long tot = 0;
    for (int i = 0; i < n; ++i) {
      const int v = verts[i];
      if (v < 0 || v >= net->nv) return itnbp_fail(ctx, ITNBP_ERR_ARG, "vertex out of range");
      if (used[v]) return itnbp_fail(ctx, ITNBP_ERR_ARG, "the vertices of one site-gate call must be distinct");
      used[v] = 1;
      const int d = net->phys[v];
      if (d > AP_SITE_D) return itnbp_fail(ctx, ITNBP_ERR_UNSUPPORTED, "one-site gates support d <= 16");
      off[i] = tot;
      tot += (long long)d * d;
    }
    DevBuf b;
    const size_t ob = ((size_t)n * 4 + 255) & ~(size_t)255, oo = ((size_t)n * 8 + 255) & ~(size_t)255;
    ITNBP_RETCHK(ensure_buf(ctx, b, ob + 2 * oo + (size_t)tot * 8));
    char* p = (char*)b.p;
    int* d_v = (int*)p;
    long long* d_off = (long long*)(p + ob);
    double* d_nrm = (double*)(p + ob + oo);
    double* d_ops = (double*)(p + ob + 2 * oo);
    std::vector<double> nrm(n);
    hipError_t e = hipMemcpyAsync(d_v, verts, (size_t)n * 4, hipMemcpyHostToDevice, ctx->stream);
    if (e == hipSuccess) e = hipMemcpyAsync(d_off, off.data(), (size_t)n * 8, hipMemcpyHostToDevice, ctx->stream);
    if (e == hipSuccess) e = hipMemcpyAsync(d_ops, ops, (size_t)tot * 8, hipMemcpyHostToDevice, ctx->stream);
    if (e == hipSuccess) {
      const int pm0 = prof_mark(ctx);
      hipLaunchKernelGGL(k_apply_site, dim3(n), dim3(256), 0, ctx->stream, (const int*)d_v, net->d_vdesc,
                         (double*)net->d_psi, (const double*)d_ops, (const long long*)d_off, normalize, d_nrm);
      e = hipGetLastError();
      prof_add(ctx, "apply_site", pm0, prof_mark(ctx));
    }
    if (e == hipSuccess) e = hipMemcpyAsync(nrm.data(), d_nrm, (size_t)n * 8, hipMemcpyDeviceToHost, ctx->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(ctx->stream);
    free_buf(b);
    if (e != hipSuccess) return itnbp_fail(ctx, ITNBP_ERR_HIP, std::string("apply_site_gates: ") + hipGetErrorString(e));
    invalidate_fast_state(net);
    if (norms) std::copy(nrm.begin(), nrm.end(), norms);
    for (int i = 0; i < n; ++i)
      if (!std::isfinite(nrm[i])) return itnbp_fail(ctx, ITNBP_ERR_NONFINITE, "apply_site_gates: non-finite result");
    return ITNBP_OK;
  });
}

extern "C" int itnbp_apply_gates_noalloc(itnbp_net* net, int n, const int* edge_ids, const double* gates,
                                         int maxdim, double cutoff, int normalize, double* truncerr,
                                         double* svals, int max_keep, int* kept) {
  if (!net || n < 0 || (n > 0 && (!edge_ids || !gates || !truncerr))) return ITNBP_ERR_ARG;
  if (n == 0) return ITNBP_OK;
  itnbp_ctx* ctx = net->ctx;
  return itnbp_guarded(ctx, [&]() -> int {
    if (n > NOALLOC_MAX_GATES)
      return itnbp_fail(ctx, ITNBP_ERR_UNSUPPORTED,
                        "apply_gates_noalloc: at most " + std::to_string(NOALLOC_MAX_GATES) + " gates per call");
    const int mk = svals ? max_keep : 1;
    if (mk > NOALLOC_MAX_KEEP)
      return itnbp_fail(ctx, ITNBP_ERR_UNSUPPORTED,
                        "apply_gates_noalloc: max_keep at most " + std::to_string(NOALLOC_MAX_KEEP));
    std::vector<ApplyItem> items;
    long long goff = 0;
    // no allocation, so no resizing: every bond keeps its dimension and fewer
    // kept values are zero-padded
    ITNBP_RETCHK(prepare_apply(net, n, edge_ids, maxdim, cutoff, svals, max_keep, net->chi, true, items, goff));
    if (goff > (long long)n * NOALLOC_MAX_GATE_ELEMS)
      return itnbp_fail(ctx, ITNBP_ERR_UNSUPPORTED,
                        "apply_gates_noalloc: gate matrices larger than (d_u d_v)^2 = 256 elements");
    void* base = nullptr;
    {
      std::lock_guard<std::mutex> lk(g_noalloc_mu);
      if (ctx->device >= 0 && ctx->device < NOALLOC_MAX_DEVICES && g_noalloc_done[ctx->device])
        base = g_noalloc_ptr[ctx->device];
    }
    if (!base)
      return itnbp_fail(ctx, ITNBP_ERR_HIP, "apply_gates_noalloc: the workspace address of this device is unknown");
    size_t sz[7];
    apply_buf_sizes(n, goff, mk, sz);
    size_t total = 0;
    for (size_t b : sz) total += b;
    if (total > noalloc_bytes())
      return itnbp_fail(ctx, ITNBP_ERR_UNSUPPORTED, "apply_gates_noalloc: call exceeds the workspace");
    return run_apply(net, n, items, gates, goff, maxdim, cutoff, normalize, truncerr, svals, mk, kept,
                     carve_apply_bufs((char*)base, n, goff, mk));
  });
}

// ============================================================================
// Adjoint of the gate application (vector-Jacobian product of
// simple_update_bp, src/apply.jl:33-95, with the normalisation of :134-137).
//
// The kernel recomputes each bond's forward pass in a gauge of its own and
// pulls the cotangents of psi_u', psi_v' back to psi_u, psi_v, the gate and
// every environment message.  With X = psi (x) sqrt(env) as the E x n matrix of
// a side (E external, n = d chi_b) the QR factor only enters through a gauge
// that cancels between Theta and the rebuild, so:
//   - a tall side (E >= n) uses R = C^{1/2}, C = X^T X, and the rebuild factor
//     W = psi_P C^{-1/2}, psi_P = psi (x) P with P the projector on the kept
//     environment eigenvectors (S Si = P);
//   - a wide side (E < n) uses R = X and W = (x) Si.
// Theta = G (R_u R_v), thin SVD U S V^T, F_u = U_k sqrt(S_k), F_v = V_k sqrt(S_k),
// psi_u' = W_u F_u times the bond signs of the forward gauge, then normalised.
// Pullbacks, in reverse: normalisation; W F products; sqrt(S); the thin SVD
// (full-rank formula with the kept/discarded couplings, 1/(s_j^2 - s_i^2)
// broadened by 1e-12 s_max^2 against degenerate values); the contraction with
// the gate; R = C^{1/2} and C^{-1/2} through the eigenbasis of C with the
// divided differences 1/(s_i + s_j) and -1/(s_i s_j (s_i + s_j)); X = psi (x) S;
// sqrt and inverse sqrt of every environment through its eigenbasis (kept
// eigenvalues; a dropped one contributes nothing).  P is taken as constant.
// One workgroup per bond, FP64, intermediates in a global workspace per bond.
// ============================================================================
namespace {

constexpr int VJ_SM = 1024;
constexpr int VJ_ENV = 64 * 6 + 16;  // per external axis: V, S, Si, Sb, Sib, tmp (8x8 each) + w
// per side: 9 matrices of up to AP_XY, 8 of up to 1024, 3 environments
constexpr long long VJ_SIDE = 9LL * AP_XY + 8LL * VJ_SM + AP_MAXEXT * VJ_ENV + 64;
// shared: 14 matrices of up to 1024 and small vectors
constexpr long long VJ_SHARED = 14LL * VJ_SM + 6 * 64;
constexpr long long VJ_GATE = 2 * VJ_SIDE + VJ_SHARED;

struct VjpIo {
  long long out_u, out_v;  // cotangents of psi_u', psi_v' (new bond dimension keep)
  long long in_u, in_v;    // cotangents of psi_u, psi_v
  long long dgate;         // cotangent of the gate
  int keep, pad;
};

__device__ inline void bsync() {
  __threadfence_block();
  __syncthreads();
}

// C (m x n, ld ldc) = op(A) op(B) (+ C if acc), column-major; A m x k (or k x m
// transposed), B k x n (or n x k transposed)
__device__ void gmm(int m, int n, int k, const double* A, int lda, bool ta, const double* B, int ldb, bool tb,
                    double* C, int ldc, bool acc = false) {
  for (int idx = threadIdx.x; idx < m * n; idx += blockDim.x) {
    const int i = idx % m, j = idx / m;
    double s = 0;
    for (int l = 0; l < k; ++l) {
      const double a = ta ? A[l + (long long)lda * i] : A[i + (long long)lda * l];
      const double b = tb ? B[j + (long long)ldb * l] : B[l + (long long)ldb * j];
      s += a * b;
    }
    C[i + (long long)ldc * j] = acc ? C[i + (long long)ldc * j] + s : s;
  }
  bsync();
}

// Y = X with the symmetric chi x chi matrix Mt (row-major) on external axis pa
__device__ void ext_mp_g(const SideGeom& g, int pa, const double* X, double* Y, int cols, const double* Mt) {
  const int stride = (int)g.fst[pa].d;
  const int chi = g.dims[g.ext[pa]];
  for (int idx = threadIdx.x; idx < g.E * cols; idx += blockDim.x) {
    const int c = (int)g.fE.div(idx), e = idx - c * g.E;
    const int q = (int)g.fst[pa].div(e), lo = e - q * stride;
    const int hi = (int)g.fchi[pa].div(q), b2 = q - hi * chi;
    double acc = 0;
    for (int b = 0; b < chi; ++b) acc += X[(lo + stride * (b + chi * hi)) + (long long)g.E * c] * Mt[b * chi + b2];
    Y[idx] = acc;
  }
  bsync();
}

// Symmetric eigendecomposition of one chi x chi message by one wave (the Jacobi
// of env_roots_wave): V (row-major, V[r * chi + m] = component r of eigenvector
// m), w[m], and the kept mask of map_eigvals' truncation (cutoff on |w|).
__device__ unsigned env_eig_wave(const double* M, int chi, double cutoff, double* Vout, double* wout) {
  const int l = threadIdx.x & 63;
  const int ne = chi + (chi & 1);
  const bool live = l < ne * ne;
  const int i = live ? l / ne : 0, j = live ? l % ne : 0;
  const bool in = live && i < chi && j < chi;
  double a = in ? 0.5 * (M[i + chi * j] + M[j + chi * i]) : 0.0;
  double v = (live && i == j) ? 1.0 : 0.0;
  if (chi > 1) {
    auto rot = [&](int p, int q, double& c, double& sn) {
      const double app = __shfl(a, p * ne + p), aqq = __shfl(a, q * ne + q), apq = __shfl(a, p * ne + q);
      c = 1.0;
      sn = 0.0;
      if (q < chi && apq != 0.0) {
        const double zeta = (aqq - app) / (2 * apq);
        const double t = (zeta >= 0 ? 1.0 : -1.0) / (fabs(zeta) + sqrt(1 + zeta * zeta));
        c = 1 / sqrt(1 + t * t);
        sn = c * t;
      }
    };
    double prev = INFINITY;
    for (int sweep = 0; sweep < 40; ++sweep) {
      double off = (in && i != j) ? a * a : 0.0, diag = (in && i == j) ? a * a : 0.0;
      for (int m = 32; m > 0; m >>= 1) {
        off += __shfl_xor(off, m);
        diag += __shfl_xor(diag, m);
      }
      // converged, or the off-diagonal mass no longer decreases (rounding level)
      if (off <= 1e-30 * diag || off == 0.0 || off >= prev) break;
      prev = off;
      for (int st = 0; st < ne - 1; ++st) {
        // (x - 1 - st) lies in (-(ne - 1), ne - 1) and (pp - 1 + st) in [0, 2 (ne - 1)):
        // conditional corrections instead of modulos
        auto partner = [&](int x) {
          int t = x - 1 - st;
          if (t < 0) t += ne - 1;
          const int pos = x == 0 ? 0 : 1 + t;
          const int pp = ne - 1 - pos;
          int u = pp - 1 + st;
          if (u >= ne - 1) u -= ne - 1;
          return pp == 0 ? 0 : 1 + u;
        };
        const int ri = partner(i), cj = partner(j);
        double cr, sr, cc, sc;
        rot(i < ri ? i : ri, i < ri ? ri : i, cr, sr);
        rot(j < cj ? j : cj, j < cj ? cj : j, cc, sc);
        const double ao = __shfl(a, ri * ne + j);
        const double ar = i < ri ? cr * a - sr * ao : sr * ao + cr * a;
        const double aro = __shfl(ar, i * ne + cj), vo = __shfl(v, i * ne + cj);
        a = j < cj ? cc * ar - sc * aro : sc * aro + cc * ar;
        v = j < cj ? cc * v - sc * vo : sc * vo + cc * v;
      }
    }
  }
  double w[AP_ENV];
#pragma unroll
  for (int m = 0; m < AP_ENV; ++m) w[m] = __shfl(a, (m < ne ? m : 0) * ne + (m < ne ? m : 0));
  int order[AP_ENV];
  for (int m = 0; m < chi; ++m) order[m] = m;
  for (int x = 0; x < chi; ++x)
    for (int y = x + 1; y < chi; ++y)
      if (fabs(w[order[y]]) > fabs(w[order[x]])) {
        const int t = order[x];
        order[x] = order[y];
        order[y] = t;
      }
  double tot = 0;
  for (int m = 0; m < chi; ++m) tot += fabs(w[m]);
  int keep = chi;
  double disc = 0;
  while (keep > 1 && tot > 0 && (disc + fabs(w[order[keep - 1]])) / tot <= cutoff) {
    disc += fabs(w[order[keep - 1]]);
    --keep;
  }
  unsigned kmask = 0;
  for (int m = 0; m < keep; ++m) kmask |= 1u << order[m];
  if (in) Vout[i * chi + j] = v;
  if (l < chi) wout[l] = w[l];
  return kmask;
}

// S = V f(w) V^T over the kept eigenvalues (row-major chi x chi), f = sqrt
// (which = 0), 1/sqrt (1) or the indicator (2)
__device__ void env_fun(const double* V, const double* w, unsigned kmask, int chi, int which, double* out) {
  for (int idx = threadIdx.x & 63; idx < chi * chi; idx += 64) {
    const int r = idx / chi, c = idx % chi;
    double s = 0;
    for (int m = 0; m < chi; ++m)
      if ((kmask >> m) & 1u) {
        const double f = which == 0 ? sqrt(w[m]) : which == 1 ? 1.0 / sqrt(w[m]) : 1.0;
        s += V[r * chi + m] * V[c * chi + m] * f;
      }
    out[idx] = s;
  }
}

// Mbar (row-major, chi x chi, symmetrised) = V [(V^T Sb V) o K1 + (V^T Sib V) o K2] V^T
// with the divided differences of sqrt and 1/sqrt on the kept eigenvalues
__device__ void env_pullback(const double* V, const double* w, unsigned kmask, int chi, const double* Sb,
                             const double* Sib, double* tmp, double* Mb) {
  const int l = threadIdx.x & 63;
  // tmp = V^T (Sb_sym) V o K1 + V^T (Sib_sym) V o K2   (eigenbasis, row-major)
  for (int idx = l; idx < chi * chi; idx += 64) {
    const int p = idx / chi, q = idx % chi;
    double a = 0, b = 0;
    for (int r = 0; r < chi; ++r)
      for (int c = 0; c < chi; ++c) {
        const double vv = V[r * chi + p] * V[c * chi + q];
        a += vv * 0.5 * (Sb[r * chi + c] + Sb[c * chi + r]);
        b += vv * 0.5 * (Sib[r * chi + c] + Sib[c * chi + r]);
      }
    const bool kp = (kmask >> p) & 1u, kq = (kmask >> q) & 1u;
    double k1 = 0, k2 = 0;
    if (kp && kq) {
      const double sp = sqrt(w[p]), sq = sqrt(w[q]);
      k1 = 1.0 / (sp + sq);
      k2 = -1.0 / (sp * sq * (sp + sq));
    } else if (kp || kq) {
      // one kept (f(x)), one dropped (f = 0): (f(w_p) - f(w_q)) / (w_p - w_q)
      const double wk = kp ? w[p] : w[q], wd = kp ? w[q] : w[p];
      const double den = wk - wd;
      if (den != 0.0) {
        k1 = sqrt(wk) / den;
        k2 = 1.0 / sqrt(wk) / den;
      }
    }
    tmp[idx] = a * k1 + b * k2;
  }
  __threadfence_block();
  for (int idx = l; idx < chi * chi; idx += 64) {
    const int r = idx / chi, c = idx % chi;
    double s = 0, t = 0;
    for (int p = 0; p < chi; ++p)
      for (int q = 0; q < chi; ++q) {
        s += V[r * chi + p] * tmp[p * chi + q] * V[c * chi + q];
        t += V[c * chi + p] * tmp[p * chi + q] * V[r * chi + q];
      }
    Mb[idx] = 0.5 * (s + t);
  }
}

__global__ __launch_bounds__(256) void k_apply_vjp(const ApplyItem* __restrict__ items, const VjpIo* __restrict__ io,
                                                   const VDesc* __restrict__ vds, const double* __restrict__ psi,
                                                   const double* __restrict__ msg, const double* __restrict__ gates,
                                                   ApplyParams prm, const double* __restrict__ dout,
                                                   double* __restrict__ din, double* __restrict__ dgate,
                                                   double* __restrict__ dmsg, double* __restrict__ work,
                                                   int* __restrict__ status) {
  __shared__ double red[8];
  __shared__ int order[AP_TH];
  __shared__ int sh_keep;
  __shared__ unsigned kmask[2][AP_MAXEXT];
  const ApplyItem it = items[blockIdx.x];
  const VjpIo o = io[blockIdx.x];
  const int tid = threadIdx.x;
  SideGeom gs[2] = {side_geom(vds[it.u], it.ju), side_geom(vds[it.v], it.jv)};
  const int vtx[2] = {it.u, it.v};
  double* base = work + (long long)blockIdx.x * VJ_GATE;
  // per side areas
  double *X[2], *Pt[2], *A[2], *W[2], *Xb[2], *Pb[2], *Yb[2], *T1[2], *T2[2];
  double *Z[2], *R[2], *B[2], *Rb[2], *Bb[2], *Cb[2], *Sg[2], *Wb[2], *env[2];
  for (int s = 0; s < 2; ++s) {
    double* p = base + s * VJ_SIDE;
    X[s] = p; Pt[s] = p + AP_XY; A[s] = p + 2 * AP_XY; W[s] = p + 3 * AP_XY; Xb[s] = p + 4 * AP_XY;
    Pb[s] = p + 5 * AP_XY; Yb[s] = p + 6 * AP_XY; T1[s] = p + 7 * AP_XY; T2[s] = p + 8 * AP_XY;
    double* q = p + 9LL * AP_XY;
    Z[s] = q; R[s] = q + VJ_SM; B[s] = q + 2 * VJ_SM; Rb[s] = q + 3 * VJ_SM; Bb[s] = q + 4 * VJ_SM;
    Cb[s] = q + 5 * VJ_SM; Sg[s] = q + 6 * VJ_SM; Wb[s] = q + 7 * VJ_SM;
    env[s] = q + 8 * VJ_SM;
  }
  double* sh = base + 2 * VJ_SIDE;
  double *Th = sh, *Tt = sh + VJ_SM, *As = sh + 2 * VJ_SM, *Vs = sh + 3 * VJ_SM, *Fu = sh + 4 * VJ_SM,
         *Fv = sh + 5 * VJ_SM, *Fub = sh + 6 * VJ_SM, *Fvb = sh + 7 * VJ_SM, *Thb = sh + 8 * VJ_SM,
         *Ttb = sh + 9 * VJ_SM, *Um = sh + 10 * VJ_SM, *Vm = sh + 11 * VJ_SM, *M1 = sh + 12 * VJ_SM,
         *Q2 = sh + 13 * VJ_SM;
  double* svec = sh + 14 * VJ_SM;  // thin singular values (sorted)
  double* sbar = svec + 64;
  double* sgn = sbar + 64;
  double* rot = sgn + 64;  // 128
  auto env_p = [&](int s, int pa, int which) { return env[s] + pa * VJ_ENV + which * 64; };
  // env slots: 0 V, 1 S, 2 Si, 3 Sbar, 4 Sibar, 5 tmp; w at 6 * 64

  // ---- forward -------------------------------------------------------------
  // F1. eigendecompositions of the environments, one wave each
  {
    const int wv = tid >> 6;
    for (int q = wv; q < gs[0].next + gs[1].next; q += (int)blockDim.x / 64) {
      const int s = q < gs[0].next ? 0 : 1;
      const int pa = s == 0 ? q : q - gs[0].next;
      const SideGeom& g = gs[s];
      const int a = g.ext[pa];
      const int chi = g.dims[a];
      double* V = env_p(s, pa, 0);
      double* w = env[s] + pa * VJ_ENV + 6 * 64;
      const unsigned km = env_eig_wave(msg + vds[vtx[s]].in_msg[a], chi, prm.eig_cutoff, V, w);
      __threadfence_block();
      env_fun(V, w, km, chi, 0, env_p(s, pa, 1));
      env_fun(V, w, km, chi, 1, env_p(s, pa, 2));
      env_fun(V, w, km, chi, 2, env_p(s, pa, 5));  // P in the tmp slot until the pullback
      for (int i = (tid & 63); i < 64; i += 64) {
        env_p(s, pa, 3)[i] = 0.0;
        env_p(s, pa, 4)[i] = 0.0;
      }
      if ((tid & 63) == 0) kmask[s][pa] = km;
    }
    bsync();
  }
  // F2-F3. X = psi (x) S, Pt = psi (x) P, R and W per side
  for (int s = 0; s < 2; ++s) {
    const SideGeom& g = gs[s];
    for (int idx = tid; idx < g.E * g.n; idx += blockDim.x) {
      const int e = idx % g.E, c = idx / g.E;
      const double x = psi[g.psi_off + nat_off(g, c % g.d, e, c / g.d)];
      X[s][idx] = x;
      Pt[s][idx] = x;
    }
    bsync();
    for (int pa = 0; pa < g.next; ++pa) {
      ext_mp_g(g, pa, X[s], T1[s], g.n, env_p(s, pa, 1));
      for (int i = tid; i < g.E * g.n; i += blockDim.x) X[s][i] = T1[s][i];
      ext_mp_g(g, pa, Pt[s], T1[s], g.n, env_p(s, pa, 5));
      for (int i = tid; i < g.E * g.n; i += blockDim.x) Pt[s][i] = T1[s][i];
      bsync();
    }
    if (g.E >= g.n) {
      // tall: singular values and right vectors of X give C = Z diag(sigma^2) Z^T
      for (int i = tid; i < g.E * g.n; i += blockDim.x) A[s][i] = X[s][i];
      bsync();
      jacobi_svd(A[s], g.E, g.n, Z[s], rot, red);
      bsync();
      for (int j = tid; j < g.n; j += blockDim.x) {
        double t = 0;
        for (int i = 0; i < g.E; ++i) t += A[s][i + (long long)g.E * j] * A[s][i + (long long)g.E * j];
        Sg[s][j] = sqrt(t);
      }
      bsync();
      for (int idx = tid; idx < g.n * g.n; idx += blockDim.x) {
        const int i = idx % g.n, j = idx / g.n;
        double r = 0, b = 0;
        for (int m = 0; m < g.n; ++m) {
          const double zz = Z[s][i + g.n * m] * Z[s][j + g.n * m];
          r += zz * Sg[s][m];
          b += Sg[s][m] > 0 ? zz / Sg[s][m] : 0.0;
        }
        R[s][idx] = r;  // C^{1/2}, r = n rows
        B[s][idx] = b;  // C^{-1/2}
      }
      bsync();
      gmm(g.E, g.n, g.n, Pt[s], g.E, false, B[s], g.n, false, W[s], g.E);  // W = Pt C^{-1/2}
    } else {
      // wide: R = X (r = E rows), W = (x) Si as an E x E matrix
      for (int i = tid; i < g.E * g.n; i += blockDim.x) R[s][i] = X[s][i];
      for (int idx = tid; idx < g.E * g.E; idx += blockDim.x) {
        const int e = idx % g.E, f = idx / g.E;
        double w = 1.0;
        int re = e, rf = f;
        for (int pa = 0; pa < g.next; ++pa) {
          const int chi = g.dims[g.ext[pa]];
          w *= env_p(s, pa, 2)[(re % chi) * chi + (rf % chi)];
          re /= chi;
          rf /= chi;
        }
        W[s][idx] = w;
      }
      bsync();
    }
  }
  const int du = gs[0].d, dv = gs[1].d;
  const int ru = gs[0].E >= gs[0].n ? gs[0].n : gs[0].E, rv = gs[1].E >= gs[1].n ? gs[1].n : gs[1].E;
  const int nu = gs[0].n, nv = gs[1].n, chib = gs[0].chib;
  const int Mr = ru * du, Nc = rv * dv, dd = du * dv;
  const double* G = gates + it.gate;
  // F4. Tt[(ru + r su), (rv + r sv)] = sum_b R_u[ru, su + du b] R_v[rv, sv + dv b]; Theta = G Tt
  for (int idx = tid; idx < Mr * Nc; idx += blockDim.x) {
    const int row = idx % Mr, col = idx / Mr;
    const int a = row % ru, su = row / ru, c = col % rv, sv = col / rv;
    double t = 0;
    for (int b = 0; b < chib; ++b) t += R[0][a + ru * (su + du * b)] * R[1][c + rv * (sv + dv * b)];
    Tt[idx] = t;
  }
  bsync();
  for (int idx = tid; idx < Mr * Nc; idx += blockDim.x) {
    const int row = idx % Mr, col = idx / Mr;
    const int a = row % ru, sup = row / ru, c = col % rv, svp = col / rv;
    double t = 0;
    for (int su = 0; su < du; ++su)
      for (int sv = 0; sv < dv; ++sv)
        t += G[(sup + du * svp) + dd * (su + du * sv)] * Tt[(a + ru * su) + Mr * (c + rv * sv)];
    Th[idx] = t;
  }
  bsync();
  // F5. thin SVD of Theta (one-sided Jacobi on the taller orientation)
  const bool tr = Mr < Nc;
  const int Ms = tr ? Nc : Mr, Ns = tr ? Mr : Nc;  // Ns = p
  const int p = Ns;
  for (int idx = tid; idx < Mr * Nc; idx += blockDim.x) {
    const int row = idx % Mr, col = idx / Mr;
    if (tr) As[col + Nc * row] = Th[idx];
    else As[idx] = Th[idx];
  }
  bsync();
  jacobi_svd(As, Ms, Ns, Vs, rot, red);
  bsync();
  for (int j = tid; j < Ns; j += blockDim.x) {
    double t = 0;
    for (int i = 0; i < Ms; ++i) t += As[i + Ms * j] * As[i + Ms * j];
    sbar[j] = sqrt(t);  // unsorted singular values (sbar reused below)
  }
  bsync();
  if (tid == 0) {
    for (int i = 0; i < Ns; ++i) order[i] = i;
    for (int i = 0; i < Ns; ++i)
      for (int j = i + 1; j < Ns; ++j)
        if (sbar[order[j]] > sbar[order[i]]) {
          const int t = order[i];
          order[i] = order[j];
          order[j] = t;
        }
    double tot = 0;
    for (int i = 0; i < Ns; ++i) tot += sbar[i] * sbar[i];
    int keep = Ns;
    if (prm.maxdim > 0 && keep > prm.maxdim) keep = prm.maxdim;
    double disc = 0;
    for (int i = keep; i < Ns; ++i) disc += sbar[order[i]] * sbar[order[i]];
    if (prm.cutoff >= 0 && tot > 0)
      while (keep > 1 && (disc + sbar[order[keep - 1]] * sbar[order[keep - 1]]) / tot <= prm.cutoff) {
        disc += sbar[order[keep - 1]] * sbar[order[keep - 1]];
        --keep;
      }
    int st = 0;
    if (keep != o.keep) st = 1;
    if (!isfinite(tot)) st = 2;
    for (int i = 0; i < keep; ++i)
      if (!(sbar[order[i]] > 0)) st = 3;
    status[blockIdx.x] = st;
    sh_keep = st ? -1 : keep;
  }
  __syncthreads();
  const int keep = sh_keep;
  if (keep < 0) return;
  // sorted thin factors: Um (Mr x p), Vm (Nc x p), svec (p)
  for (int idx = tid; idx < Mr * p; idx += blockDim.x) {
    const int i = idx % Mr, j = idx / Mr, oj = order[j];
    const double sj = sbar[oj];
    Um[idx] = tr ? Vs[i + Ns * oj] : (sj > 0 ? As[i + Ms * oj] / sj : 0.0);
  }
  for (int idx = tid; idx < Nc * p; idx += blockDim.x) {
    const int i = idx % Nc, j = idx / Nc, oj = order[j];
    const double sj = sbar[oj];
    Vm[idx] = tr ? (sj > 0 ? As[i + Ms * oj] / sj : 0.0) : Vs[i + Ns * oj];
  }
  bsync();
  for (int j = tid; j < p; j += blockDim.x) svec[j] = sbar[order[j]];
  bsync();
  // F6. F_u = U_k sqrt(S), F_v = V_k sqrt(S)
  for (int idx = tid; idx < Mr * keep; idx += blockDim.x) Fu[idx] = Um[idx] * sqrt(svec[idx / Mr]);
  for (int idx = tid; idx < Nc * keep; idx += blockDim.x) Fv[idx] = Vm[idx] * sqrt(svec[idx / Nc]);
  bsync();
  // F7. pre-gauge outputs Y_s[e, s' + d j] = sum_r W[e, r] F[r + r_s s', j] into T2
  const int rs[2] = {ru, rv};
  const double* Fs[2] = {Fu, Fv};
  for (int s = 0; s < 2; ++s) {
    const SideGeom& g = gs[s];
    const int r = rs[s];
    for (int idx = tid; idx < g.E * g.d * keep; idx += blockDim.x) {
      const int e = idx % g.E, c = idx / g.E, sp = c % g.d, j = c / g.d;
      double t = 0;
      for (int q = 0; q < r; ++q) t += W[s][e + (long long)g.E * q] * Fs[s][(q + r * sp) + (long long)rs[s] * g.d * j];
      T2[s][idx] = t;
    }
    bsync();
  }
  // bond signs from psi_u' (largest |entry| of every slice, first in natural order)
  if (tid < keep) {
    const SideGeom& g = gs[0];
    const int j = tid;
    double best = -1, val = 0;
    int best_off = 0x7fffffff;
    for (int e = 0; e < g.E; ++e)
      for (int s2 = 0; s2 < g.d; ++s2) {
        const double x = T2[0][e + (long long)g.E * (s2 + g.d * j)];
        const int off = nat_off(g, s2, e, j);
        if (fabs(x) > best || (fabs(x) == best && off < best_off)) {
          best = fabs(x);
          best_off = off;
          val = x;
        }
      }
    sgn[j] = val < 0 ? -1.0 : 1.0;
  }
  bsync();

  // ---- backward ------------------------------------------------------------
  // B1-B3. cotangents of the pre-gauge outputs: read, undo the normalisation, the signs
  for (int s = 0; s < 2; ++s) {
    const SideGeom& g = gs[s];
    SideGeom gk = g;
    gk.dims[g.j] = keep;
    const double* dsrc = dout + (s == 0 ? o.out_u : o.out_v);
    const int cols = g.d * keep;
    double n2 = 0, dot = 0;
    for (int idx = tid; idx < g.E * cols; idx += blockDim.x) {
      const int e = idx % g.E, c = idx / g.E;
      const double y = T2[s][idx] * sgn[c / g.d];
      const double yb = dsrc[nat_off(gk, c % g.d, e, c / g.d)];
      Yb[s][idx] = yb;
      n2 += y * y;
      dot += y * yb;
    }
    n2 = block_sum_d(n2, red);
    dot = block_sum_d(dot, red);
    const double nrm = sqrt(n2);
    const bool nz = prm.normalize && n2 > 0;
    for (int idx = tid; idx < g.E * cols; idx += blockDim.x) {
      const double y = T2[s][idx] * sgn[(idx / g.E) / g.d];
      double yb = Yb[s][idx];
      if (nz) yb = (yb - y * dot / n2) / nrm;  // pullback of y / ||y||
      Yb[s][idx] = yb * sgn[(idx / g.E) / g.d];
    }
    bsync();
  }
  // B4. Wbar (E x r) and Fbar (r d x keep)
  double* Fbs[2] = {Fub, Fvb};
  for (int s = 0; s < 2; ++s) {
    const SideGeom& g = gs[s];
    const int r = rs[s];
    for (int idx = tid; idx < g.E * r; idx += blockDim.x) {
      const int e = idx % g.E, q = idx / g.E;
      double t = 0;
      for (int j = 0; j < keep; ++j)
        for (int sp = 0; sp < g.d; ++sp)
          t += Yb[s][e + (long long)g.E * (sp + g.d * j)] * Fs[s][(q + r * sp) + (long long)r * g.d * j];
      T1[s][idx] = t;  // Wbar
    }
    for (int idx = tid; idx < r * g.d * keep; idx += blockDim.x) {
      const int row = idx % (r * g.d), j = idx / (r * g.d);
      const int q = row % r, sp = row / r;
      double t = 0;
      for (int e = 0; e < g.E; ++e) t += W[s][e + (long long)g.E * q] * Yb[s][e + (long long)g.E * (sp + g.d * j)];
      Fbs[s][idx] = t;
    }
    bsync();
  }
  // B5. Ubar = Fbar_u sqrt(S), Vbar = Fbar_v sqrt(S) (zero beyond keep), sbar
  for (int idx = tid; idx < Mr * p; idx += blockDim.x) {
    const int j = idx / Mr;
    M1[idx] = j < keep ? Fub[idx] * sqrt(svec[j]) : 0.0;  // Ubar
  }
  for (int idx = tid; idx < Nc * p; idx += blockDim.x) {
    const int j = idx / Nc;
    Q2[idx] = j < keep ? Fvb[idx] * sqrt(svec[j]) : 0.0;  // Vbar
  }
  for (int j = tid; j < p; j += blockDim.x) {
    double t = 0;
    if (j < keep) {
      for (int i = 0; i < Mr; ++i) t += Fub[i + Mr * j] * Um[i + Mr * j];
      for (int i = 0; i < Nc; ++i) t += Fvb[i + Nc * j] * Vm[i + Nc * j];
      t /= 2 * sqrt(svec[j]);
    }
    sbar[j] = t;
  }
  bsync();
  // B6. thin SVD pullback.  J = U^T Ubar, K = V^T Vbar (p x p) in Ttb, Thb
  gmm(p, p, Mr, Um, Mr, true, M1, Mr, false, Ttb, p);
  gmm(p, p, Nc, Vm, Nc, true, Q2, Nc, false, Thb, p);
  {
    const double smax = svec[0];
    const double eps2 = 1e-24 * smax * smax * smax * smax;
    // Inner (p x p) into Fu (free after B4), then M1' = U Inner + (Ubar - U J) S^-1
    for (int idx = tid; idx < p * p; idx += blockDim.x) {
      const int i = idx % p, j = idx / p;
      double v = i == j ? sbar[i] : 0.0;
      if (i != j) {
        const double dfr = svec[j] * svec[j] - svec[i] * svec[i];
        const double f = dfr / (dfr * dfr + eps2);
        v += f * (Ttb[i + p * j] - Ttb[j + p * i]) * svec[j] + svec[i] * f * (Thb[i + p * j] - Thb[j + p * i]);
      }
      Fu[idx] = v;
    }
    bsync();
  }
  // Fv <- U Inner (Mr x p); As <- U J (Mr x p)
  gmm(Mr, p, p, Um, Mr, false, Fu, p, false, Fv, Mr);
  gmm(Mr, p, p, Um, Mr, false, Ttb, p, false, As, Mr);
  for (int idx = tid; idx < Mr * p; idx += blockDim.x) {
    const int j = idx / Mr;
    const double inv = (j < keep && svec[j] > 0) ? 1.0 / svec[j] : 0.0;
    Fv[idx] += (M1[idx] - As[idx]) * inv;  // U Inner + (I - U U^T) Ubar S^-1
  }
  // Vs <- S^-1 (Vbar^T - K^T V^T) (p x Nc)
  bsync();
  gmm(p, Nc, p, Thb, p, true, Vm, Nc, true, Vs, p);  // K^T V^T
  for (int idx = tid; idx < p * Nc; idx += blockDim.x) {
    const int j = idx % p, c = idx / p;
    const double inv = (j < keep && svec[j] > 0) ? 1.0 / svec[j] : 0.0;
    Vs[idx] = (Q2[c + Nc * j] - Vs[idx]) * inv;
  }
  bsync();
  // Thetabar = Fv V^T + U Vs (Mr x Nc)
  gmm(Mr, Nc, p, Fv, Mr, false, Vm, Nc, true, Thb, Mr);
  gmm(Mr, Nc, p, Um, Mr, false, Vs, p, false, Thb, Mr, true);
  // B7. Ttbar and Gbar
  for (int idx = tid; idx < Mr * Nc; idx += blockDim.x) {
    const int row = idx % Mr, col = idx / Mr;
    const int a = row % ru, su = row / ru, c = col % rv, sv = col / rv;
    double t = 0;
    for (int sup = 0; sup < du; ++sup)
      for (int svp = 0; svp < dv; ++svp)
        t += G[(sup + du * svp) + dd * (su + du * sv)] * Thb[(a + ru * sup) + Mr * (c + rv * svp)];
    Ttb[idx] = t;
  }
  for (int idx = tid; idx < dd * dd; idx += blockDim.x) {
    const int i = idx % dd, jj = idx / dd;
    const int sup = i % du, svp = i / du, su = jj % du, sv = jj / du;
    double t = 0;
    for (int a = 0; a < ru; ++a)
      for (int c = 0; c < rv; ++c) t += Thb[(a + ru * sup) + Mr * (c + rv * svp)] * Tt[(a + ru * su) + Mr * (c + rv * sv)];
    dgate[o.dgate + idx] = t;
  }
  bsync();
  // B8. Rbar
  for (int idx = tid; idx < ru * nu; idx += blockDim.x) {
    const int a = idx % ru, cu = idx / ru, su = cu % du, b = cu / du;
    double t = 0;
    for (int c = 0; c < rv; ++c)
      for (int sv = 0; sv < dv; ++sv) t += Ttb[(a + ru * su) + Mr * (c + rv * sv)] * R[1][c + rv * (sv + dv * b)];
    Rb[0][idx] = t;
  }
  for (int idx = tid; idx < rv * nv; idx += blockDim.x) {
    const int c = idx % rv, cv = idx / rv, sv = cv % dv, b = cv / dv;
    double t = 0;
    for (int a = 0; a < ru; ++a)
      for (int su = 0; su < du; ++su) t += Ttb[(a + ru * su) + Mr * (c + rv * sv)] * R[0][a + ru * (su + du * b)];
    Rb[1][idx] = t;
  }
  bsync();
  // B9-B11 per side
  for (int s = 0; s < 2; ++s) {
    const SideGeom& g = gs[s];
    const int n = g.n;
    if (g.E >= n) {
      // Bbar = Pt^T Wbar (n x n); Ptbar = Wbar B (E x n) into Pb
      gmm(n, n, g.E, Pt[s], g.E, true, T1[s], g.E, false, Bb[s], n);
      gmm(g.E, n, n, T1[s], g.E, false, B[s], n, false, Pb[s], g.E);
      // Cbar = Z [(Z^T Rbar_s Z) o K1 + (Z^T Bbar_s Z) o K2] Z^T
      for (int idx = tid; idx < n * n; idx += blockDim.x) {
        const int i = idx % n, j = idx / n;
        Cb[s][idx] = 0.5 * (Rb[s][i + n * j] + Rb[s][j + n * i]);
        A[s][idx] = 0.5 * (Bb[s][i + n * j] + Bb[s][j + n * i]);
      }
      bsync();
      gmm(n, n, n, Z[s], n, true, Cb[s], n, false, T2[s], n);
      gmm(n, n, n, T2[s], n, false, Z[s], n, false, Cb[s], n);  // Z^T Rbar Z
      gmm(n, n, n, Z[s], n, true, A[s], n, false, T2[s], n);
      gmm(n, n, n, T2[s], n, false, Z[s], n, false, A[s], n);   // Z^T Bbar Z
      for (int idx = tid; idx < n * n; idx += blockDim.x) {
        const int i = idx % n, j = idx / n;
        const double si = Sg[s][i], sj = Sg[s][j];
        const double k1 = (si + sj) > 0 ? 1.0 / (si + sj) : 0.0;
        const double k2 = (si > 0 && sj > 0) ? -1.0 / (si * sj * (si + sj)) : 0.0;
        T2[s][idx] = Cb[s][idx] * k1 + A[s][idx] * k2;
      }
      bsync();
      gmm(n, n, n, Z[s], n, false, T2[s], n, false, A[s], n);
      gmm(n, n, n, A[s], n, false, Z[s], n, true, Cb[s], n);    // Cbar (symmetric)
      // Xbar = 2 X Cbar
      gmm(g.E, n, n, X[s], g.E, false, Cb[s], n, false, Xb[s], g.E);
      for (int i = tid; i < g.E * n; i += blockDim.x) Xb[s][i] *= 2.0;
      bsync();
    } else {
      for (int i = tid; i < g.E * n; i += blockDim.x) {
        Xb[s][i] = Rb[s][i];
        Pb[s][i] = 0.0;
      }
      bsync();
      // Sibar_a from Wbar (E x E) with W = (x) Si
      for (int pa = 0; pa < g.next; ++pa) {
        const int chi = g.dims[g.ext[pa]];
        double* Sib = env_p(s, pa, 4);
        // every (e, f) pair with e_pa = x, f_pa = y
        for (int idx = tid; idx < chi * chi; idx += blockDim.x) {
          const int x = idx / chi, y = idx % chi;
          double t = 0;
          for (int e = 0; e < g.E; ++e)
            for (int f = 0; f < g.E; ++f) {
              int re = e, rf = f;
              bool ok = true;
              double w = 1.0;
              for (int qa = 0; qa < g.next; ++qa) {
                const int c2 = g.dims[g.ext[qa]];
                const int ea = re % c2, fa = rf % c2;
                re /= c2;
                rf /= c2;
                if (qa == pa) ok = ok && ea == x && fa == y;
                else w *= env_p(s, qa, 2)[ea * c2 + fa];
              }
              if (ok) t += T1[s][e + (long long)g.E * f] * w;
            }
          Sib[x * chi + y] = t;
        }
        bsync();
      }
    }
    // Sbar_a = sum Xbar[e (e_a = x), c] (psi (x)_{others} S)[e (e_a = y), c]
    // (Xbar, Pb intact; T2, A, W, Pt are free)
    for (int pa = 0; pa < g.next; ++pa) {
      double* yc = T2[s];
      double* yo = A[s];
      for (int idx = tid; idx < g.E * n; idx += blockDim.x) {
        const int e = idx % g.E, c = idx / g.E;
        yc[idx] = psi[g.psi_off + nat_off(g, c % g.d, e, c / g.d)];
      }
      bsync();
      for (int qa = 0; qa < g.next; ++qa) {
        if (qa == pa) continue;
        ext_mp_g(g, qa, yc, yo, n, env_p(s, qa, 1));
        double* t = yc;
        yc = yo;
        yo = t;
      }
      int stride = 1;
      for (int i = 0; i < pa; ++i) stride *= g.dims[g.ext[i]];
      const int chi = g.dims[g.ext[pa]];
      double* Sb = env_p(s, pa, 3);
      for (int idx = tid; idx < chi * chi; idx += blockDim.x) {
        const int x = idx / chi, y = idx % chi;
        double t = 0;
        for (int c = 0; c < n; ++c)
          for (int rest = 0; rest < g.E / chi; ++rest) {
            const int lo = rest % stride, hi = rest / stride;
            t += Xb[s][(lo + stride * (x + chi * hi)) + (long long)g.E * c] *
                 yc[(lo + stride * (y + chi * hi)) + (long long)g.E * c];
          }
        Sb[x * chi + y] = t;
      }
      bsync();
    }
    // psibar = Xbar (x) S (+ Ptbar (x) P on a tall side), to the natural layout
    {
      const double* src = Xb[s];
      double* bufs2[2] = {T2[s], A[s]};
      int bi = 0;
      for (int pa = 0; pa < g.next; ++pa) {
        ext_mp_g(g, pa, src, bufs2[bi], n, env_p(s, pa, 1));
        src = bufs2[bi];
        bi ^= 1;
      }
      const double* srcp = nullptr;
      if (g.E >= n) {
        srcp = Pb[s];
        double* bufs3[2] = {W[s], Pt[s]};
        int bj = 0;
        for (int pa = 0; pa < g.next; ++pa) {
          ext_mp_g(g, pa, srcp, bufs3[bj], n, env_p(s, pa, 5));
          srcp = bufs3[bj];
          bj ^= 1;
        }
      }
      double* dst = din + (s == 0 ? o.in_u : o.in_v);
      for (int idx = tid; idx < g.E * n; idx += blockDim.x) {
        const int e = idx % g.E, c = idx / g.E;
        dst[nat_off(g, c % g.d, e, c / g.d)] = src[idx] + (srcp ? srcp[idx] : 0.0);
      }
      bsync();
    }
    // environment pullbacks into dmsg (accumulated; every message of a call belongs to one bond)
    {
      const int wv = tid >> 6;
      for (int pa = wv; pa < g.next; pa += (int)blockDim.x / 64) {
        const int a = g.ext[pa];
        const int chi = g.dims[a];
        double* Mb = env_p(s, pa, 5);
        env_pullback(env_p(s, pa, 0), env[s] + pa * VJ_ENV + 6 * 64, kmask[s][pa], chi, env_p(s, pa, 3),
                     env_p(s, pa, 4), env_p(s, pa, 2), Mb);
        __threadfence_block();
        const long long off = vds[vtx[s]].in_msg[a];
        for (int idx = tid & 63; idx < chi * chi; idx += 64) {
          const int i = idx % chi, j = idx / chi;  // message layout M[i + chi j]
          dmsg[off + idx] += Mb[i * chi + j];
        }
      }
      bsync();
    }
  }
}

}  // namespace

extern "C" int itnbp_apply_vjp(itnbp_net* net, int n, const int* edge_ids, const double* gates, int maxdim,
                               double cutoff, int normalize, const int* kept, const double* dpsi_out,
                               double* dpsi_in, double* dgates, double* dmsgs) {
  if (!net || n < 0 || (n > 0 && (!edge_ids || !gates || !kept || !dpsi_out || !dpsi_in || !dgates || !dmsgs)))
    return ITNBP_ERR_ARG;
  if (n == 0) return ITNBP_OK;
  itnbp_ctx* ctx = net->ctx;
  return itnbp_guarded(ctx, [&]() -> int {
    std::vector<ApplyItem> items;
    long long goff = 0;
    ITNBP_RETCHK(prepare_apply(net, n, edge_ids, maxdim, cutoff, nullptr, 1, net->chi, false, items, goff));
    std::vector<VjpIo> io(n);
    long long out_tot = 0, in_tot = 0;
    for (int i = 0; i < n; ++i) {
      const ApplyItem& it = items[i];
      const int e = edge_ids[i];
      const int chib = net->chi[e];
      if (kept[i] < 1) return itnbp_fail(ctx, ITNBP_ERR_ARG, "apply_vjp: kept must be >= 1");
      for (int side = 0; side < 2; ++side) {
        const int x = side == 0 ? it.u : it.v;
        const long long D = net->vdesc[x].D;
        const long long E = D / ((long long)net->phys[x] * chib);
        if (E * net->phys[x] * kept[i] > AP_XY)
          return itnbp_fail(ctx, ITNBP_ERR_UNSUPPORTED, "apply_vjp: the new site tensor is too large");
        const long long Dn = D / chib * kept[i];
        if (side == 0) {
          io[i].out_u = out_tot;
          io[i].in_u = in_tot;
        } else {
          io[i].out_v = out_tot;
          io[i].in_v = in_tot;
        }
        out_tot += Dn;
        in_tot += D;
      }
      io[i].dgate = it.gate;
      io[i].keep = kept[i];
      io[i].pad = 0;
    }
    DevBuf b_items, b_io, b_gates, b_out, b_in, b_dg, b_dm, b_work, b_st;
    struct Guard {
      DevBuf* b[9];
      ~Guard() {
        for (DevBuf* x : b) free_buf(*x);
      }
    } guard{{&b_items, &b_io, &b_gates, &b_out, &b_in, &b_dg, &b_dm, &b_work, &b_st}};
    ITNBP_RETCHK(upload(ctx, b_items, items.data(), n * sizeof(ApplyItem)));
    ITNBP_RETCHK(upload(ctx, b_io, io.data(), n * sizeof(VjpIo)));
    ITNBP_RETCHK(upload(ctx, b_gates, gates, goff * 8));
    ITNBP_RETCHK(upload(ctx, b_out, dpsi_out, out_tot * 8));
    ITNBP_RETCHK(upload(ctx, b_dm, dmsgs, net->msg_total * 8));
    ITNBP_RETCHK(ensure_buf(ctx, b_in, in_tot * 8));
    ITNBP_RETCHK(ensure_buf(ctx, b_dg, goff * 8));
    ITNBP_RETCHK(ensure_buf(ctx, b_work, (size_t)n * VJ_GATE * 8));
    ITNBP_RETCHK(ensure_buf(ctx, b_st, n * sizeof(int)));
    ApplyParams prm;
    prm.maxdim = maxdim;
    prm.cutoff = cutoff;
    prm.normalize = normalize;
    prm.eig_cutoff = 10 * 2.220446049250313e-16;
    prm.max_keep = 1;
    const int pm0 = prof_mark(ctx);
    hipLaunchKernelGGL(k_apply_vjp, dim3(n), dim3(256), 0, ctx->stream, (const ApplyItem*)b_items.p,
                       (const VjpIo*)b_io.p, net->d_vdesc, (const double*)net->d_psi, net->d_msg[net->cur],
                       (const double*)b_gates.p, prm, (const double*)b_out.p, (double*)b_in.p, (double*)b_dg.p,
                       (double*)b_dm.p, (double*)b_work.p, (int*)b_st.p);
    ITNBP_HIPCHK(ctx, hipGetLastError());
    prof_add(ctx, "apply_vjp", pm0, prof_mark(ctx));
    std::vector<int> st(n);
    ITNBP_HIPCHK(ctx, hipMemcpyAsync(st.data(), b_st.p, n * sizeof(int), hipMemcpyDeviceToHost, ctx->stream));
    ITNBP_HIPCHK(ctx, hipMemcpyAsync(dpsi_in, b_in.p, in_tot * 8, hipMemcpyDeviceToHost, ctx->stream));
    ITNBP_HIPCHK(ctx, hipMemcpyAsync(dgates, b_dg.p, goff * 8, hipMemcpyDeviceToHost, ctx->stream));
    ITNBP_HIPCHK(ctx, hipMemcpyAsync(dmsgs, b_dm.p, net->msg_total * 8, hipMemcpyDeviceToHost, ctx->stream));
    ITNBP_HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
    for (int i = 0; i < n; ++i) {
      if (st[i] == 1)
        return itnbp_fail(ctx, ITNBP_ERR_ARG, "apply_vjp: kept differs from the rank the truncation keeps");
      if (st[i] == 2) return itnbp_fail(ctx, ITNBP_ERR_NONFINITE, "apply_vjp: non-finite two-site tensor");
      if (st[i] == 3)
        return itnbp_fail(ctx, ITNBP_ERR_UNSUPPORTED, "apply_vjp: a kept singular value is zero (no derivative)");
    }
    return ITNBP_OK;
  });
}
