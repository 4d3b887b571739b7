// Gate application for bonds past the LDS kernel's limits (external bonds up
// to 32, d chi_b <= 64, Theta up to 128 x 128): the steps of simple_update_bp
// (src/apply.jl:33-95) as a sequence of launches over all gates of a call, so
// that the passes over the site tensors fill the device instead of running on
// one workgroup per bond.  One side of a gate: psi as the E x n matrix of its
// external bonds (E) and (s, b) = physical index and gate bond (n = d chi_b).
//
//   roots     sqrt(M), M^{-1/2} of every external environment message (and the
//             projector P on its kept eigenvectors where some are dropped)
//   mode x3   X = psi with sqrt(M) on the external bonds, in place per bond
//   gram      partial G = X^T X per block of rows
//   chol1     G -> X1 = X T with orthonormal columns up to rounding, R0: X = X1 R0
//   gram      partial G1 = X1^T X1 (X1 in registers only)
//   chol2     G1 = R1^T R1: R = R1 R0, Tq = T R1^{-1}, so X = Q R with Q = X Tq
//   theta     gate * (R_u R_v)
//   svd       pivoted QR, one-sided Jacobi, truncation
//   factors   W = Tq [U sqrt(S)] and Tq [V sqrt(S)] (n x d keep)
//   mode x3   only where P != 1: psi with P on that bond (into X)
//   rebuild   psi' = psi W in place, with the largest entry of every new-bond
//             slice and the norm per block
//   signs, scale
//
// M^{-1/2} is never applied to a tall side: Q = X Tq with X = psi sqrt(M), and
// sqrt(M) M^{-1/2} = P, which is the identity unless map_eigvals drops
// eigenvalues, so psi' = (psi P) Tq F.  A wide side (E <= n) of full rank needs no
// QR: R = X, Q = 1 and psi' = M^{-1/2} F.
//
// Bound: the launches over the site tensors move about 12 times their bytes
// (three read + write passes, two Gram reads, rebuild, scale) and are HBM-bound
// at chi = 32; the per-gate kernels (roots, chol, svd) are latency-bound, one
// workgroup each.  One round with the copies in and out, against one workgroup
// per bond through all steps: 8x8 chi = 16 (4 classes of 28 gates) 44.1 -> 8.9 ms,
// 5x4 chi = 32 (4 classes of 6 to 10) 447 -> 26.6 ms; per class there, svd 0.51 and
// 2.12 ms, rebuild 88 and 343 us, roots 75 and 197 us, grams 89 and 347 us, chol 81
// and 476 us, the three mode passes 50 and 124 us.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <string>
#include <vector>

#include "itnbp_apply.hpp"
#include "itnbp_ops.hpp"

namespace {

constexpr double EPS = 2.220446049250313e-16;
constexpr int GB_ROWS = 64;    // external rows of one chunk
constexpr int GB_PITCH = 66;   // LDS pitch of a chunk's columns: 2 mod 32 doubles, conflict-free MFMA operands
constexpr int GB_N = AP_N_BIG; // 64
constexpr int GB_ROOT = AP_ENV_BIG * AP_ENV_BIG;
constexpr int GB_LD = CholLds<4>::LD;

struct GbSide {
  long long psi_off;             // site tensor
  long long x_off;               // X in the workspace (natural layout of the site tensor)
  long long msg_off[AP_MAXEXT];  // environment messages
  int ext_dim[AP_MAXEXT], ext_st[AP_MAXEXT];  // external bonds: dimension, stride in the site tensor
  int ext_est[AP_MAXEXT];                     // and in the external index e
  int next, d, chib, lay;  // chib: bond dimension before the call; lay: of its layout (>= chib)
  int lo, E, n, wide, D;   // lo: product of the bonds before the gate bond
  FastDiv fd, fn, flo, fdlo, flay;
};

// written by the kernels
struct GbInfo {
  int r;                  // rows of R
  int trunc[AP_MAXEXT];   // the environment dropped eigenvalues (P != 1)
};
struct GbGate {
  long long gate_off;
  int slot, pad;
};
struct GbOut {
  int keep;   // -1: refused, tensors untouched
  int pad;
};

struct GbWork {  // device pointers
  const GbSide* side;
  const GbGate* gate;
  GbInfo* info;
  GbOut* out;
  double* roots;   // per side: AP_MAXEXT x (S, Si, P) x GB_ROOT
  double* T;       // per side n x r
  double* R0;      // per side r x n
  double* R;       // per side r x n
  double* Tq;      // per side n x r
  double* W;       // per side n x (d keep); wide: E x (d keep)
  double* theta;   // per gate M x N
  double* V;       // per gate N x keep
  double* sv;      // per gate, sorted
  double* part;    // per side nsplit x n x n
  double* normp;   // per side gxr
  double* cmax;    // per gate gxr x mcols
  int* coff;
  double* sgn;     // per gate AP_KEEP_BIG
  double* scale;   // per side
  double* X;
  int nsplit, gxr, mcols;  // mcols: stride of cmax and coff
  int lcols;               // the most columns d keep of a tall side
};

constexpr int GB_SQ = GB_N * GB_N;
constexpr int GB_W = AP_TH_BIG * AP_KEEP_BIG;

__device__ inline int gb_nat(const GbSide& g, int s, int e, int b) {
  const int hi = (int)g.flo.div(e), lo = e - hi * g.lo;
  return s + g.d * (lo + g.lo * (b + g.lay * hi));
}

// ---- environment roots -----------------------------------------------------
// One workgroup per environment (block_jacobi_eigh, M scaled to order 1 by an even
// power of two); stopping rule and eigenvalue truncation of env_roots_wave.
__global__ __launch_bounds__(256) void k_gb_roots(GbWork w, const double* __restrict__ msg, double cutoff) {
  const GbSide& g = w.side[blockIdx.y];
  const int pa = blockIdx.x;
  if (pa >= g.next) return;
  constexpr int LD = AP_ENV_BIG + 1;
  __shared__ double A[AP_ENV_BIG * LD], V[AP_ENV_BIG * LD], rc[16], rs[16], red[8];
  __shared__ int rank[AP_ENV_BIG], byr[AP_ENV_BIG];
  const int tid = threadIdx.x, chi = g.ext_dim[pa];
  const double* M = msg + g.msg_off[pa];
  double a[4], mx = 0;
#pragma unroll
  for (int h = 0; h < 4; ++h) {
    const int i = (tid >> 5) + 8 * h, j = tid & 31;
    a[h] = (i < chi && j < chi) ? 0.5 * (M[i + chi * j] + M[j + chi * i]) : 0.0;
    V[i * LD + j] = i == j ? 1.0 : 0.0;
    mx = fmax(mx, fabs(a[h]));
  }
  for (int m = 32; m > 0; m >>= 1) mx = fmax(mx, __shfl_xor(mx, m));
  if ((tid & 63) == 0) red[tid >> 6] = mx;
  __syncthreads();
  mx = fmax(fmax(red[0], red[1]), fmax(red[2], red[3]));
  const int ex = mx > 0 && isfinite(mx) ? ilogb(mx) & ~1 : 0;
#pragma unroll
  for (int h = 0; h < 4; ++h) A[((tid >> 5) + 8 * h) * LD + (tid & 31)] = ldexp(a[h], -ex);
  __syncthreads();
  block_jacobi_eigh<LD>(A, V, chi, 1e-30, rc, rs, red);
  // truncation: rank |lambda| descending (ties by index); drop from the small
  // end while the dropped weight / total <= cutoff (keep >= 1)
  if (tid < chi) {
    const double wl = fabs(A[tid * LD + tid]);
    int r = 0;
    for (int m = 0; m < chi; ++m) {
      const double wm = fabs(A[m * LD + m]);
      if (wm > wl || (wm == wl && m < tid)) ++r;
    }
    rank[tid] = r;
  }
  __syncthreads();
  if (tid < chi) byr[tid] = tid;  // a NaN spectrum ranks nothing: every index stays valid
  __syncthreads();
  if (tid < chi) byr[rank[tid]] = tid;
  __syncthreads();
  double tot = 0;
  for (int m = 0; m < chi; ++m) tot += fabs(A[m * LD + m]);
  int keep = chi;
  double disc = 0;
  while (keep > 1 && tot > 0) {
    const int m = byr[keep - 1];
    const double x = fabs(A[m * LD + m]);
    if (!((disc + x) / tot <= cutoff)) break;
    disc += x;
    --keep;
  }
  double* S = w.roots + ((long long)blockIdx.y * AP_MAXEXT + pa) * 3 * GB_ROOT;
  for (int o = tid; o < chi * chi; o += 256) {
    const int i = o / chi, j = o - i * chi;
    double sv = 0, siv = 0, pv = 0;
    for (int m = 0; m < chi; ++m) {
      if (rank[m] >= keep) continue;
      const double sq = sqrt(A[m * LD + m]);  // NaN for a kept negative eigenvalue
      const double vv = V[i * LD + m] * V[j * LD + m];
      sv += vv * sq;
      siv += vv / sq;
      pv += vv;
    }
    S[o] = ldexp(sv, ex / 2);
    S[GB_ROOT + o] = ldexp(siv, -ex / 2);
    S[2 * GB_ROOT + o] = pv;
  }
  if (tid == 0) w.info[blockIdx.y].trunc[pa] = keep < chi;
}

// ---- mode products -----------------------------------------------------------
// Bond pa of a side: Y[.. b' ..] = sum_b src[.. b ..] K[b][b'] (K symmetric), src
// and Y in the site tensor's layout.  A wave owns 16 fibres (consecutive, so its
// loads and stores are runs of min(16, stride) doubles): it loads their chi
// entries as the B operands of v_mfma_f64_16x16x4f64 (B[k = b][fibre]), the
// matrix stays in registers as the A operands (A[b'][b]), and every fibre is
// written back by the wave that read it, so the product runs in place.
// PROJ = false: K = sqrt(M), psi -> X on bond 0, then X in place.  PROJ = true:
// K = P of a truncated environment, psi -> X on the first truncated bond of the
// side, then X in place; most sides have none and return.
template <bool PROJ>
__global__ __launch_bounds__(256) void k_gb_mode(GbWork w, const double* __restrict__ psi, int pa) {
  const GbSide& g = w.side[blockIdx.y];
  const double* src = psi + g.psi_off;
  double* dst = w.X + g.x_off;
  if constexpr (PROJ) {
    const GbInfo& in = w.info[blockIdx.y];
    if (g.wide || pa >= g.next || !in.trunc[pa] || w.out[blockIdx.y >> 1].keep < 0) return;
    for (int a = 0; a < pa; ++a)
      if (in.trunc[a]) src = dst;
  } else {
    if (pa >= g.next) {
      if (pa == 0)  // no external bond: X = psi
        for (int i = blockIdx.x * 256 + threadIdx.x; i < g.D; i += gridDim.x * 256) dst[i] = src[i];
      return;
    }
    if (pa > 0) src = dst;
  }
  const double* K = w.roots + ((long long)blockIdx.y * AP_MAXEXT + pa) * 3 * GB_ROOT + (PROJ ? 2 * GB_ROOT : 0);
  const int l = threadIdx.x & 63, li = l & 15, lk = l >> 4;
  const int chi = g.ext_dim[pa], st = g.ext_st[pa], nq = (chi + 3) >> 2;
  const int nfib = g.D / chi, ngrp = (nfib + 15) >> 4;
  const FastDiv fst = fast_div((unsigned)st);
  double am[2][8];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int b = 4 * q + lk, b2 = 16 * t + li;
      am[t][q] = (b < chi && b2 < chi) ? K[b * chi + b2] : 0.0;
    }
  for (int gr = blockIdx.x * 4 + (threadIdx.x >> 6); gr < ngrp; gr += gridDim.x * 4) {
    const int f = 16 * gr + li;
    const bool fin = f < nfib;
    const int hi = (int)fst.div(fin ? f : 0);
    const long long base = (fin ? f - hi * st : 0) + (long long)st * chi * hi;
    double x[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int b = 4 * q + lk;
      x[q] = (q < nq && fin && b < chi) ? src[base + (long long)st * b] : 0.0;
    }
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      if (16 * t >= chi) break;
      f64x4 acc = {0, 0, 0, 0};
#pragma unroll
      for (int q = 0; q < 8; ++q)
        if (q < nq) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(am[t][q], x[q], acc, 0, 0, 0);
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int b2 = 16 * t + 4 * v + lk;
        if (fin && b2 < chi) dst[base + (long long)st * b2] = acc[v];
      }
    }
  }
}

// ---- chunks of external rows --------------------------------------------------
// tile[c * GB_PITCH + r] = src(row e0 + r, column c = s + d b) for b < chib, zero
// past E and n; 16 nt columns.  Loads follow the site tensor's memory order.
__device__ inline void gb_load_tile(const GbSide& g, const double* __restrict__ src, int e0, int nt, double* tile) {
  const int tid = threadIdx.x;
  if (g.lo >= 16) {
    const int tot = g.d * GB_ROWS * g.chib;
#pragma unroll 4
    for (int i = tid; i < tot; i += 256) {
      const int t = (int)g.fd.div(i), s = i - t * g.d, r = t & (GB_ROWS - 1), b = t / GB_ROWS;
      const int e = e0 + r;
      tile[(s + g.d * b) * GB_PITCH + r] = e < g.E ? src[gb_nat(g, s, e, b)] : 0.0;
    }
  } else {
    const int tot = g.n * GB_ROWS;
#pragma unroll 4
    for (int i = tid; i < tot; i += 256) {
      const int r = (int)g.fn.div(i), c = i - r * g.n;
      const int b = (int)g.fd.div(c), s = c - b * g.d;
      const int e = e0 + r;
      tile[c * GB_PITCH + r] = e < g.E ? src[gb_nat(g, s, e, b)] : 0.0;
    }
  }
  for (int i = tid; i < (16 * nt - g.n) * GB_ROWS; i += 256)
    tile[(g.n + i / GB_ROWS) * GB_PITCH + (i & (GB_ROWS - 1))] = 0.0;
}

// Partial Gram of the chunks blockIdx.x, blockIdx.x + gridDim.x, .. of a side:
// wave w takes rows 16 w .. of every chunk; the upper-triangle 16 x 16 tiles
// (ti <= tj) accumulate in registers, one LDS value per lane feeding a tile row
// as A operand (A[i = column][k = row]) and a tile column as B operand.  SECOND:
// of X1 = X T, whose 16 x 16 tiles come out of the MFMA as D[4 v + l / 16][l % 16],
// which is the operand of K-step v, so X1 stays in registers.
template <int NT, bool SECOND>
__device__ void gb_gram_body(const GbWork& w, const GbSide& g, int r, double* sm) {
  const int tid = threadIdx.x, l = tid & 63, wv = tid >> 6, li = l & 15, lk = l >> 4;
  double* tile = sm;
  double* Tl = sm + GB_N * GB_PITCH;
  const double* X = w.X + g.x_off;
  const int side = blockIdx.y;
  const int rn = SECOND ? r : g.n;  // size of the Gram
  if constexpr (SECOND) {
    const double* T = w.T + (long long)side * GB_SQ;
    for (int i = tid; i < GB_N * GB_N; i += 256) {
      const int c = i & 63, k = i >> 6;
      Tl[c * GB_PITCH + k] = (c < g.n && k < r) ? T[c + g.n * k] : 0.0;
    }
  }
  f64x4 acc[NT * (NT + 1) / 2];
#pragma unroll
  for (int t = 0; t < NT * (NT + 1) / 2; ++t) acc[t] = f64x4{0, 0, 0, 0};
  const int nch = (g.E + GB_ROWS - 1) / GB_ROWS;
  for (int ch = blockIdx.x; ch < nch; ch += gridDim.x) {
    __syncthreads();  // the previous chunk is consumed
    gb_load_tile(g, X, ch * GB_ROWS, NT, tile);
    __syncthreads();
    f64x4 x1[NT];
    if constexpr (SECOND) {
#pragma unroll
      for (int t = 0; t < NT; ++t) x1[t] = f64x4{0, 0, 0, 0};
#pragma unroll 4
      for (int q = 0; q < 4 * NT; ++q) {
        const double a = tile[(4 * q + lk) * GB_PITCH + 16 * wv + li];
#pragma unroll
        for (int t = 0; t < NT; ++t)
          x1[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, Tl[(4 * q + lk) * GB_PITCH + 16 * t + li], x1[t], 0, 0, 0);
      }
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      double op[NT];
#pragma unroll
      for (int t = 0; t < NT; ++t)
        op[t] = SECOND ? x1[t][v] : tile[(16 * t + li) * GB_PITCH + 16 * wv + 4 * v + lk];
      int k = 0;
#pragma unroll
      for (int ti = 0; ti < NT; ++ti)
#pragma unroll
        for (int tj = ti; tj < NT; ++tj, ++k)
          acc[k] = __builtin_amdgcn_mfma_f64_16x16x4f64(op[ti], op[tj], acc[k], 0, 0, 0);
    }
  }
  // the four waves' tiles, summed in wave order
  for (int q = 0; q < 4; ++q) {
    __syncthreads();
    if (wv == q) {
#pragma unroll
      for (int k = 0; k < NT * (NT + 1) / 2; ++k)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          double* p = tile + k * 256 + v * 64 + l;
          *p = (q == 0 ? 0.0 : *p) + acc[k][v];
        }
    }
  }
  __syncthreads();
  double* out = w.part + ((long long)side * w.nsplit + blockIdx.x) * GB_SQ;
  int k = 0;
  for (int ti = 0; ti < NT; ++ti)
    for (int tj = ti; tj < NT; ++tj, ++k) {
      // thread tid: value v = tid / 64 of lane tid % 64
      const int row = 16 * ti + 4 * wv + lk, col = 16 * tj + li;
      const double x = tile[k * 256 + tid];
      if (row < rn && col < rn) {
        out[row + rn * col] = x;
        if (ti != tj) out[col + rn * row] = x;
      }
    }
}

template <bool SECOND>
__global__ __launch_bounds__(256) void k_gb_gram(GbWork w) {
  extern __shared__ __align__(16) double sm[];
  const GbSide& g = w.side[blockIdx.y];
  if (g.wide || (int)blockIdx.x * GB_ROWS >= g.E) return;
  const int r = SECOND ? w.info[blockIdx.y].r : g.n;
  switch ((g.n + 15) >> 4) {
    case 1: gb_gram_body<1, SECOND>(w, g, r, sm); break;
    case 2: gb_gram_body<2, SECOND>(w, g, r, sm); break;
    case 3: gb_gram_body<3, SECOND>(w, g, r, sm); break;
    default: gb_gram_body<4, SECOND>(w, g, r, sm); break;
  }
}

// ---- Cholesky -----------------------------------------------------------------
__device__ inline void gb_sum_parts(const GbWork& w, int side, int np, int n, double (&g)[4][4]) {
  const int ti = threadIdx.x & 15, tj = threadIdx.x >> 4;
  const double* p = w.part + (long long)side * w.nsplit * GB_SQ;
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < 4; ++b) g[a][b] = 0;
  for (int q = 0; q < np; ++q, p += GB_SQ)
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
      for (int a = 0; a < 4; ++a) {
        const int i = ti + 16 * a, j = tj + 16 * b;
        if (i < n && j < n) g[a][b] += p[i + n * j];
      }
}

// X X^T of a wide side (E <= n <= 64) from R = X
__device__ inline void gb_wide_gram(const GbWork& w, int side, double (&g)[4][4]) {
  const GbSide& sd = w.side[side];
  const int ti = threadIdx.x & 15, tj = threadIdx.x >> 4, E = sd.E;
  const double* R = w.R + (long long)side * GB_SQ;
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const int i = ti + 16 * a, j = tj + 16 * b;
      g[a][b] = 0;
      if (i < E && j < E)
        for (int c = 0; c < sd.n; ++c) g[a][b] += R[i + E * c] * R[j + E * c];
    }
}

// R <- V_r^T R (r x n) in place, V E x E in LDS
__device__ inline void gb_wide_rank(const GbWork& w, int side, int r, const double* V, const int* keep_idx) {
  const GbSide& g = w.side[side];
  const int tid = threadIdx.x, E = g.E;
  double* R = w.R + (long long)side * GB_SQ;
  double t[16];
#pragma unroll
  for (int q = 0; q < 16; ++q) {
    const int i = tid + 256 * q, k = i % r, c = i / r;
    t[q] = 0;
    if (i < r * g.n)
      for (int e = 0; e < E; ++e) t[q] += V[e + E * keep_idx[k]] * R[e + E * c];
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < 16; ++q)
    if (tid + 256 * q < r * g.n) R[tid + 256 * q] = t[q];
}

// The first factorisation of a side.  The Cholesky factor is used while its
// pivots span at most 1e-10 (R's diagonal 1e-5); a side past that,
// rank-deficient ones among them, takes the eigendecomposition G = V diag(l) V^T by one-sided Jacobi instead, dropping
// directions with l <= n eps l_max: T = V_r l_r^{-1/2}, R0 = l_r^{1/2} V_r^T,
// exact inverses of each other however graded l is.  A wide side keeps R = X, Q = 1
// unless X X^T fails the same test: then R = V_r^T X and Q = V_r with its
// eigenvectors, so that noise directions stay out of Theta.
__global__ __launch_bounds__(256) void k_gb_chol1(GbWork w) {
  extern __shared__ __align__(16) double sm[];
  const int side = blockIdx.x, tid = threadIdx.x;
  const GbSide& g = w.side[side];
  const int n = g.wide ? g.E : g.n;
  double* T = w.T + (long long)side * GB_SQ;
  double* R0 = w.R0 + (long long)side * GB_SQ;
  if (g.wide) {  // R = X
    const double* X = w.X + g.x_off;
    double* R = w.R + (long long)side * GB_SQ;
    for (int i = tid; i < g.E * g.n; i += 256) {
      const int c = i / g.E, e = i - c * g.E, b = (int)g.fd.div(c), s = c - b * g.d;
      R[i] = X[gb_nat(g, s, e, b)];
    }
    __syncthreads();
  }
  const CholLds<4> L(sm);
  double *U = L.U, *Mi = L.Mi, *piv = L.piv;
  const int nch = (g.E + GB_ROWS - 1) / GB_ROWS, np = nch < w.nsplit ? nch : w.nsplit;
  double a[4][4];
  if (g.wide)
    gb_wide_gram(w, side, a);
  else
    gb_sum_parts(w, side, np, n, a);
  bool bad = false;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) bad = bad || !isfinite(a[i][j]);
  if (__syncthreads_or(bad)) {
    // a NaN or Inf in psi or an environment: carried to Theta, which reports it
    for (int i = tid; !g.wide && i < n * n; i += 256) {
      T[i] = 0.0;
      R0[i] = NAN;
    }
    if (tid == 0) w.info[side].r = n;
    return;
  }
  chol_eliminate<4>(a, n, 0.0, L);
  double pmin = INFINITY, pmax = 0;
  for (int k = 0; k < n; ++k) {
    pmin = fmin(pmin, piv[k]);
    pmax = fmax(pmax, piv[k]);
  }
  if (pmin > 1e-10 * pmax) {
    for (int i = tid; !g.wide && i < n * n; i += 256) {
      const int c = i % n, k = i / n;
      T[i] = c <= k ? Mi[k * GB_LD + c] / sqrt(piv[k]) : 0.0;  // T[c + n k]
      R0[i] = c <= k ? U[c * GB_LD + k] / sqrt(piv[c]) : 0.0;  // R0[c + n k], row c, column k
    }
    if (tid == 0) w.info[side].r = n;
    return;
  }
  __syncthreads();
  if (g.wide)
    gb_wide_gram(w, side, a);
  else
    gb_sum_parts(w, side, np, n, a);
  double* G = U;
  double* V = Mi;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int r = (tid & 15) + 16 * i, c = (tid >> 4) + 16 * j;
      if (r < n && c < n) G[r + n * c] = a[i][j];
    }
  __syncthreads();
  __shared__ double red[4];
  __shared__ int keep_idx[GB_N], s_rank;
  double* lam = piv;
  jacobi_svd(G, n, n, V, nullptr, red);
  for (int j = tid; j < n; j += 256) {  // eigenvalues of the PSD G: the column norms of U diag(l)
    double t = 0;
    for (int i = 0; i < n; ++i) t += G[i + n * j] * G[i + n * j];
    lam[j] = sqrt(t);
  }
  __syncthreads();
  if (tid == 0) {
    double lmax = 0;
    for (int j = 0; j < n; ++j) lmax = lam[j] > lmax ? lam[j] : lmax;
    int r = 0;
    for (int j = 0; j < n; ++j)
      if (lam[j] > g.n * EPS * lmax) keep_idx[r++] = j;
    if (r == 0) keep_idx[r++] = 0;  // X = 0: one zero direction, R = 0
    s_rank = r;
    w.info[side].r = r;
  }
  __syncthreads();
  const int r = s_rank;
  if (g.wide) {  // R = V_r^T X, Q = V_r
    double* Tq = w.Tq + (long long)side * GB_SQ;
    for (int i = tid; i < n * r; i += 256) Tq[i] = V[i % n + n * keep_idx[i / n]];
    gb_wide_rank(w, side, r, V, keep_idx);
    return;
  }
  for (int i = tid; i < n * r; i += 256) {
    const int c = i % n, k = i / n, kk = keep_idx[k];
    const double l = lam[kk];
    T[c + n * k] = l > 0 ? V[c + n * kk] / sqrt(l) : 0.0;
    R0[k + r * c] = sqrt(l) * V[c + n * kk];
  }
}

// The second factorisation: G1 = X1^T X1 = R1^T R1 (a non-positive pivot, a zero
// column of X1, gives a unit diagonal and a zero row), R = R1 R0, Tq = T R1^{-1}.
__global__ __launch_bounds__(256) void k_gb_chol2(GbWork w) {
  extern __shared__ __align__(16) double sm[];
  const int side = blockIdx.x, tid = threadIdx.x;
  const GbSide& g = w.side[side];
  if (g.wide) return;
  const int n = g.n, r = w.info[side].r;
  const CholLds<4> L(sm);
  double *U = L.U, *Mi = L.Mi, *piv = L.piv;
  const int nch = (g.E + GB_ROWS - 1) / GB_ROWS, np = nch < w.nsplit ? nch : w.nsplit;
  double a[4][4];
  gb_sum_parts(w, side, np, r, a);
  chol_eliminate<4>(a, r, 0.0, L);
  // R1 and R1^{-1} in place
  for (int i = tid; i < r * r; i += 256) {
    const int k = i / r, j = i % r;
    const bool ok = piv[k] > 0;
    const double sc = ok ? 1 / sqrt(piv[k]) : 1.0;
    U[k * GB_LD + j] = j < k ? 0.0 : (j == k && !ok ? 1.0 : (ok ? U[k * GB_LD + j] * sc : 0.0));
    Mi[k * GB_LD + j] = j > k ? 0.0 : Mi[k * GB_LD + j] * sc;  // R1^{-1}[j][k]
  }
  __syncthreads();
  const double* T = w.T + (long long)side * GB_SQ;
  const double* R0 = w.R0 + (long long)side * GB_SQ;
  double* R = w.R + (long long)side * GB_SQ;
  double* Tq = w.Tq + (long long)side * GB_SQ;
  for (int i = tid; i < r * n; i += 256) {
    const int k = i % r, c = i / r;
    double t = 0;
    for (int j = k; j < r; ++j) t += U[k * GB_LD + j] * R0[j + r * c];
    R[k + r * c] = t;
  }
  for (int i = tid; i < n * r; i += 256) {
    const int c = i % n, k = i / n;
    double t = 0;
    for (int j = 0; j <= k; ++j) t += T[c + n * j] * Mi[k * GB_LD + j];
    Tq[c + n * k] = t;
  }
}

// ---- Theta ----------------------------------------------------------------------
// Theta[(ru, su'), (rv, sv')] = sum G[(su', sv'), (su, sv)] Ru[ru, su + du b] Rv[rv, sv + dv b],
// stored M x N column-major in the taller orientation; a block of the entries per workgroup
__global__ __launch_bounds__(256) void k_gb_theta(GbWork w, const double* __restrict__ gates) {
  extern __shared__ __align__(16) double sm[];
  const int gt = blockIdx.y, tid = threadIdx.x;
  const GbSide& gu = w.side[2 * gt];
  const GbSide& gv = w.side[2 * gt + 1];
  const int ru = w.info[2 * gt].r, rv = w.info[2 * gt + 1].r;
  const int du = gu.d, dv = gv.d, chib = gu.chib, dd = du * dv;
  const int Mr = ru * du, Nc = rv * dv;
  const bool tr = Mr < Nc;
  double* Ru = sm;
  double* Rv = sm + GB_SQ;
  for (int i = tid; i < ru * gu.n; i += 256) Ru[i] = w.R[(long long)(2 * gt) * GB_SQ + i];
  for (int i = tid; i < rv * gv.n; i += 256) Rv[i] = w.R[(long long)(2 * gt + 1) * GB_SQ + i];
  __syncthreads();
  const double* G = gates + w.gate[gt].gate_off;
  double* Th = w.theta + (long long)gt * AP_TH_BIG * AP_TH_BIG;
  for (int idx = blockIdx.x * 256 + tid; idx < Mr * Nc; idx += gridDim.x * 256) {
    const int row = idx % Mr, col = idx / Mr;
    const int a = row % ru, sup = row / ru, c = col % rv, svp = col / rv;
    double acc = 0;
    for (int su = 0; su < du; ++su)
      for (int sv = 0; sv < dv; ++sv) {
        const double gval = G[(sup + du * svp) + dd * (su + du * sv)];
        if (gval == 0.0) continue;
        double rr = 0;
        for (int b = 0; b < chib; ++b) rr += Ru[a + ru * (su + du * b)] * Rv[c + rv * (sv + dv * b)];
        acc += gval * rr;
      }
    Th[tr ? col + Nc * row : idx] = acc;
  }
}

// ---- SVD ------------------------------------------------------------------------
// Theta of one gate by one workgroup (gate_svd); the kept right singular vectors
// and values go to the workspace
template <int NP>
__global__ __launch_bounds__(8 * NP) void k_gb_svd(GbWork w, ApplyParams prm, double* __restrict__ truncerr,
                                                   double* __restrict__ svals, int* __restrict__ kept,
                                                   int* __restrict__ status) {
  extern __shared__ __align__(16) double sm[];
  const SvdLds<NP> L(sm);
  const int gt = blockIdx.x, tid = threadIdx.x;
  const GbSide& gu = w.side[2 * gt];
  const GbSide& gv = w.side[2 * gt + 1];
  const int Mr = w.info[2 * gt].r * gu.d, Nc = w.info[2 * gt + 1].r * gv.d;
  const int M = Mr < Nc ? Nc : Mr, N = Mr < Nc ? Mr : Nc;
  const double* Th = w.theta + (long long)gt * AP_TH_BIG * AP_TH_BIG;
  const int c = tid >> 3, h = tid & 7;
  double a[NP / 8];
#pragma unroll
  for (int i = 0; i < NP / 8; ++i) {
    const int row = h + 8 * i;
    a[i] = (c < N && row < M) ? Th[row + M * c] : 0.0;
  }
  const int keep = gate_svd<NP>(a, M, N, L, prm, gu.lay, w.gate[gt].slot, truncerr, svals, kept, status);
  if (tid == 0) w.out[gt].keep = keep;
  if (keep < 0) return;
  double* Vg = w.V + (long long)gt * GB_W;
  for (int i = tid; i < N * keep; i += 8 * NP) {
    const int row = i % N, k = i / N, o = L.order[k];
    Vg[L.perm[row] + N * k] = L.X[row + SvdLds<NP>::LD * o];
    if (row == 0) w.sv[gt * AP_KEEP_BIG + k] = L.svec[o];
  }
}

// ---- factors ----------------------------------------------------------------------
// One side of a gate per workgroup: F = V sqrt(S) on the shorter side of Theta,
// Theta V / sqrt(S) = U sqrt(S) on the taller one (rows (r, s'), r fastest); then
// W = Tq F as n x (d keep), column s' + d b' (F is r x (d keep) in the same
// storage).  A wide side: W = F (rank-deficient: V_r F) with M^{-1/2} on its
// external bonds.
__global__ __launch_bounds__(256) void k_gb_factors(GbWork w) {
  extern __shared__ __align__(16) double F[];
  const int side = blockIdx.x, gt = side >> 1, tid = threadIdx.x;
  const int keep = w.out[gt].keep;
  if (keep < 0) return;
  const GbSide& g = w.side[side];
  const int r = w.info[side].r, n = g.n, cols = g.d * keep;
  const int Mr = w.info[2 * gt].r * w.side[2 * gt].d, Nc = w.info[2 * gt + 1].r * w.side[2 * gt + 1].d;
  const bool tr = Mr < Nc;
  const int M = tr ? Nc : Mr, N = tr ? Mr : Nc;
  const double* Th = w.theta + (long long)gt * AP_TH_BIG * AP_TH_BIG;
  const double* V = w.V + (long long)gt * GB_W;
  const double* sv = w.sv + gt * AP_KEEP_BIG;
  const int l = tid & 63, wv = tid >> 6, li = l & 15, lk = l >> 4;
  if ((side & 1) == (tr ? 0 : 1)) {
    for (int i = tid; i < N * keep; i += 256) F[i] = V[i] * sqrt(sv[i / N]);
  } else {
    const int nr = (M + 15) >> 4, ncol = (keep + 15) >> 4;
    for (int t = wv; t < nr * ncol; t += 4) {
      const int row = 16 * (t % nr) + li, col = 16 * (t / nr) + li;
      f64x4 acc = {0, 0, 0, 0};
#pragma unroll 4
      for (int k0 = 0; k0 < N; k0 += 4) {
        const int k = k0 + lk;
        const double a = (row < M && k < N) ? Th[row + M * k] : 0.0;
        const double b = (col < keep && k < N) ? V[k + N * col] : 0.0;
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, acc, 0, 0, 0);
      }
      if (col < keep) {
        const double s = sv[col], sc = s > 0 ? 1 / sqrt(s) : 0.0;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int i = 16 * (t % nr) + 4 * v + lk;
          if (i < M) F[i + M * col] = acc[v] * sc;
        }
      }
    }
  }
  __syncthreads();
  double* W = w.W + (long long)side * GB_W;
  if (!g.wide) {
    const double* Tq = w.Tq + (long long)side * GB_SQ;
    const int nr = (n + 15) >> 4, ncol = (cols + 15) >> 4;
    for (int t = wv; t < nr * ncol; t += 4) {
      const int row = 16 * (t % nr) + li, col = 16 * (t / nr) + li;
      f64x4 acc = {0, 0, 0, 0};
#pragma unroll 4
      for (int k0 = 0; k0 < r; k0 += 4) {
        const int k = k0 + lk;
        const double a = (row < n && k < r) ? Tq[row + n * k] : 0.0;
        const double b = (col < cols && k < r) ? F[k + r * col] : 0.0;
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, acc, 0, 0, 0);
      }
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int i = 16 * (t % nr) + 4 * v + lk;
        if (i < n && col < cols) W[i + n * col] = acc[v];
      }
    }
    return;
  }
  if (r < g.E) {  // Q = V_r
    const double* Tq = w.Tq + (long long)side * GB_SQ;
    for (int i = tid; i < g.E * cols; i += 256) {
      const int e = i % g.E, c = i / g.E;
      double t = 0;
      for (int k = 0; k < r; ++k) t += Tq[e + g.E * k] * F[k + r * c];
      W[i] = t;
    }
    __syncthreads();
    for (int i = tid; i < g.E * cols; i += 256) F[i] = W[i];
    __syncthreads();
  }
  for (int pa = 0; pa < g.next; ++pa) {
    const double* Si = w.roots + ((long long)side * AP_MAXEXT + pa) * 3 * GB_ROOT + GB_ROOT;
    const int chi = g.ext_dim[pa], st = g.ext_est[pa], per = g.E / chi;
    for (int f = tid; f < per * cols; f += 256) {
      const int cc = f / per, q = f - cc * per, hi = q / st;
      double* x = F + g.E * cc + (q - hi * st) + st * chi * hi;
      double in[AP_ENV_BIG];
#pragma unroll
      for (int b = 0; b < AP_ENV_BIG; ++b) in[b] = b < chi ? x[st * b] : 0.0;
      for (int b2 = 0; b2 < chi; ++b2) {
        double t = 0;
#pragma unroll
        for (int b = 0; b < AP_ENV_BIG; ++b)
          if (b < chi) t += in[b] * Si[b2 * chi + b];
        x[st * b2] = t;
      }
    }
    __syncthreads();
  }
  for (int i = tid; i < g.E * cols; i += 256) W[i] = F[i];
}

// ---- rebuild ----------------------------------------------------------------------
// (value, offset) of the larger |value|; ties: the smaller offset
__device__ inline void gb_better(double& v, int& o, double v2, int o2) {
  if (fabs(v2) > fabs(v) || (fabs(v2) == fabs(v) && o2 < o)) {
    v = v2;
    o = o2;
  }
}

// psi'(e, (s', b')) = sum_c psi(e, c) W[c][(s', b')] in place: a workgroup reads
// all columns of its 64 rows (psi, or X where the environment's projector was
// applied), then writes all columns of the layout (zeros past the kept rank),
// through LDS in the site tensor's memory order.  Also, per block: the sum of
// squares and, for the edge's first site, the largest entry of every column.
__global__ __launch_bounds__(256) void k_gb_rebuild(GbWork w, double* psi) {
  extern __shared__ __align__(16) double sm[];
  const int side = blockIdx.y, gt = side >> 1, tid = threadIdx.x;
  const int keep = w.out[gt].keep;
  const GbSide& g = w.side[side];
  if (keep < 0 || (int)blockIdx.x * GB_ROWS >= g.E) return;
  const int l = tid & 63, wv = tid >> 6, li = l & 15, lk = l >> 4;
  const int n = g.n, cols = g.d * keep, mcols = w.mcols, lcols = w.lcols;
  double* tile = sm;
  double* red = tile + GB_N * GB_PITCH;
  double* cv = red + 4;                                    // per wave: largest entry of each column
  int* co = reinterpret_cast<int*>(cv + 4 * lcols);        // and its offset
  double* Wl = reinterpret_cast<double*>(co + 4 * lcols);  // n x cols
  const double* W = w.W + (long long)side * GB_W;
  double* dst = psi + g.psi_off;
  const bool first = (side & 1) == 0;
  double* cmax = w.cmax + ((long long)gt * w.gxr + blockIdx.x) * mcols;
  int* coff = w.coff + ((long long)gt * w.gxr + blockIdx.x) * mcols;
  double nrm2 = 0;
  if (g.wide) {
    for (int cc = tid; cc < g.d * g.lay; cc += 256) {
      const int b = (int)g.fd.div(cc), s = cc - b * g.d;
      double best = 0;
      int boff = 0x7fffffff;
      for (int e = 0; e < g.E; ++e) {
        const double x = cc < cols ? W[e + g.E * cc] : 0.0;
        const int off = gb_nat(g, s, e, b);
        dst[off] = x;
        nrm2 += x * x;
        gb_better(best, boff, x, off);
      }
      if (first && cc < cols) {
        cmax[cc] = best;
        coff[cc] = boff;
      }
    }
  } else {
    for (int i = tid; i < 4 * lcols; i += 256) {
      cv[i] = 0.0;
      co[i] = 0x7fffffff;
    }
    const double* src = dst;
    for (int a = 0; a < g.next; ++a)
      if (w.info[side].trunc[a]) src = w.X + g.x_off;
    for (int i = tid; i < n * cols; i += 256) Wl[i] = W[i];
    const int nt = (n + 15) >> 4, nq = 4 * nt;
    const int bstep = GB_ROWS / g.d;  // bond values of one pass: at most 64 columns
    const int nch = (g.E + GB_ROWS - 1) / GB_ROWS;
    for (int ch = blockIdx.x; ch < nch; ch += gridDim.x) {
      const int e0 = ch * GB_ROWS;
      __syncthreads();
      gb_load_tile(g, src, e0, nt, tile);
      __syncthreads();
      double av[16];
#pragma unroll
      for (int q = 0; q < 16; ++q) av[q] = q < nq ? tile[(4 * q + lk) * GB_PITCH + 16 * wv + li] : 0.0;
      for (int b0 = 0; b0 < g.lay; b0 += bstep) {
        const int bs = g.lay - b0 < bstep ? g.lay - b0 : bstep;
        const int c0 = b0 * g.d, nc = bs * g.d;
        __syncthreads();  // tile read (first pass) or written out
        for (int t = 0; 16 * t < nc; ++t) {
          // the last tile's columns past nc (d = 3, 5, 6, 7) belong to the next pass
          const int cc = c0 + 16 * t + li;
          const bool in = 16 * t + li < nc && cc < cols;
          f64x4 acc = {0, 0, 0, 0};
#pragma unroll
          for (int q = 0; q < 16; ++q)
            if (q < nq) {
              const int c = 4 * q + lk;
              const double b = (c < n && in) ? Wl[c + n * cc] : 0.0;
              acc = __builtin_amdgcn_mfma_f64_16x16x4f64(av[q], b, acc, 0, 0, 0);
            }
          double best = 0;
          int boff = 0x7fffffff;
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            const int r = 16 * wv + 4 * v + lk, e = e0 + r;
            if (16 * t + li < GB_ROWS) tile[(16 * t + li) * GB_PITCH + r] = acc[v];
            nrm2 += acc[v] * acc[v];
            if (first && e < g.E && in) {
              const int b = (int)g.fd.div(cc);
              gb_better(best, boff, acc[v], gb_nat(g, cc - b * g.d, e, b));
            }
          }
          if (first) {
            gb_better(best, boff, __shfl_xor(best, 16), __shfl_xor(boff, 16));
            gb_better(best, boff, __shfl_xor(best, 32), __shfl_xor(boff, 32));
            if (lk == 0 && in) gb_better(cv[wv * lcols + cc], co[wv * lcols + cc], best, boff);
          }
        }
        __syncthreads();
        const int rows = g.E - e0 < GB_ROWS ? g.E - e0 : GB_ROWS;
        if (g.lo >= 16) {
          for (int i = tid; i < nc * GB_ROWS; i += 256) {
            const int t = (int)g.fd.div(i), s = i - t * g.d, r = t & (GB_ROWS - 1), b = t / GB_ROWS;
            if (r < rows) dst[gb_nat(g, s, e0 + r, b0 + b)] = tile[(s + g.d * b) * GB_PITCH + r];
          }
        } else {
          const FastDiv fnc = fast_div((unsigned)nc);
          for (int i = tid; i < nc * rows; i += 256) {
            const int r = (int)fnc.div(i), c = i - r * nc;
            const int b = (int)g.fd.div(c), s = c - b * g.d;
            dst[gb_nat(g, s, e0 + r, b0 + b)] = tile[c * GB_PITCH + r];
          }
        }
      }
    }
  }
  nrm2 = block_sum_d(nrm2, red);
  if (tid == 0) w.normp[(long long)side * w.gxr + blockIdx.x] = nrm2;
  if (first && !g.wide)
    for (int cc = tid; cc < cols; cc += 256) {
      double v = cv[cc];
      int o = co[cc];
      for (int q = 1; q < 4; ++q) gb_better(v, o, cv[q * lcols + cc], co[q * lcols + cc]);
      cmax[cc] = v;
      coff[cc] = o;
    }
}

// the sign of every new-bond slice (the largest entry of the first site's slice
// becomes positive) and the scale of each side
__global__ __launch_bounds__(256) void k_gb_signs(GbWork w, int normalize) {
  const int gt = blockIdx.x, tid = threadIdx.x;
  const int keep = w.out[gt].keep;
  if (keep < 0) return;
  __shared__ double red[4];
  const GbSide& gu = w.side[2 * gt];
  auto blocks = [&](const GbSide& g) {
    const int nch = (g.E + GB_ROWS - 1) / GB_ROWS;
    return g.wide ? 1 : (nch < w.gxr ? nch : w.gxr);
  };
  const int nb = blocks(gu);
  for (int k = tid; k < keep; k += 256) {
    double v = 0;
    int o = 0x7fffffff;
    for (int q = 0; q < nb; ++q)
      for (int s = 0; s < gu.d; ++s) {
        const long long at = ((long long)gt * w.gxr + q) * w.mcols + s + gu.d * k;
        gb_better(v, o, w.cmax[at], w.coff[at]);
      }
    w.sgn[gt * AP_KEEP_BIG + k] = v < 0 ? -1.0 : 1.0;
  }
  for (int sd = 0; sd < 2; ++sd) {
    const int side = 2 * gt + sd, m = blocks(w.side[side]);
    double t = 0;
    for (int q = tid; q < m; q += 256) t += w.normp[(long long)side * w.gxr + q];
    t = block_sum_d(t, red);
    if (tid == 0) w.scale[side] = (normalize && t > 0) ? 1.0 / sqrt(t) : 1.0;
  }
}

__global__ __launch_bounds__(256) void k_gb_scale(GbWork w, double* __restrict__ psi) {
  const int side = blockIdx.y, gt = side >> 1;
  const int keep = w.out[gt].keep;
  if (keep < 0) return;
  const GbSide& g = w.side[side];
  __shared__ double f[AP_KEEP_BIG];
  for (int k = threadIdx.x; k < keep; k += 256) f[k] = w.sgn[gt * AP_KEEP_BIG + k] * w.scale[side];
  __syncthreads();
  double* x = psi + g.psi_off;
  for (int i = blockIdx.x * 256 + threadIdx.x; i < g.D; i += gridDim.x * 256) {
    const int b = (int)g.flay.mod(g.fdlo.div(i));
    if (b < keep) x[i] *= f[b];
  }
}

// ---- host ------------------------------------------------------------------------
// what the workspace's layout depends on
struct GbNeed {
  int gates = 0, mcols = 1, lcols = 1, max_th = 1, max_w = 1;  // max_w: the most entries of a tall side's W
  long long xtot = 0, maxD = 1, maxE = 1;
};
struct GbPlan {
  std::vector<GbSide> side;
  std::vector<GbGate> gate;
  GbNeed need;
  int nsplit, gxr;
  size_t off[20], total;
};

// side sd of a gate; x_off is left to the caller
GbSide gb_side(const itnbp_net* net, const ApplyItem& it, int sd) {
  GbSide g{};
  const VDesc& V = net->vdesc[sd == 0 ? it.u : it.v];
  const int j = sd == 0 ? it.ju : it.jv;
  g.psi_off = V.psi_off;
  g.d = V.dims[0];
  g.chib = it.chib_in;
  g.lay = V.dims[j];
  g.lo = 1;
  g.E = 1;
  int st = g.d;
  for (int a = 1; a <= V.k; ++a) {
    if (a < j) g.lo *= V.dims[a];
    if (a != j) {
      g.ext_dim[g.next] = V.dims[a];
      g.ext_st[g.next] = st;
      g.ext_est[g.next] = g.E;
      g.msg_off[g.next++] = V.in_msg[a];
      g.E *= V.dims[a];
    }
    st *= V.dims[a];
  }
  g.n = g.d * g.chib;
  g.wide = g.E <= g.n;
  g.D = V.D;
  g.fd = fast_div(g.d);
  g.fn = fast_div(g.n);
  g.flo = fast_div(g.lo);
  g.fdlo = fast_div(g.d * g.lo);
  g.flay = fast_div(g.lay);
  return g;
}

void gb_count(const GbSide& g, GbNeed& q) {
  q.xtot += (g.D + 31) & ~31LL;
  q.maxE = std::max<long long>(q.maxE, g.E);
  q.maxD = std::max<long long>(q.maxD, g.D);
  const int cols = g.d * std::min(g.lay, AP_KEEP_BIG);
  q.mcols = std::max(q.mcols, cols);
  if (!g.wide) {  // n d <= 128 (Theta's limit), so n cols <= GB_W
    q.lcols = std::max(q.lcols, cols);
    q.max_w = std::max(q.max_w, g.n * cols);
  }
  q.max_th = std::max(q.max_th, std::min(g.E, g.n) * g.d);
}

void gb_layout(const GbNeed& q, GbPlan& p) {
  p.need = q;
  // row blocks per side: about two workgroups per CU over all sides, at most one
  // per chunk and 48 partial Grams (one workgroup sums them)
  const int nb = q.gates, ns = 2 * nb, nch = (int)((q.maxE + GB_ROWS - 1) / GB_ROWS);
  p.nsplit = std::max(1, std::min({512 / ns + 1, 48, nch}));
  p.gxr = std::max(1, std::min({512 / ns + 1, 128, nch}));
  size_t at = 0;
  int k = 0;
  auto take = [&](size_t bytes) {
    p.off[k++] = at;
    at += (bytes + 255) & ~(size_t)255;
  };
  take(ns * sizeof(GbSide));
  take(nb * sizeof(GbGate));
  take(ns * sizeof(GbInfo));
  take(nb * sizeof(GbOut));
  take((size_t)ns * AP_MAXEXT * 3 * GB_ROOT * 8);
  for (int q4 = 0; q4 < 4; ++q4) take((size_t)ns * GB_SQ * 8);  // T, R0, R, Tq
  take((size_t)ns * GB_W * 8);
  take((size_t)nb * AP_TH_BIG * AP_TH_BIG * 8);
  take((size_t)nb * GB_W * 8);
  take((size_t)nb * AP_KEEP_BIG * 8);
  take((size_t)ns * p.nsplit * GB_SQ * 8);
  take((size_t)ns * p.gxr * 8);
  take((size_t)nb * p.gxr * q.mcols * 8);
  take((size_t)nb * p.gxr * q.mcols * 4);
  take((size_t)nb * AP_KEEP_BIG * 8);
  take((size_t)ns * 8);
  take((size_t)q.xtot * 8);
  p.total = at;
}

}  // namespace

std::vector<int> apply_big_chunks(const itnbp_net* net, const ApplyItem* items, int nb, size_t budget, size_t& bytes) {
  std::vector<int> ends;
  GbNeed have;
  GbPlan p;
  size_t last = 0;
  bytes = 0;
  for (int i = 0; i < nb; ++i) {
    const GbSide u = gb_side(net, items[i], 0), v = gb_side(net, items[i], 1);
    for (;;) {
      GbNeed q = have;
      gb_count(u, q);
      gb_count(v, q);
      ++q.gates;
      gb_layout(q, p);
      if (have.gates > 0 && p.total > budget) {  // a new sequence starts with this gate
        ends.push_back(i);
        bytes = std::max(bytes, last);
        have = GbNeed{};
        continue;
      }
      have = q;
      last = p.total;
      break;
    }
  }
  if (nb > 0) ends.push_back(nb);
  bytes = std::max(bytes, last);
  return ends;
}

int apply_big_run(itnbp_net* net, const ApplyItem* items, int nb, const double* d_gates, const ApplyParams& prm,
                  void* work, double* truncerr, double* svals, int* kept, int* status,
                  std::vector<std::vector<char>>& tables) {
  itnbp_ctx* ctx = net->ctx;
  GbPlan p;
  GbNeed need;
  p.side.reserve(2 * nb);
  p.gate.reserve(nb);
  for (int i = 0; i < nb; ++i) {
    for (int sd = 0; sd < 2; ++sd) {
      GbSide g = gb_side(net, items[i], sd);
      g.x_off = need.xtot;
      gb_count(g, need);
      p.side.push_back(g);
    }
    GbGate gt{};
    gt.gate_off = items[i].gate;
    gt.slot = items[i].slot;
    p.gate.push_back(gt);
    ++need.gates;
  }
  gb_layout(need, p);
  char* base = (char*)work;
  GbWork w;
  w.side = (const GbSide*)(base + p.off[0]);
  w.gate = (const GbGate*)(base + p.off[1]);
  w.info = (GbInfo*)(base + p.off[2]);
  w.out = (GbOut*)(base + p.off[3]);
  w.roots = (double*)(base + p.off[4]);
  w.T = (double*)(base + p.off[5]);
  w.R0 = (double*)(base + p.off[6]);
  w.R = (double*)(base + p.off[7]);
  w.Tq = (double*)(base + p.off[8]);
  w.W = (double*)(base + p.off[9]);
  w.theta = (double*)(base + p.off[10]);
  w.V = (double*)(base + p.off[11]);
  w.sv = (double*)(base + p.off[12]);
  w.part = (double*)(base + p.off[13]);
  w.normp = (double*)(base + p.off[14]);
  w.cmax = (double*)(base + p.off[15]);
  w.coff = (int*)(base + p.off[16]);
  w.sgn = (double*)(base + p.off[17]);
  w.scale = (double*)(base + p.off[18]);
  w.X = (double*)(base + p.off[19]);
  w.nsplit = p.nsplit;
  w.gxr = p.gxr;
  w.mcols = need.mcols;
  w.lcols = need.lcols;
  hipStream_t s = ctx->stream;
  tables.emplace_back(p.off[2]);
  std::vector<char>& up = tables.back();
  std::memcpy(up.data(), p.side.data(), p.side.size() * sizeof(GbSide));
  std::memcpy(up.data() + p.off[1], p.gate.data(), p.gate.size() * sizeof(GbGate));
  ITNBP_HIPCHK(ctx, hipMemcpyAsync(base, up.data(), up.size(), hipMemcpyHostToDevice, s));
  const int ns = 2 * nb;
  double* psi = (double*)net->d_psi;
  const size_t lds_gram = sizeof(double) * GB_N * GB_PITCH;
  const size_t lds_chol = CholLds<4>::bytes();
  const size_t lds_reb = sizeof(double) * (GB_N * GB_PITCH + 4 + 6 * need.lcols + need.max_w);
  const size_t lds_svd = need.max_th <= 32 ? SvdLds<32>::bytes() : need.max_th <= 64 ? SvdLds<64>::bytes() : SvdLds<128>::bytes();
  const struct {
    const void* f;
    size_t lds;
  } attr[] = {{(const void*)k_gb_gram<true>, 2 * lds_gram},
              {(const void*)k_gb_chol1, lds_chol},
              {(const void*)k_gb_chol2, lds_chol},
              {(const void*)k_gb_theta, 2 * GB_SQ * sizeof(double)},
              {(const void*)k_gb_svd<128>, SvdLds<128>::bytes()},
              {(const void*)k_gb_factors, GB_W * sizeof(double)},
              {(const void*)k_gb_rebuild, lds_reb}};
  for (const auto& a : attr)
    ITNBP_HIPCHK(ctx, hipFuncSetAttribute(a.f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)a.lds));
  const int pm0 = prof_mark(ctx);
  hipLaunchKernelGGL(k_gb_roots, dim3(AP_MAXEXT, ns), dim3(256), 0, s, w, (const double*)net->d_msg[net->cur],
                     prm.eig_cutoff);
  const dim3 gmode((unsigned)std::max<long long>(1, std::min<long long>((need.maxD / 16 + 63) / 64, 2048 / ns + 1)), ns);
  for (int pa = 0; pa < AP_MAXEXT; ++pa)
    hipLaunchKernelGGL(k_gb_mode<false>, gmode, dim3(256), 0, s, w, (const double*)psi, pa);
  hipLaunchKernelGGL(k_gb_gram<false>, dim3(p.nsplit, ns), dim3(256), lds_gram, s, w);
  hipLaunchKernelGGL(k_gb_chol1, dim3(ns), dim3(256), lds_chol, s, w);
  hipLaunchKernelGGL(k_gb_gram<true>, dim3(p.nsplit, ns), dim3(256), 2 * lds_gram, s, w);
  hipLaunchKernelGGL(k_gb_chol2, dim3(ns), dim3(256), lds_chol, s, w);
  hipLaunchKernelGGL(k_gb_theta, dim3(16, nb), dim3(256), 2 * GB_SQ * sizeof(double), s, w, d_gates);
  if (need.max_th <= 32)
    hipLaunchKernelGGL(k_gb_svd<32>, dim3(nb), dim3(256), lds_svd, s, w, prm, truncerr, svals, kept, status);
  else if (need.max_th <= 64)
    hipLaunchKernelGGL(k_gb_svd<64>, dim3(nb), dim3(512), lds_svd, s, w, prm, truncerr, svals, kept, status);
  else
    hipLaunchKernelGGL(k_gb_svd<128>, dim3(nb), dim3(1024), lds_svd, s, w, prm, truncerr, svals, kept, status);
  hipLaunchKernelGGL(k_gb_factors, dim3(ns), dim3(256), GB_W * sizeof(double), s, w);
  for (int pa = 0; pa < AP_MAXEXT; ++pa)
    hipLaunchKernelGGL(k_gb_mode<true>, gmode, dim3(256), 0, s, w, (const double*)psi, pa);
  hipLaunchKernelGGL(k_gb_rebuild, dim3(p.gxr, ns), dim3(256), lds_reb, s, w, psi);
  hipLaunchKernelGGL(k_gb_signs, dim3(nb), dim3(256), 0, s, w, prm.normalize);
  hipLaunchKernelGGL(k_gb_scale,
                     dim3((unsigned)std::max<long long>(1, std::min<long long>((need.maxD + 1023) / 1024, 2048 / ns + 1)), ns),
                     dim3(256), 0, s, w, psi);
  ITNBP_HIPCHK(ctx, hipGetLastError());
  prof_add(ctx, "apply_gates_split", pm0, prof_mark(ctx));
  return ITNBP_OK;
}
