// Jacobi sweeps of the sites whose bonds are all <= 16: the sites whose tensor
// fits in LDS as tasks of k_site.hip, two messages per task, and the larger ones
// by the per-vertex eigenbasis kernels below
// (updated_message, src/caches/abstractbeliefpropagationcache.jl:225-239):
//
//   1. every incoming message M_c (symmetric) -> M_c = U_c diag(l_c) U_c^T by a
//      wave-level cyclic Jacobi;
//   2. psi_v rotated into the eigenbasis of every bond, a pair of bonds per pass,
//      in a scratch tensor in global memory;
//   3. per bond c: T'_c[r, r'] = sum over the fibres along c of
//      prod_{e != c} l_e[r_e] Y[.., r, ..] Y[.., r', ..], both bonds of a pair per pass;
//   4. T_c = U_c T'_c U_c^T, symmetrised, normalised, message_diff / residual.
//
// That is d prod(chi) (k chi + k chi) multiply-adds per vertex for all k
// messages, versus k (k - 1) chi d prod(chi) for k independent contractions.  The
// absorbed form is recovered exactly for any orthogonal U_c (eigenvalues of
// either sign), so the result is the reference's update for symmetric messages.
#include <algorithm>
#include <cstdlib>
#include <vector>

#include "itnbp_jacobi.hpp"
#include "itnbp_ops.hpp"

namespace {

typedef double f64x4 __attribute__((ext_vector_type(4)));

constexpr int SV_MAXCHI = 16;
constexpr int SV_LD = SV_MAXCHI + 1;
constexpr int SV_THREADS = 256;

// A site whose tensor does not fit in LDS (physical dimension <= 8 and bonds <= 16,
// so at least three bonds), by pairs of neighbouring bonds (a, b = a + 1): the last pair of an odd number of bonds starts with a bond that the pair
// before has rotated (rot_a = 0).  Entry (r, p, q) of a pair: p and q its two bond
// indices, r = lo + sa hi the others (lo < sa in memory before bond a, hi after b).
// A workgroup takes chunks of L values of lo by H of hi.
struct BigPair {
  int a, na, nb;              // axis of the first bond, dimensions
  int sa, nhi, L, H, ncl, nchunk;
  int rot_a, want_b;          // first bond still to be rotated; second bond's Gram in this pair's pass
  SmallDiv fL, fLr, fab, fa;  // L and the remainder sa % L, na nb, na
};
struct BigSite {
  int v, inst, k, m;          // degree, pairs
  long long psi_off, yoff;    // site tensor, scratch tensor
  long long part;             // partial Grams: 256 per bond and workgroup
  int dims[ITNBP_MAXR];
  long long out[ITNBP_MAXK];  // outgoing message on bond axis a + 1
  int slot[ITNBP_MAXK];
  long long in[ITNBP_MAXK];   // incoming message
  int useed[ITNBP_MAXK];      // its id (eigenvector slot)
  int pair_of[ITNBP_MAXK];    // the pair whose pass computes the bond's Gram
  BigPair pr[(ITNBP_MAXK + 1) / 2];
};

__device__ inline void wave_sync() {
  __builtin_amdgcn_s_waitcnt(0);
  __builtin_amdgcn_wave_barrier();
}

// Symmetric n x n (n <= 16) eigendecomposition in LDS by one wave: A (ld
// SV_LD, entries of order 1) is overwritten by diag(l), V receives the
// eigenvectors as columns.  With init_v = false, V holds an orthogonal seed onto
// which the rotations accumulate.  Lane l takes index l % 16 of a row or column and
// the pairs l / 16 and l / 16 + 4 of a step.
__device__ void wave_jacobi_small(double* A, double* V, int n, double* rc, double* rs, int* rp, int* rq,
                                  bool init_v = true) {
  const int l = threadIdx.x & 63, j = l & 15, g = l >> 4;
  const int ne = n + (n & 1), np = ne / 2;
  if (init_v)
#pragma unroll
    for (int h = 0; h < 4; ++h) {
      const int i = g + 4 * h;
      if (i < n && j < n) V[i * SV_LD + j] = (i == j) ? 1.0 : 0.0;
    }
  wave_sync();
  double prev = INFINITY;
  for (int sweep = 0; sweep < 30; ++sweep) {
    double off = 0, dg = 0;
#pragma unroll
    for (int h = 0; h < 4; ++h) {
      const int i = g + 4 * h;
      const double a = i < n && j < n ? A[i * SV_LD + j] : 0.0;
      if (i != j) off += a * a;
      else dg += a * a;
    }
    for (int m = 32; m > 0; m >>= 1) {
      off += __shfl_xor(off, m);
      dg += __shfl_xor(dg, m);
    }
    // converged (off-diagonal mass at rounding level) or no longer decreasing
    if (off <= 1e-28 * dg || off == 0.0 || off >= prev) break;
    prev = off;
    for (int st = 0; st < ne - 1; ++st) {
      if (l < np) {
        int p, q;
        rr_pair(ne, st, l, p, q);
        double c = 1, s = 0;
        if (q < n) {
          const double apq = A[p * SV_LD + q];
          if (fabs(apq) > 1e-150) jacobi_rotation(A[p * SV_LD + p], A[q * SV_LD + q], apq, c, s);
        }
        rc[l] = c;
        rs[l] = s;
        rp[l] = p;
        rq[l] = q;
      }
      wave_sync();
      int p[2], q[2];
      double c[2], s[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int i = g + 4 * h;
        const bool in = i < np && j < n && rq[i] < n;
        p[h] = in ? rp[i] : -1;
        q[h] = rq[i < np ? i : 0];
        c[h] = rc[i < np ? i : 0];
        s[h] = rs[i < np ? i : 0];
        if (p[h] >= 0) {  // rows: A <- J^T A
          const double ap = A[p[h] * SV_LD + j], aq = A[q[h] * SV_LD + j];
          A[p[h] * SV_LD + j] = c[h] * ap - s[h] * aq;
          A[q[h] * SV_LD + j] = s[h] * ap + c[h] * aq;
        }
      }
      wave_sync();
#pragma unroll
      for (int h = 0; h < 2; ++h)
        if (p[h] >= 0) {  // columns: A <- A J, V <- V J
          const double ap = A[j * SV_LD + p[h]], aq = A[j * SV_LD + q[h]];
          const double vp = V[j * SV_LD + p[h]], vq = V[j * SV_LD + q[h]];
          A[j * SV_LD + p[h]] = c[h] * ap - s[h] * aq;
          A[j * SV_LD + q[h]] = s[h] * ap + c[h] * aq;
          V[j * SV_LD + p[h]] = c[h] * vp - s[h] * vq;
          V[j * SV_LD + q[h]] = s[h] * vp + c[h] * vq;
        }
      wave_sync();
    }
  }
}

constexpr int SEED_LD = SV_MAXCHI;  // row stride of a stored eigenvector seed

// n x n product by one wave into registers: lane l holds elements (l / 16 + 4 h,
// l % 16), C[i][j] = sum_k X(i, k) Y(k, j), X read transposed when tx
__device__ inline void wave_mm(const double* X, bool tx, const double* Y, int n, double (&c)[4]) {
  const int l = threadIdx.x & 63, j = l & 15, g = l >> 4;
#pragma unroll
  for (int h = 0; h < 4; ++h) {
    const int i = g + 4 * h;
    double s = 0.0;
    if (i < n && j < n)
      for (int kk = 0; kk < n; ++kk) s += (tx ? X[kk * SV_LD + i] : X[i * SV_LD + kk]) * Y[kk * SV_LD + j];
    c[h] = s;
  }
}

// Eigendecomposition of the symmetrised message M (n x n, column-major) on one
// bond by one wave: eigenvectors to U (columns, ld SV_LD), eigenvalues to lamv,
// A (ld SV_LD) as work.  With warm, the previous sweep's eigenvectors U0 (in
// seed, ld SEED_LD) start it: Jacobi diagonalises the symmetrised U0^T S U0 and
// its rotations accumulate onto U0; near a BP fixed point that matrix is
// nearly diagonal and takes one or two sweeps instead of a cold start's six to
// ten.  The eigenvectors are stored back to seed for the next sweep.
template <typename TM>
__device__ void bond_eigh(const TM* M, int n, double* A, double* U, double* lamv, double* seed, int warm,
                          double* rc, double* rs, int* rp, int* rq) {
  const int l = threadIdx.x & 63, j = l & 15, g = l >> 4;
  double c[4], mx = 0;
#pragma unroll
  for (int h = 0; h < 4; ++h) {
    const int i = g + 4 * h;
    c[h] = i < n && j < n ? 0.5 * ((double)M[i + n * j] + (double)M[j + n * i]) : 0.0;
    mx = fmax(mx, fabs(c[h]));
  }
  for (int m = 32; m > 0; m >>= 1) mx = fmax(mx, __shfl_xor(mx, m));
  const int ex = mx > 0 && isfinite(mx) ? ilogb(mx) : 0;  // to order 1 for jacobi_rotation
  auto put = [&](double* X) {
#pragma unroll
    for (int h = 0; h < 4; ++h)
      if (g + 4 * h < n && j < n) X[(g + 4 * h) * SV_LD + j] = c[h];
    wave_sync();
  };
#pragma unroll
  for (int h = 0; h < 4; ++h) {
    c[h] = ldexp(c[h], -ex);
    if (warm && g + 4 * h < n && j < n) U[(g + 4 * h) * SV_LD + j] = seed[(g + 4 * h) * SEED_LD + j];
  }
  put(A);
  if (warm) {
    wave_mm(A, false, U, n, c);  // S U0
    wave_sync();
    put(A);
    wave_mm(U, true, A, n, c);  // U0^T (S U0)
    wave_sync();
    put(A);
#pragma unroll
    for (int h = 0; h < 4; ++h) {  // symmetrise
      const int i = g + 4 * h;
      if (i < n && j < n) c[h] = 0.5 * (A[i * SV_LD + j] + A[j * SV_LD + i]);
    }
    wave_sync();
    put(A);
  }
  wave_jacobi_small(A, U, n, rc, rs, rp, rq, !warm);
  if (l < n) lamv[l] = ldexp(A[l * SV_LD + l], ex);
#pragma unroll
  for (int h = 0; h < 4; ++h)
    if (g + 4 * h < n && j < n) seed[(g + 4 * h) * SEED_LD + j] = U[(g + 4 * h) * SV_LD + j];
  wave_sync();
}

__device__ inline double block_sum(double v, double* red) {
  for (int m = 32; m > 0; m >>= 1) v += __shfl_xor(v, m);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  double s = 0;
  for (int i = 0; i < SV_THREADS / 64; ++i) s += red[i];
  return s;
}

// ---- sites too large for LDS -------------------------------------------------------
// Sweep: k_big_eigh (every incoming message), k_big_pass<.., false> per pair of
// bonds (rotation, the last pair's Grams with it), k_big_pass<.., true> for the Grams
// of the other pairs, k_big_final.  A chunk of a pair's entries is staged through LDS
// in the site tensor's memory order; per r the 16 x 16 tile [p][q] is then two
// products on the matrix cores,
//   D1[p][q'] = sum_q X[p][q] U_b[q][q'],   D2[p'][q'] = sum_p U_a[p][p'] D1[p][q'],
// where D1 leaves the MFMA in the operand layout of the second product (value v of
// lane l is row drow(l, v), column l % 16: the contracted row index is the K index).
// The Gram of bond b contracts D2's rows the same way, that of bond a the rows of
// D2^T, the same product with the operands exchanged.  FP32 Grams accumulate 4 r (64
// fibres) in FP32 and are carried in FP64.
//
// Bound: the passes over psi and Y, for two pairs read + write, read + write, read:
// five times the tensor.  A batched FP32 set of about 700 chi = 12 and 16 sites, 241
// MB, per sweep: eigh 37 us, passes 2 x 114 and 63 (4.1 TB/s over them), final 14.
// One workgroup per site through every step (12 passes over Y, their latency
// exposed) took 970 us.
constexpr int BIG_R32 = 32, BIG_R64 = 16;  // r per chunk
constexpr int BIG_ROWS = 32768;            // sites per plane of a pass's grid
constexpr int BIG_Q = 17, BIG_T = 16 * BIG_Q + 1;  // LDS pitch of q, of r

template <typename TA>
struct Mma;
template <>
struct Mma<float> {
  typedef float V __attribute__((ext_vector_type(4)));
  __device__ static V mm(float a, float b, V c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
  __device__ static int drow(int lk, int v) { return 4 * lk + v; }
};
template <>
struct Mma<double> {
  typedef double V __attribute__((ext_vector_type(4)));
  __device__ static V mm(double a, double b, V c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }
  __device__ static int drow(int lk, int v) { return 4 * v + lk; }
};

// pairs, chunks of at most R values of r
void big_pairs(const VDesc& V, int R, BigSite& t) {
  t.k = V.k;
  t.m = (V.k + 1) / 2;
  t.psi_off = V.psi_off;
  for (int a = 0; a <= V.k; ++a) t.dims[a] = V.dims[a];
  for (int i = 0; i < t.m; ++i) {
    BigPair& p = t.pr[i];
    const bool odd = i == t.m - 1 && (V.k & 1);
    p.a = odd ? V.k - 1 : 2 * i + 1;
    p.na = V.dims[p.a];
    p.nb = V.dims[p.a + 1];
    p.rot_a = !odd;
    p.want_b = !(i == t.m - 2 && (V.k & 1));  // else that bond's Gram comes from the last pair
    p.sa = 1;
    for (int a = 0; a < p.a; ++a) p.sa *= V.dims[a];
    p.nhi = V.D / (p.sa * p.na * p.nb);
    p.L = std::min(R, p.sa);
    p.H = p.sa <= R ? std::max(1, std::min(R / p.sa, p.nhi)) : 1;
    p.ncl = (p.sa + p.L - 1) / p.L;
    p.nchunk = p.ncl * ((p.nhi + p.H - 1) / p.H);
    p.fL = small_div(p.L);
    p.fLr = small_div(std::max(1, p.sa % p.L));
    p.fab = small_div(p.na * p.nb);
    p.fa = small_div(p.na);
    t.pair_of[p.a - 1] = i;
    if (p.want_b) t.pair_of[p.a] = i;
  }
}

template <typename TM>
__global__ __launch_bounds__(SV_THREADS) void k_big_eigh(const BigSite* __restrict__ sites, const TM* __restrict__ msg,
                                                         double* __restrict__ seeds, double* __restrict__ lam,
                                                         int warm, const int* __restrict__ active,
                                                         const long long* __restrict__ sweep_ctr) {
  __shared__ double A[4][SV_LD * SV_LD], U[4][SV_LD * SV_LD], rc[32], rs[32];
  __shared__ int rp[32], rq[32];
  const BigSite& t = sites[blockIdx.x];
  // batched update: a finished instance's messages were carried over already
  if (active && !active[t.inst]) return;
  if (sweep_ctr) warm = (*sweep_ctr % 16) != 0;
  const int wv = threadIdx.x >> 6;
  for (int a = wv; a < t.k; a += 4)
    bond_eigh(msg + t.in[a], t.dims[a + 1], A[wv], U[wv], lam + (long long)t.useed[a] * SEED_LD,
              seeds + (long long)t.useed[a] * SEED_LD * SEED_LD, warm, rc + 8 * wv, rs + 8 * wv, rp + 8 * wv,
              rq + 8 * wv);
}

// grid (workgroups per site, rows of sites, planes): a batched set may hold more sites
// than a grid has rows
template <typename TS, typename TA, bool GRAM>
__global__ __launch_bounds__(SV_THREADS) void k_big_pass(const BigSite* __restrict__ sites, int nsites, int pass,
                                                         const TS* __restrict__ psi, TA* __restrict__ scratch,
                                                         const double* __restrict__ seeds,
                                                         const double* __restrict__ lam, double* __restrict__ part,
                                                         const int* __restrict__ active) {
  typedef typename Mma<TA>::V V4;
  constexpr int R = sizeof(TA) == 4 ? BIG_R32 : BIG_R64;
  __shared__ TA slab[R * BIG_T];
  __shared__ TA wr[R];
  __shared__ double ls[ITNBP_MAXK][SV_MAXCHI];
  const int site = blockIdx.y + gridDim.y * blockIdx.z;
  if (site >= nsites) return;
  const BigSite& t = sites[site];
  // a site's last pair gets its Grams with the rotation
  if (pass >= (GRAM ? t.m - 1 : t.m) || (active && !active[t.inst])) return;
  const BigPair& P = t.pr[pass];
  if ((int)blockIdx.x >= P.nchunk) return;
  const bool grams = GRAM || pass == t.m - 1;
  const int tid = threadIdx.x, l = tid & 63, wv = tid >> 6, li = l & 15, lk = l >> 4;
  const int na = P.na, nb = P.nb, nab = na * nb, sa = P.sa;
  const TS* src = psi + t.psi_off;
  TA* Y = scratch + t.yoff;
  for (int i = tid; i < R * BIG_T; i += SV_THREADS) slab[i] = 0;
  for (int i = tid; i < t.k * SV_MAXCHI; i += SV_THREADS) {
    const int a = i / SV_MAXCHI, j = i % SV_MAXCHI;
    ls[a][j] = j < t.dims[a + 1] ? lam[(long long)t.useed[a] * SEED_LD + j] : 0.0;
  }
  // operands: U_b rows 4 v + lk, U_a rows drow, the weights of D2's and D2^T's rows
  TA ub[4], ua[4], wa[4], wb[4];
  {
    const double* Ua = seeds + (long long)t.useed[P.a - 1] * SEED_LD * SEED_LD;
    const double* Ub = seeds + (long long)t.useed[P.a] * SEED_LD * SEED_LD;
    const double* la = lam + (long long)t.useed[P.a - 1] * SEED_LD;
    const double* lb = lam + (long long)t.useed[P.a] * SEED_LD;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int q = 4 * v + lk, r = Mma<TA>::drow(lk, v);
      ub[v] = q < nb && li < nb ? (TA)Ub[q * SEED_LD + li] : (TA)0;
      ua[v] = P.rot_a ? (r < na && li < na ? (TA)Ua[r * SEED_LD + li] : (TA)0) : (TA)(r == li && r < na);
      wa[v] = r < na ? (TA)la[r] : (TA)0;
      wb[v] = r < nb ? (TA)lb[r] : (TA)0;
    }
  }
  V4 acca = {0, 0, 0, 0}, accb = {0, 0, 0, 0};
  double ga[4] = {0, 0, 0, 0}, gb[4] = {0, 0, 0, 0};
  for (int c = blockIdx.x; c < P.nchunk; c += gridDim.x) {
    const int ch = c / P.ncl, cl = c - ch * P.ncl;
    const int lo0 = cl * P.L, nl = min(P.L, sa - lo0), hi0 = ch * P.H, nh = min(P.H, P.nhi - hi0);
    const SmallDiv fl = nl == P.L ? P.fL : P.fLr, fab = P.fab, fa = P.fa;
    const int nr = nl * nh, ne = nr * nab;
    // entry i of the chunk in memory order: lo fastest, then the pair, then hi
    auto locate = [&](int i, int& mem, int& at) {
      const int u = (int)fl.div(i), lo = i - u * nl, hi = (int)fab.div(u), pq = u - hi * nab;
      const int q = (int)fa.div(pq);
      mem = lo0 + lo + sa * (pq + nab * (hi0 + hi));
      at = (lo + nl * hi) * BIG_T + q * BIG_Q + pq - q * na;
    };
    __syncthreads();  // the slab is free
    if (GRAM || pass > 0) {
#pragma unroll 8
      for (int i = tid; i < ne; i += SV_THREADS) {
        int mem, at;
        locate(i, mem, at);
        slab[at] = Y[mem];
      }
    } else {
#pragma unroll 8
      for (int i = tid; i < ne; i += SV_THREADS) {
        int mem, at;
        locate(i, mem, at);
        slab[at] = load_as<TA>(src, mem);
      }
    }
    if (grams && tid < nr) {
      const int h = (int)fl.div(tid);
      int lo = (lo0 + tid - h * nl) / t.dims[0], hi = hi0 + h;
      double w = 1.0;
      for (int a = 1; a < P.a; ++a) {
        w *= ls[a - 1][lo % t.dims[a]];
        lo /= t.dims[a];
      }
      for (int a = P.a + 2; a <= t.k; ++a) {
        w *= ls[a - 1][hi % t.dims[a]];
        hi /= t.dims[a];
      }
      wr[tid] = (TA)w;
    }
    __syncthreads();
    int run = 0;
    for (int r = wv; r < nr; r += 4) {
      TA* x = slab + r * BIG_T;
      const TA w = grams ? wr[r] : (TA)0;
      if constexpr (GRAM) {
        TA xa[4], xb[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int row = Mma<TA>::drow(lk, v);
          xb[v] = x[li * BIG_Q + row];
          xa[v] = x[row * BIG_Q + li];
        }
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          acca = Mma<TA>::mm(xa[v] * (wb[v] * w), xa[v], acca);
          if (P.want_b) accb = Mma<TA>::mm(xb[v] * (wa[v] * w), xb[v], accb);
        }
      } else {
        V4 d1 = {0, 0, 0, 0}, d2 = {0, 0, 0, 0};
        TA xa[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) xa[v] = x[(4 * v + lk) * BIG_Q + li];
#pragma unroll
        for (int v = 0; v < 4; ++v) d1 = Mma<TA>::mm(xa[v], ub[v], d1);
#pragma unroll
        for (int v = 0; v < 4; ++v) d2 = Mma<TA>::mm(ua[v], d1[v], d2);
#pragma unroll
        for (int v = 0; v < 4; ++v) x[li * BIG_Q + Mma<TA>::drow(lk, v)] = d2[v];
        if (grams) {
          V4 dt = {0, 0, 0, 0};
#pragma unroll
          for (int v = 0; v < 4; ++v) dt = Mma<TA>::mm(d1[v], ua[v], dt);
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            acca = Mma<TA>::mm(dt[v] * (wb[v] * w), dt[v], acca);
            accb = Mma<TA>::mm(d2[v] * (wa[v] * w), d2[v], accb);
          }
        }
      }
      if (grams && sizeof(TA) == 4 && ++run == 4) {
        run = 0;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          ga[v] += (double)acca[v];
          gb[v] += (double)accb[v];
          acca[v] = accb[v] = 0;
        }
      }
    }
    // a chunk of fewer r, or what is left of one
    if (grams && sizeof(TA) == 4 && run > 0) {
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        ga[v] += (double)acca[v];
        gb[v] += (double)accb[v];
        acca[v] = accb[v] = 0;
      }
    }
    if constexpr (!GRAM) {
      __syncthreads();
#pragma unroll 8
      for (int i = tid; i < ne; i += SV_THREADS) {
        int mem, at;
        locate(i, mem, at);
        Y[mem] = slab[at];
      }
    }
  }
  if (!grams) return;
  // the four waves' Grams, then one partial per workgroup
  double* sum = reinterpret_cast<double*>(slab);
  static_assert(sizeof(TA) * R * BIG_T >= 4 * 256 * 8, "the wave partials must fit the slab");
  for (int b = 0; b < 2; ++b) {
    if (b == 1 && !P.want_b) continue;
    __syncthreads();
#pragma unroll
    for (int v = 0; v < 4; ++v)
      sum[wv * 256 + 16 * Mma<TA>::drow(lk, v) + li] = b == 0 ? ga[v] + (double)acca[v] : gb[v] + (double)accb[v];
    __syncthreads();
    part[t.part + ((long long)(P.a - 1 + b) * gridDim.x + blockIdx.x) * 256 + tid] =
        (sum[tid] + sum[256 + tid]) + (sum[512 + tid] + sum[768 + tid]);
  }
}

// The Gram of one bond from the partials, back from the eigenbasis, normalised, with
// its statistics.
template <typename TM>
__global__ __launch_bounds__(SV_THREADS) void k_big_final(const BigSite* __restrict__ sites,
                                                          const int* __restrict__ bonds, int nsplit,
                                                          const double* __restrict__ seeds,
                                                          const double* __restrict__ part,
                                                          const TM* __restrict__ msg_in, TM* __restrict__ msg_out,
                                                          MsgStat* __restrict__ stats, int normalize,
                                                          const int* __restrict__ active) {
  __shared__ double U[SV_LD * SV_LD], Tp[SV_LD * SV_LD], X[SV_LD * SV_LD], red[4];
  const int a = bonds[blockIdx.x] % ITNBP_MAXK, tid = threadIdx.x;
  const BigSite& t = sites[bonds[blockIdx.x] / ITNBP_MAXK];
  if (active && !active[t.inst]) return;
  const int n = t.dims[a + 1], nn = n * n;
  {
    const int np = min(nsplit, t.pr[t.pair_of[a]].nchunk);
    const double* p = part + t.part + (long long)a * nsplit * 256 + tid;
    double s = 0;
    for (int q = 0; q < np; ++q) s += p[256 * q];
    Tp[(tid >> 4) * SV_LD + (tid & 15)] = s;
    U[(tid >> 4) * SV_LD + (tid & 15)] = seeds[(long long)t.useed[a] * SEED_LD * SEED_LD + tid];
  }
  __syncthreads();
  if (tid < nn) {
    const int b = tid % n, rr = tid / n;
    double s = 0;
    for (int q = 0; q < n; ++q) s += U[b * SV_LD + q] * Tp[q * SV_LD + rr];
    X[b * SV_LD + rr] = s;  // (U T')[b][r']
  }
  __syncthreads();
  double tval = 0;
  if (tid < nn) {
    const int i = tid % n, j = tid / n;  // message layout M[i + n j]
    double sij = 0, sji = 0;
    for (int q = 0; q < n; ++q) {
      sij += X[i * SV_LD + q] * U[j * SV_LD + q];
      sji += X[j * SV_LD + q] * U[i * SV_LD + q];
    }
    tval = 0.5 * (sij + sji);
  }
  const double n2 = block_sum(tval * tval, red);
  const double nrm = sqrt(n2);
  const double sc = (normalize && nrm != 0.0) ? 1.0 / nrm : 1.0;
  const long long off = t.out[a];
  double dot = 0, o2 = 0, d2 = 0, bad = 0;
  if (tid < nn) {
    const double nv = tval * sc;
    const double ov = (double)msg_in[off + tid];
    if (!isfinite(nv)) bad = 1;
    dot = ov * nv;
    o2 = ov * ov;
    d2 = (nv - ov) * (nv - ov);
    msg_out[off + tid] = (TM)nv;
  }
  dot = block_sum(dot, red);
  o2 = block_sum(o2, red);
  d2 = block_sum(d2, red);
  bad = block_sum(bad, red);
  const int slot = t.slot[a];
  if (tid == 0 && slot >= 0) {
    const double nn2 = n2 * sc * sc;
    MsgStat stt;
    stt.diff = 1.0 - (dot * dot) / (o2 * nn2);
    stt.res2 = nn2 > 0 ? d2 / nn2 : 0.0;
    stt.norm = nrm;
    stt.bad = (bad > 0 || !isfinite(nrm)) ? 1.0 : 0.0;
    stats[slot] = stt;
  }
}

constexpr int QUEUE_STRIDE = 64;

struct SmallState {
  // LDS-resident sites: tasks of k_site.hip in launches of similar LDS need
  std::vector<SiteTask> tasks;
  int nsites = 0;  // sites the tasks cover
  DevBuf d_tasks;
  std::vector<SiteLaunch> launches;
  int queue_grid[SITE_CLASSES + 1] = {0};  // resident workgroups of the persistent form (0: not yet sized)
  // sites too large for LDS, with scratch tensors and the partial Grams of bsplit
  // workgroups per site; bonds: one (site, bond) index per final workgroup
  std::vector<BigSite> big;
  std::vector<int> bonds;
  DevBuf d_big, ybuf, part, lam;
  long long ytotal = 0;  // scratch elements
  int bsplit = 1, bpairs = 0;
  // eigenvector seeds, one SEED_LD x SEED_LD slot per message id; valid after the
  // first sweep since the last prepare, and every 16th sweep starts cold so that
  // rounding in the accumulated rotations cannot build up
  DevBuf seeds;
  long long sweeps = 0;
  // batched update: instance of every vertex (empty: 0), the per-instance
  // active flags the kernels skip finished instances by, and the device sweep
  // counter the warm start is taken from (both null outside the batched update)
  std::vector<int> vinst;
  const int* active = nullptr;
  const long long* sweep_ctr = nullptr;
  // persistent form of the LDS-resident launches: a task counter each
  // (QUEUE_STRIDE ints apart), and the autotuner's choice between it and one
  // workgroup per task (-1: untuned, one per task)
  DevBuf queue;
  int site_queue = -1;
};

// ITNBP_VERTEX_QUEUE=0/1 forces the small-site launch form, else the
// autotuner's choice, else one workgroup per task
bool use_queue(const SmallState* st) {
  if (const char* e = getenv("ITNBP_VERTEX_QUEUE")) return atoi(e) != 0;
  return st->site_queue == 1;
}

SmallState* small_of(itnbp_net* net) { return reinterpret_cast<SmallState*>(net->small); }

// the LDS-resident sites: one workgroup per task, or the persistent queue form
hipError_t launch_small(itnbp_net* net, SmallState* st, int acc_f64, const void* psi, int psi_dtype,
                        const void* msg_in, void* msg_out, MsgStat* stats, int normalize, bool queue,
                        hipStream_t stream) {
  for (size_t i = 0; i < st->launches.size(); ++i) {
    const SiteLaunch& L = st->launches[i];
    int* q = queue && st->queue.p ? (int*)st->queue.p + i * QUEUE_STRIDE : nullptr;
    if (q && st->queue_grid[i] == 0) {
      // every workgroup of the grid resident at once
      int per_cu = 0;
      hipError_t e = site_queue_occupancy(psi_dtype, acc_f64, L.threads, L.lds, L.staged, &per_cu);
      if (e != hipSuccess) return e;
      st->queue_grid[i] = std::max(1, std::min((int)L.count, std::max(1, per_cu) * net->ctx->num_cu));
    }
    hipError_t e = launch_site(psi_dtype, acc_f64, (const SiteTask*)st->d_tasks.p + L.begin, (int)L.count, psi, msg_in,
                               msg_out, stats, 1, normalize, L.threads, L.lds, L.staged, st->active, q, st->queue_grid[i], stream);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

template <typename TS, typename TA, typename TM>
hipError_t launch_big_sites(itnbp_net* net, SmallState* st, const void* psi, const void* msg_in, void* msg_out,
                            MsgStat* stats, int normalize) {
  if (st->big.empty()) return hipSuccess;
  const int warm = (st->sweeps % 16) != 0 ? 1 : 0, ns = (int)st->big.size();
  hipStream_t stream = net->ctx->stream;
  const BigSite* sites = (const BigSite*)st->d_big.p;
  const int* bonds = (const int*)(sites + ns);
  double* seeds = (double*)st->seeds.p;
  double* lam = (double*)st->lam.p;
  double* part = (double*)st->part.p;
  TA* y = (TA*)st->ybuf.p;
  hipLaunchKernelGGL(k_big_eigh<TM>, dim3(ns), dim3(SV_THREADS), 0, stream, sites, (const TM*)msg_in, seeds, lam, warm,
                     st->active, st->sweep_ctr);
  const int rows = std::min(ns, BIG_ROWS);
  const dim3 grid(st->bsplit, rows, (ns + rows - 1) / rows);
  for (int p = 0; p < st->bpairs; ++p)
    hipLaunchKernelGGL((k_big_pass<TS, TA, false>), grid, dim3(SV_THREADS), 0, stream, sites, ns, p, (const TS*)psi,
                       y, (const double*)seeds, (const double*)lam, part, st->active);
  for (int p = 0; p + 1 < st->bpairs; ++p)
    hipLaunchKernelGGL((k_big_pass<TS, TA, true>), grid, dim3(SV_THREADS), 0, stream, sites, ns, p, (const TS*)psi,
                       y, (const double*)seeds, (const double*)lam, part, st->active);
  hipLaunchKernelGGL(k_big_final<TM>, dim3((unsigned)st->bonds.size()), dim3(SV_THREADS), 0, stream, sites, bonds,
                     st->bsplit, (const double*)seeds, (const double*)part, (const TM*)msg_in, (TM*)msg_out, stats,
                     normalize, st->active);
  return hipGetLastError();
}

}  // namespace

bool small_path_enabled(const itnbp_net* net) {
  const char* e = getenv("ITNBP_DISABLE_VERTEX");
  return net->msgs_sym && !(e && e[0] == '1');
}

int small_prepare(itnbp_net* net, const std::vector<int>& seq, int acc_f64, std::vector<char>& handled) {
  itnbp_ctx* ctx = net->ctx;
  SmallState* st = small_of(net);
  if (!st) {
    st = new SmallState();
    net->small = st;
  }
  st->tasks.clear();
  st->big.clear();
  st->bonds.clear();
  st->launches.clear();
  st->nsites = 0;
  st->ytotal = 0;
  st->sweeps = 0;
  if (!small_path_enabled(net)) return ITNBP_OK;
  std::vector<int> pos(2 * net->ne, -1);
  for (size_t i = 0; i < seq.size(); ++i) pos[seq[i]] = (int)i;
  const size_t eb = acc_f64 ? 8 : 4;
  for (int v = 0; v < net->nv; ++v) {
    const VDesc& V = net->vdesc[v];
    if (V.k < 1 || V.k > ITNBP_MAXK) continue;
    bool ok = true;
    for (int a = 1; a <= V.k && ok; ++a) ok = V.dims[a] <= SV_MAXCHI;
    if (!ok) continue;
    const bool fits = site_fits(V, (int)eb);
    BigSite t{};
    t.v = v;
    t.inst = st->vinst.empty() ? 0 : st->vinst[v];
    for (int a = 1; a <= V.k && ok; ++a) {
      const int e = net->inc_edge[net->inc_ptr[v] + a - 1];
      const int w = net->edges[2 * e] == v ? net->edges[2 * e + 1] : net->edges[2 * e];
      const int m = msg_id_into(net, e, w);
      if (pos[m] < 0 || handled[pos[m]]) ok = false;
      else {
        t.out[a - 1] = net->msg_off[m];
        t.slot[a - 1] = pos[m];
        t.useed[a - 1] = msg_id_into(net, e, v);
        t.in[a - 1] = V.in_msg[a];
      }
    }
    if (!ok) continue;
    for (int a = 0; a < V.k; ++a) handled[t.slot[a]] = 1;
    if (fits) {
      // pairs of neighbouring bonds, both messages of a pair from one task; the
      // last of an odd number of bonds as the second of a pair of its own
      ++st->nsites;
      for (int p = 1; p <= V.k; p += 2) {
        const int q = p < V.k ? p : (V.k == 1 ? 1 : p - 1), want = p < V.k ? 3 : (V.k == 1 ? 1 : 2);
        SiteTask s = site_task(V, q, want, (int)eb);
        s.inst = t.inst;
        for (int o = 0; o < 2; ++o)
          if ((want >> o) & 1) {
            s.out[o] = s.old[o] = t.out[q + o - 1];
            s.slot[o] = t.slot[q + o - 1];
            s.normalize[o] = 1;
          }
        st->tasks.push_back(s);
      }
    } else {
      t.yoff = st->ytotal;
      st->ytotal += V.D;
      big_pairs(V, acc_f64 ? BIG_R64 : BIG_R32, t);
      st->big.push_back(t);
    }
  }
  // the largest sites first, so that the short ones fill in behind them
  std::stable_sort(st->big.begin(), st->big.end(),
                   [&](const BigSite& x, const BigSite& y) { return net->vdesc[x.v].D > net->vdesc[y.v].D; });
  // workgroups per site: about 8 per CU over all sites (4 are resident), at most one per chunk
  int most = 1;
  st->bpairs = 0;
  for (const BigSite& b : st->big)
    for (int p = 0; p < b.m; ++p) {
      most = std::max(most, b.pr[p].nchunk);
      st->bpairs = std::max(st->bpairs, b.m);
    }
  st->bsplit = std::min(most, std::max(1, 8 * net->ctx->num_cu / std::max(1, (int)st->big.size())));
  for (size_t i = 0; i < st->big.size(); ++i) {
    st->big[i].part = (long long)st->bonds.size() * st->bsplit * 256;
    for (int a = 0; a < st->big[i].k; ++a) st->bonds.push_back((int)i * ITNBP_MAXK + a);
  }
  st->launches = site_group(st->tasks, (int)eb, net->ctx->num_cu);
  std::fill(st->queue_grid, st->queue_grid + SITE_CLASSES + 1, 0);
  if (!st->big.empty()) {
    const size_t nb = st->big.size() * sizeof(BigSite), nbond = st->bonds.size();
    ITNBP_RETCHK(ensure_buf(ctx, st->seeds, (size_t)std::max(1, 2 * net->ne) * SEED_LD * SEED_LD * 8));
    ITNBP_RETCHK(ensure_buf(ctx, st->lam, (size_t)std::max(1, 2 * net->ne) * SEED_LD * 8));
    ITNBP_RETCHK(ensure_buf(ctx, st->part, nbond * st->bsplit * 256 * 8));
    ITNBP_RETCHK(ensure_buf(ctx, st->d_big, nb + nbond * sizeof(int)));
    ITNBP_RETCHK(ensure_buf(ctx, st->ybuf, (size_t)st->ytotal * eb));
    ITNBP_HIPCHK(ctx, hipMemcpyAsync(st->d_big.p, st->big.data(), nb, hipMemcpyHostToDevice, ctx->stream));
    ITNBP_HIPCHK(ctx, hipMemcpyAsync((char*)st->d_big.p + nb, st->bonds.data(), nbond * sizeof(int),
                                     hipMemcpyHostToDevice, ctx->stream));
    ITNBP_HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
  }
  if (!st->tasks.empty()) {
    ITNBP_RETCHK(ensure_buf(ctx, st->queue, (SITE_CLASSES + 1) * QUEUE_STRIDE * sizeof(int)));
    ITNBP_RETCHK(ensure_buf(ctx, st->d_tasks, st->tasks.size() * sizeof(SiteTask)));
    ITNBP_HIPCHK(ctx, hipMemcpyAsync(st->d_tasks.p, st->tasks.data(), st->tasks.size() * sizeof(SiteTask),
                                     hipMemcpyHostToDevice, ctx->stream));
    ITNBP_HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
  }
  return ITNBP_OK;
}

void small_set_batch(itnbp_net* net, const std::vector<int>& vinst, const int* active, const long long* sweep_ctr) {
  SmallState* st = small_of(net);
  if (!st) {
    st = new SmallState();
    net->small = st;
  }
  st->vinst = vinst;
  st->active = active;
  st->sweep_ctr = sweep_ctr;
}

// Times one launch of the LDS-resident sites in each form (one workgroup per
// task; the persistent queue) on scratch outputs and keeps the faster.
static int autotune_small(itnbp_net* net, SmallState* st, int acc_f64, const void* psi, int psi_dtype,
                          const void* msg_in, int normalize) {
  itnbp_ctx* ctx = net->ctx;
  DevBuf out, stats;
  auto cleanup = [&]() {
    free_buf(out);
    free_buf(stats);
  };
  int rc = ensure_buf(ctx, out, (size_t)net->msg_total * (acc_f64 ? 8 : 4));
  if (rc == ITNBP_OK) rc = ensure_buf(ctx, stats, sizeof(MsgStat) * (size_t)std::max(1, 2 * net->ne));
  if (rc != ITNBP_OK) {
    cleanup();
    return rc;
  }
  float best = INFINITY;
  int best_q = 0;
  for (int rep = 0; rep < 2; ++rep)
    for (int q = 0; q < 2; ++q) {
      hipError_t e = hipEventRecord(ctx->ev0, ctx->stream);
      if (e == hipSuccess)
        e = launch_small(net, st, acc_f64, psi, psi_dtype, msg_in, out.p, (MsgStat*)stats.p, normalize, q == 1,
                         ctx->stream);
      if (e == hipSuccess) e = hipEventRecord(ctx->ev1, ctx->stream);
      if (e == hipSuccess) e = hipEventSynchronize(ctx->ev1);
      float ms = 0;
      if (e == hipSuccess) e = hipEventElapsedTime(&ms, ctx->ev0, ctx->ev1);
      if (e != hipSuccess) {
        cleanup();
        return itnbp_fail(ctx, ITNBP_ERR_HIP, std::string("vertex autotune: ") + hipGetErrorString(e));
      }
      if (rep == 1 && ms < best) {
        best = ms;
        best_q = q;
      }
    }
  cleanup();
  st->site_queue = best_q;
  return ITNBP_OK;
}

int small_autotune(itnbp_net* net, int acc_f64, const void* psi, int psi_dtype, const void* msg_in, int normalize) {
  SmallState* st = small_of(net);
  if (st && !st->tasks.empty() && st->queue.p) {
    const int rc = autotune_small(net, st, acc_f64, psi, psi_dtype, msg_in, normalize);
    if (rc != ITNBP_OK) return rc;
  }
  return ITNBP_OK;
}

bool small_queue_used(itnbp_net* net) {
  SmallState* st = small_of(net);
  return st && !st->tasks.empty() && st->queue.p && use_queue(st);
}

int small_task_count(itnbp_net* net) {
  SmallState* st = small_of(net);
  return st ? st->nsites + (int)st->big.size() : 0;
}

int small_sweep(itnbp_net* net, int acc_f64, const void* psi, int psi_dtype, const void* msg_in, void* msg_out,
                MsgStat* stats, int normalize) {
  itnbp_ctx* ctx = net->ctx;
  SmallState* st = small_of(net);
  if (!st || (st->tasks.empty() && st->big.empty())) return ITNBP_OK;
  const int e0 = prof_mark(ctx);
  hipError_t e = hipSuccess;
  // the big sites (the longest workgroups) first, so that the LDS-resident
  // sites fill in behind them
  if (!st->big.empty()) {
    if (acc_f64) {
      switch (psi_dtype) {
        case ITNBP_F64: e = launch_big_sites<double, double, double>(net, st, psi, msg_in, msg_out, stats, normalize); break;
        case ITNBP_F32: e = launch_big_sites<float, double, double>(net, st, psi, msg_in, msg_out, stats, normalize); break;
        default: e = launch_big_sites<bf16_t, double, double>(net, st, psi, msg_in, msg_out, stats, normalize); break;
      }
    } else {
      switch (psi_dtype) {
        case ITNBP_F64: e = launch_big_sites<double, float, float>(net, st, psi, msg_in, msg_out, stats, normalize); break;
        case ITNBP_F32: e = launch_big_sites<float, float, float>(net, st, psi, msg_in, msg_out, stats, normalize); break;
        default: e = launch_big_sites<bf16_t, float, float>(net, st, psi, msg_in, msg_out, stats, normalize); break;
      }
    }
  }
  if (e == hipSuccess && !st->tasks.empty())
    e = launch_small(net, st, acc_f64, psi, psi_dtype, msg_in, msg_out, stats, normalize, use_queue(st), ctx->stream);
  prof_add(ctx, "vertex_eig", e0, prof_mark(ctx));
  ITNBP_HIPCHK(ctx, e);
  ++st->sweeps;
  return ITNBP_OK;
}

void release_small_state(itnbp_net* net) {
  SmallState* st = small_of(net);
  if (!st) return;
  free_buf(st->d_tasks);
  free_buf(st->queue);
  free_buf(st->d_big);
  free_buf(st->ybuf);
  free_buf(st->part);
  free_buf(st->lam);
  free_buf(st->seeds);
  delete st;
  net->small = nullptr;
}
