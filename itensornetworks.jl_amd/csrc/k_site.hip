// Message updates out of one site, every bond <= 16 and the site tensor in LDS
// (updated_message, src/caches/abstractbeliefpropagationcache.jl:225-239), by
// direct contraction on the matrix cores.  One workgroup runs one SiteTask:
//
//   1. P = psi with the messages of every bond but a neighbouring pair (p, q)
//      absorbed: one mode product per bond, the first from global memory into
//      LDS, the others in place (a wave owns the fibres it reads and writes);
//   2. over the blocks [p][q] of P and psi (one per value of the other indices):
//      T_p += (P M_q) psi^T and T_q += (P^T M_p) psi.  The product with M comes out
//      of the MFMA with its rows in operand order, so it feeds the Gram's MFMA
//      from registers;
//   3. the waves' partial T are summed in a fixed order, (symmetrised,)
//      normalised and compared with the previous message.
//
// A Jacobi sweep runs a site of degree 4 as two tasks, (1,2) and (3,4): four mode
// products and four absorb + Gram steps for all four messages, against twelve
// absorptions and four Grams for independent messages.  The messages need not be
// symmetric.  Sums over a site run in FP64 (the products with M in the
// accumulator type, at most 16 terms each).
//
// The eigenbasis form this replaces (rotate every bond into its message's
// eigenvectors, weighted Grams) needs a Jacobi eigendecomposition per message
// first, a serial chain of some 30 us per workgroup, and ran one workgroup per
// site.  Bound: a fixed chain of about 6 us (launch, task, inputs, stores), then LDS
// and MFMA latency; blocks of bonds <= 8 leave half of each 16 x 16 tile idle in the
// mode products and the absorptions.
// One Jacobi sweep, eigenbasis form -> this: 16x16 PEPS chi = 8 FP64 103 -> 39 us
// (two launches), heavy-hex 9x7 chi 5..16 FP32 189 -> 15 us, 8x8 chi = 4 FP64 40 -> 9
// us.  A level of a sequential sweep of a 9x7 chi 3..8 PEPS takes 13 us.
#include <algorithm>
#include <cstdlib>
#include <vector>

#include "itnbp_site.hpp"

namespace {

typedef double f64x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// 16x16x4 MFMA of the accumulator type: A[i][k] in lane i + 16 k, B[k][j] in lane
// j + 16 k.  Value v of lane l of the result is row 4 v + l / 16 for FP64 and
// 4 (l / 16) + v for FP32; feeding row a_row(i) of A into lane i makes both
// 4 v + l / 16, which is K-step v of a following MFMA.
template <typename T>
struct Mf;
template <>
struct Mf<double> {
  typedef f64x4 V;
  static __device__ inline V mma(double a, double b, V c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }
  static __device__ inline int a_row(int i) { return i; }
};
template <>
struct Mf<float> {
  typedef f32x4 V;
  static __device__ inline V mma(float a, float b, V c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
  static __device__ inline int a_row(int i) { return 4 * (i & 3) + (i >> 2); }
};

__device__ inline double site_wave_sum(double v) {
  for (int m = 32; m > 0; m >>= 1) v += __shfl_xor(v, m);
  return v;
}

// A operand of a product with the message at msg (n x n, column-major):
// A[b'][b] = M[b][b'] for output row b' = a_row(lane) and K-steps b = 4 q + l / 16.
// msg < 0: none, ones (the missing second bond of a site of one; else not used)
template <typename TA, typename TM>
__device__ inline void site_msg(const TM* msg_in, long long msg, int n, TA (&a)[4]) {
  const int l = threadIdx.x & 63, lk = l >> 4, r = Mf<TA>::a_row(l & 15);
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int b = 4 * q + lk;
    a[q] = (b < n && r < n) ? (msg < 0 ? (TA)1 : (TA)msg_in[msg + b + n * r]) : (TA)0;
  }
}

// LDS layout of a site tensor: the stride of bond p padded from sp to sps, so that
// element a sits at a + (sps - sp) (a / sp).  Blocks and fibres along outer bonds
// otherwise step by powers of two of 32 and more elements (chi = 4, 8, 16), which
// puts the lanes of a load on one or two banks (site_task picks the padding).

// P[.. b' ..] = sum_b src[.. b ..] M[b][b'] on one bond (n <= 16), 16 fibres per
// MFMA column set and two sets in flight per wave; src in LDS, or psi itself.
// FULL: no remainder in the bond or the fibres, so no lane is masked.
template <typename TA, bool LDS, bool FULL, typename TSrc>
__device__ inline void site_mode_body(const SiteTask* __restrict__ tk, const SiteTask::Mode& md, const TA (&a)[4],
                                      const TSrc* src, TA* P) {
  const int l = threadIdx.x & 63, li = l & 15, lk = l >> 4, wv = threadIdx.x >> 6, nw = blockDim.x >> 6;
  const int n = md.n, st = (int)md.fst.d, pst = md.pst, nk = (n + 3) >> 2, above = md.above;
  const int nfib = md.nfib, ngrp = (nfib + 15) >> 4, pad = tk->sps - (int)tk->fsp.d;
  int off[4], goff[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int b = 4 * q + lk < n ? 4 * q + lk : 0;
    off[q] = pst * b;
    goff[q] = st * b;
  }
  for (int g0 = wv; g0 < ngrp; g0 += 2 * nw) {
    TA x[2][4];
    int base[2];
    bool in[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int f0 = 16 * (g0 + u * nw) + li;
      in[u] = FULL ? g0 + u * nw < ngrp : f0 < nfib;
      const int f = in[u] ? f0 : 0;
      const int hi = (int)md.fst.div(f), lo = f - hi * st;
      base[u] = above ? lo + pad * (int)tk->fsp.div(lo) + pst * n * hi : lo + st * n * hi + pad * (int)md.fg.div(hi);
      const int gb = lo + st * n * hi;
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (q < nk) {
          const TA t = load_as<TA>(src, LDS ? base[u] + off[q] : gb + goff[q]);
          x[u][q] = FULL || (in[u] && 4 * q + lk < n) ? t : (TA)0;
        }
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      if (FULL && u == 1 && !in[1]) continue;
      typename Mf<TA>::V acc = {0, 0, 0, 0};
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (q < nk) acc = Mf<TA>::mma(a[q], x[u][q], acc);
#pragma unroll
      for (int v = 0; v < 4; ++v)
        if (v < nk && (FULL || (in[u] && 4 * v + lk < n))) P[base[u] + off[v]] = acc[v];
    }
  }
}

template <typename TA, bool LDS, typename TSrc>
__device__ inline void site_mode(const SiteTask* __restrict__ tk, int m, const TA (&a)[4], const TSrc* src, TA* P) {
  const SiteTask::Mode& md = tk->mode[m];
  if (((md.n & 3) | (md.nfib & 15)) == 0)
    site_mode_body<TA, LDS, true>(tk, md, a, src, P);
  else
    site_mode_body<TA, LDS, false>(tk, md, a, src, P);
}

// The blocks of a pair.  Lane column li is index li % 2^lsh of block li / 2^lsh of
// the tile.  FULL: tiles without remainder.  ld(at, gl): psi at LDS position at /
// element gl.
template <bool FULL, typename TA, typename F>
__device__ inline void site_blocks(const SiteTask* __restrict__ tk, const TA* P, const TA (&mp)[4], const TA (&mq)[4],
                                   F ld, f64x4& tp, f64x4& tq) {
  const int l = threadIdx.x & 63, li = l & 15, lk = l >> 4, wv = threadIdx.x >> 6, nw = blockDim.x >> 6;
  const int np = tk->np, nq = tk->nq, want = tk->want, lsh = tk->lsh, nb = tk->nb;
  const int sp = (int)tk->fsp.d, sq = sp * np, sps = tk->sps, sqs = sps * np;
  const int pk = 16 >> lsh, idx = li & ((1 << lsh) - 1), blk = li >> lsh;
  const int npk = (nb + pk - 1) >> (4 - lsh);
  // one output: x = its bond as the lane column, b = the other bond as K-row
  auto output = [&](int base, int gb, bool in, int nx, int nbb, int sx, int sb, int gx, int gbb, const TA(&m)[4],
                    f64x4& acc) {
    const int kb = (nbb + 3) >> 2;
    TA x[4], y[4];
#pragma unroll
    for (int q = 0; q < 4; ++q)
      if (q < kb) {
        const int b = 4 * q + lk;
        const bool ok = FULL || (in && idx < nx && b < nbb);
        const int at = base + (ok ? sx * idx + sb * b : 0);
        x[q] = P[at];
        y[q] = ld(at, gb + (ok ? gx * idx + gbb * b : 0));
        if (!ok) x[q] = y[q] = (TA)0;
      }
    typename Mf<TA>::V d = {0, 0, 0, 0};
#pragma unroll
    for (int q = 0; q < 4; ++q)
      if (q < kb) d = Mf<TA>::mma(m[q], x[q], d);
#pragma unroll
    for (int v = 0; v < 4; ++v)
      if (v < kb) acc = __builtin_amdgcn_mfma_f64_16x16x4f64((double)d[v], (double)y[v], acc, 0, 0, 0);
  };
  for (int t = wv; t < npk; t += nw) {
    const int r0 = t * pk + blk;
    const bool in = FULL || r0 < nb;
    const int r = in ? r0 : 0;
    const int hi = (int)tk->fsp.div(r), lo = r - hi * sp;
    const int base = lo + hi * (sqs * nq), gb = lo + hi * (sq * nq);
    if (want & 1) output(base, gb, in, np, nq, sps, sqs, sp, sq, mq, tp);
    if (want & 2) output(base, gb, in, nq, np, sqs, sps, sq, sp, mp, tq);
  }
}

// STAGE: psi is staged in LDS as well (behind P)
template <bool STAGE, typename TS, typename TA, typename TM>
__device__ __forceinline__ void site_run(const SiteTask* __restrict__ tk, const TS* __restrict__ psi_all,
                                         const TM* msg_in, TM* msg_out, MsgStat* __restrict__ stats, int sym,
                                         int normalize, unsigned char* smem) {
  // the task's cache lines, all at once: its fields are read one by one below,
  // and each first touch of a line would be a round trip of its own
  {
    const int* w = reinterpret_cast<const int*>(tk);
    int touch = 0;
#pragma unroll
    for (int i = 0; i < (int)sizeof(SiteTask) / 4; i += 16) touch += w[i];
    asm volatile("" ::"s"(touch));
  }
  const int tid = threadIdx.x, l = tid & 63, li = l & 15, lk = l >> 4, wv = tid >> 6, nw = blockDim.x >> 6;
  const int D = tk->D, nmode = tk->nmode, want = tk->want;
  const int np = tk->np, nq = tk->nq;
  TA* P = reinterpret_cast<TA*>(smem);
  TA* Y = P + tk->Ds;
  const int sp = (int)tk->fsp.d, pad = tk->sps - sp;
  const TS* psi = psi_all + tk->psi_off;
  // everything the task reads from global memory is asked for at once: psi, the
  // messages in, and (waves 0 and 1) the previous messages out
  TA a[4], mp[4], mq[4];
  if (nmode > 0) site_msg(msg_in, tk->mode[0].msg, tk->mode[0].n, a);
  site_msg(msg_in, tk->mp, np, mp);
  site_msg(msg_in, tk->mq, nq, mq);
  double ov[4] = {0, 0, 0, 0};
  const int fin = wv < 2 && ((want >> wv) & 1);  // this wave finishes output wv
  const long long old = fin ? tk->old[wv] : -1;
  const int no = wv == 0 ? np : nq;
  if (old >= 0)
#pragma unroll
    for (int c = 0; c < 4; ++c)
      if (l + 64 * c < no * no) ov[c] = (double)msg_in[old + l + 64 * c];
  if constexpr (STAGE) {
#pragma unroll 4
    for (int i = tid; i < D; i += blockDim.x) Y[i + pad * (int)tk->fsp.div(i)] = load_as<TA>(psi, i);
    __syncthreads();
  }
  // 1. mode products
  if (nmode == 0) {
    if constexpr (STAGE)
      P = Y;
    else
      for (int i = tid; i < D; i += blockDim.x) P[i + pad * (int)tk->fsp.div(i)] = load_as<TA>(psi, i);
  }
  for (int m = 0; m < nmode; ++m) {
    TA an[4] = {0, 0, 0, 0};
    if (m + 1 < nmode) site_msg(msg_in, tk->mode[m + 1].msg, tk->mode[m + 1].n, an);
    if (m > 0)
      site_mode<TA, true>(tk, m, a, P, P);
    else if constexpr (STAGE)
      site_mode<TA, true>(tk, 0, a, Y, P);
    else
      site_mode<TA, false>(tk, 0, a, psi, P);
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 4; ++q) a[q] = an[q];
  }
  if (!STAGE && nmode == 0) __syncthreads();
  // 2. blocks
  auto ld = [&](int at, int gl) -> TA {
    if constexpr (STAGE)
      return Y[at];
    else
      return load_as<TA>(psi, gl);
  };
  f64x4 tp = {0, 0, 0, 0}, tq = {0, 0, 0, 0};
  const int lsh = tk->lsh, pk = 16 >> lsh;
  if (np == (1 << lsh) && nq == np && np >= 4 && (tk->nb & (pk - 1)) == 0)
    site_blocks<true, TA>(tk, P, mp, mq, ld, tp, tq);
  else
    site_blocks<false, TA>(tk, P, mp, mq, ld, tp, tq);
  __syncthreads();  // P and psi are read; their place takes the partial T
  // 3. red[wave][output][row * 16 + col]
  double* red = reinterpret_cast<double*>(smem);
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    red[(wv * 2 + 0) * 256 + (4 * v + lk) * 16 + li] = tp[v];
    red[(wv * 2 + 1) * 256 + (4 * v + lk) * 16 + li] = tq[v];
  }
  __syncthreads();
  for (int e = tid; e < 512; e += blockDim.x) {
    double s = red[e];
    for (int w = 1; w < nw; ++w) s += red[w * 512 + e];
    red[e] = s;
  }
  __syncthreads();
  if (fin) {
    const int n = no, nn = n * n;
    const double* T = red + wv * 256;
    const long long off = tk->out[wv];
    double tv[4], n2 = 0;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const int e = l + 64 * c;
      tv[c] = 0;
      if (e < nn) {
        const int i = e % n, j = e / n;  // message layout M[i + n j]
        double tij = 0, tji = 0;
        for (int b = 0; b < pk; ++b) {
          const int o = b << lsh;
          tij += T[(o + i) * 16 + o + j];
          tji += T[(o + j) * 16 + o + i];
        }
        tv[c] = sym ? 0.5 * (tij + tji) : tij;
        n2 += tv[c] * tv[c];
      }
    }
    n2 = site_wave_sum(n2);
    const double nrm = sqrt(n2);
    const double sc = (normalize && tk->normalize[wv] && nrm != 0.0) ? 1.0 / nrm : 1.0;
    double dot = 0, o2 = 0, d2 = 0, bad = 0;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const int e = l + 64 * c;
      if (e < nn) {
        const double nv = tv[c] * sc;
        if (!isfinite(nv)) bad = 1;
        if (old >= 0) {
          dot += ov[c] * nv;
          o2 += ov[c] * ov[c];
          d2 += (nv - ov[c]) * (nv - ov[c]);
        }
        msg_out[off + e] = (TM)nv;
      }
    }
    dot = site_wave_sum(dot);
    o2 = site_wave_sum(o2);
    d2 = site_wave_sum(d2);
    bad = site_wave_sum(bad);
    const int slot = tk->slot[wv];
    if (l == 0 && slot >= 0) {
      const double nn2 = n2 * sc * sc;
      MsgStat st;
      st.diff = old >= 0 ? 1.0 - (dot * dot) / (o2 * nn2) : 0.0;
      st.res2 = old >= 0 && nn2 > 0 ? d2 / nn2 : 0.0;
      st.norm = nrm;
      st.bad = (bad > 0 || !isfinite(nrm)) ? 1.0 : 0.0;
      stats[slot] = st;
    }
  }
}

template <bool STAGE, typename TS, typename TA, typename TM>
__global__ __launch_bounds__(STAGE ? 1024 : 512) void k_site(const SiteTask* __restrict__ tasks, const TS* __restrict__ psi,
                                              const TM* msg_in, TM* msg_out, MsgStat* __restrict__ stats, int sym,
                                              int normalize, const int* __restrict__ active) {
  extern __shared__ __align__(16) unsigned char smem[];
  const SiteTask* tk = tasks + blockIdx.x;
  // batched update: a finished instance's messages were carried over already
  if (active && !active[tk->inst]) return;
  site_run<STAGE, TS, TA, TM>(tk, psi, msg_in, msg_out, stats, sym, normalize, smem);
}

// Persistent form: a grid of resident workgroups takes the (cost-sorted) tasks
// in order from a device counter that k_site_reset clears before the launch;
// every workgroup leaves once the counter has passed ntasks, so the grid
// drains without any wait on another workgroup.
template <bool STAGE, typename TS, typename TA, typename TM>
__global__ __launch_bounds__(STAGE ? 1024 : 512) void k_site_queue(const SiteTask* __restrict__ tasks, int ntasks,
                                                    int* __restrict__ queue, const TS* __restrict__ psi,
                                                    const TM* msg_in, TM* msg_out, MsgStat* __restrict__ stats,
                                                    int sym, int normalize, const int* __restrict__ active) {
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ int next;
  for (;;) {
    if (threadIdx.x == 0) next = atomicAdd(queue, 1);
    __syncthreads();
    const int t = next;
    __syncthreads();  // every thread has read next before thread 0 takes the following task
    if (t >= ntasks) return;
    if (!(active && !active[tasks[t].inst])) 
      site_run<STAGE, TS, TA, TM>(tasks + t, psi, msg_in, msg_out, stats, sym, normalize, smem);
    __syncthreads();  // the task's last LDS reads come before the next task's writes
  }
}

// clears the task counter of k_site_queue (a kernel, so that it can sit in a
// captured graph; one lane writes)
__global__ void k_site_reset(int* __restrict__ queue) {
  if (threadIdx.x == 0) queue[0] = 0;
}

template <bool STAGE, typename TS, typename TA, typename TM>
hipError_t launch_impl(const SiteTask* d_tasks, int n, const void* psi, const void* msg_in, void* msg_out,
                       MsgStat* stats, int sym, int normalize, int threads, size_t lds, const int* active, int* queue, int grid,
                       hipStream_t s) {
  if (!queue) {
    auto kern = k_site<STAGE, TS, TA, TM>;
    hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(kern, dim3((unsigned)n), dim3((unsigned)threads), lds, s, d_tasks, (const TS*)psi,
                       (const TM*)msg_in, (TM*)msg_out, stats, sym, normalize, active);
    return hipGetLastError();
  }
  auto kern = k_site_queue<STAGE, TS, TA, TM>;
  hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_site_reset, dim3(1), dim3(64), 0, s, queue);
  hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3((unsigned)threads), lds, s, d_tasks, n, queue, (const TS*)psi,
                     (const TM*)msg_in, (TM*)msg_out, stats, sym, normalize, active);
  return hipGetLastError();
}

template <bool STAGE, typename TS, typename TA, typename TM>
hipError_t occ_impl(int threads, size_t lds, int* per_cu) {
  auto kern = k_site_queue<STAGE, TS, TA, TM>;
  hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (e != hipSuccess) return e;
  return hipOccupancyMaxActiveBlocksPerMultiprocessor(per_cu, (const void*)kern, threads, lds);
}

}  // namespace

bool site_enabled() {
  const char* e = getenv("ITNBP_DISABLE_VERTEX");
  return !(e && e[0] == '1');
}

namespace {
// LDS elements of one padded site tensor, by its elements alone (an upper bound:
// site_task keeps the padding within it)
long long site_pad(long long D) { return D + D / 8 + 32; }
constexpr size_t SITE_LDS = 160 * 1024 - 256;  // less the static LDS of the persistent form
}  // namespace

bool site_stageable(long long D, int elem_bytes) { return (size_t)(2 * site_pad(D) * elem_bytes) <= SITE_LDS; }

int site_class(long long D, int elem_bytes) {
  const size_t b = (size_t)site_pad(D) * elem_bytes;
  return D < 2048 ? 0 : b <= 40 * 1024 ? 1 : b <= 80 * 1024 ? 2 : 3;
}

// Workgroup size by the tensor's elements: below 2048 four waves have their blocks, and
// unstaged tasks want many workgroups per CU; one staged workgroup has its CU to
// itself.  Sweeps of 10x10 (staged) and 24x24 (unstaged) FP64 grids, us:
//   D (chi)      staged 256 / 512 / 1024 threads   unstaged 256 / 512
//   512 (4)       8.6 /  8.2 /  8.5                13.3 / 20.0
//   1250 (5)     15.1 / 11.9 / 12.6                25.5 / 31.0
//   2592 (6)     20.3 / 15.0 / 13.7                43.6 / 46.0
//   4802 (7)     27.2 / 19.1 / 17.2                78.5 / 60.2
//   8192 (8)     29.1 / 20.8 / 18.8                77.7 / 65.2
// The lines suit the unstaged form; staged tasks would gain from 512 threads at 1250 and
// 1024 at 2592 elements.
int site_threads(long long D, bool staged) { return D < 2048 ? 256 : staged && D >= 4096 ? 1024 : 512; }

size_t site_lds_bytes(long long D, int elem_bytes, bool staged) {
  const size_t red = (size_t)(site_threads(D, staged) / 64) * 512 * 8;
  return std::max((size_t)site_pad(D) * elem_bytes * (staged ? 2 : 1), red);
}

bool site_fits(const VDesc& V, int elem_bytes) {
  if (V.k < 1 || V.k > ITNBP_MAXK) return false;
  for (int a = 1; a <= V.k; ++a)
    if (V.dims[a] > SITE_MAXCHI) return false;
  return site_lds_bytes(V.D, elem_bytes, false) <= SITE_LDS;
}

namespace {
// Padding of bond p's LDS stride sp: among paddings that grow the tensor by at
// most an eighth, the smallest with the fewest LDS cycles for the two operand
// loads of a block (lane column (block, index) x 4 K-rows), counted as the most
// lanes on one bank of elem_bytes.
int site_padding(int sp, int np, int nq, int lsh, int elem_bytes) {
  struct Key {
    int sp, np, nq, pad;
  };
  static thread_local std::vector<Key> known[2];
  std::vector<Key>& seen = known[elem_bytes == 8];
  for (const Key& k : seen)
    if (k.sp == sp && k.np == np && k.nq == nq) return k.pad;
  const int banks = 256 / elem_bytes, pk = 16 >> lsh;
  int best = 0, best_cost = 1 << 30;
  for (int pad = 0; pad <= sp / 8 && pad < banks; ++pad) {
    const int s1 = sp + pad, s2 = s1 * np;
    int cost = 0;
    for (int o = 0; o < 2; ++o) {
      int hit[64] = {0}, most = 0;
      const int ni = o == 0 ? np : nq, nk = o == 0 ? nq : np, si = o == 0 ? s1 : s2, sk = o == 0 ? s2 : s1;
      for (int blk = 0; blk < pk; ++blk)
        for (int i = 0; i < ni; ++i)
          for (int b = 0; b < std::min(4, nk); ++b) {
            const int base = blk % sp + blk / sp * s2 * nq;
            most = std::max(most, ++hit[(base + i * si + b * sk) % banks]);
          }
      cost += most;
    }
    if (cost < best_cost) {
      best_cost = cost;
      best = pad;
    }
  }
  if (seen.size() < 512) seen.push_back(Key{sp, np, nq, best});
  return best;
}
}  // namespace

SiteTask site_task(const VDesc& V, int p, int want, int elem_bytes) {
  SiteTask t{};
  t.D = V.D;
  t.psi_off = V.psi_off;
  t.want = want;
  const int q = p < V.k ? p + 1 : 0;
  t.np = V.dims[p];
  t.nq = q ? V.dims[q] : 1;
  t.nb = V.D / (t.np * t.nq);
  int lsh = 0;
  while ((1 << lsh) < std::max(t.np, t.nq)) ++lsh;
  t.lsh = lsh;
  int sp = V.dims[0];
  for (int a = 1; a < p; ++a) sp *= V.dims[a];
  t.fsp = fast_div((unsigned)sp);
  t.sps = sp + site_padding(sp, t.np, t.nq, lsh, elem_bytes);
  t.Ds = V.D / sp * t.sps;
  // only what an output absorbs: another workgroup of the launch may be writing the
  // message into the site on a lone output's own bond
  t.mp = (want & 2) ? V.in_msg[p] : -1;
  t.mq = q && (want & 1) ? V.in_msg[q] : -1;
  t.slot[0] = t.slot[1] = -1;
  t.old[0] = t.old[1] = -1;
  int st = V.dims[0];
  for (int a = 1; a <= V.k; ++a) {
    if (a != p && a != q) {
      SiteTask::Mode& m = t.mode[t.nmode++];
      m.n = V.dims[a];
      m.nfib = V.D / m.n;
      m.fst = fast_div((unsigned)st);
      m.msg = V.in_msg[a];
      m.above = a > p;
      m.pst = m.above ? st / sp * t.sps : st;
      m.fg = fast_div((unsigned)(m.above ? 1 : sp / (st * m.n)));
    }
    st *= V.dims[a];
  }
  return t;
}

hipError_t launch_site(int psi_dtype, int acc_f64, const SiteTask* d_tasks, int n, const void* psi, const void* msg_in,
                       void* msg_out, MsgStat* stats, int sym, int normalize, int threads, size_t lds, bool staged, const int* active,
                       int* queue, int grid, hipStream_t s) {
  if (n <= 0) return hipSuccess;
#define SITE_GO(TS, TA)                                                                                              \
  (staged ? launch_impl<true, TS, TA, TA>(d_tasks, n, psi, msg_in, msg_out, stats, sym, normalize, threads, lds,     \
                                          active, queue, grid, s)                                                    \
          : launch_impl<false, TS, TA, TA>(d_tasks, n, psi, msg_in, msg_out, stats, sym, normalize, threads, lds,    \
                                           active, queue, grid, s))
  if (acc_f64) switch (psi_dtype) {
      case ITNBP_F64: return SITE_GO(double, double);
      case ITNBP_F32: return SITE_GO(float, double);
      default: return SITE_GO(bf16_t, double);
    }
  switch (psi_dtype) {
    case ITNBP_F64: return SITE_GO(double, float);
    case ITNBP_F32: return SITE_GO(float, float);
    default: return SITE_GO(bf16_t, float);
  }
#undef SITE_GO
}

hipError_t site_queue_occupancy(int psi_dtype, int acc_f64, int threads, size_t lds, bool staged, int* per_cu) {
#define SITE_OCC(TS, TA) \
  (staged ? occ_impl<true, TS, TA, TA>(threads, lds, per_cu) : occ_impl<false, TS, TA, TA>(threads, lds, per_cu))
  if (acc_f64) switch (psi_dtype) {
      case ITNBP_F64: return SITE_OCC(double, double);
      case ITNBP_F32: return SITE_OCC(float, double);
      default: return SITE_OCC(bf16_t, double);
    }
  switch (psi_dtype) {
    case ITNBP_F64: return SITE_OCC(double, float);
    case ITNBP_F32: return SITE_OCC(float, float);
    default: return SITE_OCC(bf16_t, float);
  }
#undef SITE_OCC
}

std::vector<SiteLaunch> site_group(std::vector<SiteTask>& tasks, int elem_bytes, int num_cu) {
  std::vector<SiteTask> cls[SITE_CLASSES + 1];  // the staged ones first
  size_t nst = 0;
  for (const SiteTask& t : tasks) nst += site_stageable(t.D, elem_bytes);
  const bool stage = nst <= (size_t)num_cu;
  for (const SiteTask& t : tasks)
    cls[stage && site_stageable(t.D, elem_bytes) ? 0 : 1 + site_class(t.D, elem_bytes)].push_back(t);
  auto cost = [](const SiteTask& t) {
    long long s = (long long)(t.np + t.nq) * (t.want == 3 ? 2 : 1);
    for (int m = 0; m < t.nmode; ++m) s += t.mode[m].n;
    return (long long)t.D * s;
  };
  std::vector<SiteLaunch> out;
  tasks.clear();
  for (int c : {4, 3, 2, 1, 0}) {
    if (cls[c].empty()) continue;
    std::stable_sort(cls[c].begin(), cls[c].end(),
                     [&](const SiteTask& x, const SiteTask& y) { return cost(x) > cost(y); });
    long long dmax = 1;
    for (const SiteTask& t : cls[c]) dmax = std::max<long long>(dmax, t.D);
    const bool st = c == 0;
    out.push_back(SiteLaunch{tasks.size(), cls[c].size(), site_threads(dmax, st), site_lds_bytes(dmax, elem_bytes, st), st});
    tasks.insert(tasks.end(), cls[c].begin(), cls[c].end());
  }
  return out;
}
