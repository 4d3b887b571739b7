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
// site.  Bound: latency of the LDS and MFMA chains; blocks of bonds <= 8 leave half
// of each 16 x 16 tile idle in the mode products and the absorptions.
// One Jacobi sweep, eigenbasis form -> this: 16x16 PEPS chi = 8 FP64 103 -> 42 us,
// heavy-hex 9x7 chi 5..16 FP32 189 -> 31 us, 8x8 chi = 4 FP64 40 -> 9 us (two launches
// where the sites fall into two classes).  A sequential run of a 9x7 chi 3..8 PEPS
// takes 10 us a launch, 21 us on the generic LDS kernel.
#include <algorithm>
#include <cstdlib>

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

// P[.. b' ..] = sum_b src[.. b ..] K[b][b'] on one bond (n <= 16), 16 fibres per
// MFMA column set and two sets in flight per wave
template <typename TA, typename TSrc, typename TM>
__device__ inline void site_mode(const SiteTask::Mode& md, int D, const TSrc* src, TA* P, const TM* msg_in) {
  const int l = threadIdx.x & 63, li = l & 15, lk = l >> 4, wv = threadIdx.x >> 6, nw = blockDim.x >> 6;
  const int n = md.n, st = (int)md.fst.d, nk = (n + 3) >> 2;
  const TM* K = msg_in + md.msg;
  TA a[4];
  const int r = Mf<TA>::a_row(li);
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int b = 4 * q + lk;
    a[q] = (b < n && r < n) ? (TA)K[b + n * r] : (TA)0;
  }
  const int nfib = D / n, ngrp = (nfib + 15) >> 4;
  for (int g0 = wv; g0 < ngrp; g0 += 2 * nw) {
    TA x[2][4];
    int base[2];
    bool in[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int f = 16 * (g0 + u * nw) + li;
      in[u] = f < nfib;
      base[u] = in[u] ? f + (int)md.fst.div(f) * st * (n - 1) : 0;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int b = 4 * q + lk;
        x[u][q] = (q < nk && in[u] && b < n) ? load_as<TA>(src, base[u] + st * b) : (TA)0;
      }
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      typename Mf<TA>::V acc = {0, 0, 0, 0};
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (q < nk) acc = Mf<TA>::mma(a[q], x[u][q], acc);
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int b2 = 4 * v + lk;
        if (v < nk && in[u] && b2 < n) P[base[u] + st * b2] = acc[v];
      }
    }
  }
}

template <typename TS, typename TA, typename TM>
__device__ __forceinline__ void site_run(const SiteTask* __restrict__ tk, const TS* __restrict__ psi_all,
                                         const TM* msg_in, TM* msg_out, MsgStat* __restrict__ stats, int sym,
                                         int normalize, unsigned char* smem) {
  TA* P = reinterpret_cast<TA*>(smem);
  const int tid = threadIdx.x, l = tid & 63, li = l & 15, lk = l >> 4, wv = tid >> 6, nw = blockDim.x >> 6;
  const int D = tk->D;
  const TS* psi = psi_all + tk->psi_off;
  // 1. mode products
  if (tk->nmode == 0)
    for (int i = tid; i < D; i += blockDim.x) P[i] = load_as<TA>(psi, i);
  for (int m = 0; m < tk->nmode; ++m) {
    if (m == 0)
      site_mode<TA>(tk->mode[0], D, psi, P, msg_in);
    else
      site_mode<TA>(tk->mode[m], D, P, P, msg_in);
    if (m + 1 < tk->nmode) __syncthreads();
  }
  // 2. blocks: lane column li is index li % 2^lsh of block li / 2^lsh of the tile
  const int np = tk->np, nq = tk->nq, want = tk->want, lsh = tk->lsh, nb = tk->nb;
  const int sp = (int)tk->fsp.d, sq = sp * np;
  const int pk = 16 >> lsh, idx = li & ((1 << lsh) - 1), blk = li >> lsh;
  const int kp = (np + 3) >> 2, kq = (nq + 3) >> 2;
  TA mq[4], mp[4];
  {
    const int r = Mf<TA>::a_row(li);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int b = 4 * q + lk;
      mq[q] = (b < nq && r < nq) ? (tk->mq < 0 ? (TA)1 : (TA)msg_in[tk->mq + b + nq * r]) : (TA)0;
      mp[q] = (b < np && r < np) ? (TA)msg_in[tk->mp + b + np * r] : (TA)0;
    }
  }
  __syncthreads();
  f64x4 tp = {0, 0, 0, 0}, tq = {0, 0, 0, 0};
  const int npk = (nb + pk - 1) / pk;
  for (int t = wv; t < npk; t += nw) {
    const int r = t * pk + blk;
    const bool in = r < nb;
    const int base = in ? r + (int)tk->fsp.div(r) * sp * (np * nq - 1) : 0;
    if (want & 1) {
      TA x[4], y[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int b = 4 * q + lk;
        const bool ok = q < kq && in && idx < np && b < nq;
        const int at = base + sp * idx + sq * b;
        x[q] = ok ? P[at] : (TA)0;
        y[q] = ok ? load_as<TA>(psi, at) : (TA)0;
      }
      typename Mf<TA>::V d = {0, 0, 0, 0};
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (q < kq) d = Mf<TA>::mma(mq[q], x[q], d);
#pragma unroll
      for (int v = 0; v < 4; ++v)
        if (v < kq) tp = __builtin_amdgcn_mfma_f64_16x16x4f64((double)d[v], (double)y[v], tp, 0, 0, 0);
    }
    if (want & 2) {
      TA x[4], y[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int b = 4 * q + lk;
        const bool ok = q < kp && in && idx < nq && b < np;
        const int at = base + sp * b + sq * idx;
        x[q] = ok ? P[at] : (TA)0;
        y[q] = ok ? load_as<TA>(psi, at) : (TA)0;
      }
      typename Mf<TA>::V d = {0, 0, 0, 0};
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (q < kp) d = Mf<TA>::mma(mp[q], x[q], d);
#pragma unroll
      for (int v = 0; v < 4; ++v)
        if (v < kp) tq = __builtin_amdgcn_mfma_f64_16x16x4f64((double)d[v], (double)y[v], tq, 0, 0, 0);
    }
  }
  __syncthreads();  // P is read; its place takes the partial T
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
  if (wv < 2 && ((want >> wv) & 1)) {
    const int n = wv == 0 ? np : nq, nn = n * n;
    const double* T = red + wv * 256;
    const long long off = tk->out[wv], old = tk->old[wv];
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
          const double ov = (double)msg_in[old + e];
          dot += ov * nv;
          o2 += ov * ov;
          d2 += (nv - ov) * (nv - ov);
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

template <typename TS, typename TA, typename TM>
__global__ __launch_bounds__(512) void k_site(const SiteTask* __restrict__ tasks, const TS* __restrict__ psi,
                                              const TM* msg_in, TM* msg_out, MsgStat* __restrict__ stats, int sym,
                                              int normalize, const int* __restrict__ active) {
  extern __shared__ __align__(16) unsigned char smem[];
  const SiteTask* tk = tasks + blockIdx.x;
  // batched update: a finished instance's messages were carried over already
  if (active && !active[tk->inst]) return;
  site_run<TS, TA, TM>(tk, psi, msg_in, msg_out, stats, sym, normalize, smem);
}

// Persistent form: a grid of resident workgroups takes the (cost-sorted) tasks
// in order from a device counter that k_site_reset clears before the launch;
// every workgroup leaves once the counter has passed ntasks, so the grid
// drains without any wait on another workgroup.
template <typename TS, typename TA, typename TM>
__global__ __launch_bounds__(512) void k_site_queue(const SiteTask* __restrict__ tasks, int ntasks,
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
      site_run<TS, TA, TM>(tasks + t, psi, msg_in, msg_out, stats, sym, normalize, smem);
    __syncthreads();  // the task's last LDS reads come before the next task's writes
  }
}

// clears the task counter of k_site_queue (a kernel, so that it can sit in a
// captured graph; one lane writes)
__global__ void k_site_reset(int* __restrict__ queue) {
  if (threadIdx.x == 0) queue[0] = 0;
}

template <typename TS, typename TA, typename TM>
hipError_t launch_impl(const SiteTask* d_tasks, int n, const void* psi, const void* msg_in, void* msg_out,
                       MsgStat* stats, int sym, int normalize, int threads, size_t lds, const int* active, int* queue, int grid,
                       hipStream_t s) {
  if (!queue) {
    auto kern = k_site<TS, TA, TM>;
    hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(kern, dim3((unsigned)n), dim3((unsigned)threads), lds, s, d_tasks, (const TS*)psi,
                       (const TM*)msg_in, (TM*)msg_out, stats, sym, normalize, active);
    return hipGetLastError();
  }
  auto kern = k_site_queue<TS, TA, TM>;
  hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_site_reset, dim3(1), dim3(64), 0, s, queue);
  hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3((unsigned)threads), lds, s, d_tasks, n, queue, (const TS*)psi,
                     (const TM*)msg_in, (TM*)msg_out, stats, sym, normalize, active);
  return hipGetLastError();
}

template <typename TS, typename TA, typename TM>
hipError_t occ_impl(int threads, size_t lds, int* per_cu) {
  auto kern = k_site_queue<TS, TA, TM>;
  hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (e != hipSuccess) return e;
  return hipOccupancyMaxActiveBlocksPerMultiprocessor(per_cu, (const void*)kern, threads, lds);
}

}  // namespace

bool site_enabled() {
  const char* e = getenv("ITNBP_DISABLE_VERTEX");
  return !(e && e[0] == '1');
}

int site_class(long long D, int elem_bytes) {
  const long long b = D * elem_bytes;
  return D < 2048 ? 0 : b <= 40 * 1024 ? 1 : b <= 80 * 1024 ? 2 : 3;
}

int site_threads(long long D) { return D >= 2048 ? 512 : 256; }

size_t site_lds_bytes(long long D, int elem_bytes) {
  const size_t red = (size_t)(site_threads(D) / 64) * 512 * 8;
  return std::max((size_t)D * elem_bytes, red);
}

bool site_fits(const VDesc& V, int elem_bytes) {
  if (V.k < 1 || V.k > ITNBP_MAXK) return false;
  for (int a = 1; a <= V.k; ++a)
    if (V.dims[a] > SITE_MAXCHI) return false;
  return site_lds_bytes(V.D, elem_bytes) + 256 <= 160 * 1024;  // + the static LDS of the persistent form
}

SiteTask site_task(const VDesc& V, int p, int want) {
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
  t.mp = V.in_msg[p];
  t.mq = q ? V.in_msg[q] : -1;
  t.slot[0] = t.slot[1] = -1;
  t.old[0] = t.old[1] = -1;
  int st = V.dims[0];
  for (int a = 1; a <= V.k; ++a) {
    if (a == p) t.fsp = fast_div((unsigned)st);
    if (a != p && a != q) {
      SiteTask::Mode& m = t.mode[t.nmode++];
      m.n = V.dims[a];
      m.fst = fast_div((unsigned)st);
      m.msg = V.in_msg[a];
    }
    st *= V.dims[a];
  }
  return t;
}

hipError_t launch_site(int psi_dtype, int acc_f64, const SiteTask* d_tasks, int n, const void* psi, const void* msg_in,
                       void* msg_out, MsgStat* stats, int sym, int normalize, int threads, size_t lds, const int* active, int* queue,
                       int grid, hipStream_t s) {
  if (n <= 0) return hipSuccess;
#define SITE_GO(TS, TA) \
  launch_impl<TS, TA, TA>(d_tasks, n, psi, msg_in, msg_out, stats, sym, normalize, threads, lds, active, queue, grid, s)
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

hipError_t site_queue_occupancy(int psi_dtype, int acc_f64, int threads, size_t lds, int* per_cu) {
  if (acc_f64) switch (psi_dtype) {
      case ITNBP_F64: return occ_impl<double, double, double>(threads, lds, per_cu);
      case ITNBP_F32: return occ_impl<float, double, double>(threads, lds, per_cu);
      default: return occ_impl<bf16_t, double, double>(threads, lds, per_cu);
    }
  switch (psi_dtype) {
    case ITNBP_F64: return occ_impl<double, float, float>(threads, lds, per_cu);
    case ITNBP_F32: return occ_impl<float, float, float>(threads, lds, per_cu);
    default: return occ_impl<bf16_t, float, float>(threads, lds, per_cu);
  }
}
