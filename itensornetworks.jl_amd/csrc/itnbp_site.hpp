// Message updates out of one site on the matrix cores (k_site.hip): the task
// of one workgroup and its host-side construction.
#pragma once
#include <vector>

#include "itnbp_internal.hpp"

constexpr int SITE_MAXCHI = 16;

// Every bond but two neighbouring ones (p, q = p + 1) is absorbed into psi by a
// mode product; the outgoing messages on p and / or q then come from the
// np x nq blocks that remain.  A site of one bond has q = none (nq = 1).
struct SiteTask {
  int inst;   // batched update: instance of the vertex (0 otherwise)
  int D, nmode, np, nq;
  int nb;     // blocks: D / (np nq)
  int lsh;    // 16 >> lsh blocks share one 16 x 16 tile
  int want;   // bit 0: message on p, bit 1: on q
  long long psi_off;
  long long mp, mq;      // messages into the site on p (for the output on q) and q (< 0: not read)
  long long out[2];      // messages out on p and q
  long long old[2];      // previous messages out (-1: none to compare with)
  int slot[2];           // statistics slots (-1: none)
  int normalize[2];
  FastDiv fsp;           // stride sp of bond p in the site tensor
  int sps, Ds;           // its padded stride in LDS, and the elements of the padded tensor
  struct Mode {
    long long msg;
    int n, nfib, pst;    // dimension, fibres, padded stride
    int above;           // the bond lies above p
    FastDiv fst;         // stride in the site tensor
    FastDiv fg;          // below p: sp / (stride n)
  } mode[ITNBP_MAXK - 1];
};

struct TaskPlan {
  std::vector<OcTask> tasks;
  std::vector<SiteTask> sites;  // site-kernel groups; uploaded behind the tasks
  std::vector<LaunchGroup> groups;
  size_t scratch_bytes = 0, partial_bytes = 0;
  int acc_f64 = 1;
};

// true when the update of vertex v fits: every bond <= 16, the site tensor in LDS
bool site_fits(const VDesc& V, int elem_bytes);
// task of vertex V for the messages on bond axis p and p + 1 (1-based; want as
// above); out, old, slot and normalize are left to the caller
SiteTask site_task(const VDesc& V, int p, int want, int elem_bytes);
// ITNBP_DISABLE_VERTEX=1 keeps message updates on the generic kernels
bool site_enabled();
// Launches of a set of tasks.  While the tasks whose two tensors (P and psi) fit
// in LDS are no more than the CUs, each has a CU to itself: one launch of them,
// with psi staged in LDS (shortest task: no global load after the first).  More
// tasks than that are bound by throughput: psi is read from global memory a second
// time, so that more workgroups share a CU, in launches of similar LDS need (below
// 2048 elements 256 threads; P of at most 40, 80 and 160 KB 512 threads).  A sweep,
// staged / unstaged: FP64 chi = 8 grids of 158 to 260 tasks 18.6 / 27.5 us, 308 20.5 / 27.6,
// 388 35.1 / 36.2, 508 36.9 / 36.9; FP32 chi = 16 heavy-hex lattices of 165 to 340 tasks
// 16.3 / 22.2, 625 26.3 / 28.9; FP64 chi = 4 grids 8.5 / 8.3 at every size.  The line at one
// task per CU is on the safe side: the forms meet between 1.3 and 2.
constexpr int SITE_CLASSES = 4;
struct SiteLaunch {
  size_t begin, count;
  int threads;
  size_t lds;
  bool staged;
};
// reorders the tasks launch by launch, the costliest first
std::vector<SiteLaunch> site_group(std::vector<SiteTask>& tasks, int elem_bytes, int num_cu);
// queue != null: a persistent grid of `grid` workgroups takes the n tasks in
// order from the counter at queue (cleared by the launch); active: skip the
// tasks of finished instances
hipError_t launch_site(int psi_dtype, int acc_f64, const SiteTask* d_tasks, int n, const void* psi, const void* msg_in,
                       void* msg_out, MsgStat* stats, int sym, int normalize, int threads, size_t lds, bool staged, const int* active,
                       int* queue, int grid, hipStream_t s);
// resident workgroups of the persistent form on the current device
hipError_t site_queue_occupancy(int psi_dtype, int acc_f64, int threads, size_t lds, bool staged, int* per_cu);
