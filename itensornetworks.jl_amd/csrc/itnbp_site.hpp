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
  long long mp, mq;      // messages into the site on p and q (mq < 0: none)
  long long out[2];      // messages out on p and q
  long long old[2];      // previous messages out (-1: none to compare with)
  int slot[2];           // statistics slots (-1: none)
  int normalize[2];
  FastDiv fsp;           // stride of bond p
  struct Mode {
    long long msg;
    int n, pad;
    FastDiv fst;         // stride of the bond
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
SiteTask site_task(const VDesc& V, int p, int want);
// ITNBP_DISABLE_VERTEX=1 keeps message updates on the generic kernels
bool site_enabled();
// launches group tasks of similar LDS need: below 2048 elements (256 threads),
// then site tensors of at most 40, 80 and 160 KB (4, 2 and 1 workgroups per CU)
constexpr int SITE_CLASSES = 4;
int site_class(long long D, int elem_bytes);
// threads and dynamic LDS of a launch whose largest task has D elements
int site_threads(long long D);
size_t site_lds_bytes(long long D, int elem_bytes);
// queue != null: a persistent grid of `grid` workgroups takes the n tasks in
// order from the counter at queue (cleared by the launch); active: skip the
// tasks of finished instances
hipError_t launch_site(int psi_dtype, int acc_f64, const SiteTask* d_tasks, int n, const void* psi, const void* msg_in,
                       void* msg_out, MsgStat* stats, int sym, int normalize, int threads, size_t lds, const int* active, int* queue,
                       int grid, hipStream_t s);
// resident workgroups of the persistent form on the current device
hipError_t site_queue_occupancy(int psi_dtype, int acc_f64, int threads, size_t lds, int* per_cu);
