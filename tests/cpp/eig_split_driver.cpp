// eig_split_driver A B: one FP64 sweep of an A x B grid of chi = 32 on a runtime without
// a device: the workgroups of its rot34 launch.  Prints a JSON summary.
#include <cstdio>
#include <cstdlib>
#include <string>

#include "fake_hip.hpp"
#include "itnbp.h"

int main(int argc, char** argv) {
  if (argc != 3) return 2;
  const int A = std::atoi(argv[1]), B = std::atoi(argv[2]), nv = A * B;
  std::vector<int> edges, ptr{0}, ie;
  std::vector<std::vector<int>> inc(nv);
  auto link = [&](int a, int b) {
    inc[a].push_back((int)edges.size() / 2);
    inc[b].push_back((int)edges.size() / 2);
    edges.push_back(a);
    edges.push_back(b);
  };
  for (int j = 0; j < B; ++j)
    for (int i = 0; i < A; ++i) {
      if (i + 1 < A) link(i + A * j, i + 1 + A * j);
      if (j + 1 < B) link(i + A * j, i + A * (j + 1));
    }
  const int ne = (int)edges.size() / 2;
  std::vector<int> chi(ne, 32), phys(nv, 2);
  for (const auto& v : inc) {
    ie.insert(ie.end(), v.begin(), v.end());
    ptr.push_back((int)ie.size());
  }
  itnbp_ctx* ctx = nullptr;
  itnbp_net* net = nullptr;
  int rc = itnbp_create(0, &ctx);
  if (rc == ITNBP_OK)
    rc = itnbp_net_create(ctx, nv, ne, edges.data(), ptr.data(), ie.data(), chi.data(), phys.data(), ITNBP_F64, &net);
  if (rc == ITNBP_OK) rc = itnbp_init_identity_messages(net);
  itnbp_update_opts o = {ITNBP_SCHED_PARALLEL, 1, -1, -1, ITNBP_PREC_F64, 0, 1, 0, nullptr, 0};
  itnbp_update_result r{};
  if (rc == ITNBP_OK) rc = itnbp_update(net, &o, &r);
  unsigned wgs = 0;
  for (const auto& l : fake::launches)
    if (std::string(l.kernel).find("k_rot34_f64ILb1E") != std::string::npos) wgs = l.grid.x;
  std::printf("{\"rc\": %d, \"workgroups\": %u}\n", rc, wgs);
  itnbp_net_destroy(net);
  itnbp_destroy(ctx);
  return 0;
}
