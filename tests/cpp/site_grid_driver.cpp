// One parallel sweep over 65600 sites too large for LDS (a ring with chords, bonds of
// 16, physical dimension 5, FP64) without a device: the launches' grids.  Prints a JSON
// summary.
#include <cstdio>

#include "fake_hip.hpp"
#include "itnbp.h"

int main() {
  const int nv = 65600;
  std::vector<int> edges;
  std::vector<std::vector<int>> inc(nv);
  auto link = [&](int a, int b) {
    inc[a].push_back((int)edges.size() / 2);
    inc[b].push_back((int)edges.size() / 2);
    edges.push_back(a);
    edges.push_back(b);
  };
  for (int i = 0; i < nv; ++i) link(i, (i + 1) % nv);
  for (int i = 0; i < nv / 2; ++i) link(i, i + nv / 2);
  const int ne = (int)edges.size() / 2;
  std::vector<int> ptr{0}, ie, chi(ne, 16), phys(nv, 5);
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
  const size_t before = fake::launches.size();
  itnbp_update_opts o = {ITNBP_SCHED_PARALLEL, 1, -1, -1, ITNBP_PREC_F64, 0, 1, 0, nullptr, 0};
  itnbp_update_result r{};
  if (rc == ITNBP_OK) rc = itnbp_update(net, &o, &r);
  unsigned long long x = 0, y = 0, z = 0;
  for (size_t i = before; i < fake::launches.size(); ++i) {
    x = std::max<unsigned long long>(x, fake::launches[i].grid.x);
    y = std::max<unsigned long long>(y, fake::launches[i].grid.y);
    z = std::max<unsigned long long>(z, fake::launches[i].grid.z);
  }
  std::printf("{\"rc\": %d, \"path\": \"%s\", \"launches\": %zu, \"x\": %llu, \"y\": %llu, \"z\": %llu}\n", rc,
              itnbp_last_path(ctx), fake::launches.size() - before, x, y, z);
  itnbp_net_destroy(net);
  itnbp_destroy(ctx);
  return rc;
}
