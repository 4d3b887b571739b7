// One- and two-site density matrices of a 3x3 grid of chi = 32 through the eigenbasis
// rotations, on a runtime without a device.  Prints a JSON summary.
#include <cstdio>
#include <cstdlib>

#include "fake_hip.hpp"
#include "itnbp.h"

int main() {
  setenv("ITNBP_RDM_FAST_MIN", "1", 1);
  const int L = 3, nv = L * L;
  std::vector<int> edges, ptr{0}, ie;
  std::vector<std::vector<int>> inc(nv);
  auto link = [&](int a, int b) {
    inc[a].push_back((int)edges.size() / 2);
    inc[b].push_back((int)edges.size() / 2);
    edges.push_back(a);
    edges.push_back(b);
  };
  for (int j = 0; j < L; ++j)
    for (int i = 0; i < L; ++i) {
      if (i + 1 < L) link(i + L * j, i + 1 + L * j);
      if (j + 1 < L) link(i + L * j, i + L * (j + 1));
    }
  const int ne = (int)edges.size() / 2;
  std::vector<int> chi(ne, 32), phys(nv, 2), verts(nv), eids(ne);
  for (const auto& v : inc) {
    ie.insert(ie.end(), v.begin(), v.end());
    ptr.push_back((int)ie.size());
  }
  for (int i = 0; i < nv; ++i) verts[i] = i;
  for (int i = 0; i < ne; ++i) eids[i] = i;
  itnbp_ctx* ctx = nullptr;
  itnbp_net* net = nullptr;
  int rc = itnbp_create(0, &ctx);
  if (rc == ITNBP_OK)
    rc = itnbp_net_create(ctx, nv, ne, edges.data(), ptr.data(), ie.data(), chi.data(), phys.data(), ITNBP_F64, &net);
  if (rc == ITNBP_OK) rc = itnbp_init_identity_messages(net);
  std::vector<double> rho(4 * (size_t)nv), pair(16 * (size_t)ne);
  size_t launches = fake::launches.size();
  if (rc == ITNBP_OK) rc = itnbp_rdm1(net, nv, verts.data(), rho.data());
  if (rc == ITNBP_OK) rc = itnbp_rdm2(net, ne, eids.data(), pair.data());
  std::printf("{\"rc\": %d, \"launches\": %zu, \"changed_copies\": %d}\n", rc, fake::launches.size() - launches,
              fake::changed_copies);
  itnbp_net_destroy(net);
  itnbp_destroy(ctx);
  return 0;
}
