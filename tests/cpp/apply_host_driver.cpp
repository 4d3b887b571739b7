// apply_host_driver GATES FREE_MIB: one call of GATES gates for the split pipeline (every
// other bond of a chain, chi = 10) with FREE_MIB MiB of free device memory, on a runtime
// without a device.  Prints a JSON summary.
#include <chrono>
#include <cstdio>
#include <cstdlib>

#include "fake_hip.hpp"
#include "itnbp.h"

int main(int argc, char** argv) {
  if (argc != 3) return 2;
  const int n = std::atoi(argv[1]), nv = 2 * n + 2, ne = nv - 1;
  fake::free_bytes = (size_t)std::atoi(argv[2]) << 20;
  std::vector<int> edges, ptr{0}, ie, chi(ne, 10), phys(nv, 2), gate_edges;
  for (int i = 0; i < ne; ++i) {
    edges.push_back(i);
    edges.push_back(i + 1);
  }
  for (int v = 0; v < nv; ++v) {
    if (v > 0) ie.push_back(v - 1);
    if (v < ne) ie.push_back(v);
    ptr.push_back((int)ie.size());
  }
  for (int i = 0; i < n; ++i) gate_edges.push_back(2 * i + 1);
  itnbp_ctx* ctx = nullptr;
  itnbp_net* net = nullptr;
  int rc = itnbp_create(0, &ctx);
  if (rc == ITNBP_OK)
    rc = itnbp_net_create(ctx, nv, ne, edges.data(), ptr.data(), ie.data(), chi.data(), phys.data(), ITNBP_F64, &net);
  if (rc == ITNBP_OK) rc = itnbp_init_identity_messages(net);
  std::vector<double> gates(16 * (size_t)n, 0.5), err(n), sv(16 * (size_t)n);
  std::vector<int> kept(n);
  const size_t before = fake::launches.size();
  fake::largest_alloc = 0;
  const auto t0 = std::chrono::steady_clock::now();
  if (rc == ITNBP_OK)
    rc = itnbp_apply_gates(net, n, gate_edges.data(), gates.data(), 10, -1, 1, err.data(), sv.data(), 16, kept.data());
  const double us = std::chrono::duration<double, std::micro>(std::chrono::steady_clock::now() - t0).count();
  std::printf("{\"rc\": %d, \"launches\": %zu, \"us\": %.1f, \"largest_alloc\": %zu, \"changed_copies\": %d}\n", rc,
              fake::launches.size() - before, us, fake::largest_alloc, fake::changed_copies);
  itnbp_net_destroy(net);
  itnbp_destroy(ctx);
  return 0;
}
