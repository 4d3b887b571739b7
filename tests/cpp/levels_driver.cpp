// Checks itnbp_graph::sequential_levels on random graphs and sequences (with
// repeated messages) against the definition; prints a JSON summary.
#include <cstdio>
#include <random>
#include <vector>

#include "../../itensornetworks.jl_amd/csrc/itnbp_graph.hpp"

using namespace itnbp_graph;

int main() {
  std::mt19937 rng(5);
  int failures = 0, cases = 0, shorter = 0;
  for (int c = 0; c < 300; ++c) {
    const int nv = 2 + (int)(rng() % 14);
    std::vector<int> edges;
    std::vector<std::vector<int>> inc(nv);
    for (int a = 0; a < nv; ++a)
      for (int b = a + 1; b < nv; ++b)
        if ((b == a + 1 || rng() % 4 == 0) && inc[a].size() < 6 && inc[b].size() < 6) {
          const int e = (int)edges.size() / 2;
          edges.push_back(rng() % 2 ? a : b);
          edges.push_back(edges.back() == a ? b : a);
          inc[a].push_back(e);
          inc[b].push_back(e);
        }
    std::vector<int> ptr{0}, ie;
    for (const auto& v : inc) {
      ie.insert(ie.end(), v.begin(), v.end());
      ptr.push_back((int)ie.size());
    }
    const int ne = (int)edges.size() / 2;
    if (ne == 0) continue;
    const Topo t{nv, ne, edges.data(), ptr.data(), ie.data()};
    std::vector<int> seq;
    if (c % 3 == 0)
      default_sequence(t, false, seq);
    else
      for (int i = 0; i < 4 * ne; ++i) seq.push_back((int)(rng() % (2 * ne)));
    const int n = (int)seq.size();
    std::vector<int> order;
    std::vector<std::pair<int, int>> bounds;
    sequential_levels(t, seq, order, bounds);
    auto reads = [&](int r, int m) { return msg_dst(t, m) == msg_src(t, r) && msg_src(t, m) != msg_dst(t, r); };
    auto conflict = [&](int i, int j) {
      return seq[i] == seq[j] || reads(seq[i], seq[j]) || reads(seq[j], seq[i]);
    };
    std::vector<int> level(n, -1);
    int at = 0;
    for (size_t l = 0; l < bounds.size(); ++l) {
      if (bounds[l].first != at || bounds[l].second <= at) ++failures;
      for (int k = bounds[l].first; k < bounds[l].second; ++k) {
        if (order[k] < 0 || order[k] >= n || level[order[k]] >= 0) ++failures;
        else level[order[k]] = (int)l;
      }
      at = bounds[l].second;
    }
    if (at != n) ++failures;
    for (int i = 0; i < n; ++i) {
      int want = 0;  // the longest chain of conflicting earlier positions
      for (int j = 0; j < i; ++j)
        if (conflict(i, j)) want = std::max(want, level[j] + 1);
      if (level[i] != want) ++failures;
    }
    shorter += bounds.size() < sequential_runs(t, seq).size();
    if (bounds.size() > sequential_runs(t, seq).size()) ++failures;
    ++cases;
  }
  std::printf("{\"failures\": %d, \"cases\": %d, \"shorter\": %d}\n", failures, cases, shorter);
  return 0;
}
