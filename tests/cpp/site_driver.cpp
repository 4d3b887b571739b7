// The messages a task of the site kernel reads (site_task): those absorbed on the bonds
// outside the pair, plus, per output, the one into the site on the pair's other bond -
// never the message into the site on the bond whose output is the only one: a
// sequential level updates messages in place and does not order it against that one.
// Prints a JSON summary.
#include <algorithm>
#include <cstdio>
#include <random>
#include <vector>

#include "../../itensornetworks.jl_amd/csrc/itnbp_site.hpp"

int main() {
  std::mt19937 rng(3);
  int failures = 0, cases = 0;
  for (int c = 0; c < 200; ++c) {
    VDesc V{};
    V.k = 1 + (int)(rng() % ITNBP_MAXK);
    V.dims[0] = 1 + (int)(rng() % 3);
    V.D = V.dims[0];
    for (int a = 1; a <= V.k; ++a) {
      V.dims[a] = 1 + (int)(rng() % 4);
      V.D *= V.dims[a];
      V.in_msg[a] = 100 * a;
    }
    for (int p = 1; p <= V.k; ++p)
      for (int want = 1; want <= 3; ++want) {
        const bool pair = p < V.k;
        if (!pair && (want != 1 || V.k > 1)) continue;  // a single bond is alone; the last one comes as q
        const SiteTask t = site_task(V, p, want, 8);
        std::vector<long long> got;
        if (t.mp >= 0) got.push_back(t.mp);
        if (t.mq >= 0) got.push_back(t.mq);
        for (int m = 0; m < t.nmode; ++m) got.push_back(t.mode[m].msg);
        std::vector<long long> need;
        for (int a = 1; a <= V.k; ++a)
          if ((a != p || (want & 2)) && (a != p + 1 || (want & 1))) need.push_back(V.in_msg[a]);
        std::sort(got.begin(), got.end());
        if (got != need) ++failures;
        ++cases;
      }
  }
  std::printf("{\"failures\": %d, \"cases\": %d}\n", failures, cases);
  return 0;
}
