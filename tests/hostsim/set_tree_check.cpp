// wx::set_tree against the plain loop that copies the same arrays: prints the
// shortest times of both in microseconds.  TEST SCAFFOLDING.
//   set_tree_check NBLOCKS
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "../../walicxe2d_amd/csrc/wx_runtime.h"

using namespace wx;
using Clock = std::chrono::steady_clock;

int main(int argc, char **argv) {
  const int n = argc > 1 ? atoi(argv[1]) : 10000;
  wx_params p{};
  p.neq = 5; p.nblocks = n; p.nbrootx = n / 16; p.nbrooty = 16; p.nlevs = 1;
  Mesh m;
  m.init(p);
  if (basegrid_tree(&m)) return 3;
  const int nb = m.nbmax;
  std::vector<int32_t> lp((size_t)nb * 8), leaf(nb), ic((size_t)nb * 2);
  int32_t nbmax = 0, nbleafs = 0;
  if (get_tree(&m, lp.data(), leaf.data(), ic.data(), nb, &nbmax, &nbleafs)) return 3;
  std::vector<int32_t> lp2((size_t)(nb + 1) * 8), ic2((size_t)(nb + 1) * 2);
  std::vector<uint8_t> leaf2(nb + 1);
  double best[2] = {1e30, 1e30};
  for (int r = 0; r < 60; ++r) {
    for (int32_t &x : ic) x += 16;   // another tree each time
    const auto t0 = Clock::now();
    bool changed = false;
    if (set_tree(&m, lp.data(), leaf.data(), ic.data(), nb, nb, nbleafs, &changed) || !changed) return 3;
    const auto t1 = Clock::now();
    std::fill(lp2.begin(), lp2.end(), 0);
    std::fill(leaf2.begin(), leaf2.end(), 0);
    std::fill(ic2.begin(), ic2.end(), 0);
    for (int b = 1; b <= nb; ++b) {
      for (int k = 0; k < 8; ++k) lp2[(size_t)b * 8 + k] = lp[(size_t)k * nb + b - 1];
      leaf2[b] = leaf[b - 1] != 0;
      ic2[(size_t)b * 2] = ic[b - 1];
      ic2[(size_t)b * 2 + 1] = ic[(size_t)nb + b - 1];
    }
    const auto t2 = Clock::now();
    best[0] = std::min(best[0], std::chrono::duration<double, std::micro>(t1 - t0).count());
    best[1] = std::min(best[1], std::chrono::duration<double, std::micro>(t2 - t1).count());
    if (lp2 != std::vector<int32_t>(m.lp.begin(), m.lp.begin() + lp2.size()) || ic2[2] != m.icoord[2]) return 4;
  }
  printf("%.2f %.2f\n", best[0], best[1]);
  return 0;
}
