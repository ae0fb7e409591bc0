// Segments of the tiles' output blocks: whatever partial sums the explicit product and the chained
// kernels have, the finer cut of a long list never makes chm_heff_apply_noalloc refuse a site that
// the coarser one fits. Exit code 0: all cases.
#include <cstdio>
#include <random>

#include "../../chemps2_amd/csrc/segments.hpp"

using namespace chm;

static int64_t partials(const std::vector<SegBlock>& b, const std::vector<int>& s) {
  int64_t n = 0;
  for (size_t q = 0; q < b.size(); q++)
    if (s[q] > 1) n += (int64_t)s[q] * b[q].rows * b[q].cols;
  return n;
}

int main() {
  std::mt19937 rng(5);
  int finer = 0, coarser = 0;
  for (int rep = 0; rep < 4000; rep++) {
    std::vector<SegBlock> b(1 + rng() % 3000);
    const int dmax = 1 + rng() % 100;
    for (auto& k : b) k = {(int64_t)(rng() % 200000), 1 + (int)(rng() % dmax), 1 + (int)(rng() % dmax)};
    const int64_t room = NOALLOC_DOUBLES + NOALLOC_RESERVE;
    const int64_t ep = (int64_t)(rng() % 1000) * room / 1000, cp = (int64_t)(rng() % 1000) * (room - ep) / 1000;
    std::vector<int> coarse, seg;
    choose_segments(b, false, 8192, 64, ep, cp, coarse);
    choose_segments(b, true, 8192, 64, ep, cp, seg);
    (seg == coarse ? coarser : finer)++;
    for (int s : seg)
      if (s < 1 || s > 64) return std::printf("%d segments\n", s), 1;
    if (partials(b, coarse) + ep + cp <= NOALLOC_DOUBLES && partials(b, seg) + ep + cp > NOALLOC_DOUBLES)
      return std::printf("case %d: %lld of segments, %lld explicit, %lld chained\n", rep, (long long)partials(b, seg), (long long)ep, (long long)cp), 1;
  }
  return finer > 100 && coarser > 100 ? 0 : (std::printf("%d finer, %d coarser\n", finer, coarser), 1);
}
