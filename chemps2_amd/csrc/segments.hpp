// Segments of the output blocks of the Heff tiles' second phase (host only).
#pragma once
#include <algorithm>
#include <cstdint>
#include <vector>

namespace chm {

// Doubles of partial sums that chm_heff_apply_noalloc holds (256 MiB), and what of it the
// segments leave to the lower states (at most 1024 partial sums each) and to alignment.
constexpr int64_t NOALLOC_DOUBLES = (int64_t)1 << 25;
constexpr int64_t NOALLOC_RESERVE = (int64_t)4 << 20;

struct SegBlock {
  int64_t work;  // 16-deep chunks of its products, per tile
  int rows, cols;
  bool small() const { return rows <= 32 && cols <= 32; }  // a wavefront's tile
};

// Segments of ws chunks (small blocks) or wl chunks (the others), at least `least`, at most 64 a
// block; returns the partial sums they need.
inline int64_t cut_segments(const std::vector<SegBlock>& blocks, int64_t ws, int64_t wl, int64_t least,
                            std::vector<int>& seg) {
  int64_t part = 0;
  for (size_t b = 0; b < blocks.size(); b++) {
    const SegBlock& k = blocks[b];
    seg[b] = (int)std::max<int64_t>(1, std::min<int64_t>(k.work / std::max(least, k.small() ? ws : wl), 64));
    if (seg[b] > 1) part += (int64_t)seg[b] * k.rows * k.cols;
  }
  return part;
}

// A long list gets enough segments of either kind to fill the device (a wavefront takes one of the
// small blocks': four times as many; 11.3 -> 10.6 ms a product at the L = 32, D = 2000 middle
// site), unless their partial sums, with those of the explicit product and of the chained
// kernels, would not fit chm_heff_apply_noalloc; then, and in a short list, one target over both
// kinds.
inline void choose_segments(const std::vector<SegBlock>& blocks, bool longlist, int64_t target, int64_t least,
                            int64_t explicit_part, int64_t chained_part, std::vector<int>& seg) {
  int64_t wsmall = 0, wlarge = 0;
  for (const SegBlock& k : blocks)
    (k.small() ? wsmall : wlarge) += k.work * ((k.rows + 63) / 64) * ((k.cols + 63) / 64);
  seg.assign(blocks.size(), 1);
  const int64_t room = NOALLOC_DOUBLES - NOALLOC_RESERVE - explicit_part - chained_part;
  if (longlist && cut_segments(blocks, wsmall / (2 * target), wlarge / target, least, seg) <= room) return;
  cut_segments(blocks, (wsmall + wlarge) / target, (wsmall + wlarge) / target, least, seg);
}

}  // namespace chm
