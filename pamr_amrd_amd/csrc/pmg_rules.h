// pmg_rules.h -- how a level's sizes become launch shapes.  Plain C++ with no
// HIP in it, so that the host can go through the sizes by itself.
#pragma once
#include <algorithm>
#include <cstddef>

namespace pmg {

// Residual: RTX x RTY columns a block.  z planes a block marches: long marches
// on big levels (HBM reuse), a sixteenth of the planes on small ones (latency:
// a block's planes are processed one after another).
constexpr int RTX = 64, RTY = 8, RZC = 16;
inline int residual_blocks(const int *n, int zchunk) {
  return ((n[0] - 2 + RTX - 1) / RTX) * ((n[1] - 2 + RTY - 1) / RTY) * ((n[2] - 2 + zchunk - 1) / zchunk);
}
// ... and no more blocks than there is room for partial norms: a wide flat grid
// has enough of them with longer marches (1025 x 1025 x 33: 32768 with two
// planes each)
inline int residual_planes(const int *n, int cap) {
  int z = std::max(1, std::min(std::min(RZC, std::max(2, (n[2] - 2 + 15) / 16)), n[2] - 2));
  while (z < RZC && residual_blocks(n, z) > cap) z = std::min(2 * z, RZC);
  return z;
}

// Room for the partial norms of the launches over a finest level of n points:
// its residual in the longest march, and 64 x 8 x 8 points a block.
inline int norm_room(const int *n) {
  const int rblk = ((n[0] + RTX - 1) / RTX) * ((n[1] + RTY - 1) / RTY) * ((n[2] + RZC - 1) / RZC);
  const int sblk = ((n[0] + 61) / 64) * ((n[1] + 5) / 8) * ((n[2] + 5) / 8);
  return std::max(1 << 14, std::max(rblk, sblk) + 64);
}

}  // namespace pmg
