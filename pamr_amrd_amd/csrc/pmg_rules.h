// pmg_rules.h -- how a level's sizes become launch shapes.  Plain C++ with no
// HIP in it, so that the host can go through the sizes by itself.
#pragma once
#include <algorithm>
#include <cstddef>

namespace pmg {

// Rows of at most this many points: byte offsets within a tile of up to 36 rows
// of doubles fit 32 bits.  Longer ones take kernels with 64-bit offsets, on the
// narrowest tiles (no one has them in earnest; they run, that is all).
constexpr int kLongRow = 1 << 23;

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

// Fused finest residual + injection (streamed): kRrCX x kRrCY coarse columns a
// block ([0] FP64, [1] FP32), columns 0 .. cn-2 -- the last ones lie on a face.
constexpr int kRrCX[2] = {16, 32}, kRrCY = 8;
constexpr int rr_tiles(int cn, int c) { return cn > 1 ? (cn - 1 + c - 1) / c : 1; }
inline int rr_blocks(const int *cn, int pi, int cz) {
  return rr_tiles(cn[0], kRrCX[pi]) * rr_tiles(cn[1], kRrCY) * ((cn[2] + cz - 1) / cz);
}
// Coarse planes a block marches: 6 (FP64) and 4 (FP32) on a coarse level of 129
// planes, 8 from 257 planes on, the fastest measured.  On smaller grids a block's
// march is the time: halved while it makes fewer than 1000 blocks, down to two
// planes, and to one where those make fewer than 500.  FP64, us with 6, 3, 2 and
// 1 (blocks with 2): 161 x 97 x 129 fine points 47 with 8, 18 with 2 (990);
// 81 x 49 x 257 24.8, 17.9, 16.5, 18.2 (585); 65 x 65 x 257 19.8, 14.6, 12.8, 15.5
// (520); 97^3 25.1, 17.8, 14.5, 14.0 (450); 33 x 65 x 257 19.7, 12.1, 11.4, 9.9
// (260).  FP32, with 4, 2 and 1: 65 x 65 x 257 17.9, 12.8, 11.2 (260).
inline int resid_restrict_planes(const int *cn, int pi) {
  if (cn[2] >= 257) return 8;
  int cz = cn[2] < 129 ? 8 : pi ? 4 : 6;
  while (cz > 2 && rr_blocks(cn, pi, cz) < 1000) cz = std::max(2, cz / 2);
  return cz == 2 && rr_blocks(cn, pi, cz) < 500 ? 1 : cz;
}

// Tile variant and z chunk of a level that was never tuned, from what the
// tuned sizes show.  From 200^3 points on, where memory is the bound: 128 x 16
// columns, 64 x 16 where 128 would leave more than a sixth of the tile outside;
// with the variable coefficient, whose LDS ring doubles the block's LDS, 64 x 16
// in FP64 (257^3: 170 us, 32 x 16 181, 128 x 16 without the ring 211) and the
// five-plane 128 x 8 in FP32 (92 us, 128 x 16 103).  The longest march that
// leaves a block a CU; in FP32, where a CU holds two of them, at most 16 planes
// (32 with the coefficient): neighbours drift apart on a long march and no
// longer find each other's rows in the L2 (513^3: 453 us with 16 planes, 484
// with 32, 503 with 64).  Below 200^3: 32 x 16 columns, the longest march of 64
// .. 2 planes that makes 400 workgroups -- fewer leave CUs without work, shorter
// marches repeat the prologue (129^3: 14.9 us at 8 planes and 512 workgroups;
// 65^3: 6.6 us at 2 planes, 7.6 at 4).  Not the best of a full search where a
// side is no 2^m + 1 (back to back): 225^3 FP64 81 us against 73 on 32 x 16 x 32,
// FP32 58 against 47 on 64 x 32 x 16, FP64 with the coefficient 186 against 140 on 32
// x 16 x 16; 321 x 257 x 257 FP64 132 against 118 on 64 x 16 x 16; nor at 257^3 FP64,
// 80 against 75 on the five-plane 128 x 8 x 64, which the tuned table has.
inline void default_sweep(const int *n, int op, int pi, int *variant, int *zchunk) {
  const size_t size = (size_t)n[0] * n[1] * n[2];
  int tx = 32, ty = 16, want = 400, z = 64;
  *variant = 2;
  if (size >= 8000000) {
    const int w = n[0] - 2, w128 = (w + 127) / 128 * 128;
    const bool ring64 = op == 1 && pi == 0;
    tx = ring64 || 6 * (w128 - w) > w128 ? 64 : 128;
    *variant = tx == 64 ? 1 : (op == 1 ? 11 : 5);
    if (*variant == 11) ty = 8;
    want = tx == 64 && !ring64 ? 400 : 256;
    if (pi == 1) z = op == 1 ? 32 : 16;
  }
  auto columns = [&] { return ((n[0] - 2 + tx - 1) / tx) * ((n[1] - 2 + ty - 1) / ty); };
  if (columns() > 1 << 14) {  // a thin grid: narrow columns alone outnumber the partial norms (norm_room)
    tx = std::max(tx, 64);
    *variant = *variant == 2 ? 1 : *variant;
  }
  const int cols = columns();
  while (z > 2 && cols * ((n[2] - 2 + z - 1) / z) < want) z /= 2;
  *zchunk = z;
}

// Room for the partial norms of the launches over a finest level of n points:
// its residual in the longest march, and 64 x 8 x 8 points a block.
inline int norm_room(const int *n) {
  const int rblk = ((n[0] + RTX - 1) / RTX) * ((n[1] + RTY - 1) / RTY) * ((n[2] + RZC - 1) / RZC);
  const int sblk = ((n[0] + 61) / 64) * ((n[1] + 5) / 8) * ((n[2] + 5) / 8);
  return std::max(1 << 14, std::max(rblk, sblk) + 64);
}

}  // namespace pmg
