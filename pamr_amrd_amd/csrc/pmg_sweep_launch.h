// pmg_sweep_launch.h -- launch of the fused red-black sweep, one tile variant
// of k_sweep per table row.  Every variant is instantiated for both spacings
// and both right-hand sides, so each (type, operator) pair is a translation
// unit of its own (pmg_sweep_*.hip): they compile in parallel.
#pragma once
#include "pmg_kernels.h"

namespace pmg {

// sweep tile variants (TX, TY, NT, planes in flight, LDS ring planes)
#define PMG_SWEEP_VARIANTS(X)                                                                                   \
  X(0, 64, 8, 256, 1, 4) X(1, 64, 16, 512, 1, 4) X(2, 32, 16, 512, 1, 4) X(3, 128, 8, 512, 1, 4)             \
  X(4, 64, 32, 512, 1, 4) X(5, 128, 16, 1024, 1, 4) X(6, 128, 16, 1024, 2, 4) X(7, 64, 16, 512, 2, 4)        \
  X(8, 128, 8, 512, 2, 4) X(9, 128, 16, 1024, 2, 5) X(10, 128, 16, 1024, 1, 5) X(11, 128, 8, 512, 1, 5)
constexpr int kNumSweepVariants = 12;

// n workgroups beyond cap (the partial-norm workspace): -3, nothing launched
template <typename T, int OP, bool EX>
int launch_sweep(hipStream_t stream, int variant, SweepP<T> P, bool p2, bool rhs0);

#ifdef PMG_SWEEP_IMPL
template <typename T, int OP, bool EX, bool P2, bool RHS0>
int launch_sweep_v(hipStream_t stream, int variant, SweepP<T> P) {
  P.zchunk = std::max(1, std::min(P.zchunk, P.nz - 2));
  int tx = 64, ty = 8;
  const bool wide = P.nx > kLongRow;  // 64-bit offsets, in the tile of variant 0
  switch (wide ? 0 : variant) {
#define PMG_TXY(V, TXV, TYV, NTV, PFV, RGV) case V: tx = TXV; ty = TYV; break;
    PMG_SWEEP_VARIANTS(PMG_TXY)
#undef PMG_TXY
    default: return -1;
  }
  dim3 grid(((P.nx - 2 + tx - 1) / tx) * ((P.ny - 2 + ty - 1) / ty) * ((P.nz - 2 + P.zchunk - 1) / P.zchunk));
  P.nb = (int)grid.x;
  if (P.nb > P.ws.cap) return -3;
  if (wide) {
    hipLaunchKernelGGL((k_sweep<T, OP, EX, P2, RHS0, 64, 8, 256, 1, 4, size_t>), grid, dim3(256), 0, stream, P);
    PMG_HOST_CHECK(hipGetLastError());
    return 0;
  }
  switch (variant) {
#define PMG_LSW(V, TXV, TYV, NTV, PFV, RGV)                                                         \
  case V:                                                                                           \
    hipLaunchKernelGGL((k_sweep<T, OP, EX, P2, RHS0, TXV, TYV, NTV, PFV, RGV>), grid, dim3(NTV), 0, \
                       stream, P);                                                               \
    break;
    PMG_SWEEP_VARIANTS(PMG_LSW)
#undef PMG_LSW
  }
  PMG_HOST_CHECK(hipGetLastError());
  return 0;
}

template <typename T, int OP, bool EX>
int launch_sweep(hipStream_t stream, int v, SweepP<T> P, bool p2, bool rhs0) {
  if (p2) return rhs0 ? launch_sweep_v<T, OP, EX, true, true>(stream, v, P) : launch_sweep_v<T, OP, EX, true, false>(stream, v, P);
  return rhs0 ? launch_sweep_v<T, OP, EX, false, true>(stream, v, P) : launch_sweep_v<T, OP, EX, false, false>(stream, v, P);
}
#endif  // PMG_SWEEP_IMPL

}  // namespace pmg
