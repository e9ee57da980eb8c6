// pmg_small.h -- both legs of the V-cycle on a small level, one launch each.
//
// On a level of up to a few 10^5 points the cycle's cost is not bytes but
// launches and the march: two sweeps, L_op / rhs and the residual were five
// launches of 5-11 us each, and a marching sweep of such a level is a chain of
// dependent planes on a few workgroups.  Here a workgroup takes an 8^3 tile
// with everything the leg needs around it into LDS and runs the whole leg
// there: the halo shrinks by one point per colour pass, so no workgroup waits
// for another.  The redundant halo updates are the owner's operations on the
// owner's values, so the results are the same bits as the separate kernels'.
//
//   down: L_op + compute_MG_rhs (levels below the finest), two red-black
//         sweeps, the residual (amrd/mg.c:84-133 on one level)
//   up:   the coarse-grid correction (amrd/mg.c:323-355), two red-black
//         sweeps (or the sweeps alone)
//
// Both read u from one buffer and write the other (neighbours read halos of
// the first), so a down and an up leg return u to where it was.  The residual
// of a level below the finest goes to a buffer of its own: its f_res, read
// around every tile for the rhs, is still being read by the neighbours (the
// cycle overwrites that f_res with the correction afterwards).
//
// Geometry: local coordinates 0..15 per axis are the tile (4..11) and a
// 4-point halo; LDS holds one more point on each side.  Thread t owns the
// column (t % 16, t / 16 % 16) and eight consecutive z of it, its rho and rhs
// in registers; a colour pass updates four of the eight.
#pragma once
#include "pmg_kernels.h"

namespace pmg {

constexpr int kSmT = 8, kSmH = 4, kSmR = kSmT + 2 * kSmH, kSmL = kSmR + 2;
constexpr int kSmNT = kSmR * kSmR * 2, kSmP = kSmR / 2;  // threads; points per thread
constexpr int kSmC = kSmR / 2 + 2;                       // coarse points per axis around a tile

// The largest level whose legs run as one launch each.  A cycle with separate
// kernels and with legs on every level, us (FP64 plain / FP64 variable coefficient
// / FP32 iteration plain / variable): 33^3 146 -> 124, 169 -> 143, 85 -> 75, 141 ->
// 117; 65^3 187 -> 163, 231 -> 221, 125 -> 107, 189 -> 162; 81^3 663 -> 653, 430 ->
// 467, 224 -> 206, 296 -> 270; 97^3 1417 -> 1426, 1957 -> 2100, 300 -> 299, 327 ->
// 341.  The line is FP64's with the variable coefficient, the first to lose: the
// others would still gain at 81^3.
constexpr size_t kSmallPoints = 300000;

template <typename T>
struct SmallP {
  const T *uin;
  T *uout;
  const T *rho, *a, *c;
  T *rhs;          // down: written (below the finest); up: read (below the finest)
  const T *res;    // down, below the finest: the injected f_res
  T *res_out;      // down: the residual
  T *lop;          // down, below the finest: written
  const T *cu, *clop;
  T *cres;         // up with the correction: the coarse level; its f_res gets the correction (null: not stored)
  const uint8_t *chr;
  int nx, ny, nz, cnx, cny, cnz;
  int bx0, bx1, by0, by1, bz0, bz1;  // relax / residual box
  int cx0, cx1, cy0, cy1, cz0, cz1;  // child-mask ON box (down, below the finest)
  T w0_r, w0_i;
  Spacing<T> sp;
  NormWs ws;
  int slot;
  int nb;
};

// LDS offset of local point (x, y, z), -1 <= x, y, z <= 16
__device__ __forceinline__ int sm_at(int x, int y, int z) { return ((z + 1) * kSmL + y + 1) * kSmL + x + 1; }

template <typename T, int OP, bool P2>
__device__ __forceinline__ T sm_lop(const T *U, const T *A, int q, T cc, T rho, const Spacing<T> &sp, T *jac) {
  constexpr int sy = kSmL, sz = kSmL * kSmL;
  if constexpr (OP == 0) {
    if (jac) *jac = sp.jac;
    return lop_poisson<T, P2>(U[q], U[q + 1], U[q - 1], U[q + sy], U[q - sy], U[q + sz], U[q - sz], rho, sp);
  } else {
    return lop_varcoef<T, P2>(U[q], U[q + 1], U[q - 1], U[q + sy], U[q - sy], U[q + sz], U[q - sz], A[q], A[q + 1],
                              A[q - 1], A[q + sy], A[q - sy], A[q + sz], A[q - sz], cc, rho, sp, jac);
  }
}

// What a thread knows of its eight points (bit s: local z = 8 * half + s)
template <typename T, int OP>
struct SmCol {
  int x, y, zb;        // local position of point 0
  int i, j, kb;        // its global position
  unsigned in, upd, own;  // in the grid; updatable; stored by this block (tile and adjoining faces)
  unsigned tile;          // in the tile proper (counted in the norms)
  size_t p0, sz;          // element of point 0 (0 when out of the grid) and the z stride
  T rho[kSmP], rhs[kSmP], cc[OP == 1 ? kSmP : 1];
};

template <typename T, int OP, bool EX>
__device__ __forceinline__ void sm_col(const SmallP<T> &P, int x0, int y0, int z0, SmCol<T, OP> &C) {
  const int t = threadIdx.x;
  C.x = t % kSmR;
  C.y = (t / kSmR) % kSmR;
  C.zb = (t / (kSmR * kSmR)) * kSmP;
  C.i = x0 - kSmH + C.x;
  C.j = y0 - kSmH + C.y;
  C.kb = z0 - kSmH + C.zb;
  const bool gxy = C.i >= 0 && C.i < P.nx && C.j >= 0 && C.j < P.ny;
  const bool bxy = C.i >= P.bx0 && C.i <= P.bx1 && C.j >= P.by0 && C.j <= P.by1;
  // own: the tile, and the faces next to it
  auto own1 = [](int v, int o, int n) { return (v >= o && v < o + kSmT && v <= n - 2) || (v == 0 && o == 1) || (v == n - 1 && o + kSmT >= n - 1); };
  const bool oxy = own1(C.i, x0, P.nx) && own1(C.j, y0, P.ny);
  const bool txy = C.x >= kSmH && C.x < kSmH + kSmT && C.y >= kSmH && C.y < kSmH + kSmT;
  C.sz = (size_t)P.nx * P.ny;
  C.p0 = gxy ? (size_t)C.i + (size_t)P.nx * C.j : 0;
  C.in = C.upd = C.own = C.tile = 0;
#pragma unroll
  for (int s = 0; s < kSmP; s++) {
    const int k = C.kb + s;
    const bool in = gxy && k >= 0 && k < P.nz;
    bool upd = in && bxy && k >= P.bz0 && k <= P.bz1;
    if constexpr (EX) upd = upd && !P.chr[in ? C.p0 + (size_t)k * C.sz : 0];
    C.in |= (unsigned)in << s;
    C.upd |= (unsigned)upd << s;
    C.own |= (unsigned)(in && oxy && own1(k, z0, P.nz)) << s;
    C.tile |= (unsigned)(txy && C.zb + s >= kSmH && C.zb + s < kSmH + kSmT) << s;
  }
}
template <typename T, int OP>
__device__ __forceinline__ size_t sm_p(const SmCol<T, OP> &C, int s) {
  return (C.in >> s) & 1 ? C.p0 + (size_t)(C.kb + s) * C.sz : 0;
}

// two red-black sweeps in LDS; pass q acts on local [q + off, 16 - q - off)
template <typename T, int OP, bool P2, bool RHS0>
__device__ __forceinline__ void sm_sweeps(const SmallP<T> &P, SmCol<T, OP> &C, T *U, const T *A, int off, bool count,
                                          double &sum, double &cnt) {
#pragma unroll
  for (int q = 0; q < 4; q++) {
    const int lo = q + off, hi = kSmR - 1 - lo;
    // pass (q & 1) takes the points with (i + j + k + 3 + pass) even
    const int o = (C.i + C.j + C.kb + 3 + q) & 1;
    const bool xy = C.x >= lo && C.x <= hi && C.y >= lo && C.y <= hi;
#pragma unroll
    for (int h = 0; h < kSmP / 2; h++) {
      const int s = 2 * h + o, z = C.zb + s;
      if (!(xy && z >= lo && z <= hi && ((C.upd >> s) & 1))) continue;
      const int at = sm_at(C.x, C.y, z);
      const T rho = o ? C.rho[2 * h + 1] : C.rho[2 * h];
      T cc = T(0);
      if constexpr (OP == 1) cc = o ? C.cc[2 * h + 1] : C.cc[2 * h];
      T jac;
      const T L = sm_lop<T, OP, P2>(U, A, at, cc, rho, P.sp, &jac);
      T r;
      if constexpr (RHS0) r = L - T(0);
      else r = L - (o ? C.rhs[2 * h + 1] : C.rhs[2 * h]);
      if constexpr (std::is_same<T, float>::value && OP == 0) U[at] = U[at] - r * P.sp.ijac;
      else U[at] = U[at] - div_jac<T, OP>(r, jac, P.sp);
      if (count && q >= 2 && ((C.tile >> s) & 1)) {
        sum += (double)r * (double)r;
        cnt += 1.0;
      }
    }
    __syncthreads();
  }
}

__device__ __forceinline__ void sm_tile(int nx, int ny, int &x0, int &y0, int &z0) {
  const int tile = xcd_tile(blockIdx.x, gridDim.x);
  const int ntx = (nx - 2 + kSmT - 1) / kSmT, nty = (ny - 2 + kSmT - 1) / kSmT;
  x0 = 1 + (tile % ntx) * kSmT;
  y0 = 1 + ((tile / ntx) % nty) * kSmT;
  z0 = 1 + (tile / (ntx * nty)) * kSmT;
}

template <typename T, int OP, bool EX, bool P2, bool FINE>
__global__ __launch_bounds__(kSmNT) void k_small_down(SmallP<T> P) {
  __shared__ T U[kSmL * kSmL * kSmL];
  __shared__ T Ab[OP == 1 ? kSmL * kSmL * kSmL : 1];
  int x0, y0, z0;
  sm_tile(P.nx, P.ny, x0, y0, z0);
  SmCol<T, OP> C;
  sm_col<T, OP, EX>(P, x0, y0, z0, C);
  // every load of the leg is requested before any is used (positions outside
  // the grid read element 0; no updatable point reads them)
  constexpr int NL = (kSmL * kSmL * kSmL + kSmNT - 1) / kSmNT;
  T lu[NL], la[OP == 1 ? NL : 1];
#pragma unroll
  for (int m = 0; m < NL; m++) {
    const int q = threadIdx.x + m * kSmNT;
    const int i = x0 - kSmH - 1 + q % kSmL, j = y0 - kSmH - 1 + (q / kSmL) % kSmL, k = z0 - kSmH - 1 + q / (kSmL * kSmL);
    const bool ok = q < kSmL * kSmL * kSmL && i >= 0 && i < P.nx && j >= 0 && j < P.ny && k >= 0 && k < P.nz;
    const size_t p = ok ? ix3(i, j, k, P.nx, P.ny) : 0;
    lu[m] = P.uin[p];
    if constexpr (OP == 1) la[m] = P.a[p];
  }
  T res[FINE ? 1 : kSmP];
#pragma unroll
  for (int s = 0; s < kSmP; s++) {
    const size_t p = sm_p(C, s);
    C.rho[s] = P.rho[p];
    if constexpr (OP == 1) C.cc[s] = P.c[p];
    if constexpr (!FINE) res[s] = P.res[p];
  }
#pragma unroll
  for (int m = 0; m < NL; m++) {
    const int q = threadIdx.x + m * kSmNT;
    if (q < kSmL * kSmL * kSmL) {
      U[q] = lu[m];
      if constexpr (OP == 1) Ab[q] = la[m];
    }
  }
  __syncthreads();
  if constexpr (!FINE) {
    // L_op + compute_MG_rhs (k_lop_rhs)
    const bool cxy = C.i >= P.cx0 && C.i <= P.cx1 && C.j >= P.cy0 && C.j <= P.cy1;
    const bool ixy = C.i >= 1 && C.i <= P.nx - 2 && C.j >= 1 && C.j <= P.ny - 2;
#pragma unroll
    for (int s = 0; s < kSmP; s++) {
      const int k = C.kb + s, at = sm_at(C.x, C.y, C.zb + s);
      const bool on = cxy && k >= P.cz0 && k <= P.cz1;
      T lopv = T(0);
      bool act = ((C.in >> s) & 1) && on && ixy && k >= 1 && k <= P.nz - 2;
      if constexpr (EX) act = act && !P.chr[sm_p(C, s)];
      if (act) lopv = sm_lop<T, OP, P2>(U, Ab, at, OP == 1 ? C.cc[s] : T(0), C.rho[s], P.sp, nullptr);
      C.rhs[s] = on ? (-res[s]) * P.w0_r + lopv : T(0);
      if ((C.own >> s) & 1) {
        const size_t p = sm_p(C, s);
        P.rhs[p] = C.rhs[s];
        P.lop[p] = U[at];
      }
    }
    __syncthreads();
  }
  double s2 = 0.0, cnt = 0.0, u1 = 0.0, u2 = 0.0;
  sm_sweeps<T, OP, P2, FINE>(P, C, U, Ab, 0, false, u1, u2);
#pragma unroll
  for (int s = 0; s < kSmP; s++) {
    if (!((C.own >> s) & 1)) continue;
    const size_t p = sm_p(C, s);
    const int at = sm_at(C.x, C.y, C.zb + s);
    P.uout[p] = U[at];
    if ((C.upd >> s) & 1) {
      const T L = sm_lop<T, OP, P2>(U, Ab, at, OP == 1 ? C.cc[s] : T(0), C.rho[s], P.sp, nullptr);
      T r;
      if constexpr (FINE) r = L - T(0);
      else r = L - C.rhs[s];
      P.res_out[p] = r;
      s2 += (double)r * (double)r;
      cnt += 1.0;
    } else if constexpr (FINE) {
      // excised interior points hold 0, faces are not written (k_residual)
      if ((C.tile >> s) & 1) P.res_out[p] = T(0);
    } else {
      P.res_out[p] = res[s];  // the injected value stays
    }
  }
  norm_partial<kSmNT>(s2, cnt, P.ws, P.slot, blockIdx.x, P.nb);
}

template <typename T, int OP, bool EX, bool P2, bool FINE, bool CGC>
__global__ __launch_bounds__(kSmNT) void k_small_up(SmallP<T> P) {
  __shared__ T U[kSmL * kSmL * kSmL];
  __shared__ T Ab[OP == 1 ? kSmL * kSmL * kSmL : 1];
  __shared__ T D[CGC ? kSmC * kSmC * kSmC : 1];
  int x0, y0, z0;
  sm_tile(P.nx, P.ny, x0, y0, z0);
  SmCol<T, OP> C;
  sm_col<T, OP, EX>(P, x0, y0, z0, C);
  T u[kSmP], av[OP == 1 ? kSmP : 1];
#pragma unroll
  for (int s = 0; s < kSmP; s++) {
    const size_t p = sm_p(C, s);
    u[s] = P.uin[p];
    C.rho[s] = P.rho[p];
    if constexpr (!FINE) C.rhs[s] = P.rhs[p];
    if constexpr (OP == 1) {
      C.cc[s] = P.c[p];
      av[s] = P.a[p];
    }
  }
  if constexpr (CGC) {
    // the coarse correction (u - lop) / w0_i around the tile; this block
    // stores the coarse points under the fine points it owns
    const int ca0 = (x0 - kSmH) >> 1, cb0 = (y0 - kSmH) >> 1, cc0 = (z0 - kSmH) >> 1;
    auto own1 = [](int c, int o, int n) {
      const int f = 2 * c;
      return (f >= o && f < o + kSmT && f <= n - 2) || (f == 0 && o == 1) || (f == n - 1 && o + kSmT >= n - 1);
    };
    for (int q = threadIdx.x; q < kSmC * kSmC * kSmC; q += kSmNT) {
      const int a = ca0 + q % kSmC, b = cb0 + (q / kSmC) % kSmC, c = cc0 + q / (kSmC * kSmC);
      T d = T(0);
      if (a >= 0 && a < P.cnx && b >= 0 && b < P.cny && c >= 0 && c < P.cnz) {
        const size_t p = ix3(a, b, c, P.cnx, P.cny);
        d = (P.cu[p] - P.clop[p]) / P.w0_i;
        if (P.cres && own1(a, x0, P.nx) && own1(b, y0, P.ny) && own1(c, z0, P.nz)) P.cres[p] = d;
      }
      D[q] = d;
    }
    __syncthreads();
    // the trilinear phases of k_cgc: x, then y, then z
    const T c0 = T(1 - (1 * 1.0) / 2), c1 = T((1 * 1.0) / 2);
    const int ai = (C.i >> 1) - ca0, aj = (C.j >> 1) - cb0;
    const bool ri = C.i & 1, rj = C.j & 1;
    // z0 is odd, so the thread's first point is odd: points 0 and 1 lie
    // between coarse planes 0, 1 and on 1, points 2 and 3 between 1, 2, ...
    const int ak = (C.kb >> 1) - cc0;
    auto Y = [&](int pl) -> T {
      const T *S = D + ((ak + pl) * kSmC + aj) * kSmC + ai;
      auto X = [&](int b) -> T { return ri ? c0 * S[b * kSmC] + c1 * S[b * kSmC + 1] : S[b * kSmC]; };
      return rj ? c0 * X(0) + c1 * X(1) : X(0);
    };
    T y0v = Y(0);
#pragma unroll
    for (int h = 0; h < kSmP / 2; h++) {
      const T y1v = Y(h + 1);
      T v0 = c0 * y0v + c1 * y1v, v1 = y1v;
      if constexpr (EX) {
        if (P.chr[sm_p(C, 2 * h)]) v0 = T(0);
        if (P.chr[sm_p(C, 2 * h + 1)]) v1 = T(0);
      }
      u[2 * h] = u[2 * h] + v0;
      u[2 * h + 1] = u[2 * h + 1] + v1;
      y0v = y1v;
    }
  }
#pragma unroll
  for (int s = 0; s < kSmP; s++) {
    const int at = sm_at(C.x, C.y, C.zb + s);
    U[at] = u[s];
    if constexpr (OP == 1) Ab[at] = av[s];
  }
  __syncthreads();
  double s2 = 0.0, cnt = 0.0;
  sm_sweeps<T, OP, P2, FINE>(P, C, U, Ab, 1, true, s2, cnt);
#pragma unroll
  for (int s = 0; s < kSmP; s++)
    if ((C.own >> s) & 1) P.uout[sm_p(C, s)] = U[sm_at(C.x, C.y, C.zb + s)];
  norm_partial<kSmNT>(s2, cnt, P.ws, P.slot, blockIdx.x, P.nb);
}

inline int small_blocks(int nx, int ny, int nz) {
  auto t = [](int n) { return (n - 2 + kSmT - 1) / kSmT; };
  return t(nx) * t(ny) * t(nz);
}

// leg: 0 down, 1 up with the coarse-grid correction, 2 up without
template <typename T>
int launch_small(hipStream_t stream, int leg, SmallP<T> P, int op, bool ex, bool fine);

#ifdef PMG_SMALL_IMPL
template <typename T, int OP, bool EX, bool P2, bool FINE>
int launch_small_v(hipStream_t stream, int leg, SmallP<T> P) {
  const dim3 grid(small_blocks(P.nx, P.ny, P.nz)), blk(kSmNT);
  P.nb = (int)grid.x;
  if (P.nb > P.ws.cap) return -3;
  if (leg == 0) hipLaunchKernelGGL((k_small_down<T, OP, EX, P2, FINE>), grid, blk, 0, stream, P);
  else if (leg == 1) hipLaunchKernelGGL((k_small_up<T, OP, EX, P2, FINE, true>), grid, blk, 0, stream, P);
  else hipLaunchKernelGGL((k_small_up<T, OP, EX, P2, FINE, false>), grid, blk, 0, stream, P);
  PMG_HOST_CHECK(hipGetLastError());
  return 0;
}
template <typename T, int OP, bool EX>
int launch_small_e(hipStream_t st, int leg, const SmallP<T> &P, bool fine) {
  if (P.sp.pow2) return fine ? launch_small_v<T, OP, EX, true, true>(st, leg, P) : launch_small_v<T, OP, EX, true, false>(st, leg, P);
  return fine ? launch_small_v<T, OP, EX, false, true>(st, leg, P) : launch_small_v<T, OP, EX, false, false>(st, leg, P);
}
template <typename T>
int launch_small(hipStream_t st, int leg, SmallP<T> P, int op, bool ex, bool fine) {
  if (op == 0) return ex ? launch_small_e<T, 0, true>(st, leg, P, fine) : launch_small_e<T, 0, false>(st, leg, P, fine);
  return ex ? launch_small_e<T, 1, true>(st, leg, P, fine) : launch_small_e<T, 1, false>(st, leg, P, fine);
}
#endif  // PMG_SMALL_IMPL

}  // namespace pmg
