// pmg_transfer.hip -- device versions of the m_util_r8 transfer routines.
//
// Each extern "C" entry point takes exactly the arguments of the Fortran
// routine it replaces (src/m_util_r8.f; prototypes include/m_util_r8.h),
// by value, with u1/u2/chr1 being device pointers, plus a HIP stream.  The
// silent early returns of the Fortran bounds checks are kept (return 0,
// nothing written); launch errors return -1.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "pamr_mg_gpu.h"

#include "pmg_ops.h"

using namespace pmg;

namespace {

constexpr int NT = 256;

// dmcopy3d, src/m_util_r8.f:20-50
template <typename T>
__global__ __launch_bounds__(NT) void k_copy3d(const T *u1, T *u2, int nx1, int ny1, int nx2,
                                               int ny2, int i1, int j1, int k1, int i2, int j2,
                                               int k2, int ni, int nj, int nk, int si1, int sj1,
                                               int sk1, int si2, int sj2, int sk2, BoxPts bp) {
  for_box(bp, [&](int i, int j, int k) {
    u2[ix3(i2 - 1 + i * si2, j2 - 1 + j * sj2, k2 - 1 + k * sk2, nx2, ny2)] =
        u1[ix3(i1 - 1 + i * si1, j1 - 1 + j * sj1, k1 - 1 + k * sk1, nx1, ny1)];
  });
}

// dmfwr3d / dmhwr3d over an ni x nj x nk target segment
template <typename T, int KIND, bool EXC>
__global__ __launch_bounds__(NT) void k_restrict3d(const T *u1, T *u2, const T *chr1, T ex,
                                                   int nx1, int ny1, int nz1, int nx2, int ny2,
                                                   int i1, int j1, int k1, int i2, int j2,
                                                   int k2, int ni, int nj, int nk, int si1,
                                                   int sj1, int sk1, int si2, int sj2,
                                                   int sk2, BoxPts bp) {
  for_box(bp, [&](int i, int j, int k) {
    const int i0 = i1 + i * si1, j0 = j1 + j * sj1, k0 = k1 + k * sk1;
    T v;
    if constexpr (KIND == 3) {
      if constexpr (EXC) v = fw_point_ex<T>(u1, chr1, ex, nx1, ny1, nz1, i0, j0, k0, i + 1);
      else v = fw_point<T>(u1, nx1, ny1, nz1, i0, j0, k0);
    } else {
      v = hw_point<T, EXC>(u1, chr1, ex, nx1, ny1, nz1, i0, j0, k0);
    }
    u2[ix3(i2 - 1 + i * si2, j2 - 1 + j * sj2, k2 - 1 + k * sk2, nx2, ny2)] = v;
  });
}

// dminterp3d with ord = 2 and no excision: the three line phases of
// src/m_util_r8.f:518-634 composed per target point.  Along each axis the
// phase value is c0*v(a) + c1*v(a+1) (dvi2q1d, :350-357) with
// sg=(r*1.0)/rho, c0=1-sg, c1=sg, applied x first, then y, then z, on the
// previous phase's values -- the same IEEE operations in the same order.
template <typename T>
__device__ __forceinline__ T interp_coef(int r, int rho, T *c1) {
  double sg = (r * 1.0) / rho;
  *c1 = (T)sg;
  return (T)(1 - sg);
}

// R2: all three ratios are 2 (shifts for the divisions, 0.5 for both weights)
template <typename T, bool R2>
__global__ __launch_bounds__(NT) void k_interp3d(const T *u1, T *u2, int nx1, int ny1, int nx2,
                                                 int ny2, int i1, int j1, int k1, int i2,
                                                 int j2, int k2, int ni, int nj, int nk,
                                                 int si1, int sj1, int sk1, int irho, int jrho,
                                                 int krho, BoxPts bp) {
  if (R2) irho = jrho = krho = 2;
  for_box(bp, [&](int fi, int fj, int fk) {
    const int ai = fi / irho, ri = fi % irho, aj = fj / jrho, rj = fj % jrho, ak = fk / krho, rk = fk % krho;
    auto U = [&](int a, int b, int c) -> T {
      return u1[ix3(i1 - 1 + a * si1, j1 - 1 + b * sj1, k1 - 1 + c * sk1, nx1, ny1)];
    };
    T cx1 = T(0.5), cy1 = T(0.5), cz1 = T(0.5), cx0 = T(0.5), cy0 = T(0.5), cz0 = T(0.5);
    if constexpr (!R2) {
      cx0 = interp_coef<T>(ri, irho, &cx1);
      cy0 = interp_coef<T>(rj, jrho, &cy1);
      cz0 = interp_coef<T>(rk, krho, &cz1);
    }
    auto X = [&](int b, int c) -> T {
      return ri == 0 ? U(ai, b, c) : cx0 * U(ai, b, c) + cx1 * U(ai + 1, b, c);
    };
    auto Y = [&](int c) -> T { return rj == 0 ? X(aj, c) : cy0 * X(aj, c) + cy1 * X(aj + 1, c); };
    u2[ix3(i2 - 1 + fi, j2 - 1 + fj, k2 - 1 + fk, nx2, ny2)] = rk == 0 ? Y(ak) : cz0 * Y(ak) + cz1 * Y(ak + 1);
  });
}

// ---- fourth-order interpolation (dminterp3d, ord = 4, no excision) ------
// (vi4_point, one point of dvi4q1d, is in pmg_ops.h)

// The three line phases of dminterp3d (src/m_util_r8.f:518-634), one launch
// each, one thread per written point.  A phase writes only points off the
// anchor lattice of its axis and reads only points on it (inside or just
// outside the segment), so its points are independent; phases run in the
// reference's order x, y, z on u2 after the common points were copied.
template <int AX, bool R2>
__global__ __launch_bounds__(NT) void k_interp4(double *u2, int nx2, int ny2, int nz2, int i2, int j2, int k2, int ni,
                                                int nj, int nk, int irho, int jrho, int krho, BoxPts bp) {
  if (R2) irho = jrho = krho = 2;
  // offsets from (i2, j2, k2); axes behind the phase's own are still coarse
  for_box(bp, [&](int fi, int fj, int fk) {
    if (AX < 1) fj *= jrho;
    if (AX < 2) fk *= krho;
    const int f = AX == 0 ? fi : (AX == 1 ? fj : fk), rho = AX == 0 ? irho : (AX == 1 ? jrho : krho);
    if (f % rho == 0) return;
    auto A = [&](int a) -> double {
      return u2[ix3(i2 - 1 + (AX == 0 ? a * irho : fi), j2 - 1 + (AX == 1 ? a * jrho : fj),
                    k2 - 1 + (AX == 2 ? a * krho : fk), nx2, ny2)];
    };
    u2[ix3(i2 - 1 + fi, j2 - 1 + fj, k2 - 1 + fk, nx2, ny2)] =
        AX == 0 ? vi4_point(ni, irho, i2, nx2, f, A) : (AX == 1 ? vi4_point(nj, jrho, j2, ny2, f, A) : vi4_point(nk, krho, k2, nz2, f, A));
  });
}

// ---- excision interpolation -------------------------------------------
// Line view: v(q) for q = 1..n1 (1-based) at stride sv elements.
template <typename T, typename CHR>
__device__ void line_vi2q1d_ex(T *v, int i1, int n1, int n, int irho, int s1, int s2,
                               const CHR &chr, int i3, int s3, T ex) {
#define LV(q) v[((size_t)(q)-1)]
#define LC(q) chr((q)-1)
  for (int i = 1; i <= n; i++) {
    int i10 = (i - 1) * s1 + i1, i30 = (i - 1) * s3 + i3;
    if (LC(i30) == ex) {
      if (i10 > 3 * s1 && LC(i30 - s3) != ex && LC(i30 - 2 * s3) != ex && LC(i30 - 3 * s3) != ex)
        LV(i10) = 3 * (LV(i10 - s1) - LV(i10 - 2 * s1)) + LV(i10 - 3 * s1);
      else if (i10 <= (n1 - 3 * s1) && LC(i30 + s3) != ex && LC(i30 + 2 * s3) != ex &&
               LC(i30 + 3 * s3) != ex)
        LV(i10) = 3 * (LV(i10 + s1) - LV(i10 + 2 * s1)) + LV(i10 + 3 * s1);
      else if (i10 > 2 * s1 && LC(i30 - s3) != ex && LC(i30 - 2 * s3) != ex)
        LV(i10) = 2 * LV(i10 - s1) - LV(i10 - 2 * s1);
      else if (i10 <= (n1 - 2 * s1) && LC(i30 + s3) != ex && LC(i30 + 2 * s3) != ex)
        LV(i10) = 2 * LV(i10 + s1) - LV(i10 + 2 * s1);
      else if (i10 > s1 && LC(i30 - s3) != ex)
        LV(i10) = LV(i10 - s1);
      else if (i10 <= (n1 - s1) && LC(i30 + s3) != ex)
        LV(i10) = LV(i10 + s1);
    }
    // v2(irho*(i-1)*s2+i2) = v1(i10): in place with s1 == irho*s2, i1 == i2
  }
  for (int j = 1; j <= irho - 1; j++) {
    double sg = (j * 1.0) / irho;
    T c0 = (T)(1 - sg), c1 = (T)sg;
    for (int i = 0; i <= n - 2; i++) LV((irho * i + j) * s2 + i1) = c0 * LV(i * s1 + i1) + c1 * LV((i + 1) * s1 + i1);
  }
#undef LV
#undef LC
}

// dvi4q1d_ex (src/m_util_r8.f:146-319) on one line, in place (v1 = v2 with
// s1 == irho*s2, so the common-point copy is a no-op): the extension of the
// anchor range by up to 3 anchors each side, the dvi2q1d_ex pass when a
// non-excised run is shorter than 4 anchors, extrapolation into excised
// anchors, then the first / last / interior cubic cells -- in the
// reference's order, with its conditions as written.
template <typename T, typename CHR>
__device__ void line_vi4q1d_ex(T *v, int i1, int n1, int n, int irho, int s1, int s2, const CHR &chr, int i3,
                               int s3, T ex) {
#define LV(q) v[((size_t)(q)-1)]
#define LC(q) chr((q)-1)
  const double half = 0.5, mhalf = -0.5, sixth = 0.1666666666666667, msixth = -0.1666666666666667;
  int i = 3, i1s = i1;
  while (i > 0 && i1s > s1) {
    i1s -= s1;
    i--;
  }
  i = 3;
  int i1e = i1 + (n - 1) * s1;
  while (i > 0 && i1e < (n1 - s1)) {
    i1e += s1;
    i--;
  }
  int cn = 0;
  bool init_2 = false;
  for (i = i1s; i <= i1e; i += s1) {
    if (LC((i - i1) * s3 / s1 + i3) == ex || i == i1e) {
      if (cn > 0 && cn < 4) init_2 = true;
      else cn = 0;
    } else {
      cn++;
    }
  }
  if (init_2) line_vi2q1d_ex<T>(v, i1, n1, n, irho, s1, s2, chr, i3, s3, ex);
  for (i = i1s; i <= i1e; i += s1) {
    if (LC(i3 + s3 * (i - i1) / s1) == ex) {
      if (i >= (i1s + 3 * s1) && LC(i3 + s3 * (i - s1 - i1) / s1) != ex && LC(i3 + s3 * (i - 2 * s1 - i1) / s1) != ex &&
          LC(i3 + s3 * (i - 3 * s1 - i1) / s1) != ex) {
        if (i >= (i1s + 4 * s1) && LC(i3 + s3 * (i - 4 * s1 - i1) / s1) != ex)
          LV(i) = 4 * (LV(i - s1) + LV(i - 3 * s1)) - 6 * LV(i - 2 * s1) - LV(i - 4 * s1);
        else
          LV(i) = 3 * (LV(i - s1) - LV(i - 2 * s1)) + LV(i - 3 * s1);
      } else if (i <= (i1e - 3 * s1) && LC(i3 + s3 * (i + s1 - i1) / s1) != ex &&
                 LC(i3 + s3 * (i + 2 * s1 - i1) / s1) != ex && LC(i3 + s3 * (i + 3 * s1 - i1) / s1) != ex) {
        if (i <= (i1s - 4 * s1) && LC(i3 + s3 * (i + 4 * s1 - i1) / s1) != ex)
          LV(i) = 4 * (LV(i + s1) + LV(i + 3 * s1)) - 6 * LV(i + 2 * s1) - LV(i + 4 * s1);
        else
          LV(i) = 3 * (LV(i + s1) - LV(i + 2 * s1)) + LV(i + 3 * s1);
      }
    }
  }
  auto coef = [&](double sg, double *c) {
    c[0] = msixth * (sg - 1.0) * (sg - 2.0) * (sg - 3.0);
    c[1] = half * sg * (sg - 2.0) * (sg - 3.0);
    c[2] = mhalf * sg * (sg - 1.0) * (sg - 3.0);
    c[3] = sixth * sg * (sg - 1.0) * (sg - 2.0);
  };
  double c[4];
  for (i = 1; i <= n - 1; i++) {  // first cells of non-excised runs
    const int i10 = (i - 1) * s1 + i1, i30 = (i - 1) * s3 + i3, j0 = (i - 1) * irho * s2 + i1;
    if (i10 <= (i1e - 3 * s1) && LC(i30 + s3) != ex && LC(i30 + 2 * s3) != ex &&
        ((i == 1 && i10 == i1s) || (i10 >= (i1s + s1) && LC(i30) != ex && LC(i30 - s3) == ex) || LC(i30) == ex)) {
      for (int j = 1; j <= irho - 1; j++) {
        coef((j * 1.0) / irho, c);
        LV(j * s2 + j0) = c[0] * LV(i10) + c[1] * LV(s1 + i10) + c[2] * LV(2 * s1 + i10) + c[3] * LV(3 * s1 + i10);
      }
    }
  }
  for (i = 1; i <= n - 1; i++) {  // last cells of non-excised runs
    const int i10 = (i - 1) * s1 + i1, i30 = (i - 1) * s3 + i3, j0 = (i - 1) * irho * s2 + i1;
    if (i10 >= (i1s + 2 * s1) && LC(i30 - s3) != ex &&
        ((i == (n - 1) && i10 == (i1e - s1)) || (i10 <= (i1e - s1) && LC(i30) != ex && LC(i30 + s3) == ex))) {
      for (int j = 1; j <= irho - 1; j++) {
        coef(2.0 + (j * 1.0) / irho, c);
        LV(j * s2 + j0) = c[0] * LV(i10 - 2 * s1) + c[1] * LV(i10 - s1) + c[2] * LV(i10) + c[3] * LV(i10 + s1);
      }
    }
  }
  for (i = 1; i <= n; i++) {  // interior cells
    const int i10 = (i - 1) * s1 + i1, i30 = (i - 1) * s3 + i3, j0 = (i - 1) * irho * s2 + i1;
    if (LC(i30) != ex && i10 >= (i1s + s1) && LC(i30 - s3) != ex && i10 <= (i1e - 2 * s1) && LC(i30 + s3) != ex) {
      for (int j = 1; j <= irho - 1; j++) {
        coef(1.0 + (j * 1.0) / irho, c);
        LV(j0 + j * s2) = c[0] * LV(i10 - s1) + c[1] * LV(i10) + c[2] * LV(i10 + s1) + c[3] * LV(i10 + 2 * s1);
      }
    }
  }
#undef LV
#undef LC
}

// chrt of src/m_util_r8.f:426-456 evaluated on demand: init_chrt copies
// column c0, each and_chrt folds one more column (ex only if both are ex).
template <typename T>
struct ChrtCols {
  const T *c[4];
  size_t stride;
  T ex;
  __device__ T operator()(int m) const {
    size_t off = (size_t)m * stride;
    T v = c[0][off];
    for (int q = 1; q < 4; q++)
      if (c[q]) v = (v == ex && c[q][off] == ex) ? ex : ex + 1;
    return v;
  }
};

// One line phase of the second-order excised interpolation, one thread per
// point.  dvi2q1d_ex walks a line: it first replaces the value of every
// excised anchor that has non-excised neighbours by an extrapolation from
// them, then interpolates between anchors.  The extrapolations read only
// non-excised anchors, which it never changes, so each anchor's value -- and
// each point between two anchors -- follows from the line as it was before:
// no order along the line is needed.  (A thread per line left most of the
// chip idle behind a serial walk: 89 + 66 + 131 us for the x, y and z lines of
// 161 x 97 x 129 points, now 7 + 5 + 9.)  In place on u2: an anchor is written
// only if its extrapolation succeeded, and no other point reads it then.
template <typename T, typename CHR>
__device__ __forceinline__ bool anchor_ex(const T *v, long long i10, long long n1, long long s1, const CHR &chr, int i30,
                                          int s3, T ex, T &val) {
#define LV(q) v[(q)-1]
#define LC(q) chr((q)-1)
  if (LC(i30) == ex) {
    if (i10 > 3 * s1 && LC(i30 - s3) != ex && LC(i30 - 2 * s3) != ex && LC(i30 - 3 * s3) != ex)
      val = 3 * (LV(i10 - s1) - LV(i10 - 2 * s1)) + LV(i10 - 3 * s1);
    else if (i10 <= (n1 - 3 * s1) && LC(i30 + s3) != ex && LC(i30 + 2 * s3) != ex && LC(i30 + 3 * s3) != ex)
      val = 3 * (LV(i10 + s1) - LV(i10 + 2 * s1)) + LV(i10 + 3 * s1);
    else if (i10 > 2 * s1 && LC(i30 - s3) != ex && LC(i30 - 2 * s3) != ex)
      val = 2 * LV(i10 - s1) - LV(i10 - 2 * s1);
    else if (i10 <= (n1 - 2 * s1) && LC(i30 + s3) != ex && LC(i30 + 2 * s3) != ex)
      val = 2 * LV(i10 + s1) - LV(i10 + 2 * s1);
    else if (i10 > s1 && LC(i30 - s3) != ex)
      val = LV(i10 - s1);
    else if (i10 <= (n1 - s1) && LC(i30 + s3) != ex)
      val = LV(i10 + s1);
    else {
      val = LV(i10);
      return false;
    }
    return true;
  }
  val = LV(i10);
  return false;
#undef LV
#undef LC
}

// R2: all ratios are 2, as between PAMR's levels; the divisions by them are
// then shifts (six a point; 161 x 97 x 129: 28 + 15 + 11 -> 21 + 14 + 9 us).
template <typename T, int AX, bool R2>
__global__ __launch_bounds__(NT) void k_interp_ex2(T *u2, const T *chr1, T ex, int nx1, int ny1, int nx2, int ny2,
                                                   int nz2, int i1, int j1, int k1, int i2, int j2, int k2, int ni,
                                                   int nj, int nk, int si1, int sj1, int sk1, int irho, int jrho,
                                                   int krho, BoxPts bp) {
  if (R2) irho = jrho = krho = 2;
  for_box(bp, [&](int fi, int fj, int fk) {
    if (AX < 1) fj *= jrho;
    if (AX < 2) fk *= krho;
    // the line's column(s) of chr: those of the anchors on either side along
    // the axes already interpolated (init_chrt / and_chrt)
    const int ic = i1 + si1 * (fi / irho), jc = j1 + sj1 * (fj / jrho), kc = k1 + sk1 * (fk / krho);
    const bool oi = AX >= 1 && fi % irho != 0, oj = AX >= 2 && fj % jrho != 0;
    const size_t stride = AX == 0 ? 1 : (AX == 1 ? (size_t)nx1 : (size_t)nx1 * ny1);
    const T *c0 = chr1 + ix3(AX == 0 ? 0 : ic - 1, AX == 1 ? 0 : jc - 1, AX == 2 ? 0 : kc - 1, nx1, ny1);
    const size_t di = si1, dj = (size_t)sj1 * nx1;
    auto chr = [&](int m) -> T {
      const T *c = c0 + (size_t)m * stride;
      bool x = c[0] == ex;
      if (oi) x = x && c[di] == ex;
      if (oj) x = x && c[dj] == ex;
      if (oi && oj) x = x && c[di + dj] == ex;
      return x ? ex : ex + 1;
    };
    // the line itself, at stride s2, its first anchor at 1-based position p0
    const long long s2 = AX == 0 ? 1 : (AX == 1 ? (long long)nx2 : (long long)nx2 * ny2);
    const int rho = AX == 0 ? irho : (AX == 1 ? jrho : krho), n2 = AX == 0 ? nx2 : (AX == 1 ? ny2 : nz2);
    const int o2 = AX == 0 ? i2 : (AX == 1 ? j2 : k2), o1 = AX == 0 ? i1 : (AX == 1 ? j1 : k1);
    const int so = AX == 0 ? si1 : (AX == 1 ? sj1 : sk1), f = AX == 0 ? fi : (AX == 1 ? fj : fk);
    T *line = u2 + ix3(AX == 0 ? 0 : i2 - 1 + fi, AX == 1 ? 0 : j2 - 1 + fj, AX == 2 ? 0 : k2 - 1 + fk, nx2, ny2);
    const long long p0 = 1 + (o2 - 1) * s2, n1 = s2 * (n2 - 1) + 1, s1 = rho * s2;
    const int a = f / rho, r = f % rho;
    T v0, v1;
    const bool changed = anchor_ex(line, p0 + a * s1, n1, s1, chr, o1 + a * so, so, ex, v0);
    if (r == 0) {
      if (changed) line[p0 + a * s1 - 1] = v0;
      return;
    }
    anchor_ex(line, p0 + (a + 1) * s1, n1, s1, chr, o1 + (a + 1) * so, so, ex, v1);
    const double sg = (r * 1.0) / rho;
    line[p0 + f * s2 - 1] = (T)(1 - sg) * v0 + (T)sg * v1;
  });
}

// ---- fourth order with excision: one thread per line -------------------
// x lines through anchor (j,k): in place on u2
template <typename T>
__global__ void k_interp_ex_x(T *u2, const T *chr1, T ex, int nx1, int ny1, int nx2, int ny2,
                              int i1, int j1, int k1, int i2, int j2, int k2, int ni, int nj,
                              int nk, int si1, int sj1, int sk1, int irho, int jrho, int krho) {
  int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= nj * nk) return;
  int jj = q % nj, kk = q / nj;
  int j = j2 + jj * jrho, k = k2 + kk * krho;
  T *line = u2 + ix3(0, j - 1, k - 1, nx2, ny2);
  ChrtCols<T> cl{{chr1 + ix3(0, j1 + sj1 * (j - j2) / jrho - 1, k1 + sk1 * (k - k2) / krho - 1,
                             nx1, ny1), nullptr, nullptr, nullptr}, 1, ex};
  line_vi4q1d_ex<T>(line, i2, nx2, ni, irho, irho, 1, cl, i1, si1, ex);
}

// y lines for every fine i at anchor k; chrt staged in a per-thread column
template <typename T>
__global__ void k_interp_ex_y(T *u2, const T *chr1, T ex, int nx1, int ny1,
                              int nx2, int ny2, int i1, int j1, int k1, int i2, int j2, int k2,
                              int ni, int nj, int nk, int si1, int sj1, int sk1, int irho,
                              int jrho, int krho) {
  const int mi = (ni - 1) * irho + 1;
  int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= mi * nk) return;
  int ii = q % mi, kk = q / mi;
  int i = i2 + ii, k = k2 + kk * krho;
  int ic = i1 + si1 * ((i - i2) / irho), kc = k1 + sk1 * ((k - k2) / krho);
  ChrtCols<T> ch{{chr1 + ix3(ic - 1, 0, kc - 1, nx1, ny1),
                  ((i - i2) % irho != 0) ? chr1 + ix3(ic - 1 + si1, 0, kc - 1, nx1, ny1) : nullptr,
                  nullptr, nullptr},
                 (size_t)nx1, ex};
  T *col = u2 + ix3(i - 1, 0, k - 1, nx2, ny2);
  line_vi4q1d_ex<T>(col, 1 + (j2 - 1) * nx2, nx2 * (ny2 - 1) + 1, nj, jrho, jrho * nx2, nx2, ch, j1, sj1, ex);
}

// z lines for every fine (i,j)
template <typename T>
__global__ void k_interp_ex_z(T *u2, const T *chr1, T ex, int nx1, int ny1,
                              int nz1, int nx2, int ny2, int nz2, int i1, int j1, int k1, int i2,
                              int j2, int k2, int ni, int nj, int nk, int si1, int sj1, int sk1,
                              int irho, int jrho, int krho) {
  const int mi = (ni - 1) * irho + 1, mj = (nj - 1) * jrho + 1;
  int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= mi * mj) return;
  int ii = q % mi, jj = q / mi;
  int i = i2 + ii, j = j2 + jj;
  int ic = i1 + si1 * ((i - i2) / irho), jc = j1 + sj1 * ((j - j2) / jrho);
  bool oi = (i - i2) % irho != 0, oj = (j - j2) % jrho != 0;
  ChrtCols<T> ch{{chr1 + ix3(ic - 1, jc - 1, 0, nx1, ny1),
                  oi ? chr1 + ix3(ic - 1 + si1, jc - 1, 0, nx1, ny1) : nullptr,
                  oj ? chr1 + ix3(ic - 1, jc - 1 + sj1, 0, nx1, ny1) : nullptr,
                  (oi && oj) ? chr1 + ix3(ic - 1 + si1, jc - 1 + sj1, 0, nx1, ny1) : nullptr},
                 (size_t)nx1 * ny1, ex};
  (void)nz1;
  T *col = u2 + ix3(i - 1, j - 1, 0, nx2, ny2);
  const int s2 = nx2 * ny2;
  line_vi4q1d_ex<T>(col, (k2 - 1) * s2 + 1, s2 * (nz2 - 1) + 1, nk, krho, krho * s2, s2, ch, k1, sk1, ex);
}

}  // namespace

extern "C" {

int pmg_dmcopy3d(const double *u1, double *u2, int nx1, int ny1, int nz1, int nx2, int ny2,
                 int nz2, int i1, int j1, int k1, int i2, int j2, int k2, int ni, int nj,
                 int nk, int si1, int sj1, int sk1, int si2, int sj2, int sk2,
                 hipStream_t stream) {
  if (i1 < 1 || (i1 + (ni - 1) * si1) > nx1) return 0;
  if (i2 < 1 || (i2 + (ni - 1) * si2) > nx2) return 0;
  if (j1 < 1 || (j1 + (nj - 1) * sj1) > ny1) return 0;
  if (j2 < 1 || (j2 + (nj - 1) * sj2) > ny2) return 0;
  if (k1 < 1 || (k1 + (nk - 1) * sk1) > nz1) return 0;
  if (k2 < 1 || (k2 + (nk - 1) * sk2) > nz2) return 0;
  if (ni < 1 || nj < 1 || nk < 1) return 0;
  return box_launch(ni, nj, nk, [&](dim3 grid, const BoxPts &b) {
    hipLaunchKernelGGL(k_copy3d<double>, grid, dim3(NT), 0, stream, u1, u2, nx1, ny1,
                       nx2, ny2, i1, j1, k1, i2, j2, k2, ni, nj, nk, si1, sj1, sk1, si2, sj2, sk2, b);
  });
}

static int restrict_launch(int kind, const double *u1, double *u2, int nx1, int ny1, int nz1,
                           int nx2, int ny2, int nz2, int i1, int j1, int k1, int i2, int j2,
                           int k2, int ni, int nj, int nk, int si1, int sj1, int sk1, int si2,
                           int sj2, int sk2, const double *chr1, double ex, int do_ex,
                           hipStream_t stream) {
  if (i1 < 1 || (i1 + (ni - 1) * si1) > nx1) return 0;
  if (i2 < 1 || (i2 + (ni - 1) * si2) > nx2) return 0;
  if (j1 < 1 || (j1 + (nj - 1) * sj1) > ny1) return 0;
  if (j2 < 1 || (j2 + (nj - 1) * sj2) > ny2) return 0;
  if (k1 < 1 || (k1 + (nk - 1) * sk1) > nz1) return 0;
  if (k2 < 1 || (k2 + (nk - 1) * sk2) > nz2) return 0;
  if (ni < 1 || nj < 1 || nk < 1) return 0;
  const bool ex1 = (do_ex == 1);
  if (ex1 && !chr1) return -1;
#define PMG_RL(K, E)                                                                           \
  hipLaunchKernelGGL((k_restrict3d<double, K, E>), grid, dim3(NT), 0, stream, u1, u2,          \
                     chr1, ex, nx1, ny1, nz1, nx2, ny2, i1, j1, k1, i2, j2, k2, ni, nj, nk,   \
                     si1, sj1, sk1, si2, sj2, sk2, b)
  return box_launch(ni, nj, nk, [&](dim3 grid, const BoxPts &b) {
    if (kind == 3) {
      if (ex1) PMG_RL(3, true); else PMG_RL(3, false);
    } else {
      if (ex1) PMG_RL(2, true); else PMG_RL(2, false);
    }
  });
#undef PMG_RL
}

int pmg_dmfwr3d(const double *u1, double *u2, int nx1, int ny1, int nz1, int nx2, int ny2,
                int nz2, int i1, int j1, int k1, int i2, int j2, int k2, int ni, int nj, int nk,
                int si1, int sj1, int sk1, int si2, int sj2, int sk2, const double *chr1,
                double ex, int do_ex, hipStream_t stream) {
  return restrict_launch(3, u1, u2, nx1, ny1, nz1, nx2, ny2, nz2, i1, j1, k1, i2, j2, k2, ni,
                         nj, nk, si1, sj1, sk1, si2, sj2, sk2, chr1, ex, do_ex, stream);
}

int pmg_dmhwr3d(const double *u1, double *u2, int nx1, int ny1, int nz1, int nx2, int ny2,
                int nz2, int i1, int j1, int k1, int i2, int j2, int k2, int ni, int nj, int nk,
                int si1, int sj1, int sk1, int si2, int sj2, int sk2, const double *chr1,
                double ex, int do_ex, hipStream_t stream) {
  return restrict_launch(2, u1, u2, nx1, ny1, nz1, nx2, ny2, nz2, i1, j1, k1, i2, j2, k2, ni,
                         nj, nk, si1, sj1, sk1, si2, sj2, sk2, chr1, ex, do_ex, stream);
}

int pmg_dminterp3d(double *u1, double *u2, int nx1, int ny1, int nz1, int nx2, int ny2, int nz2,
                   int i1, int j1, int k1, int i2, int j2, int k2, int ni, int nj, int nk,
                   int si1, int sj1, int sk1, int irho, int jrho, int krho, int ord,
                   const double *chr1, double ex, int do_ex, hipStream_t stream) {
  (void)u1;
  if (i1 < 1 || (i1 + ni - 1) * si1 > nx1) return 0;
  if (i2 < 1 || (i2 + (ni - 1) * irho) > nx2) return 0;
  if (j1 < 1 || (j1 + nj - 1) * sj1 > ny1) return 0;
  if (j2 < 1 || (j2 + (nj - 1) * jrho) > ny2) return 0;
  if (k1 < 1 || (k1 + nk - 1) * sk1 > nz1) return 0;
  if (k2 < 1 || (k2 + (nk - 1) * krho) > nz2) return 0;
  if (ord != 2 && ord != 4) {
    std::fprintf(stderr, "pmg_dminterp3d: only ord=2,4 are supported (got %d)\n", ord);
    return -2;
  }
  if (ord == 4 && do_ex == 1 && (irho > 20 || jrho > 20 || krho > 20)) {
    std::fprintf(stderr, "pmg_dminterp3d: dvi4q1d_ex expects rho <= 20\n");
    return -2;
  }
  if (do_ex == 1 && (nx1 > 3000 || ny1 > 3000 || nz1 > 3000)) {
    std::fprintf(stderr, "pmg_dminterp3d: nmax too small\n");
    return -2;
  }
  if (ni < 1 || nj < 1 || nk < 1) return 0;
  const int mi = (ni - 1) * irho + 1, mj = (nj - 1) * jrho + 1, mk = (nk - 1) * krho + 1;
  const bool r2 = irho == 2 && jrho == 2 && krho == 2;
  if (ord == 4 && do_ex != 1) {
    int rc = pmg_dmcopy3d(u1, u2, nx1, ny1, nz1, nx2, ny2, nz2, i1, j1, k1, i2, j2, k2, ni, nj, nk, si1, sj1, sk1,
                          irho, jrho, krho, stream);
    if (rc) return rc;
#define PMG_I4(AX, M1, M2)                                                                                         \
  box_launch(mi, M1, M2, [&](dim3 grid, const BoxPts &b) {                                                         \
    hipLaunchKernelGGL((r2 ? k_interp4<AX, true> : k_interp4<AX, false>), grid, dim3(NT), 0, stream, u2, nx2, ny2, \
                       nz2, i2, j2, k2, ni, nj, nk, irho, jrho, krho, b);                                          \
  })
    if ((rc = PMG_I4(0, nj, nk)) || (nj == 1 && nk == 1)) return rc;
    if ((rc = PMG_I4(1, mj, nk)) || nk == 1) return rc;
    return PMG_I4(2, mj, mk);
#undef PMG_I4
  }
  if (do_ex != 1) {
    return box_launch(mi, mj, mk, [&](dim3 grid, const BoxPts &b) {
      hipLaunchKernelGGL((r2 ? k_interp3d<double, true> : k_interp3d<double, false>), grid, dim3(NT), 0, stream, u1, u2,
                         nx1, ny1, nx2, ny2, i1, j1, k1, i2, j2, k2, ni, nj, nk, si1, sj1, sk1, irho, jrho, krho, b);
    });
  }
  if (!chr1) return -1;
  // common points, then the three line phases in place on u2
  int rc = pmg_dmcopy3d(u1, u2, nx1, ny1, nz1, nx2, ny2, nz2, i1, j1, k1, i2, j2, k2, ni, nj, nk,
                        si1, sj1, sk1, irho, jrho, krho, stream);
  if (rc) return rc;
  if (ord == 2) {
#define PMG_IX2(AX, M1, M2)                                                                                            \
  box_launch(mi, M1, M2, [&](dim3 grid, const BoxPts &b) {                                                             \
    hipLaunchKernelGGL((r2 ? k_interp_ex2<double, AX, true> : k_interp_ex2<double, AX, false>), grid, dim3(NT), 0,    \
                       stream, u2, chr1, ex, nx1, ny1, nx2, ny2, nz2, i1, j1, k1, i2, j2, k2, ni, nj, nk, si1, sj1,   \
                       sk1, irho, jrho, krho, b);                                                                      \
  })
    if ((rc = PMG_IX2(0, nj, nk)) || (nj == 1 && nk == 1)) return rc;
    if ((rc = PMG_IX2(1, mj, nk)) || nk == 1) return rc;
    return PMG_IX2(2, mj, mk);
#undef PMG_IX2
  }
  hipLaunchKernelGGL(k_interp_ex_x<double>, dim3((nj * nk + 63) / 64), dim3(64), 0, stream, u2,
                     chr1, ex, nx1, ny1, nx2, ny2, i1, j1, k1, i2, j2, k2, ni, nj, nk, si1, sj1,
                     sk1, irho, jrho, krho);
  PMG_HOST_CHECK(hipGetLastError());
  if (nj == 1 && nk == 1) return 0;
  hipLaunchKernelGGL(k_interp_ex_y<double>, dim3((mi * nk + 63) / 64), dim3(64), 0, stream, u2,
                     chr1, ex, nx1, ny1, nx2, ny2, i1, j1, k1, i2, j2, k2, ni, nj, nk,
                     si1, sj1, sk1, irho, jrho, krho);
  PMG_HOST_CHECK(hipGetLastError());
  if (nk == 1) return 0;
  hipLaunchKernelGGL(k_interp_ex_z<double>, dim3((mi * mj + 63) / 64), dim3(64), 0, stream, u2,
                     chr1, ex, nx1, ny1, nz1, nx2, ny2, nz2, i1, j1, k1, i2, j2, k2,
                     ni, nj, nk, si1, sj1, sk1, irho, jrho, krho);
  PMG_HOST_CHECK(hipGetLastError());
  return 0;
}

}  // extern "C"
