// pmg_div.h -- quotients by the squared spacings and the Jacobian without a
// division.  Compiles for the host too, where the same code is compared with the
// division bit for bit.
#pragma once
#include <type_traits>

#if defined(__HIPCC__)
#define PMG_DIV_FN __host__ __device__ __forceinline__
#else
#define PMG_DIV_FN inline
#endif

namespace pmg {

// a / b rounded to nearest from y = RN(1/b), without a division: q0 =
// RN(a y) is within 2 ulps of a/b; one correction with the exact remainder
// (an FMA), q1 = RN(q0 + (a - b q0) y), is faithful; a second one with a
// faithful quotient and a correctly rounded reciprocal returns RN(a/b)
// (P. Markstein, IA-64 and Elementary Functions, 2000, Thm. 8.10; J.-M.
// Muller et al., Handbook of Floating-Point Arithmetic, 2018, Sec. 4.7),
// absent underflow and overflow.  5 FP64 operations against the ~12 of the
// IEEE division sequence.
PMG_DIV_FN double div_rn(double a, double b, double y) {
  const double q0 = a * y;
  const double r0 = __builtin_fma(-b, q0, a);
  const double q1 = __builtin_fma(r0, y, q0);
  const double r1 = __builtin_fma(-b, q1, a);
  return __builtin_fma(r1, y, q1);
}

PMG_DIV_FN float div_rn(float a, float b, float y) {
  const float q0 = a * y;
  const float r0 = __builtin_fmaf(-b, q0, a);
  const float q1 = __builtin_fmaf(r0, y, q0);
  const float r1 = __builtin_fmaf(-b, q1, a);
  return __builtin_fmaf(r1, y, q1);
}

// |v| in [2^-E, 2^E): neither zero nor infinite, NaN or subnormal
template <int E>
PMG_DIV_FN bool mid_range(double v) {
  unsigned long long u;
  __builtin_memcpy(&u, &v, 8);
  return ((unsigned)(u >> 32) & 0x7fffffffu) - ((unsigned)(1023 - E) << 20) < ((unsigned)(2 * E) << 20);
}
template <int E>
PMG_DIV_FN bool mid_range(float v) {
  unsigned u;
  __builtin_memcpy(&u, &v, 4);
  return (u & 0x7fffffffu) - ((unsigned)(127 - E) << 23) < ((unsigned)(2 * E) << 23);
}

// x / dx2, y / dy2, z / dz2, rounded as the division rounds.  With spacings
// whose squares are powers of two (P2) the product with the inverse is that
// quotient; otherwise div_rn is, while no intermediate leaves the normal
// range: the first quotient within 2^(+-600) and the inverse within 2^(+-200)
// (FP32: 60 and 30) keep every remainder's last bit above the smallest
// subnormal.  Anything else (zeros, tiny, infinite) takes the division itself.
// 15 FP64 operations for the three instead of about 36: the sweep of a
// 161 x 97 x 129 grid with 1/160 spacing 33 -> 24 us.  The test is a branch,
// though, that waits for all three: where a thread works on one point after
// another with nothing beside it, the divisions overlap better.  A spacing of a
// type with a member type `divides` asks for them (ByDivision in pmg_common.h).
template <typename S, typename = void>
struct divides : std::false_type {};
template <typename S>
struct divides<S, std::void_t<typename S::divides>> : std::true_type {};
template <typename T, bool P2, typename S>
PMG_DIV_FN void div3(T &x, T &y, T &z, const S &sp) {
  if constexpr (P2) {
    x = x * sp.idx2;
    y = y * sp.idy2;
    z = z * sp.idz2;
  } else if constexpr (divides<S>::value) {
    x = x / sp.dx2;
    y = y / sp.dy2;
    z = z / sp.dz2;
  } else {
    constexpr int EQ = std::is_same<T, double>::value ? 600 : 60, EI = std::is_same<T, double>::value ? 200 : 30;
    const bool inv = mid_range<EI>(sp.idx2) && mid_range<EI>(sp.idy2) && mid_range<EI>(sp.idz2);
    if (inv && mid_range<EQ>(x * sp.idx2) && mid_range<EQ>(y * sp.idy2) && mid_range<EQ>(z * sp.idz2)) {
      x = div_rn(x, sp.dx2, sp.idx2);
      y = div_rn(y, sp.dy2, sp.idy2);
      z = div_rn(z, sp.dz2, sp.idz2);
    } else {
      x = x / sp.dx2;
      y = y / sp.dy2;
      z = z / sp.dz2;
    }
  }
}

}  // namespace pmg
