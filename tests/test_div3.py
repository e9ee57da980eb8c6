"""The three quotients by the squared spacings (div3 in csrc/pmg_ops.h): the
division-free form while the first quotients and the inverses stay in their
exponent ranges, the division otherwise -- the same operations run on the host
in both precisions, over random spacings and dividends through the guards'
edges, zeros, subnormals, infinities and NaN, and compared with the division
bit for bit."""
import subprocess

import pytest

SRC = r"""
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <string.h>
static uint64_t s = 0x9E3779B97F4A7C15ull;
static uint64_t next(void) {
  uint64_t z = (s += 0x9E3779B97F4A7C15ull);
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}
#define DEF(T, U, FMA, BIAS, MAN, EQ, EI, N)                                         \
  static int mid##N(T v, int e) {                                                   \
    U u; memcpy(&u, &v, sizeof u);                                                  \
    u &= (U)-1 >> 1;                                                                \
    return (U)(u - ((U)(BIAS - e) << MAN)) < ((U)(2 * e) << MAN);                   \
  }                                                                                 \
  static T quo##N(T a, T b) {                                                       \
    T y = (T)1 / b;                                                                 \
    T q0 = a * y;                                                                   \
    if (!(mid##N(y, EI) && mid##N(q0, EQ))) return a / b;                           \
    T r0 = FMA(-b, q0, a), q1 = FMA(r0, y, q0), r1 = FMA(-b, q1, a);                \
    return FMA(r1, y, q1);                                                          \
  }                                                                                 \
  static long run##N(int be, int ae, long n) {                                      \
    long bad = 0;                                                                   \
    T sp[] = {0, -0.0, INFINITY, -INFINITY, NAN, ldexp(1, -BIAS - MAN + 1)};        \
    for (long t = 0; t < n; t++) {                                                  \
      T b = (T)ldexp(1 + (double)(next() >> 12) * 0x1p-52, (int)(next() % (2 * be)) - be); \
      b = b * b;                                                                    \
      T a = (T)ldexp(1 + (double)(next() >> 12) * 0x1p-52, (int)(next() % (2 * ae)) - ae); \
      if (next() & 1) a = -a;                                                       \
      if (t % 16 == 0) a = sp[next() % 6];                                          \
      T x = a / b, z = quo##N(a, b);                                                \
      if (!(isnan(x) && isnan(z)) && memcmp(&x, &z, sizeof x)) bad++;               \
    }                                                                               \
    return bad;                                                                     \
  }
DEF(double, uint64_t, fma, 1023, 52, 600, 200, d)
DEF(float, uint32_t, fmaf, 127, 23, 60, 30, f)
int main(void) {
  /* everyday spacings and values, then the whole exponent range */
  printf("%ld %ld %ld %ld\n", rund(12, 60, 20000000), rund(150, 1000, 10000000), runf(12, 40, 20000000),
         runf(20, 120, 10000000));
  return 0;
}
"""


def test_div3_equals_division(tmp_path):
    (tmp_path / "t.c").write_text(SRC)
    exe = str(tmp_path / "t")
    for extra in (["-mfma"], []):
        r = subprocess.run(["gcc", "-O2", "-std=gnu99", "-ffp-contract=off", *extra, str(tmp_path / "t.c"), "-o", exe,
                            "-lm"], capture_output=True, text=True)
        if r.returncode == 0:
            break
    else:
        pytest.skip("no C compiler: " + r.stderr[-300:])
    out = subprocess.run([exe], capture_output=True, text=True, check=True).stdout.split()
    assert out == ["0"] * 4, out
