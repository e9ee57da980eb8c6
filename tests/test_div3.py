"""The three quotients by the squared spacings (div3 in csrc/pmg_div.h, compiled
here for the host): the division-free form while the first quotients and the
inverses stay in their exponent ranges, the division otherwise.  Both
precisions, over random spacings and dividends through the guards' edges,
zeros, subnormals, infinities and NaN on any of the three axes, compared with
the division bit for bit."""
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "pamr_amrd_amd" / "csrc"

SRC = r"""
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <limits>
#include "pmg_div.h"
static uint64_t s = 0x9E3779B97F4A7C15ull;
static uint64_t next() {
  uint64_t z = (s += 0x9E3779B97F4A7C15ull);
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}
template <typename T> struct Sp { T dx2, dy2, dz2, idx2, idy2, idz2; };
template <typename T> struct By : Sp<T> { using divides = void; };
template <typename T> static T any(int e) {  // random significand, exponent in [-e, e)
  return (T)std::ldexp(1 + (double)(next() >> 12) * 0x1p-52, (int)(next() % (2 * e)) - e);
}
// se, ae: exponents of the spacings and of the dividends; edge: also quotients
// just inside and outside 2^+-edge, the guard's line
template <typename T> static long run(int se, int ae, int edge, long n) {
  typedef std::numeric_limits<T> L;
  const T special[] = {0, (T)-0.0, L::infinity(), -L::infinity(), L::quiet_NaN(), L::denorm_min(), L::min(), L::max()};
  long bad = 0;
  for (long t = 0; t < n; t++) {
    T d[3], a[3], q[3];
    for (int k = 0; k < 3; k++) {
      d[k] = any<T>(se);
      d[k] = d[k] * d[k];
      a[k] = any<T>(ae);
      if (t % 4 == 0) a[k] = (T)((double)d[k] * std::ldexp(1 + (double)(next() >> 12) * 0x1p-52, (next() & 1 ? edge : -edge) - (int)(next() % 2)));
      if (next() & 1) a[k] = -a[k];
    }
    if (t % 8 == 1) a[next() % 3] = special[next() % 8];
    if (t % 32 == 2) d[next() % 3] = special[next() % 8];
    const Sp<T> sp{d[0], d[1], d[2], 1 / d[0], 1 / d[1], 1 / d[2]};
    for (int k = 0; k < 3; k++) q[k] = a[k];
    pmg::div3<T, false>(q[0], q[1], q[2], sp);
    T e[3] = {a[0], a[1], a[2]};
    pmg::div3<T, false>(e[0], e[1], e[2], By<T>{sp});
    for (int k = 0; k < 3; k++) {
      const T x = a[k] / d[k];
      if (!(std::isnan(x) && std::isnan(q[k])) && std::memcmp(&x, &q[k], sizeof x)) bad++;
      if (!(std::isnan(x) && std::isnan(e[k])) && std::memcmp(&x, &e[k], sizeof x)) bad++;
    }
  }
  return bad;
}
int main() {
  // everyday spacings and values, then the whole exponent range
  std::printf("%ld %ld %ld %ld\n", run<double>(12, 60, 600, 8000000), run<double>(150, 1070, 600, 6000000),
              run<float>(12, 40, 60, 8000000), run<float>(30, 146, 60, 6000000));
}
"""


def build(tmp_path, src, csrc):
    (tmp_path / "t.cpp").write_text(src)
    exe = str(tmp_path / "t")
    for extra in (["-mfma"], []):
        r = subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", *extra, f"-I{csrc}", str(tmp_path / "t.cpp"),
                            "-o", exe], capture_output=True, text=True)
        if r.returncode == 0:
            return exe
    if "g++" in r.stderr and "not found" in r.stderr:
        pytest.skip("no C++ compiler")
    raise AssertionError(r.stderr[-2000:])


def test_div3_equals_division(tmp_path):
    exe = build(tmp_path, SRC, CSRC)
    out = subprocess.run([exe], capture_output=True, text=True, check=True).stdout.split()
    assert out == ["0"] * 4, out
