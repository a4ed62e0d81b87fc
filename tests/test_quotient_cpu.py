"""The kernels' quotients from a reciprocal, q = a y with y = RN(1/b) and one (for
b = 3) or two corrections q + (a - b q) y, against a / b: the same bits for random
operands of every mantissa, for divisors whose reciprocal rounds worst, and down
to where the remainder a - b q leaves the normal range."""
import subprocess


SRC = r"""
#include <cmath>
#include <cstdio>
#include <cstdint>
#include <limits>
template <typename R> R correct(R q, R a, R b, R y) { return std::fma(std::fma(-q, b, a), y, q); }
template <typename R> R quot2(R a, R b, R y) { return correct(correct(a * y, a, b, y), a, b, y); }
template <typename R> R quot1(R a, R b, R y) { return correct(a * y, a, b, y); }
static uint64_t s = 88172645463325252ull;
static double u() { s ^= s << 13; s ^= s >> 7; s ^= s << 17; return (s >> 11) * 0x1p-53; }
template <typename R> long run(long n) {
  const int p = std::numeric_limits<R>::digits, low = std::numeric_limits<R>::min_exponent + 2 * p;
  long bad = 0;
  for (long k = 0; k < n; k++) {
    R a = (R)((1 + u()) * (u() < 0.5 ? -1 : 1)), b = (R)(1 + u());
    if (k % 8 == 0) b = R(2) - std::ldexp(R(1 + k / 8 % 64), 1 - p);  // mantissas of (nearly) all ones
    if (k % 8 == 1) b = R(1) + std::ldexp(R(k / 8 % 64), 1 - p);
    a = std::ldexp(a, low + (int)(u() * (40 - low)));
    b = std::ldexp(b, -20 + (int)(u() * 24));
    const R y = R(1) / b, q = a / b;
    bad += quot2(a, b, y) != q;
    bad += quot1(a, R(3), R(1) / R(3)) != a / R(3);
  }
  return bad;
}
int main() { std::printf("%ld %ld\n", run<float>(4000000), run<double>(4000000)); }
"""


def test_quotients(tmp_path):
    src, exe = tmp_path / "q.cpp", str(tmp_path / "q")
    src.write_text(SRC)
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-mfma", str(src), "-o", exe], check=True)
    out = subprocess.run([exe], check=True, capture_output=True, text=True).stdout.split()
    assert out == ["0", "0"], out
