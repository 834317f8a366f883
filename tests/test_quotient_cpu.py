"""div_by, the quotient of the contact law by a shared reciprocal, against the
division it stands for, bit for bit, on the CPU: the numerators whose quotient
lies nearest to the middle between two doubles (where a rounding error shows
first), numerators just below the divisor and just below a power of two,
random operands over the range of exponents it is stated for, and the ends of
that range."""
import os
import subprocess

from _paths import PKG

PROGRAM = r"""
#include <hip/hip_runtime.h>
#include <cstdio>
#include <cstring>
#include <cstdint>
#include <cmath>
#include <random>
#include "mfixdem.h"
#include "device_physics.hpp"
typedef unsigned __int128 u128;
using mfixdem::div_by;
static long tested = 0, wrong = 0;
static void check(double a, double b) {
  const double got = div_by(a, b, 1.0 / b), want = a / b;
  tested++;
  if (std::memcmp(&got, &want, 8) != 0 && wrong++ < 10) std::printf("%a / %a: %a, not %a\n", a, b, got, want);
}
// 1 / a modulo an odd m
static uint64_t inverse(uint64_t a, uint64_t m) {
  __int128 t = 0, nt = 1, r = m, nr = a % m;
  while (nr) {
    const __int128 q = r / nr;
    __int128 x = t - q * nt; t = nt; nt = x;
    x = r - q * nr; r = nr; nr = x;
  }
  return (uint64_t)(t < 0 ? t + m : t);
}
int main() {
  std::mt19937_64 g(20240611);
  const uint64_t lo = 1ull << 52, hi = 1ull << 53;
  // 2^(e+1) A = (2 q + 1) B + t with a small t: A / B is t / B from the middle
  for (int k = 0; k < 20000; k++) {
    uint64_t B = lo + (g() % lo | 1);
    if (k % 3 == 0) B = hi - 1 - 2 * (g() % 4096);
    if (k % 3 == 1) B = lo + 1 + 2 * (g() % 4096);
    for (int e = 52; e <= 53; e++) {
      u128 x = 1;
      for (int i = 0; i <= e; i++) x = x * 2 % B;
      const uint64_t inv = inverse((uint64_t)x, B);
      for (int t = -8; t <= 8; t++) {
        const uint64_t tm = t >= 0 ? (uint64_t)t : B - (uint64_t)(-t);
        for (uint64_t A = (uint64_t)((u128)tm * inv % B), n = 0; n < 2; n++, A += B)
          if (A >= lo && A < hi && (e == 53) == (A < B)) check((double)A, (double)B);
      }
    }
    for (int j = 0; j < 16; j++) {
      if (B - 1 - j >= lo) check((double)(B - 1 - j), (double)B);
      check((double)(hi - 1 - j), (double)B);
    }
  }
  for (int i = 1; i <= 700; i++)
    for (int j = 1; j <= 700; j++) check((double)(hi - j), (double)(hi - i));
  // exponents: lengths and squares of lengths of anything from an atom to a star
  for (int k = 0; k < 3000000; k++) {
    const double a = std::ldexp((double)(lo + g() % lo), (int)(g() % 1800) - 52 - 900);
    const double b = std::ldexp((double)(lo + g() % lo), (int)(g() % 200) - 52 - 100);
    if (std::fabs(a) > 1e-290 && std::isfinite(a / b) && std::fabs(a / b) > 1e-300)
      check(g() & 1 ? a : -a, b);
  }
  for (double b : {1.0, 3.0, 1e-3, 0x1.fffffffffffffp-10}) {
    check(0.0, b);
    for (double a = 1.0e-290; a < 1.1e-290; a = std::nextafter(a * 1.0001, 1.0)) check(a, b);
    // outside: an error of the last bit at most, and a zero stays a zero
    for (double a = 1e-290; a > 1e-322; a *= 0.9) {
      const double got = div_by(a, b, 1.0 / b), want = a / b;
      tested++;
      if (std::fabs(got - want) > std::fmax(std::fabs(want) * 0x1p-52, 5e-324)) wrong++;
    }
    tested++;
    if (div_by(-0.0, b, 1.0 / b) != 0.0) wrong++;
  }
  std::printf("%ld %ld\n", tested, wrong);
  return 0;
}
"""


def test_div_by_rounds_as_the_division_does(tmp_path):
    src, exe = tmp_path / "quotient.hip", tmp_path / "quotient"
    src.write_text(PROGRAM)
    csrc = os.path.join(PKG, "csrc")
    include = os.path.join(os.path.dirname(PKG), "include")
    subprocess.run([os.environ.get("HIPCC", "/opt/rocm/bin/hipcc"), "--offload-host-only",
                    "-O2", "-std=c++17", "-ffp-contract=off", "-mfma", f"-I{csrc}", f"-I{include}",
                    "-o", str(exe), str(src)], check=True, capture_output=True, timeout=300)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True, timeout=300).stdout
    tested, wrong = map(int, out.split("\n")[-2].split())
    assert tested > 3_000_000
    assert wrong == 0, out
