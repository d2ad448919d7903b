"""The arithmetic 15-digit round trip of table values (gra_round15.h) against printf and
strtod, bit for bit: every decade and the doubles beside its powers of ten, exact ties,
and the values that take the text path."""
import os
import subprocess

from conftest import ROOT

SOURCE = r"""
#include <cstdint>
#include <cstring>
#include <random>
#include "gra_round15.h"
using namespace gra_hip;
static long bad = 0;
static void check(double v) {
  const double a = round15(v), b = round15_text(v);
  if (std::memcmp(&a, &b, sizeof a) && ++bad < 5) std::printf("%.17g: %.17g, %.17g\n", v, a, b);
}
int main() {
  std::mt19937_64 r(7);
  std::uniform_real_distribution<double> decade(-9.0, 17.0), half(0.0, 1.0);
  for (int i = 0; i < 300000; ++i) check((i & 1 ? 1 : -1) * std::pow(10.0, decade(r)) * (1 + half(r)));
  for (int k = -9; k < 17; ++k)
    for (int j = -30; j <= 30; ++j) {
      const double p = std::pow(10.0, k);
      int64_t bits;
      std::memcpy(&bits, &p, 8);
      bits += j;
      double v;
      std::memcpy(&v, &bits, 8);
      check(v);
    }
  for (int i = 0; i < 100000; ++i) {
    const double m = (double)(100000000000000ull + r() % 900000000000000ull) + 0.5;
    check(m);
    check(m / (1 << (r() % 6)));
  }
  for (double v : {0.0, -0.0, 1e-7, 1e15, 999999999999999.5, 99999999999999.95, HUGE_VAL}) check(v);
  std::printf("bad %ld\n", bad);
  return bad != 0;
}
"""


def test_round15_equals_the_text_round_trip(tmp_path):
    src, exe = tmp_path / "r.cpp", tmp_path / "r"
    src.write_text(SOURCE)
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-I",
                    os.path.join(ROOT, "graniitti_amd", "csrc"), str(src), "-o", str(exe)],
                   check=True)
    p = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert p.returncode == 0, p.stdout
