"""The kinematics' square root msq (gra_device.h), compiled for the host with a seed of 24
bits in place of the hardware's: sqrt's bits over the range that its comment states, 0 for
what is not positive, Inf for Inf. And what Inf decides: kinematics whose squares overflow
are refused, as by the oracle, in both phase-space classes."""
import os
import subprocess

import numpy as np
import pytest

from conftest import ROOT

HIP = r"""
#pragma once
#include <cmath>
#include <cstdint>
#include <cstring>
#define __device__
#define __forceinline__ inline
inline uint32_t __umulhi(uint32_t a, uint32_t b) { return (uint64_t)a * b >> 32; }
inline double __builtin_amdgcn_rsq(double x) {
  int e;
  const double m = std::frexp(1.0 / std::sqrt(x), &e);
  return std::ldexp(std::floor(m * (1 << 24)) / (1 << 24), e);
}
// the quotient q of num / den with the division's special cases
inline double __builtin_amdgcn_div_fixup(double q, double den, double num) {
  return std::isinf(num) || num == 0.0 || std::isnan(num) ? num / den : q;
}
using std::isinf;
using std::isnan;
"""

SOURCE = r"""
#include <cstdio>
#include <limits>
#include <random>
#include "gra_device.h"
static long bad = 0;
static void check(double x, double want) {
  const double got = msq(x);
  if (std::memcmp(&got, &want, sizeof got) && ++bad < 9)
    std::printf("msq(%.17g) = %.17g, not %.17g\n", x, got, want);
}
int main() {
  const double inf = std::numeric_limits<double>::infinity();
  check(inf, inf);
  check(std::numeric_limits<double>::max(), std::sqrt(std::numeric_limits<double>::max()));
  for (double x : {0.0, -0.0, -5e-324, -1.0, -1e308, -inf, std::nan("")}) check(x, 0.0);
  std::mt19937_64 r(3);
  std::uniform_real_distribution<double> half(1.0, 2.0);
  std::uniform_int_distribution<int> ex(-900, 900);
  for (int i = 0; i < 2000000; ++i) {
    const double x = std::ldexp(half(r), ex(r));
    check(x, std::sqrt(x));
    const double q = std::ldexp((double)(float)half(r), ex(r) / 2);  // exact squares and neighbours
    check(q * q, q);
    check(std::nextafter(q * q, inf), std::sqrt(std::nextafter(q * q, inf)));
  }
  for (double x : {5e-324, 1e-320, 2.2250738585072014e-308, 9e-301}) {
    const double v = msq(x);
    if (!(v >= 0.0 && v <= 1e-150) && ++bad) std::printf("msq(%g) = %g\n", x, v);
  }
  std::printf("bad %ld\n", bad);
  return bad != 0;
}
"""


def test_msq_equals_sqrt(tmp_path):
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text(HIP)
    src, exe = tmp_path / "m.cpp", tmp_path / "m"
    src.write_text(SOURCE)
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-w", "-I", str(tmp_path), "-I",
                    os.path.join(ROOT, "include"), "-I", os.path.join(ROOT, "graniitti_amd", "csrc"),
                    str(src), "-o", str(exe)], check=True)
    p = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert p.returncode == 0, p.stdout


@pytest.mark.gpu
@pytest.mark.parametrize("preset,pt_max", [(1, 1e200), (5, 1e200)])
def test_overflowing_kinematics_are_refused(preset, pt_max):
    from graniitti_amd import abi
    from graniitti_amd.process import MContinuum
    import oracle_lib as ol

    cfg = abi.cfg_default(preset)
    cfg.screening, cfg.amp_precision = 0, abi.GRA_AMP_FP64
    cfg.fwd_pt_max = pt_max
    print(f"case: preset {preset}, forward pT up to {pt_max:g}", flush=True)
    u = np.random.default_rng(17).random((4096, cfg.dim))
    with MContinuum(cfg) as P:
        Wg, _, fg = P.eval(u)
    Wo, _, fo = ol.OracleRun(cfg).eval(u)
    assert np.array_equal(fg, fo)
    assert np.array_equal(Wg == 0, Wo == 0)
