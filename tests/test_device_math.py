"""Reciprocal, quotient and square root of the device code on the CPU: rd_physics.hpp
compiled for the host with the two hardware estimates replaced by exact values off by
up to their documented 2^-22. What the code does with an estimate then shows at the
worst estimates, whichever of them a card returns.

Bounds: an IEEE operation is within 0.5 ulp of the exact value. recip, the quotient and
the square root end in one rounding of a value whose own error is at most a few 2^-60
relative: 0.5 ulp + 2^-7. 1/sqrt adds y e (0.5 + 0.375 e) to the estimate, with e
rounded from x y (half an ulp of 1, half of which reaches the result) and the sum
rounded once: 1 ulp + 2^-7."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")

SOURCE = r"""
#include <cmath>
#include <cstdio>
#include <random>
double est_rcp(double);
double est_rsq(double);
#define __builtin_amdgcn_rcp est_rcp
#define __builtin_amdgcn_rsq est_rsq
#include "rd_physics.hpp"
static double off;
static __float128 root(__float128 x)
{
  __float128 s = std::sqrt(static_cast<double>(x));
  for (int i = 0; i < 4; ++i) s = (s + x / s) / 2;
  return s;
}
double est_rcp(double x) { return static_cast<double>((1 + static_cast<__float128>(off)) / x); }
double est_rsq(double x) { return static_cast<double>((1 + static_cast<__float128>(off)) / root(x)); }
static double ulps(double v, __float128 ref)
{
  const double r = static_cast<double>(ref);
  return std::fabs(static_cast<double>((v - ref) / (std::nextafter(r, INFINITY) - r)));
}
int main()
{
  std::mt19937_64 g(1);
  std::uniform_real_distribution<double> U(1.0, 4.0), E(-0x1p-22, 0x1p-22);
  double worst[4] = {0, 0, 0, 0};
  for (int i = 0; i < 300000; ++i) {
    const double x = std::ldexp(U(g), static_cast<int>(g() % 400) - 200);
    off = i % 3 == 0 ? 0x1p-22 : (i % 3 == 1 ? -0x1p-22 : E(g));
    double s, rs;
    pdrd::sqrt_rsqrt(x, s, rs);
    worst[0] = std::fmax(worst[0], ulps(pdrd::recip(x), 1 / static_cast<__float128>(x)));
    worst[1] = std::fmax(worst[1], ulps(s, root(x)));
    worst[2] = std::fmax(worst[2], ulps(rs, 1 / root(x)));
    const double n = U(g);
    worst[3] = std::fmax(worst[3], ulps(pdrd::quotient(n, x), n / static_cast<__float128>(x)));
  }
  std::printf("%.6f %.6f %.6f %.6f\n", worst[0], worst[1], worst[2], worst[3]);
}
"""


@pytest.fixture(scope="module")
def worst(tmp_path_factory):
    d = tmp_path_factory.mktemp("math")
    src, exe = d / "math.cpp", d / "math"
    src.write_text(SOURCE)
    subprocess.run(["g++", "-O2", "-std=gnu++17", "-mfma", "-ffp-contract=off", "-w", "-D__HIP_PLATFORM_AMD__",
                    f"-I{ROCM}/include", f"-I{ROOT}/pdekit_amd/csrc/hip", "-o", str(exe), str(src)], check=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.split()
    return dict(zip(("recip", "sqrt", "rsqrt", "quotient"), map(float, out)))


@pytest.mark.parametrize("name,bound", [("recip", 0.5), ("sqrt", 0.5), ("rsqrt", 1.0), ("quotient", 0.5)])
def test_within_rounding(worst, name, bound):
    assert worst[name] <= bound + 2.0 ** -7
