"""The device arithmetic that stands in for divisions, compiled for the host from the header the kernels use
(ppk_kernel_args.h). fast_div by a fast_divisor equals integer division for dividends below 2^31: sampled at up to
5000 multiples of each of some 7400 divisors, two to each side, and at the 3000 largest dividends. row_scale equals
the IEEE division by 127 with the scale's floor: for every mantissa at exponents over the whole range (around the
floor one by one), and for every 4099th of all finite non-negative floats. (All 2^31 agree; that takes half a
minute, so the test samples.)"""
from __future__ import annotations

import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include <cstdio>
#include "ppk_kernel_args.h"
using ppk::fast_div;
static int check(uint32_t d) {
  const ppk::FastDiv f = ppk::fast_divisor(d);
  const uint64_t top = 0x7fffffffu, most = top / d;
  for (uint64_t step = most / 5000 + 1, k = 0; k <= most; k += step)
    for (int64_t e = -2; e <= 2; ++e) {
      const int64_t x = int64_t(k * d) + e;
      if (x < 0 || x > int64_t(top)) continue;
      if (fast_div(uint32_t(x), f) != uint32_t(x) / d) { std::printf("%lld / %u\n", (long long)x, d); return 1; }
    }
  for (uint32_t x = 0x7fffffffu; x > 0x7fffffffu - 3000; --x)
    if (fast_div(x, f) != x / d) { std::printf("%u / %u\n", x, d); return 1; }
  return 0;
}
int main() {
  for (uint32_t d = 1; d <= 4200; ++d) if (check(d)) return 1;
  for (uint32_t s = 0; s < 31; ++s)
    for (int e = -3; e <= 3; ++e) {
      const int64_t d = (int64_t(1) << s) + e;
      if (d >= 1 && d <= 0x7fffffff && check(uint32_t(d))) return 1;
    }
  for (uint32_t d = 4201, i = 0; i < 3000; ++i, d = d * 1664525u + 1013904223u)
    if (check((d >> 1) | 1u)) return 1;
  return 0;
}
"""


ROW_SCALE = r"""
#include <cstdio>
#include <cstring>
#include <initializer_list>
#include "ppk_kernel_args.h"
static bool wrong(uint32_t b) {
  float x;
  std::memcpy(&x, &b, 4);
  const float q = x / 127.0f, want = q > 1e-12f ? q : 1e-12f;
  return ppk::row_scale(x) != want;
}
int main() {
  uint32_t bad = 0;
  for (uint32_t e : {0u, 1u, 60u, 91u, 92u, 93u, 94u, 95u, 126u, 127u, 133u, 134u, 200u, 253u, 254u})
    for (uint32_t m = 0; m < 1u << 23; ++m) bad += wrong(e << 23 | m);
  for (uint32_t b = 0; b < 0x7f800000u; b += 4099) bad += wrong(b);
  return bad != 0;
}
"""


def run(tmp_path, source, *flags):
    src, exe = tmp_path / "check.cpp", str(tmp_path / "check")
    src.write_text(source)
    subprocess.run(["g++", "-O3", "-std=c++17", *flags, "-I", os.path.join(ROOT, "pop2-bezier_amd", "csrc"), str(src),
                    "-o", exe], check=True)
    got = subprocess.run([exe], capture_output=True, text=True)
    assert got.returncode == 0, got.stdout


def test_fast_divisor(tmp_path):
    run(tmp_path, SOURCE)


def test_row_scale_is_the_division(tmp_path):
    with open("/proc/cpuinfo") as f:
        if " fma " not in f.read():
            pytest.skip("no fused multiply-add on this CPU: the library's own takes minutes for 2^31 values")
    run(tmp_path, ROW_SCALE, "-mfma", "-ffp-contract=off")
