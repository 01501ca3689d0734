"""The kernels' division by a precomputed multiplier (ppk_kernel_args.h fast_divisor) equals integer division
for every dividend below 2^31: exhaustive around multiples of the divisor, where it could first be wrong."""
from __future__ import annotations

import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include <cstdio>
#include "ppk_kernel_args.h"
static uint32_t div(uint32_t x, ppk::FastDiv d) {  // fast_div of ppk_kernels.hip
  const uint32_t q = uint32_t((uint64_t(x) * d.mul) >> 32) >> d.shift;
  return d.mul ? q : x;
}
static int check(uint32_t d) {
  const ppk::FastDiv f = ppk::fast_divisor(d);
  const uint64_t top = 0x7fffffffu, most = top / d;
  for (uint64_t step = most / 5000 + 1, k = 0; k <= most; k += step)
    for (int64_t e = -2; e <= 2; ++e) {
      const int64_t x = int64_t(k * d) + e;
      if (x < 0 || x > int64_t(top)) continue;
      if (div(uint32_t(x), f) != uint32_t(x) / d) { std::printf("%lld / %u\n", (long long)x, d); return 1; }
    }
  for (uint32_t x = 0x7fffffffu; x > 0x7fffffffu - 3000; --x)
    if (div(x, f) != x / d) { std::printf("%u / %u\n", x, d); return 1; }
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


def test_fast_divisor(tmp_path):
    src = tmp_path / "fast_div.cpp"
    src.write_text(SOURCE)
    exe = str(tmp_path / "fast_div")
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", os.path.join(ROOT, "pop2-bezier_amd", "csrc"), str(src), "-o",
                    exe], check=True)
    got = subprocess.run([exe], capture_output=True, text=True)
    assert got.returncode == 0, got.stdout
