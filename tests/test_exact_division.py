"""div_by of csrc/routing.hip (a quotient from a shared reciprocal) on the CPU: the source's own
text, compiled with g++, equals the fp32 division bit for bit over the range that its callers
check: |x| >= 2^-60 or x = 0, 2^-40 <= d <= 2^20, |x / d| at most about 1 (a component by its
norm, an exponential by a sum of at least 1)."""
import re
import shutil
import subprocess

import pytest

MAIN = r"""
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <random>
#define __device__
#define __forceinline__ inline
using std::fmaf;
%s
static float bits(uint32_t u) { float f; memcpy(&f, &u, 4); return f; }
static long bad = 0, n = 0;
static void one(float x, float d) {
  const float r = 1.f / d;
  ++n;
  if (div_by(x, d, r) != x / d && bad++ < 5) printf("%%a / %%a\n", x, d);
}
int main() {
  std::mt19937_64 g(1);
  const uint32_t edge[] = {0, 1, 2, 3, 0x7fffff, 0x7ffffe, 0x400000, 0x3fffff, 0x400001, 0x2aaaaa, 0x555555};
  for (int e = -40; e <= 20; ++e) {
    for (uint32_t md : edge) {
      if (e == 20 && md) continue;
      const float d = bits(uint32_t(e + 127) << 23 | md);
      one(0.f, d);
      one(d, d);
      for (int k = e; k >= -60; k -= k > e - 4 || k < -56 ? 1 : 7)
        for (uint32_t mx : edge) {
          one(bits(uint32_t(k + 127) << 23 | mx), d);
          one(-bits(uint32_t(k + 127) << 23 | mx), d);
        }
    }
    for (int i = 0; i < 100000; ++i) {
      const uint64_t u = g();
      const float d = e == 20 ? 0x1p20f : bits(uint32_t(e + 127) << 23 | uint32_t(u & 0x7fffff));
      const int k = -60 + int((u >> 48) %% uint64_t(e + 61));
      one(bits(uint32_t(k + 127) << 23 | uint32_t((u >> 23) & 0x7fffff)), d);
    }
  }
  printf("%%ld of %%ld\n", bad, n);
  return bad != 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host compiler")
def test_div_by_is_the_division(fsi, tmp_path):
    from pathlib import Path

    src = (Path(fsi.__file__).parent / "csrc" / "routing.hip").read_text()
    text = re.search(r"__device__ __forceinline__ float div_by\(.*?\n}\n", src, re.S).group(0)
    (tmp_path / "d.cpp").write_text(MAIN % text)
    subprocess.run(["g++", "-O2", "-ffp-contract=off", "-o", str(tmp_path / "d"), str(tmp_path / "d.cpp")], check=True)
    out = subprocess.run([str(tmp_path / "d")], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0, out.stdout
