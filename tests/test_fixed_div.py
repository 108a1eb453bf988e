"""The two-operation division by a fixed divisor (csrc/pfs_fixed_div.h):
whatever prove_fixed_div accepts must equal IEEE division for every float
significand (scaling x by a power of two scales both operations exactly),
and keep zeros, infinities and NaN as IEEE division gives them.  CPU only:
the header itself, compiled with g++ -mfma, whose fmaf is the GPU's fused
multiply-add.
"""
from __future__ import annotations

import os
import shutil
import subprocess
import tempfile

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "probabilistic_fluid_simulation_amd", "csrc")
SRC = r"""
#include "pfs_fixed_div.h"
#include <cstdio>
#include <cstdlib>
#include <initializer_list>
#include <cstring>
static uint32_t bits(float f) { uint32_t u; std::memcpy(&u, &f, 4); return u; }
static float d2(float x, const pfs::FixedDiv &d) { const float t = x * d.lo; return std::fmaf(x, d.hi, t); }
int main(int, char **argv) {
  const int n = std::atoi(argv[1]);
  uint64_t s = 88172645463325252ULL;
  long bad = 0, special = 0; int refused = 0, tried = 0, ints = 0;
  for (int k = 1; k <= 131072; ++k) ints += pfs::prove_fixed_div((float)k).ok;
  for (int t = 0; t < n; ++t) {
    s ^= s << 13; s ^= s >> 7; s ^= s << 17;
    const float b = t % 2 ? (float)(1 + (s >> 20) % 131072) : std::ldexp(1.0f + (float)((s >> 40) & 0x7fffff) * 0x1p-23f, (int)(s % 6));
    const pfs::FixedDiv d = pfs::prove_fixed_div(b);
    if (!d.ok) { ++refused; continue; }
    ++tried;
    #pragma omp parallel for reduction(+:bad)
    for (uint32_t m = 1u << 23; m < 1u << 24; ++m) {
      const float x = (float)m;
      if (bits(d2(x, d)) != bits(x / b) || bits(d2(-x, d)) != bits(-x / b)) ++bad;
    }
    for (float x : {0.0f, -0.0f, INFINITY, -INFINITY, 3.4028235e38f, -3.4028235e38f, 0x1p-96f})
      special += bits(d2(x, d)) != bits(x / b);
    special += !std::isnan(d2(NAN, d));
  }
  int outside = 0;
  for (float b : {0.0f, 0.5f, -1.0f, NAN, INFINITY, 0x1p18f}) outside += pfs::prove_fixed_div(b).ok;
  std::printf("%ld %ld %d %d %d %d\n", bad, special, refused, tried, ints, outside);
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_proven_divisors_divide_exactly():
    with tempfile.TemporaryDirectory() as d:
        src, exe = os.path.join(d, "div.cpp"), os.path.join(d, "div")
        with open(src, "w") as f:
            f.write(SRC)
        subprocess.run(["g++", "-O2", "-std=c++17", "-mfma", "-ffp-contract=off", "-fopenmp",
                        "-I", CSRC, src, "-o", exe], check=True)
        out = subprocess.run([exe, "60"], capture_output=True, text=True, check=True).stdout
    bad, special, refused, tried, ints, outside = (int(t) for t in out.split())
    assert bad == 0 and special == 0
    assert tried >= 40 and refused < 20   # most divisors are proven
    assert ints == 131072                 # every field side up to 2^17 is
    assert outside == 0


SIDES = r"""
#include "pfs_fixed_div.h"
#include <cstdio>
#include <cstring>
#include <initializer_list>
static uint32_t bits(float f) { uint32_t u; std::memcpy(&u, &f, 4); return u; }
int main() {
  long refused = 0, bad = 0;
  #pragma omp parallel for reduction(+:refused) schedule(dynamic, 4096)
  for (int n = 131073; n <= 4159487; ++n) refused += !pfs::side_div((float)n, pfs::prove_fixed_div).ok;
  for (float n : {131072.0f, 131073.0f, 200003.0f, 262144.0f, 1000001.0f, 4159486.0f, 16777213.0f, 16777216.0f}) {
    const pfs::FixedDiv d = pfs::side_div(n, pfs::prove_fixed_div);
    if (!d.ok) { ++bad; continue; }
    #pragma omp parallel for reduction(+:bad)
    for (uint32_t m = 1u << 23; m < 1u << 24; ++m) {
      const float x = (float)m, t = x * d.lo;
      if (bits(std::fmaf(x, d.hi, t)) != bits(x / n)) ++bad;
    }
  }
  int outside = 0;
  for (float n : {16777218.0f, 33554432.0f, INFINITY, NAN}) outside += pfs::side_div(n, pfs::prove_fixed_div).ok;
  std::printf("%ld %ld %d\n", refused, bad, outside);
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_sides_past_2_17_divide_exactly():
    """Field sides above what prove_fixed_div takes: all are proven up to
    4,159,486 (the next is the first that is not), and those tried divide every
    significand exactly."""
    with tempfile.TemporaryDirectory() as d:
        src, exe = os.path.join(d, "side.cpp"), os.path.join(d, "side")
        with open(src, "w") as f:
            f.write(SIDES)
        subprocess.run(["g++", "-O2", "-std=c++17", "-mfma", "-ffp-contract=off", "-fopenmp",
                        "-I", CSRC, src, "-o", exe], check=True)
        out = subprocess.run([exe], capture_output=True, text=True, check=True).stdout
    assert out.split() == ["1", "0", "0"]
