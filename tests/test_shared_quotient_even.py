"""Quotients by a shared reciprocal (marian-dev_amd/csrc/shared_quotient.h) against the division for even divisors, on the CPU."""
import os
import subprocess

from conftest import ROOT

CSRC = os.path.join(ROOT, "marian-dev_amd", "csrc")

PROGRAM = r"""
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <cmath>
#include "shared_quotient.h"
using namespace marian_hip;
static uint32_t inverse(uint32_t x) {   // of an odd number, mod 2^32
  uint32_t y = x;
  for(int i = 0; i < 5; ++i) y *= 2 - x * y;
  return y;
}
int main() {
  // Significands a, s of 24 bits, s = 2^j t with t odd, whose quotient is a rounding edge but for k units of its last place times s:
  // a 2^shift = edge s + k, edge odd, 2^24 < edge < 2^25.  2^j divides k = 2^j k', and edge t + k' = a 2^(shift - j) is even, so k' is odd.
  // The correction errs by less than four units: k of up to 15 units and k' of up to 3 are looked at.
  unsigned long long hard = 0, wrong = 0;
  for(int j = 1; j <= 23; ++j) {
    const int most = 15 >> j > 3 ? 15 >> j : 3;
    for(uint32_t s = 1u << 23; s < 1u << 24; s += 1u << j) {
      const uint32_t t = s >> j;
      if(t % 2 == 0) continue;
      const uint32_t inv = inverse(t);
      for(int shift = 24; shift <= 25; ++shift)
        for(int k = -most; k <= most; ++k) {
          if(k % 2 == 0) continue;
          const uint32_t step = 1u << (shift - j), low = (uint32_t)-(int64_t)k * inv & (step - 1);
          for(uint64_t edge = (1u << 24) + low; edge < 1u << 25; edge += step) {
            if(edge % 2 == 0) continue;   // (where step is 2 or less all are walked)
            const int64_t a = (int64_t)(edge * t + k) >> (shift - j);
            if(a < 1 << 23 || a >= 1 << 24) continue;
            const float got = shared_quotient((float)a, (float)s, 1.0f / (float)s), want = (float)a / (float)s;
            ++hard;
            if(std::memcmp(&got, &want, 4) != 0 && wrong++ < 10) std::printf("%lld / %u: %a, not %a\n", (long long)a, s, got, want);
          }
        }
    }
  }
  std::printf("%llu hard pairs\n", hard);
  return wrong != 0 || hard < 100000000;
}
"""


def test_even_divisors(tmp_path):
    (tmp_path / "e.cpp").write_text(PROGRAM)
    exe = str(tmp_path / "e")
    subprocess.check_call(["g++", "-O2", "-mfma", "-ffp-contract=off", "-std=c++17", "-Wall", "-Werror", "-I", CSRC, "-o", exe, str(tmp_path / "e.cpp")])
    r = subprocess.run([exe], capture_output=True, text=True, timeout=240)
    print(r.stdout)
    assert r.returncode == 0, r.stdout
