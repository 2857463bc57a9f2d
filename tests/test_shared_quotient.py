"""Quotients of one divisor by its reciprocal (marian-dev_amd/csrc/shared_quotient.h) against the division, on the CPU."""
import os
import subprocess

from conftest import ROOT

CSRC = os.path.join(ROOT, "marian-dev_amd", "csrc")

PROGRAM = r"""
#include <cstdint>
#include <cstdio>
#include <cstring>
#include "shared_quotient.h"
using namespace marian_hip;
static uint32_t inverse(uint32_t x) {   // of an odd number, mod 2^32
  uint32_t y = x;
  for(int i = 0; i < 5; ++i) y *= 2 - x * y;
  return y;
}
static unsigned long long pairs = 0, wrong = 0;
static void check(float a, float s) {
  const float got = shared_quotient(a, s, 1.0f / s), want = a / s;
  ++pairs;
  if(std::memcmp(&got, &want, 4) != 0 && wrong++ < 10) std::printf("%a / %a: %a, not %a\n", a, s, got, want);
}
int main() {
  // Significands a, s of 24 bits whose quotient is a rounding edge but for k units of its last place times s:
  // a 2^shift = edge s + k, edge odd, 2^24 < edge < 2^25.  The correction errs by less than four of these units.
  for(uint32_t s = (1u << 23) + 1; s < 1u << 24; s += 2) {
    const uint32_t inv = inverse(s);
    for(int shift = 24; shift <= 25; ++shift)
      for(int k = -15; k <= 15; k += 2) {
        const uint32_t low = (uint32_t)-(int64_t)k * inv & ((1u << shift) - 1);
        for(uint64_t edge = low | 1u << 24; edge < 1u << 25; edge += 1u << 24) {
          if((edge & ((1u << shift) - 1)) != low) continue;
          const int64_t a = (int64_t)(edge * s + k) >> shift;
          if(a >= 1 << 23 && a < 1 << 24) check((float)a, (float)s);
        }
      }
  }
  const unsigned long long hard = pairs;
  uint64_t x = 1;
  for(int i = 0; i < 20000000; ++i) {   // all magnitudes that callers pass
    x = x * 6364136223846793005ull + 1442695040888963407ull;
    const float a = std::ldexp((float)((1u << 23) + (uint32_t)(x >> 41)), (int)((x >> 10) % 121) - 83);
    const float s = std::ldexp((float)((1u << 23) + (uint32_t)((x >> 18) & 0x7FFFFF)), (int)((x >> 3) % 81) - 63);
    if(std::fabs(a) >= kQuotientLeast && std::fabs(a) <= 0x1p60f && s >= kDivisorLeast && s <= kDivisorMost) check(i % 2 ? a : -a, s);
  }
  for(float s : {1.0f, 3.0f, 64.0f, 100.25f}) check(0.0f, s);
  std::printf("%llu hard pairs of %llu\n", hard, pairs);
  return wrong != 0 || hard < 20000000 || pairs < hard + 15000000;
}
"""


def test_shared_quotient_is_the_division(tmp_path):
    (tmp_path / "q.cpp").write_text(PROGRAM.replace("#include <cstring>", "#include <cstring>\n#include <cmath>\n#include <initializer_list>"))
    exe = str(tmp_path / "q")
    subprocess.check_call(["g++", "-O2", "-mfma", "-ffp-contract=off", "-std=c++17", "-Wall", "-Werror", "-I", CSRC, "-o", exe, str(tmp_path / "q.cpp")])
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout
