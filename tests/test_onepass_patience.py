"""How long the workgroups of a launch wait for one another (marian-dev_amd/csrc/onepass_patience.h), on the CPU."""
import os
import subprocess

from conftest import ROOT

CSRC = os.path.join(ROOT, "marian-dev_amd", "csrc")

PROGRAM = r"""
#include <cstdio>
#include <initializer_list>
#include "onepass_patience.h"
using namespace marian_hip;
int main() {
  // one budget for a workgroup's waits, however many there are
  for(int budget : {0, 1, 5, 64})
    for(int first : {0, 1, 3, 64, 100}) {   // the poll that finds the first words; 0: none does
      int left = budget, polls = 0;
      bool found = false;
      for(; onepass_patience(left); onepass_polled(left))
        if((found = ++polls == first)) break;
      if(found != (first > 0 && first <= budget)) { std::printf("found at poll %d of %d\n", first, budget); return 1; }
      if(found)
        for(; onepass_patience(left); onepass_polled(left)) ++polls;
      if(polls > budget + 1 || left < 0) { std::printf("%d polls of %d\n", polls, budget); return 1; }   // (the poll that finds costs none)
    }
  for(size_t n : {33ul << 10, 64ul << 10, 1ul << 20, 4ul << 20, 16ul << 20}) std::printf("%zu %d\n", n, onepass_polls(n));
  return 0;
}
"""


def test_waits_are_bounded(tmp_path):
    """One budget for all waits of a workgroup, and a budget of the order of what the wait spares: ten times the usual wait of
    1.2 us and more at the least, tens of microseconds more than it takes 256 workgroups to read the whole input each at the most."""
    (tmp_path / "p.cpp").write_text(PROGRAM)
    exe = str(tmp_path / "p")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", "-I", CSRC, "-o", exe, str(tmp_path / "p.cpp")])
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
    for line in r.stdout.split("\n"):
        if line:
            n, polls = map(int, line.split())
            us, way_out = 0.5 * polls, 256 * 4 * n / 6e12 * 1e6
            assert 20 <= us <= 40 + way_out, (n, us, way_out)
    used = open(os.path.join(CSRC, "onepass_exchange.h")).read()
    assert used.count("for(; onepass_patience(polls_left); onepass_polled(polls_left))") == 1   # (the kernels wait nowhere else)
    assert used.count("int polls_left = polls;") == 1 and used.count("while(") == 0 and used.count("for(") == 2
