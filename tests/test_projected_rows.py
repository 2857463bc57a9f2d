"""Where a workgroup of the projected attention takes an input row (proj_place_of) against the rows it takes (proj_row_of), on the CPU."""
import os
import subprocess

from conftest import ROOT

CSRC = os.path.join(ROOT, "marian-dev_amd", "csrc")

PROGRAM = r"""
#include <cstdio>
#include "operand_addressing.h"
using namespace marian_hip;
int main() {
  long long seen = 0;
  for(int n_proj = 1; n_proj <= 3; n_proj += 2)
    for(int M = 1; M <= 64; ++M)
      for(int nb = 1; nb <= M; ++nb)
        for(int len = 1; len <= 100; len += 33) {
          ProjRowPlan p = proj_row_plan(n_proj, M, 2, 2 * nb, len, 96, 20000, 160000);
          const int groups = p.shift < 0 ? (int)p.blocks_y : proj_groups(p.shift, p.sentences), chunks = (int)p.blocks_y / groups;
          for(int group = 0; group < groups; ++group)
            for(int chunk = 0; chunk < chunks; ++chunk)
              for(int row = 0; row < M; ++row) {
                int want = -1;
                for(int r = 0; r < p.per_wg << (p.shift < 0 ? 0 : p.shift); ++r)
                  if(proj_row_of(p.shift, p.sentences, p.hyps, p.per_wg, group, chunk, r) == row) want = r;
                const int got = proj_place_of(p.shift, p.sentences, p.hyps, p.per_wg, group, chunk, row);
                if(got != want) return std::printf("M %d sentences %d group %d chunk %d row %d: %d, not %d\n", M, nb, group, chunk, row, got, want), 1;
                seen += want >= 0;
              }
        }
  std::printf("%lld rows\n", seen);
  return seen < 100000;
}
"""


def test_place_of_a_row(tmp_path):
    (tmp_path / "p.cpp").write_text(PROGRAM)
    exe = str(tmp_path / "p")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", "-I", CSRC, "-o", exe, str(tmp_path / "p.cpp")])
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout
