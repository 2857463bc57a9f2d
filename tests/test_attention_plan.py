"""Which attentions of several query rows a head take the form of a wave to sixteen rows (marian-dev_amd/csrc/attention_plan.h), on the CPU."""
import os
import subprocess

from conftest import ROOT

CSRC = os.path.join(ROOT, "marian-dev_amd", "csrc")

PROGRAM = r"""
#include <cstdio>
#include "attention_plan.h"
using namespace marian_hip;
// as the entry point deals rows in the other form
static AttentionHeadsPlan plan(int64_t heads, int64_t m, int64_t len, int64_t* groups_of = nullptr) {
  const int64_t blocks = (m + 15) / 16;
  int64_t groups = heads >= 256 ? 1 : (256 + heads - 1) / heads;
  if(groups < (blocks + 3) / 4) groups = (blocks + 3) / 4;
  if(groups > blocks) groups = blocks;
  if(groups_of) *groups_of = groups;
  return attention_heads_plan(heads, groups, blocks, len);
}
int main() {
  long long taken = 0, wrong = 0;
  for(int64_t heads = 1; heads <= 1100; heads += heads < 300 ? 1 : 23)
    for(int64_t m = 8; m <= 300; ++m)
      for(int64_t len = 1; len <= 140; ++len) {
        int64_t groups = 0;
        const AttentionHeadsPlan p = plan(heads, m, len, &groups);
        if(!p.workgroups) continue;
        ++taken;
        const int64_t blocks = (m + 15) / 16, slots = p.workgroups * p.waves;
        bool ok = len <= 16 * p.tiles && slots >= blocks && slots - blocks < p.waves && p.waves >= 2 && p.waves <= 4 && heads * groups > 256;
        // no more than a quarter of the waves without rows, and less where a head has one workgroup in the other form
        if(p.waves > 2) ok = ok && (4 * (slots - blocks) < slots || (blocks == 3 && p.waves == 4 && groups == 2));
        if(!ok && wrong++ < 10) std::printf("%lld heads of %lld x %lld: %d tiles, %d waves, %lld workgroups\n", (long long)heads, (long long)m, (long long)len, p.tiles, p.waves, (long long)p.workgroups);
      }
  struct { int heads, m, len; bool taken; } const calls[] = {
      // measured faster
      {144, 64, 64, true}, {1024, 64, 64, true}, {384, 128, 128, true}, {512, 48, 48, true}, {512, 70, 70, true}, {1024, 23, 23, true}, {288, 8, 32, true},
      {288, 16, 15, true}, {144, 40, 100, true}, {144, 48, 64, true}, {288, 112, 112, true}, {288, 80, 80, true}, {288, 81, 96, true}, {640, 17, 20, true},
      // measured slower
      {288, 8, 64, false}, {288, 16, 33, false}, {1024, 8, 64, false}, {144, 30, 100, false}, {1024, 30, 100, false}, {640, 24, 128, false}, {512, 64, 80, false},
      {144, 64, 96, false}, {288, 72, 64, false}, {288, 96, 128, false}, {288, 48, 100, false}, {128, 64, 64, false}, {80, 64, 64, false}};
  for(const auto& c : calls)
    if((plan(c.heads, c.m, c.len).workgroups != 0) != c.taken) { ++wrong; std::printf("%d heads of %d x %d\n", c.heads, c.m, c.len); }
  std::printf("%lld taken\n", taken);
  return wrong != 0 || taken < 1000000;
}
"""


def test_waves_of_a_workgroup_have_rows(tmp_path):
    (tmp_path / "p.cpp").write_text(PROGRAM)
    exe = str(tmp_path / "p")
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-Wall", "-Werror", "-I", CSRC, "-o", exe, str(tmp_path / "p.cpp")])
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout
