"""Whether a stream is being recorded (marian-dev_amd/csrc/stream_recorded.h), on the CPU against a runtime of this program's own: a query that
fails leaves no error behind."""
import os
import subprocess

import pytest

from conftest import ROOT

CSRC = os.path.join(ROOT, "marian-dev_amd", "csrc")

PROGRAM = r"""
#include <cstdio>
#include "stream_recorded.h"
static hipError_t g_answer = hipSuccess, g_last = hipSuccess;
static hipStreamCaptureStatus g_status = hipStreamCaptureStatusNone;
extern "C" hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* s) {
  if(g_answer == hipSuccess) *s = g_status;
  else g_last = g_answer;
  return g_answer;
}
extern "C" hipError_t hipGetLastError() {
  const hipError_t e = g_last;
  g_last = hipSuccess;
  return e;
}
int main() {
  for(hipStreamCaptureStatus s : {hipStreamCaptureStatusNone, hipStreamCaptureStatusActive, hipStreamCaptureStatusInvalidated}) {
    g_status = s;
    if(marian_hip::recorded(nullptr) != (s == hipStreamCaptureStatusActive)) return std::printf("status %d\n", (int)s), 1;
  }
  g_answer = hipErrorStreamCaptureImplicit;
  if(marian_hip::recorded(nullptr)) return std::printf("a failed query\n"), 1;
  if(g_last != hipSuccess) return std::printf("an error is left\n"), 1;
  std::printf("ok\n");
}
"""


def test_a_failed_query_leaves_no_error(tmp_path):
    if not os.path.exists("/opt/rocm/include/hip/hip_runtime_api.h"):
        pytest.skip("HIP headers not available")
    (tmp_path / "p.cpp").write_text(PROGRAM)
    exe = str(tmp_path / "p")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-Wall", "-D__HIP_PLATFORM_AMD__=1", "-isystem", "/opt/rocm/include", "-I", CSRC,
                           "-o", exe, str(tmp_path / "p.cpp")])
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout
    # the query is asked for nowhere else
    for name in os.listdir(CSRC):
        if name.endswith((".h", ".hip", ".cpp")) and name != "stream_recorded.h":
            assert "hipStreamIsCapturing" not in open(os.path.join(CSRC, name)).read(), name
