"""What a cooperative launch's outcome means, and the pause after a refusal, on the CPU: the header that the
resident solves use, compiled with the host compiler."""

import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include "nfx_backoff.h"
using namespace nfx;
#define CHECK(c) if (!(c)) { std::printf("line %d: %s\n", __LINE__, #c); return 1; }
int main() {
  CHECK(grid_outcome(hipSuccess) == GridLaunch::ran);
  CHECK(grid_outcome(hipErrorIllegalState) == GridLaunch::busy);
  for (hipError_t e : {hipErrorCooperativeLaunchTooLarge, hipErrorLaunchOutOfResources, hipErrorOutOfMemory,
                       hipErrorNotSupported})
    CHECK(grid_outcome(e) == GridLaunch::no);
  for (hipError_t e : {hipErrorInvalidValue, hipErrorInvalidConfiguration, hipErrorInvalidDeviceFunction,
                       hipErrorIllegalAddress, hipErrorLaunchFailure, hipErrorInvalidHandle, hipErrorUnknown})
    CHECK(grid_outcome(e) == GridLaunch::error);
  static GridBackoff b;
  const int64_t now = 1000000;
  for (int d = -1; d <= GridBackoff::kDevices; ++d) CHECK(!b.waits(d, now));
  b.note(3, now, 10);
  CHECK(b.waits(3, now) && b.waits(3, now + 9) && !b.waits(3, now + 10));
  for (int d = -1; d <= GridBackoff::kDevices; ++d) CHECK(d == 3 || !b.waits(d, now));  // other devices are asked
  b.note(-1, now, 10);  // not in the table
  b.note(GridBackoff::kDevices, now, 10);
  CHECK(!b.waits(-1, now) && !b.waits(GridBackoff::kDevices, now));
  b.note(3, now + 20, 5);
  CHECK(b.waits(3, now + 24) && !b.waits(3, now + 25));
  return 0;
}
"""


def test_outcomes_and_pause(tmp_path):
    src, exe = tmp_path / "backoff.cpp", tmp_path / "backoff"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + os.path.join(ROOT, "nfempy_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout
