"""The LDS limit of a kernel is raised once on each device it runs on, whatever the device's ordinal: lds_limit.h compiled
for the host, the runtime's call replaced by one that counts."""
import os
import shutil
import subprocess

import pytest

from helpers import ROOT

PROGRAM = r"""
#include "lds_limit.h"
#include <cstdio>
static int calls, refuse;
extern "C" hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { calls++; return refuse ? hipErrorInvalidValue : hipSuccess; }
int main() {
  static dnnrt::LdsRaised raised, other;
  const int device[] = {0, 0, 1, 15, 16, 16, 63, 63, 64, 64, 1000};
  for (int d : device) printf("%d ", (int)dnnrt::raise_lds(raised, d, &raised, 100000) + 10 * calls);
  printf("%d ", (int)dnnrt::raise_lds(other, 0, &other, 100000) + 10 * calls);
  refuse = 1;
  for (int i = 0; i < 2; i++) printf("%d ", (int)dnnrt::raise_lds(raised, 2, &raised, 100000) + 10 * calls);
  refuse = 0;
  printf("%d\n", (int)dnnrt::raise_lds(raised, 2, &raised, 100000) + 10 * calls);
}
"""


def test_lds_limit_is_raised_once_per_device_and_for_any_ordinal(tmp_path):
    if not shutil.which("g++"):
        pytest.skip("no host compiler")
    (tmp_path / "t.cpp").write_text(PROGRAM)
    subprocess.check_call(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I", os.path.join(ROOT, "occamy_amd", "csrc"),
                           "-o", str(tmp_path / "t"), str(tmp_path / "t.cpp")])
    got = [int(v) for v in subprocess.check_output([str(tmp_path / "t")]).split()]
    # ten times the calls so far, and 1 for success; ordinals 64 and above are asked for each time
    assert got == [11, 11, 21, 31, 41, 41, 51, 51, 61, 71, 81, 91, 100, 110, 121]
