"""A handle's host levels hold no table of CSR positions (4 bytes per active
nonzero): capi.cpp builds its levels without it, and build_host_level without
it leaves everything else the same.  setup.cpp with g++, no GPU."""
import os
import re
import shutil
import subprocess

import pytest

from tests.conftest import REPO

CSRC = os.path.join(REPO, "parmoon_cmg_amd", "csrc")
MAIN = r"""
#include <cstdio>
#include "cd3d_internal.hpp"
using namespace cd3d;
int main() {
  int bad = 0;
  for (int order = 1; order <= 2; order++)
    for (int m = 1; m <= 3; m += 2) {
      HostLevel A, B;
      build_host_level(A, order, m, 1, false);
      build_host_level(B, order, m, 1, true);
      bad += !A.lat_perm.empty() || (int64_t)B.lat_perm.size() != B.lat_nval || A.lat_nval != B.lat_nval;
      bad += A.lat_sid != B.lat_sid || A.lat_first != B.lat_first || A.lat_node2dof != B.lat_node2dof;
      bad += A.rowptr != B.rowptr || A.kcol != B.kcol || A.diag != B.diag || A.dof_node != B.dof_node;
    }
  printf(bad ? "FAILED %d\n" : "OK\n", bad);
  return bad != 0;
}
"""


def test_handles_build_their_levels_without_it():
    src = open(os.path.join(CSRC, "capi.cpp")).read()
    calls = re.findall(r"build_host_level\(([^;]*)\);", src)
    assert calls and all(c.rstrip().endswith("false") for c in calls)


@pytest.mark.skipif(shutil.which("g++") is None or not os.path.isdir("/opt/rocm/include"),
                    reason="g++ or the ROCm headers are missing")
def test_levels_without_it_are_the_same(tmp_path):
    main, exe = str(tmp_path / "main.cpp"), str(tmp_path / "positions")
    open(main, "w").write(MAIN)
    p = subprocess.run(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I" + CSRC, main,
                        os.path.join(CSRC, "setup.cpp"), "-lpthread", "-o", exe], capture_output=True, text=True, timeout=600)
    assert p.returncode == 0, p.stderr[-3000:]
    out = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0 and out.stdout.strip() == "OK", out.stdout
