"""The levels of the one-workgroup V-cycle program on the host: uniform levels
(no per-node values) and varying ones in one program, by
tests/small_levels_host_check.cpp.  No GPU is needed."""
import os
import subprocess

import pytest

from tests.conftest import REPO

CSRC = os.path.join(REPO, "parmoon_cmg_amd", "csrc")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc is not installed")
def test_uniform_and_varying_levels_in_one_program(tmp_path):
    exe = str(tmp_path / "small_levels_host_check")
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O1", "-std=c++17", "-Xclang", "-target-feature", "-Xclang",
                    "-packed-fp32-ops", "-I", CSRC, os.path.join(REPO, "tests", "small_levels_host_check.cpp"),
                    os.path.join(CSRC, "setup.cpp"), "-o", exe], check=True, capture_output=True, timeout=600)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    print(out.stdout)
    assert out.returncode == 0 and out.stdout.strip().endswith("OK"), (out.returncode, out.stdout[-3000:])
