"""The end of a 1D electromagnetic step (csrc/em_step_end.h) compiled for the
host and run by threads of which the first is always ahead: no row of a step
lands in another step's slot."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "particleincellcodegolf.jl_amd", "csrc")


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="hipcc is not installed")
def test_rows_land_in_their_own_step(tmp_path):
    exe = tmp_path / "em_step_end_check"
    subprocess.run(["hipcc", "--offload-arch=gfx950", "-O1", "-std=c++17", "-Xclang", "-target-feature", "-Xclang",
                    "-packed-fp32-ops", "-I", CSRC, os.path.join(ROOT, "tests", "cpu_checks", "em_step_end_check.hip"),
                    "-o", str(exe)], check=True, capture_output=True, timeout=600)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0, out.stdout
