"""The staging of downloads (csrc/hostcopy.cpp) on the host alone, against a
stand-in for the HIP calls it makes, built with the address sanitizer and with
the thread sanitizer."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "particleincellcodegolf.jl_amd", "csrc")


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="hipcc is not installed")
@pytest.mark.parametrize("sanitizer", ["address", "thread"])
def test_staged_copies(tmp_path, sanitizer):
    exe = tmp_path / "hostcopy_check"
    subprocess.run(["hipcc", "-w", "--offload-arch=gfx950", "-O1", "-g", "-std=c++17", "-Xclang", "-target-feature",
                    "-Xclang", "-packed-fp32-ops", "-Xarch_host", f"-fsanitize={sanitizer}", "-I", CSRC,
                    os.path.join(ROOT, "tests", "cpu_checks", "hostcopy_check.cpp"), os.path.join(CSRC, "hostcopy.cpp"),
                    "-o", str(exe)], check=True, capture_output=True, timeout=600)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0, out.stdout + out.stderr
