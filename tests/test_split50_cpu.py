"""The two-word split of signed contributions (split50, csrc/pic_device.h),
compiled for the host, against the 128-bit fixed-point rounding it stands for."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "particleincellcodegolf.jl_amd", "csrc")


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="hipcc is not installed")
def test_split50_matches_fix_round128(tmp_path):
    exe = tmp_path / "split50_check"
    subprocess.run(["hipcc", "--offload-arch=gfx950", "-O2", "-std=c++17", "-ffp-contract=off", "-Xclang",
                    "-target-feature", "-Xclang", "-packed-fp32-ops", "-I", CSRC,
                    os.path.join(ROOT, "tests", "cpu_checks", "split50_check.hip"), "-o", str(exe)],
                   check=True, capture_output=True, timeout=600)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    print(out.stdout)
    assert out.returncode == 0, out.stdout
    assert " 0 mismatches" in out.stdout
