"""The Gaussian stencil's edges evaluated interval by interval
(csrc/gauss_edges.h) and the limb split of its contributions, compiled for the
host, against the CPU restatement's erf bit for bit."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "particleincellcodegolf.jl_amd", "csrc")


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="hipcc is not installed")
def test_edges_and_limbs_match_the_restatement(tmp_path, orc):
    lib = os.path.join(ROOT, "oracle")
    exe = tmp_path / "gauss_edges_check"
    subprocess.run(["hipcc", "--offload-arch=gfx950", "-O2", "-std=c++17", "-ffp-contract=off", "-Xclang",
                    "-target-feature", "-Xclang", "-packed-fp32-ops", "-I", CSRC,
                    os.path.join(ROOT, "tests", "cpu_checks", "gauss_edges_check.hip"), "-L", lib, "-lpicoracle",
                    f"-Wl,-rpath,{lib}", "-o", str(exe)], check=True, capture_output=True, timeout=600)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    print(out.stdout)
    assert out.returncode == 0, out.stdout
    assert " 0 mismatches" in out.stdout


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="hipcc is not installed")
def test_the_tails_unsure_band_is_wide_enough(tmp_path, orc):
    """The measurement behind tail_delta (4e9 arguments an interval there), over 5e7."""
    lib = os.path.join(ROOT, "oracle")
    exe = tmp_path / "gauss_edges_check"
    subprocess.run(["hipcc", "--offload-arch=gfx950", "-O2", "-std=c++17", "-ffp-contract=off", "-Xclang",
                    "-target-feature", "-Xclang", "-packed-fp32-ops", "-I", CSRC,
                    os.path.join(ROOT, "tests", "cpu_checks", "gauss_edges_check.hip"), "-L", lib, "-lpicoracle",
                    f"-Wl,-rpath,{lib}", "-o", str(exe)], check=True, capture_output=True, timeout=600)
    out = subprocess.run([str(exe), str(5 * 10 ** 7)], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0 and out.stdout.count("tail_delta") == 3, out.stdout
