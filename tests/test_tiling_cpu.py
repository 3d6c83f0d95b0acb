"""The default tiling of the 1D push (csrc/tiling.h): even batches keep the
tiles that fill the chip once, uneven ones take smaller tiles whose fixed work
stays below their particles'."""
import os
import random
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "particleincellcodegolf.jl_amd", "csrc")
CU = 256


@pytest.fixture(scope="module")
def tiling(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ is not installed")
    exe = tmp_path_factory.mktemp("tiling") / "tiling_check"
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", CSRC, os.path.join(ROOT, "tests", "cpu_checks", "tiling_check.cpp"),
                    "-o", str(exe)], check=True, timeout=120)

    def run(members, fp64=False, simpson=False, gauss=True, fit=2):
        args = [int(fp64), int(simpson), int(gauss), fit, CU] + [v for m in members for v in m]
        return tuple(map(int, subprocess.run([str(exe)] + [str(a) for a in args], check=True, capture_output=True,
                                             text=True, timeout=30).stdout.split()))
    return run


def per_tile(members, k):
    return -(-sum(P for _, P in members) // (CU * k))


@pytest.mark.parametrize("members", [[(4096, 2 ** 23)] * 2, [(4096, 2 ** 20)] * 8, [(4096, 2 ** 18)] * 8,
                                     [(1024, 2 ** 22)] * 2, [(256, 20000)] * 64])
def test_even_batches_fill_the_chip_once(tiling, members):
    assert tiling(members) == (per_tile(members, 2), 1024)                         # mixed
    assert tiling(members, fp64=True, fit=1) == (per_tile(members, 1), 1024)       # one block's LDS a CU
    assert tiling(members, fp64=True, fit=4) == (per_tile(members, 4), 512)


def uneven(n, seed, top=10):
    r = random.Random(seed)
    out = []
    for _ in range(n):
        N = 2 ** r.randint(5, top)
        out.append((N, N * r.randint(16, 256)))
    return out


@pytest.mark.parametrize("n", [64, 192, 500])
@pytest.mark.parametrize("fp64,fit", [(False, 2), (True, 1), (True, 4)])
def test_uneven_batches_take_smaller_tiles(tiling, n, fp64, fit):
    members = uneven(n, n)
    whole = per_tile(members, fit if fp64 else 2)
    tile, block = tiling(members, fp64=fp64, fit=fit)
    assert tile <= whole and block == (1024 if fp64 and fit == 1 else 512)
    assert tile >= min(whole, 2 * sum(N * P for N, P in members) // sum(P for _, P in members))
    # a stencil of one or two cells has too little work for more grids
    assert tiling(members, fp64=fp64, gauss=False, fit=fit) == (whole, 512 if fp64 and fit >= 2 else 1024)


def test_one_large_member_among_small_ones(tiling):
    # two grids of most particles, not of the largest member: never below
    members = [(4096, 2 ** 21)] + uneven(30, 3)
    tile, _ = tiling(members)
    assert tile >= 2 * sum(N * P for N, P in members) // sum(P for _, P in members) or tile == per_tile(members, 2)


def test_single_instances(tiling):
    assert tiling([(4096, 2 ** 24)]) == (2 ** 24 // 512, 1024)
    assert tiling([(4096, 3 * 10 ** 6)]) == (-(-3 * 10 ** 6 // 256), 1024)
    assert tiling([(64, 3 * 10 ** 6)], simpson=True) == (-(-3 * 10 ** 6 // 512), 1024)
    assert tiling([(64, 2 * 10 ** 6)], simpson=True) == (-(-2 * 10 ** 6 // 256), 1024)
    assert tiling([(4096, 3000001)], fp64=True, fit=1) == (-(-3000001 // 256), 1024)
    assert tiling([(1024, 10 ** 6)], fp64=True, fit=4) == (-(-10 ** 6 // 1024), 512)
    assert tiling([(64, 1)]) == (1, 1024)
