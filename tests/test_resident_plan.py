"""Plans of the resident FDTD steps (csrc/fwi2d_resident.h) on the CPU: every
grid point computed once, by an item of the right kind; the slabs tile the
rows and fit the LDS; no band row reads a field value that another item may
have overwritten (tests/resident_check.cpp)."""
import ctypes
import os
import random
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("resident") / "libresident_check.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-shared", "-fPIC", "-o", out,
                    "-I", os.path.join(HERE, "..", "geopvi_amd", "csrc"),
                    os.path.join(HERE, "resident_check.cpp")], check=True)
    return ctypes.CDLL(out)


@pytest.mark.parametrize("lc", [4, 5, 6, 7])
def test_plans_are_sound(lib, lc):
    rng = random.Random(lc)
    made = 0
    for _ in range(120):
        pml = rng.randint(0, 20) + lc
        nx, nz = rng.randint(10, 900), rng.randint(8, 300)
        for slabs in (1, 2, 3, 4, rng.randint(5, 32)):
            r = lib.resident_plan_check(nx + 2 * pml, nz + 2 * pml, lc, pml, slabs)
            assert r >= 0, f"{nz}x{nx} lc {lc} pml {pml} slabs {slabs}: fault {r}"
            made += r
    assert made > 60
