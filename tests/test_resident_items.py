"""Row ranges of the resident steps' items (csrc/fwi2d_resident.h) on the CPU,
as the kernel's wavefronts read them: every item that is present lies in its
slab, and every point is computed once (tests/resident_items_check.cpp).  The
heights run from the smallest grid, odd and even: where two halves of an odd
grid meet, the lower one lacks a row, which can be an item's only one."""
import ctypes
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("resident_items") / "libresident_items.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-shared", "-fPIC", "-o", out,
                    "-I", os.path.join(HERE, "..", "geopvi_amd", "csrc"),
                    os.path.join(HERE, "resident_items_check.cpp")], check=True)
    return ctypes.CDLL(out)


@pytest.mark.parametrize("lc", [4, 5, 6, 7])
@pytest.mark.parametrize("pml0", [0, 5, 10, 20])
def test_items_lie_in_their_slabs(lib, lc, pml0):
    pml, made = pml0 + lc, 0
    for nz in range(1, 41):
        for nx in (10, 40, 201):
            ntx, ntz = nx + 2 * pml, nz + 2 * pml
            for units in (1, 2, 7, 64):
                r = lib.resident_items_of_choice(ntx, ntz, lc, pml, units)
                assert r >= 0, f"{nz}x{nx} lc {lc} pml0 {pml0} {units} units: fault {r}"
                made += r
            for slabs in range(1, 9):
                r = lib.resident_items_of_plan(ntx, ntz, lc, pml, slabs)
                assert r >= 0, f"{nz}x{nx} lc {lc} pml0 {pml0} {slabs} slabs: fault {r}"
                made += r
    assert made > 0


def test_plans_that_may_run(lib):
    """Every admitted plan leaves a CU for a missing slab whatever the launches
    on the other queues hold; fewer CUs than a plan is made for are refused."""
    for queues in (1, 4, 8, 10, 16, 31, 32, 300):
        most = lib.resident_slab_limit(queues)
        assert 1 <= most <= 32 and lib.resident_admits(most, queues, 256)
        assert most == 32 or not lib.resident_admits(most + 1, queues, 256)
        for slabs in range(1, 33):
            held = queues * (slabs - 1)          # CUs of the launches' partial clusters, at most
            assert bool(lib.resident_admits(slabs, queues, 256)) == (held < 256)
    for cus in (0, 1, 32, 40, 63, 128, 255):     # a CU mask, a partition of the device
        for slabs in (1, 2, 20, 32):
            assert not lib.resident_admits(slabs, 8, cus)
