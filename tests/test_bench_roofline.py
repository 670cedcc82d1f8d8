"""bench.py's roofline entries, on the CPU: with the fields on the chip the
launches are those of up to 256 steps and the rate is operations against the
vector issue rate; HBM rates belong to step launches."""
import importlib
import os
import sys
from types import SimpleNamespace

import pytest

from geopvi_amd import synth


@pytest.fixture
def bench(monkeypatch):
    monkeypatch.setenv("GPU_MAX_HW_QUEUES", os.environ.get("GPU_MAX_HW_QUEUES", "4"))   # (bench sets it on import)
    monkeypatch.syspath_prepend(os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
    yield importlib.import_module("bench")
    sys.modules.pop("bench", None)


@pytest.mark.parametrize("ckpt,launches", [(0, 16), (98, 8 + 2 * 21), (600, 8 + 2 * (3 * 3 + 1))])
def test_entries(bench, ckpt, launches):
    p = synth.workload_params("c1")
    args = SimpleNamespace(steps=3, nsample=16, ckpt=ckpt)
    r = bench.resident_roofline(p, args, 1032.0, {"slabs": 7, "clusters": 36, "steps": 256})
    assert (r["bound"], r["unit"], r["kernel"]) == ("valu", "Tops/s", "resident_kernel")
    assert r["launches_per_step"] == launches and r["dispatches_per_launch"] == 1
    assert r["avg_launch_us"] == pytest.approx(344e3 / launches, rel=1e-3)
    # 320 units x 4000 steps x 228 x 428 points x 30 operations, and the imaging
    ops = 320 * (4000 * 228 * 428 * 30 + 1000 * 80000 * 9)
    assert r["achieved"] == pytest.approx(ops / 0.344 / 1e12, rel=1e-3)
    assert 0 < r["frac"] < 1 and r["frac"] == pytest.approx(r["achieved"] / r["peak"], abs=1e-3)
    step = bench.launch_roofline(p, args, 485.0, 4, 1, 2)
    assert (step["bound"], step["unit"], step["kernel"]) == ("hbm", "GB/s", "step_multi_kernel")
    assert step["dispatches_per_launch"] == 2
