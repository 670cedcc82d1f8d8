"""The no-allocation entry captured into a HIP graph, steps with the fields on
the chip: every replay, with eager work and other inputs between, gives what
the eager call gives."""
import ctypes

import numpy as np
import pytest
import torch

from helpers import case
from geopvi_amd import _lib
from geopvi_amd.forward.fwi2d import solver

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ckpt", [0, 30])
def test_replays_equal_eager(ckpt):
    print(f"resident capture: ckpt {ckpt}", flush=True)
    p, vt, vs = case("small", seed=3, nx=97, nz=61, Lc=4, nt=300, ns=3, ds=30, ns0=0, nr=48, dr=2, nr0=0, nt_interval=2)
    dev = torch.device("cuda", 0)
    v0 = torch.from_numpy(np.asarray(vs, np.float32).reshape(1, -1)).to(dev)
    obs = solver.forward_batch(p, torch.from_numpy(np.asarray(vt, np.float32).reshape(1, -1)).to(dev))[0].clone()
    assert solver.resident_plan(p, 1)["slabs"] > 1
    vel = v0.clone()
    syn = torch.zeros(1, p.record_len, device=dev)
    grad = torch.zeros(1, p.ni, device=dev)
    mis = torch.zeros(1, dtype=torch.float64, device=dev)
    c = p.to_c()

    def call():
        grad.zero_()
        _lib.check(_lib.load().gpvi_fwi2d_batch_static(
            ctypes.byref(c), 1, vel.data_ptr(), obs.data_ptr(), syn.data_ptr(), grad.data_ptr(), mis.data_ptr(), 1, ckpt,
            ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        call()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        call()
    for r in range(4):
        v = v0 * (1 + 0.01 * r)
        want = solver.fwi_batch(p, v, obs, ckpt_interval=ckpt)      # eager, between the replays
        torch.cuda.synchronize()
        vel.copy_(v)
        g.replay()
        torch.cuda.synchronize()
        assert torch.isfinite(want[0]).all() and want[0].abs().max() > 0
        for a, b in zip((syn, grad, mis), want):
            assert torch.equal(a, b.view_as(a)), r
