"""The resident steps on the smallest heights, where a slab of an odd grid
lacks the only row of an item (9 rows), against the per-step kernels: records
and gradients bit for bit."""
import numpy as np
import pytest
import torch

from helpers import case
from geopvi_amd import _lib
from geopvi_amd.forward.fwi2d import solver

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nz,nx,lc,pml0,ns,ckpt", [
    (8, 40, 3, 10, 2, 0), (9, 10, 3, 10, 1, 0), (9, 40, 3, 10, 2, 16), (9, 75, 6, 5, 3, 0), (9, 33, 4, 0, 2, 0),
    (10, 40, 5, 20, 2, 0), (11, 40, 3, 10, 2, 0)])
def test_smallest_heights(nz, nx, lc, pml0, ns, ckpt):
    print(f"resident small: {nz}x{nx} Lc {lc} pml0 {pml0} {ns} shots ckpt {ckpt}", flush=True)
    p, vt, vs = case("small", seed=nz + nx, nx=nx, nz=nz, Lc=lc, pml0=pml0, nt=60, ns=ns, ds=max(1, nx // ns), ns0=0,
                     nr=nx // 2, dr=2, nr0=0, depths=1, depthr=2, nt_interval=2)
    vel = torch.from_numpy(np.asarray(vs, np.float32).reshape(1, -1)).cuda()
    true = torch.from_numpy(np.asarray(vt, np.float32).reshape(1, -1)).cuda()
    old = _lib.get_tuning()
    out = []
    try:
        for variant in (0, -1):   # a given tile variant selects the per-step kernels
            _lib.set_tuning(variant, 0, 8)
            obs = solver.forward_batch(p, true)[0].clone()
            res = solver.fwi_batch(p, vel, obs, ckpt_interval=ckpt)
            torch.cuda.synchronize()
            out.append((obs, *res))
    finally:
        _lib.set_tuning(*old)
    assert torch.isfinite(out[0][1]).all() and out[0][0].abs().max() > 0 and out[0][2].abs().max() > 0
    for a, b in zip(*out):
        assert torch.equal(a, b)
