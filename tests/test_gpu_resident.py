"""The resident steps (fields on the chip, csrc/fwi2d_resident.hip) against
the per-step kernels on the same inputs: records bit for bit, misfit and
gradient to the parity bars.

The cases hold grids narrower and wider than one strip, odd row counts,
every stencil width and store interval, launches that end within a pass
(more than 256 steps), a last launch of one step, checkpoint segments of one
step, source and receiver rows in the absorbing band's neighbourhood, and
more units than the chip holds at once.
"""
import numpy as np
import pytest
import torch

from helpers import GRAD_RTOL, MISFIT_RTOL, case, rel_l2
from geopvi_amd import _lib
from geopvi_amd.forward.fwi2d import solver

pytestmark = pytest.mark.gpu

#       nz   nx  Lc  k   ns  samples  nt  ckpt
CASES = [
    (24, 40, 3, 2, 2, 1, 257, 0),
    (24, 40, 3, 1, 2, 3, 257, 64),
    (31, 53, 4, 3, 3, 2, 300, 0),
    (61, 97, 5, 3, 3, 5, 130, 0),
    (47, 211, 6, 2, 2, 2, 140, 20),
    (120, 200, 3, 2, 4, 4, 100, 0),
    (203, 401, 3, 2, 3, 2, 80, 33),
    (300, 900, 3, 2, 2, 1, 60, 0),
    (24, 40, 3, 2, 5, 30, 90, 0),     # 150 units: several per cluster
]


@pytest.mark.parametrize("nz,nx,lc,k,ns,samples,nt,ckpt", CASES)
def test_resident_equals_per_step(nz, nx, lc, k, ns, samples, nt, ckpt):
    print(f"resident: {nz}x{nx} Lc {lc} k {k} {samples} samples x {ns} shots {nt} steps ckpt {ckpt}", flush=True)
    p, vt, vs = case("small", seed=nz + nx, nx=nx, nz=nz, Lc=lc, nt=nt, ns=ns, ds=max(1, nx // ns), ns0=0,
                     nr=nx // 2, dr=2, nr0=0, nt_interval=k)
    rng = np.random.default_rng(nz)
    v = np.stack([np.asarray(vs, np.float32).reshape(-1) + rng.normal(0, 20, p.ni) for _ in range(samples)])
    vel = torch.from_numpy(v.astype(np.float32)).cuda()
    true = torch.from_numpy(np.asarray(vt, np.float32).reshape(1, -1)).cuda()
    old = _lib.get_tuning()
    out = []
    try:
        for variant in (0, -1):   # a given tile variant selects the per-step kernels
            _lib.set_tuning(variant, 0, 1)
            obs = solver.forward_batch(p, true)[0].clone()
            res = solver.fwi_batch(p, vel, obs, ckpt_interval=ckpt)
            fwd = solver.forward_batch(p, vel)
            torch.cuda.synchronize()
            out.append([t.cpu().numpy() for t in (obs, fwd, *res)])
    finally:
        _lib.set_tuning(*old)
    (obs0, fwd0, syn0, grad0, mis0), (obs1, fwd1, syn1, grad1, mis1) = out
    assert np.isfinite(syn0).all() and np.abs(obs0).max() > 0
    assert np.array_equal(obs0, obs1) and np.array_equal(fwd0, fwd1) and np.array_equal(syn0, syn1)
    assert np.abs(mis1 - mis0).max() <= MISFIT_RTOL * np.abs(mis0).max()
    for m in range(samples):
        assert rel_l2(grad1[m], grad0[m]) <= GRAD_RTOL
