"""Pseudo-spectral steps with twice the threads a workgroup (few workgroups)
against the ordinary ones: the same samples in batches of one and of many,
bit for bit, on odd and even lengths whose passes leave most threads idle or
need several rounds."""
import numpy as np
import pytest
import torch

from helpers import case
from geopvi_amd.forward.fwi2d import solver

pytestmark = pytest.mark.gpu


# padded lengths nz + 20, nx + 20
@pytest.mark.parametrize("nz,nx,samples", [(45, 79, 20), (44, 61, 20), (24, 40, 40), (200, 400, 6)])
def test_few_units_equal_many(nz, nx, samples):
    p, vt, vs = case("small", seed=nz, nx=nx, nz=nz, Lc=3, nt=12, ns=2, ds=max(1, nx // 2), ns0=0, nr=nx // 2, dr=2,
                     nr0=0, nt_interval=2, laplace_slover=1, pml0=10)
    print(f"psm threads: padded {p.nz + 20}x{p.nx + 20} {samples} samples", flush=True)
    rng = np.random.default_rng(nx)
    v = np.stack([np.asarray(vs, np.float32).reshape(-1) + rng.normal(0, 20, p.ni) for _ in range(samples)])
    vel = torch.from_numpy(v.astype(np.float32)).cuda()
    obs = solver.forward_batch(p, torch.from_numpy(np.asarray(vt, np.float32).reshape(1, -1)).cuda())[0].clone()
    syn, grad, mis = solver.fwi_batch(p, vel, obs)
    assert torch.isfinite(syn).all() and syn.abs().max() > 0
    for m in (0, samples - 1):
        s1, g1, m1 = solver.fwi_batch(p, vel[m:m + 1].contiguous(), obs)
        assert torch.equal(s1[0], syn[m]) and torch.equal(g1[0], grad[m]) and torch.equal(m1[0], mis[m])
