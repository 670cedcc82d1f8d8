"""Clusters of the resident steps whose workgroups do not all get a CU in time:
they give up before they touch anything and their steps are done through
memory, with the same bits.  A time limit below 0 makes every cluster of
several workgroups give up, one of a few microseconds some of them."""
import os

import numpy as np
import pytest
import torch

from helpers import case
from geopvi_amd import _lib
from geopvi_amd.engine import Engine, EngineJob
from geopvi_amd.forward.fwi2d import solver

pytestmark = pytest.mark.gpu


@pytest.fixture
def limit(monkeypatch):
    def put(us):
        monkeypatch.setenv("GPVI_RES_JOIN_US", str(us))
    yield put
    os.environ.pop("GPVI_RES_JOIN_US", None)


def make(nz, nx, lc, pml0, k, ns, samples, nt):
    p, vt, vs = case("small", seed=nz + nx, nx=nx, nz=nz, Lc=lc, pml0=pml0, nt=nt, ns=ns, ds=max(1, nx // ns), ns0=0,
                     nr=nx // 2, dr=2, nr0=0, nt_interval=k)
    v = np.stack([np.asarray(vs, np.float32).reshape(-1) * (1 + 0.01 * m) for m in range(samples)])
    obs = solver.forward_batch(p, torch.from_numpy(np.asarray(vt, np.float32).reshape(1, -1)).cuda())[0].clone()
    return p, torch.from_numpy(v.astype(np.float32)).cuda(), obs


#   nz   nx  Lc pml0 k  ns samples nt ckpt run_fwi
CASES = [
    (24, 40, 3, 10, 2, 2, 1, 300, 0, 1),
    (61, 97, 5, 10, 3, 3, 50, 40, 0, 1),      # two units per cluster
    (50, 70, 4, 0, 1, 2, 2, 60, 16, 0),
    (64, 90, 6, 20, 2, 3, 4, 60, 24, 1),
]


@pytest.mark.parametrize("nz,nx,lc,pml0,k,ns,samples,nt,ckpt,run_fwi", CASES)
def test_given_up_clusters_give_the_same_bits(limit, nz, nx, lc, pml0, k, ns, samples, nt, ckpt, run_fwi):
    p, vel, obs = make(nz, nx, lc, pml0, k, ns, samples, nt)
    assert _lib.get_tuning()[0] == -1
    plan = solver.resident_plan(p, samples)
    print(f"resident join: {nz}x{nx} {plan}", flush=True)
    assert plan["slabs"] > 1
    want = solver.fwi_batch(p, vel, obs, run_fwi=run_fwi, ckpt_interval=ckpt)
    torch.cuda.synchronize()
    for us in (-1, 0, 1, 3):
        limit(us)
        got = solver.fwi_batch(p, vel, obs, run_fwi=run_fwi, ckpt_interval=ckpt)
        torch.cuda.synchronize()
        assert torch.isfinite(got[0]).all() and got[0].abs().max() > 0
        for a, b in zip(want, got):
            assert torch.equal(a, b), us


def test_engine_jobs(limit):
    specs = [make(60, 100, 3, 10, 2, 2, 3, 150), make(24, 40, 5, 10, 3, 2, 1, 90)]
    print("resident join: engine", flush=True)
    want = [solver.fwi_batch(*s) for s in specs]
    torch.cuda.synchronize()
    limit(-1)
    eng = Engine(torch.cuda.current_stream(), max_units=64, max_tiles=1 << 14)
    jobs = [EngineJob(p, vel, obs, 0, 1) for p, vel, obs in specs]
    for j in jobs:
        eng.submit(j)
    while eng.active_jobs():
        eng.advance(32)
    for j in jobs:
        eng.release(j.id)
    eng.sync()
    eng.close()
    for j, w in zip(jobs, want):
        for a, b in zip((j.syn, j.grad, j.misfit), w):
            assert torch.equal(a, b.view_as(a))
