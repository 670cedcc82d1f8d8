"""Resident steps where the library says that it takes them
(gpvi_fwi2d_resident_plan, gpvi_engine_resident_jobs), against the per-step
kernels: records, misfit and gradient bit for bit.

The cases hold more units than clusters with one slab and with several, the
last units leaving clusters idle; no absorbing band, narrow and wide ones; the
gradient of given adjoint sources (run_fwi = 0); two batches at once on two
streams; and engine jobs that change between the two kinds of step."""
import numpy as np
import pytest
import torch

from helpers import case
from geopvi_amd import _lib
from geopvi_amd.engine import Engine, EngineJob
from geopvi_amd.forward.fwi2d import solver

pytestmark = pytest.mark.gpu


def make(nz, nx, lc, pml0, k, ns, samples, nt):
    p, vt, vs = case("small", seed=nz + nx, nx=nx, nz=nz, Lc=lc, pml0=pml0, nt=nt, ns=ns, ds=max(1, nx // ns), ns0=0,
                     nr=nx // 2, dr=2, nr0=0, nt_interval=k)
    rng = np.random.default_rng(nz)
    v = np.stack([np.asarray(vs, np.float32).reshape(-1) + rng.normal(0, 20, p.ni) for _ in range(samples)])
    obs = solver.forward_batch(p, torch.from_numpy(np.asarray(vt, np.float32).reshape(1, -1)).cuda())[0].clone()
    return p, torch.from_numpy(v.astype(np.float32)).cuda(), obs


class steps:
    """Step launches (variant 0) or the automatic choice (-1) inside."""

    def __init__(self, variant):
        self.variant = variant

    def __enter__(self):
        self.old = (_lib.get_tuning(), _lib.get_time_blocking())
        _lib.set_time_blocking(1)
        _lib.set_tuning(self.variant, 0, 8)

    def __exit__(self, *exc):
        _lib.set_tuning(*self.old[0])
        _lib.set_time_blocking(self.old[1])


def same(a, b):
    assert len(a) == len(b)
    for x, y in zip(a, b):
        assert torch.equal(x, y.view_as(x))


#   nz   nx  Lc pml0 k  ns samples nt ckpt run_fwi  slabs  rounds
CASES = [
    (24, 40, 3, 10, 2, 5, 52, 70, 0, 1, "one", 2),         # 260 units, one slab each
    (61, 97, 5, 10, 3, 3, 50, 60, 0, 1, "many", 2),        # 150 units, 3 slabs
    (100, 160, 3, 10, 1, 5, 26, 40, 16, 1, "many", 2),     # 130 units, 3 slabs
    (203, 401, 3, 10, 2, 4, 10, 40, 0, 0, "many", 2),      # 40 units, 12 slabs
    (50, 70, 4, 0, 2, 4, 10, 90, 0, 0, "many", 1),         # no absorbing band
    (47, 53, 3, 5, 2, 2, 3, 300, 0, 1, "many", 1),
    (64, 90, 6, 20, 2, 3, 4, 80, 24, 0, "many", 1),        # wide band, widest stencil
    (45, 300, 6, 10, 1, 2, 2, 70, 0, 1, "many", 1),
    (44, 70, 3, 20, 3, 3, 40, 60, 0, 1, "many", 1),
]


@pytest.mark.parametrize("nz,nx,lc,pml0,k,ns,samples,nt,ckpt,run_fwi,slabs,rounds", CASES)
def test_taken_and_the_same_bits(nz, nx, lc, pml0, k, ns, samples, nt, ckpt, run_fwi, slabs, rounds):
    p, vel, obs = make(nz, nx, lc, pml0, k, ns, samples, nt)
    out = []
    for variant in (0, -1):
        with steps(variant):
            plan = solver.resident_plan(p, samples)
            print(f"resident choice: {nz}x{nx} Lc {lc} pml0 {pml0} k {k} {samples}x{ns} units {nt} steps: {plan}",
                  flush=True)
            if variant < 0:
                assert plan and (plan["slabs"] == 1) == (slabs == "one")
                assert -(-samples * ns // plan["clusters"]) == rounds
            else:
                assert plan is None
            out.append((*solver.fwi_batch(p, vel, obs, run_fwi=run_fwi, ckpt_interval=ckpt),
                        solver.forward_batch(p, vel)))
            torch.cuda.synchronize()
    assert torch.isfinite(out[0][0]).all() and out[0][1].abs().max() > 0
    same(*out)


def test_two_batches_at_once():
    shapes = [(120, 200, 3, 10, 2, 4, 4, 600), (100, 160, 4, 10, 2, 5, 10, 300)]
    print("resident choice: two streams", flush=True)
    jobs = [make(*s) for s in shapes]
    want = []
    with steps(0):
        for p, vel, obs in jobs:
            want.append(solver.fwi_batch(p, vel, obs))
        torch.cuda.synchronize()
    with steps(-1):
        streams = [torch.cuda.Stream() for _ in jobs]
        got = []
        for st, (p, vel, obs) in zip(streams, jobs):
            st.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(st):
                assert solver.resident_plan(p, vel.shape[0])["slabs"] > 1
                got.append(solver.fwi_batch(p, vel, obs))
        torch.cuda.synchronize()
    for a, b in zip(want, got):
        same(a, b)


def test_engine_jobs_change_the_kind_of_step():
    few = [(60, 100, 3, 10, 2, 2, 3, 400), (24, 40, 5, 10, 3, 2, 1, 350)]
    many = [(24, 40, 3, 10, 2, 2, 1, 70)] * 6
    print("resident choice: engine", flush=True)
    with steps(0):
        specs = [make(*s) for s in few + many]
        want = [solver.fwi_batch(*s) for s in specs]
        torch.cuda.synchronize()
    with steps(-1):
        eng = Engine(torch.cuda.current_stream(), max_units=64, max_tiles=1 << 14)
        jobs = [EngineJob(p, vel, obs, 0, 1) for p, vel, obs in specs]
        seen = []
        for j in jobs[:2]:
            eng.submit(j)
        eng.advance(64)
        seen.append(eng.resident_jobs())
        for j in jobs[2:]:
            eng.submit(j)
        eng.advance(64)
        seen.append(eng.resident_jobs())
        while eng.active_jobs() > 2:
            eng.advance(64)
        eng.advance(64)
        seen.append(eng.resident_jobs())
        while eng.active_jobs():
            eng.advance(64)
        for j in jobs:
            eng.release(j.id)
        eng.sync()
        eng.close()
    print(f"resident jobs: {seen}", flush=True)
    assert seen == [2, 0, 2]
    for j, w in zip(jobs, want):
        same((j.syn, j.grad, j.misfit), w)
