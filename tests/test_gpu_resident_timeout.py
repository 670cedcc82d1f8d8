"""A wait between workgroups that runs out (forced by a time limit of 0; every
kernel ends normally) is reported: by the status of the stream, by the engine
and the server for that job alone, and by the drop-in calls; later calls are
not affected."""
import ctypes
import os
import threading

import numpy as np
import pytest
import torch

from helpers import case
from geopvi_amd import _lib
from geopvi_amd.engine import Engine, EngineJob
from geopvi_amd.forward.fwi2d import aco2d, solver
from geopvi_amd.serving import FWIServer

pytestmark = pytest.mark.gpu


@pytest.fixture
def no_wait(monkeypatch):
    """on(True): waits run out at once; on(False): the ordinary limit."""
    def on(yes):
        if yes:
            monkeypatch.setenv("GPVI_RES_WAIT_US", "0")
        else:
            monkeypatch.delenv("GPVI_RES_WAIT_US", raising=False)
    yield on
    os.environ.pop("GPVI_RES_WAIT_US", None)


@pytest.fixture(scope="module")
def job():
    p, vt, vs = case("small", seed=5, nx=200, nz=120, Lc=3, nt=200, ns=4, ds=50, ns0=0, nr=100, dr=2, nr0=0,
                     nt_interval=2)
    vel = torch.from_numpy(np.asarray(vs, np.float32).reshape(1, -1)).cuda()
    obs = solver.forward_batch(p, torch.from_numpy(np.asarray(vt, np.float32).reshape(1, -1)).cuda())[0].clone()
    assert solver.resident_plan(p, 1)["slabs"] > 1
    want = solver.fwi_batch(p, vel, obs)
    solver.check_waits()
    return p, vel, obs, want


def timed_out(fn):
    with pytest.raises(_lib.GpviError) as e:
        fn()
    assert e.value.code == _lib.GPVI_ERR_TIMEOUT, e.value


def test_batch(no_wait, job):
    p, vel, obs, want = job
    print("timeout: batch", flush=True)
    no_wait(True)
    solver.fwi_batch(p, vel, obs)
    seen = []

    def other():   # a thread without a failed call of its own
        try:
            solver.check_waits()
            seen.append("ok")
        except _lib.GpviError as e:
            seen.append(str(e))
    timed_out(solver.check_waits)
    t = threading.Thread(target=other)
    t.start()
    t.join()
    assert seen == ["ok"]
    no_wait(False)
    got = solver.fwi_batch(p, vel, obs)
    solver.check_waits()
    for a, b in zip(got, want):
        assert torch.equal(a, b)


def test_engine_job_alone(no_wait, job):
    p, vel, obs, want = job
    print("timeout: engine", flush=True)
    eng = Engine(torch.cuda.current_stream(), max_units=64, max_tiles=1 << 14)
    bad, good = EngineJob(p, vel, obs, 0, 1), EngineJob(p, vel, obs, 0, 1)
    no_wait(True)
    eng.submit(bad)
    no_wait(False)
    eng.submit(good)
    eng.advance(64)
    assert eng.resident_jobs() == 2
    while eng.active_jobs():
        eng.advance(64)
    eng.sync()
    timed_out(lambda: eng.status(bad.id))
    assert eng.status(good.id) == 1
    eng.release(bad.id)
    eng.release(good.id)
    for a, b in zip((good.syn, good.grad, good.misfit), want):
        assert torch.equal(a, b.view_as(a))
    again = EngineJob(p, vel, obs, 0, 1)   # takes the failed job's word
    eng.submit(again)
    while eng.active_jobs():
        eng.advance(256)
    eng.sync()
    assert eng.status(again.id) == 1
    eng.release(again.id)
    eng.close()


def test_server_fails_the_request_and_goes_on(no_wait, job):
    p, vel, obs, want = job
    print("timeout: server", flush=True)
    with FWIServer(steps_per_tick=64, mem_budget=2 << 30) as srv:
        no_wait(True)
        timed_out(lambda: srv.submit(p, vel, obs).result(timeout=60))
        no_wait(False)
        res = srv.submit(p, vel, obs).result(timeout=60)
        torch.cuda.synchronize()
        assert torch.equal(res.record_syn.view_as(want[0]), want[0])
        assert torch.equal(res.grad.view_as(want[1]), want[1])


def test_drop_in(no_wait, job, tmp_path):
    p, vel, obs, want = job
    print("timeout: drop-in", flush=True)
    path = str(tmp_path / "input_params.txt")
    p.write(path)
    v64, o32 = vel[0].cpu().numpy().astype(np.float64), obs.cpu().numpy()
    no_wait(True)
    timed_out(lambda: aco2d.fwi(v64, o32, paramfile=path))
    lib = _lib.load()
    pf = lambda a: a.ctypes.data_as(ctypes.POINTER(ctypes.c_float))  # noqa: E731
    v32 = v64.astype(np.float32)
    syn, grad = np.full(p.record_len, 7.0, np.float32), np.zeros(p.ni, np.float32)
    lib.fwi_2D(path.encode(), pf(v32), pf(syn), pf(o32), pf(grad), 1, 0)
    assert lib.gpvi_compat_last_status() == _lib.GPVI_ERR_TIMEOUT
    assert (syn == 7.0).all() and (grad == 0).all()   # outputs untouched
    no_wait(False)
    syn, grad = aco2d.fwi(v64, o32, paramfile=path)
    assert np.array_equal(syn, want[0][0].cpu().numpy())
    assert np.array_equal(grad, want[1][0].cpu().numpy())
