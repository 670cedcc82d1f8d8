"""Workspaces without the room that steps with the fields on the chip need
(the exchange words and a second array per velocity sample): the calls are
accepted, advance by one launch per step and give the same bits."""
import ctypes

import numpy as np
import pytest
import torch

from helpers import case
from geopvi_amd import _lib
from geopvi_amd.forward.fwi2d import solver

pytestmark = pytest.mark.gpu
SCRATCH = 64 << 20   # GPVI_STATIC_SCRATCH_BYTES


def inputs(nz, nx, ns, samples, nt):
    p, vt, vs = case("small", seed=nz + nx, nx=nx, nz=nz, Lc=3, nt=nt, ns=ns, ds=max(1, nx // ns), ns0=0, nr=nx // 2,
                     dr=2, nr0=0, nt_interval=2)
    v = np.stack([np.asarray(vs, np.float32).reshape(-1) * (1 + 0.01 * m) for m in range(samples)])
    obs = solver.forward_batch(p, torch.from_numpy(np.asarray(vt, np.float32).reshape(1, -1)).cuda())[0].clone()
    return p, torch.from_numpy(v.astype(np.float32)).cuda(), obs


def outputs(p, n):
    return (torch.empty(n, p.record_len, device="cuda"), torch.zeros(n, p.ni, device="cuda"),
            torch.empty(n, dtype=torch.float64, device="cuda"))


@pytest.mark.parametrize("ckpt,split", [(0, False), (30, False), (0, True), (30, True)])
def test_batch_without_the_room(ckpt, split):
    print(f"workspace room: ckpt {ckpt} split {split}", flush=True)
    n = 3
    p, vel, obs = inputs(60, 100, 4, n, 90)
    want = solver.fwi_batch(p, vel, obs, ckpt_interval=ckpt)
    # less than the full size by one sample's velocities: no room for the second arrays
    ws = torch.empty(solver.batch_workspace_bytes(p, n, ckpt) - p.ntp * 4, dtype=torch.uint8, device="cuda")
    syn, grad, mis = outputs(p, n)
    call = lambda phase: solver._batch_call(p, n, vel, obs, syn, grad, mis, 1, ckpt, phase, 0, ws,  # noqa: E731
                                            vel.device)
    if split:
        call(_lib.GPVI_PHASE_FORWARD)
        call(_lib.GPVI_PHASE_ADJOINT)
    else:
        call(_lib.GPVI_PHASE_ALL)
    torch.cuda.synchronize()
    for a, b in zip((syn, grad, mis), want):
        assert torch.equal(a, b.view_as(a))


def test_static_scratch_holds_what_the_launches_need():
    p, vel, obs = inputs(120, 200, 4, 1, 100)
    nt = next(t for t in range(200, 1000, 2)
              if solver.batch_workspace_bytes(p.replace(nt=t), 1, 0) > SCRATCH)
    print(f"static scratch: {nt} steps", flush=True)
    p, vel, obs = inputs(120, 200, 4, 1, nt)
    want = solver.fwi_batch(p, vel, obs)
    syn, grad, mis = outputs(p, 1)
    c = p.to_c()
    rc = _lib.load().gpvi_fwi2d_batch_static(ctypes.byref(c), 1, vel.data_ptr(), obs.data_ptr(), syn.data_ptr(),
                                             grad.data_ptr(), mis.data_ptr(), 1, 0,
                                             ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0, _lib.last_error()
    torch.cuda.synchronize()
    for a, b in zip((syn, grad, mis), want):
        assert torch.equal(a, b.view_as(a))
