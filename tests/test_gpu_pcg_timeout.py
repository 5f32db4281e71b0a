"""Expired waits between the workgroups of one PCG plane are reported: with
SEMX_PCG_NOWAIT=1 the kernel behaves as after an expired wait from its start
(no value is waited for, and it says so), and still ends by itself.
Two workgroups a plane (120 elements of np = 6).
"""
import numpy as np
import pytest

import semtex_amd as sx
from semtex_amd.mesh import rect_mesh
from semtex_amd.workloads import helmholtz_batch

pytestmark = pytest.mark.gpu

TIMEOUT = "bounded device-side wait"


@pytest.fixture(autouse=True)
def default_switches(monkeypatch):
    for v in ("SEMX_PCG_WG", "SEMX_PCG_OP", "SEMX_PCG_CHIP", "SEMX_PCG_NOWAIT"):
        monkeypatch.delenv(v, raising=False)


def test_solve_reports_expired_wait(cuda, monkeypatch, capfd):
    import torch
    print("[timeout] solve", flush=True)
    P = sx.Mesh(6, rect_mesh(12, 10, 0, 6.0, 0, 5.0))
    S = sx.ModalMatrixSys(P, 2.0, 1.0, 0, 2, 4, sx.JACPCG)
    f, b, _ = helmholtz_batch(P, 4, 2.0, 1.0, seed=1)
    f, b = (torch.from_numpy(a.ravel().copy()).to("cuda:0") for a in (f, b))
    ref, u = torch.zeros_like(f), torch.zeros_like(f)
    sx.solve(S, f, b, ref, iters=False)
    sx.helm_check(S)
    monkeypatch.setenv("SEMX_PCG_NOWAIT", "1")
    sx.solve(S, f, b, u, iters=False, step_max=50)
    with pytest.raises(sx.SemxError, match=TIMEOUT):
        sx.helm_check(S)
    assert "PCG" in capfd.readouterr().err
    sx.helm_check(S)                            # reported once
    with pytest.raises(sx.SemxError, match=TIMEOUT):
        sx.solve(S, f, b, u, step_max=50)
    monkeypatch.delenv("SEMX_PCG_NOWAIT")
    u.zero_()
    sx.solve(S, f, b, u)
    assert torch.equal(u, ref)


def test_startup_steps_report_expired_wait(cuda, monkeypatch):
    """The first steps' velocity systems, which the steady steps do not use."""
    import torch
    print("[timeout] start-up steps", flush=True)
    P = sx.Mesh(6, rect_mesh(12, 10, 0, 2 * np.pi, 0, 2 * np.pi, periodic_x=True, periodic_y=True))
    a = np.zeros((4, P.planeSize))
    a[0, :P.nPlane] = np.sin(P.x) * np.cos(P.y)
    a[2, :P.nPlane] = np.cos(P.x) * np.cos(P.y)
    f = [torch.from_numpy(a.reshape(-1).copy()).to("cuda:0") for _ in range(4)]
    D = sx.DNS(P, 4, 1.0, 1e-2, 0.05, norder=2, step_max=50)
    monkeypatch.setenv("SEMX_PCG_NOWAIT", "1")
    with pytest.raises(sx.SemxError, match=TIMEOUT):
        D.run(1, *f)
    monkeypatch.delenv("SEMX_PCG_NOWAIT")
    D.run(1, *f)                                # direct from here on; reported once
