"""Which kernel a system's PCG planes run in and on how many workgroups, as
the C ABI reports it: on chip for np 4 to 12 in FP64 and FP32 refined, k_pcg
for the rest and behind its switches; and k_pcg's balanced workgroup map,
which takes the iteration counts of on-chip solves as well.
"""
import numpy as np
import pytest

import semtex_amd as sx
from semtex_amd.mesh import rect_mesh
from semtex_amd.workloads import helmholtz_batch
from solve_helpers import rel, solved

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def default_switches(monkeypatch):
    for v in ("SEMX_PCG_WG", "SEMX_PCG_OP", "SEMX_PCG_CHIP"):
        monkeypatch.delenv(v, raising=False)


def _system(kx, ky, np_, nz, lam2=2.0):
    import torch
    P = sx.Mesh(np_, rect_mesh(kx, ky, 0, 0.5 * kx, 0, 0.5 * ky))
    S = sx.ModalMatrixSys(P, lam2, 1.0, 0, nz // 2, nz, sx.JACPCG)
    f, b, _ = helmholtz_batch(P, nz, lam2, 1.0, seed=np_)
    f, b = (torch.from_numpy(a.ravel().copy()).to("cuda:0") for a in (f, b))
    return P, S, f, b


def _set(S, prec):
    if prec == sx.PCG_FP32_REFINED:
        S.set_pcg(prec, inner_tol=1e-4, max_outer=40)
    elif prec == sx.PCG_BF16_REFINED:
        S.set_pcg(prec, inner_tol=1e-2, max_outer=120)


@pytest.mark.parametrize("np_", range(3, 14))
def test_route(cuda, np_, monkeypatch):
    import torch
    for kx, ky in ((3, 2), (17, 9)):
        P, S, f, b = _system(kx, ky, np_, 4)
        want = -(-kx * ky // (8 * (64 // np_)))     # 8 wavefronts of whole elements
        for prec in (sx.PCG_FP64, sx.PCG_FP32_REFINED, sx.PCG_BF16_REFINED):
            _set(S, prec)
            sx.solve(S, f, b, torch.zeros_like(f), tol_rel=1e-8)
            i = S.pcg_info()
            print(f"[route] np {np_} {kx}x{ky} precision {prec}: {i}", flush=True)
            assert i["on_chip"] == (4 <= np_ <= 12 and prec != sx.PCG_BF16_REFINED)
            assert not i["on_chip"] or i["workgroups"] == want
    S.set_pcg(sx.PCG_FP64)
    monkeypatch.setenv("SEMX_PCG_CHIP", "0")
    sx.solve(S, f, b, torch.zeros_like(f), tol_rel=1e-8)
    assert not S.pcg_info()["on_chip"]


def test_counts_of_on_chip_solves_balance_k_pcg(cuda):
    """FP64 solves on chip, then BF16 refinement, which runs in k_pcg: its
    first solve, captured, has the map of the counts read back before."""
    import torch
    print("[route] balanced map after on-chip solves", flush=True)
    P, S, f, b = _system(24, 24, 9, 128, lam2=0.5)
    u = torch.zeros_like(f)
    sx.solve(S, f, b, u, tol_rel=1e-10)
    ref = u.cpu().numpy().reshape(128, -1)
    i = S.pcg_info()
    assert i == dict(on_chip=True, workgroups=11)
    _set(S, sx.PCG_BF16_REFINED)
    u.zero_()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        sx.solve(S, f, b, u, tol_rel=1e-10, iters=False)
    g.replay()
    torch.cuda.synchronize()
    i = S.pcg_info()
    print(f"  k_pcg on up to {i['workgroups']} workgroups a plane", flush=True)
    assert not i["on_chip"] and i["workgroups"] > 2
    assert S.sweep_info()["pcg_w"] == i["workgroups"]
    assert rel(solved(P, u.cpu().numpy().reshape(128, -1)), solved(P, ref)) <= 1e-6
