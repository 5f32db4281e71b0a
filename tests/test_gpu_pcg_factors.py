"""The on-chip PCG takes an element's geometric factors as a constant times
the quadrature weights only where they are that to the last places: a mesh
whose elements are off a rectangle by some 6e-15 solves with its own factors,
as k_pcg does.  lambda2 = 1e6, so that the mass term, whose factor the
right-hand side has too, decides: bar 2e-15 between the two kernels' solutions
(both converged; a rounding error of 1.1e-16 in each of the few terms of a
node's equation), where factors off by 6e-15 would show.
"""
import warnings

import numpy as np
import pytest

import semtex_amd as sx
from semtex_amd.mesh import rect_mesh
from solve_helpers import rel

pytestmark = pytest.mark.gpu


def test_nearly_rectangular_elements(cuda, monkeypatch):
    import torch
    print("[pcg factors]", flush=True)
    monkeypatch.delenv("SEMX_PCG_CHIP", raising=False)
    P = sx.Mesh(8, rect_mesh(6, 5, 0, 3.0, 0, 3.0, bc=("N",) * 4, distort=1e-14))
    assert P.nsets == 1
    f = torch.from_numpy(np.concatenate([np.cos(P.x) * np.cos(P.y), np.zeros(P.planeSize - P.nPlane)]))
    f = f.to("cuda:0")
    b = torch.zeros(P.nline, dtype=torch.float64, device="cuda:0")
    us = []
    for chip in ("1", "0"):
        monkeypatch.setenv("SEMX_PCG_CHIP", chip)
        S = sx.ModalMatrixSys(P, 1e6, 1.0, 0, 1, 1, sx.JACPCG)
        u = torch.zeros_like(f)
        with warnings.catch_warnings():
            warnings.simplefilter("ignore")        # the last places may not reach 1e-16
            sx.solve(S, f, b, u, tol_rel=1e-16, step_max=60)
        assert S.pcg_info()["on_chip"] == (chip == "1")
        us.append(u.cpu().numpy()[:P.nPlane])
    r = rel(us[0], us[1])
    print(f"  on chip against k_pcg: {r:.2e}", flush=True)
    assert r <= 2e-15
