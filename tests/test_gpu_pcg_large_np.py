"""JACPCG with np = 14 to 16 in k_pcg, whose wavefront-level operator holds 192
nodes an element: FP64, FP32 and BF16 refined, against the CPU oracle's direct
solution.  Bar: relative L2 <= 1e-9 at TOL_REL 1e-12 (condition numbers below
1e3 here).
"""
import pytest

import oracle_lib as O
import semtex_amd as sx
from semtex_amd.mesh import rect_mesh
from semtex_amd.workloads import helmholtz_batch
from solve_helpers import gpu_solve, natural_lines, oracle_solve, rel, solved

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("np_", [13, 14, 15, 16])
def test_large_np(cuda, np_, monkeypatch):
    import torch
    for v in ("SEMX_PCG_WG", "SEMX_PCG_OP", "SEMX_PCG_CHIP"):
        monkeypatch.delenv(v, raising=False)
    print(f"[pcg large np] {np_}", flush=True)
    m = rect_mesh(4, 3, 0, 2.0, 0, 1.5, bc=("D", "D", "D", "N"), distort=0.1)
    P, Q = sx.Mesh(np_, m), O.Mesh(np_, m)
    f, b, _ = helmholtz_batch(P, 4, 40.0, 1.2, seed=np_)
    b = natural_lines(P, 4, b)
    uo, _ = oracle_solve(Q, 4, 40.0, 1.2, f, b, method=sx.DIRECT)
    for prec, tol, outer in ((sx.PCG_FP64, 0.5, 1), (sx.PCG_FP32_REFINED, 1e-4, 40),
                             (sx.PCG_BF16_REFINED, 1e-2, 120)):
        S = sx.ModalMatrixSys(P, 40.0, 1.2, 0, 2, 4, sx.JACPCG)
        S.set_pcg(prec, inner_tol=tol, max_outer=outer)
        ug, it = gpu_solve(torch, P, S, f, b)
        r = rel(solved(P, ug), solved(P, uo))
        print(f"  precision {prec}: {it} iterations, rel L2 {r:.2e}", flush=True)
        assert r <= 1e-9
    monkeypatch.setenv("SEMX_PCG_OP", "wave")
    S = sx.ModalMatrixSys(P, 40.0, 1.2, 0, 2, 4, sx.JACPCG)
    if np_ > 13:
        with pytest.raises(sx.SemxError, match="unsupported"):
            gpu_solve(torch, P, S, f, b)
    else:
        ug, _ = gpu_solve(torch, P, S, f, b)
        assert rel(solved(P, ug), solved(P, uo)) <= 1e-9


@pytest.mark.parametrize("np_", [14, 16])
def test_dns_start_up_with_large_np(cuda, np_, monkeypatch):
    """The first steps of N_TIME = 3, whose velocity systems are JACPCG, against
    the CPU oracle: relative L2 <= 1e-10 after five steps at TOL_REL 1e-13."""
    import ctypes as C

    import numpy as np
    import torch
    for v in ("SEMX_PCG_WG", "SEMX_PCG_OP", "SEMX_PCG_CHIP"):
        monkeypatch.delenv(v, raising=False)
    print(f"[dns large np] {np_}", flush=True)
    m = rect_mesh(3, 2, 0, 2 * np.pi, 0, 2 * np.pi, periodic_x=True, periodic_y=True)
    P, Q = sx.Mesh(np_, m), O.Mesh(np_, m)
    nz, f = 4, []
    for c in range(4):
        a = np.zeros((nz, P.planeSize))
        for k in (0, 2, 3):
            q = np.random.default_rng(10 * c + k).standard_normal(3)
            a[k, :P.nPlane] = 0.3 * q[0] * np.sin(P.x + q[1]) * np.cos(P.y + q[2]) * (c < 3)
        f.append(a)
    t = [torch.from_numpy(a.reshape(-1).copy()).to("cuda:0") for a in f]
    D = sx.DNS(P, nz, 1.0, 2e-3, 0.05, norder=3, tol_rel=1e-13, step_max=5000)
    D.run(5, *t)
    o = [np.ascontiguousarray(a.copy()) for a in f]
    Do = O.lib().orc_dns_create(C.c_void_p(Q.h), nz, 1.0, 2e-3, 0.05, 3, 0, 1e-13, 5000, 0)
    tm = C.c_double()
    O.lib().orc_dns_run(C.c_void_p(Do), 5, *(O.dp(a) for a in o), C.byref(tm))
    O.lib().orc_dns_destroy(C.c_void_p(Do))
    keep = [0, 2, 3]
    for name, g, r in zip("uvw", t, o):
        e = rel(g.cpu().numpy().reshape(r.shape)[keep, :P.nPlane], r[keep, :P.nPlane])
        print(f"  {name}: rel L2 {e:.2e}", flush=True)
        assert e <= 1e-10
