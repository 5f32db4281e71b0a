"""The elimination tree of the direct solve (the default for every direct
system) against the CPU FP64 oracle and against the band sweeps it stands
in for, through the C ABI: one region up to several stages of them, regions
that share a type and regions that are each their own, remainders of the
16-row and 8-column matrix tiles (np = 3 and 4, odd grids), strips one
element wide, periodic and natural sides, a singular mode whose pinned node
lies in one region, planes whose second plane is absent, and one to three
fields in one call.  Bar: relative L2 <= 1e-12, that of every direct solve.
"""
import numpy as np
import pytest

import oracle_lib as O
import semtex_amd as sx
from semtex_amd.mesh import rect_mesh
from semtex_amd.workloads import helmholtz_batch
from solve_helpers import drop_mode0_constant, gpu_solve, natural_lines, oracle_solve, rel

pytestmark = pytest.mark.gpu

TOL = 1e-12
TWO_PI = 2 * np.pi

CASES = [
    # name, kx, ky, np, nz, lambda2, distort, bc (P: periodic)
    ("one-element", 1, 1, 5, 2, 1.0, 0.0, "NNNN"),
    ("np3-2x2", 2, 2, 3, 1, 1.0, 0.0, "DDDD"),
    ("np4-5x3", 5, 3, 4, 6, 2.0, 0.2, "DNDD"),
    ("strip-24x1", 24, 1, 6, 4, 1.0, 0.0, "DPDP"),
    ("strip-1x9", 1, 9, 7, 8, 0.5, 0.0, "NDND"),
    ("distorted-11x7", 11, 7, 6, 12, 50.0, 0.2, "DNDD"),
    ("uniform-16x16-nz64", 16, 16, 9, 64, 20000.0, 0.0, "DDDD"),
    ("channel-20x12", 20, 12, 8, 16, 40.0, 0.0, "DPDP"),
    ("singular-13x9", 13, 9, 7, 6, 0.0, 0.0, "PPPP"),
    ("distorted-24x17", 24, 17, 7, 4, 3.0, 0.25, "NDDD"),
    ("uniform-32x32-np11", 32, 32, 11, 2, 1.0, 0.0, "DDDD"),
]


def _case(kx, ky, np_, nz, lam2, dist, bc, seed=3):
    m = rect_mesh(kx, ky, 0, TWO_PI, 0, TWO_PI, bc=tuple("D" if c == "P" else c for c in bc),
                  periodic_x=bc[1] == "P", periodic_y=bc[0] == "P", distort=dist)
    P, Q = sx.Mesh(np_, m), O.Mesh(np_, m)
    f, bcl, _ = helmholtz_batch(P, nz, lam2, 1.0, seed=seed)
    if "N" in bc:
        bcl = natural_lines(P, nz, bcl)
    return P, Q, f, bcl


@pytest.fixture(autouse=True)
def default_switches(monkeypatch):
    for v in ("SEMX_AUTOTUNE", "SEMX_BAND_COOP", "SEMX_BAND_XCOOP", "SEMX_BAND_PARTS", "SEMX_TREE"):
        monkeypatch.delenv(v, raising=False)


@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_tree_parity(cuda, case, monkeypatch):
    import torch
    name, kx, ky, np_, nz, lam2, dist, bc = case
    print(f"[tree] {name}", flush=True)
    P, Q, f, bcl = _case(kx, ky, np_, nz, lam2, dist, bc)
    nm = max(nz // 2, 1)
    S = sx.ModalMatrixSys(P, lam2, 1.0, 0, nm, nz, sx.DIRECT)
    ug, _ = gpu_solve(torch, P, S, f, bcl)
    assert S.sweep_info()["pick"][1] == 9
    ug2, _ = gpu_solve(torch, P, S, f, bcl)
    assert np.array_equal(ug, ug2)
    monkeypatch.setenv("SEMX_TREE", "0")
    B = sx.ModalMatrixSys(P, lam2, 1.0, 0, nm, nz, sx.DIRECT)
    ub, _ = gpu_solve(torch, P, B, f, bcl)
    assert 1 <= B.sweep_info()["pick"][1] <= 8 or B.sweep_info()["coop_w"] > 0
    uo, _ = oracle_solve(Q, nz, lam2, 1.0, f, bcl)
    rb = rel(ub[:, :P.nPlane], ug[:, :P.nPlane])   # the same pinned node
    if S.info["singular0"]:
        drop_mode0_constant(P, ug, uo)
    r = rel(ug[:, :P.nPlane], uo[:, :P.nPlane])
    print(f"  nsolve {P.nsolve}: rel L2 vs oracle {r:.3e}, vs band sweeps {rb:.3e}", flush=True)
    assert r <= TOL
    assert rb <= (1e-11 if S.info["singular0"] else TOL)


@pytest.mark.parametrize("nf", [1, 2, 3])
def test_tree_fields_and_mixed(cuda, nf):
    """Several fields on one system, and the direct mode 0 of a MIXED one:
    each field's bits do not depend on the others."""
    import torch
    P, Q, f, bcl = _case(9, 6, 7, 8, 2.0, 0.2, "DNDD")
    for method in (sx.DIRECT, sx.MIXED):
        S = sx.ModalMatrixSys(P, 2.0, 1.0, 0, 4, 8, method)
        dev = torch.device("cuda:0")
        fs, bcs, us, ref = [], [], [], []
        for i in range(nf):
            _, _, fi, bi = _case(9, 6, 7, 8, 2.0, 0.2, "DNDD", seed=20 + i)
            u1, _ = gpu_solve(torch, P, S, fi, bi)
            ref.append(u1)
            fs.append(torch.from_numpy(fi.ravel().copy()).to(dev))
            bcs.append(torch.from_numpy(bi.ravel().copy()).to(dev))
            us.append(torch.zeros(fi.size, dtype=torch.float64, device=dev))
        sx.solve_fields(S, fs, bcs, us)
        torch.cuda.synchronize()
        for u, r in zip(us, ref):
            g = u.cpu().numpy().reshape(r.shape)
            rows = slice(0, 1) if method == sx.MIXED else slice(None)   # PCG counts differ by map
            assert np.array_equal(g[rows], r[rows])


def test_tree_graph_replay(cuda):
    """The stages captured into a graph: four replays with eager work between
    them equal the eager solve bit for bit."""
    import torch
    P, _, f, bcl = _case(16, 16, 9, 8, 3.0, 0.0, "DDDD")
    S = sx.ModalMatrixSys(P, 3.0, 1.0, 0, 4, 8, sx.DIRECT)
    dev = torch.device("cuda:0")
    tf = torch.from_numpy(f.ravel().copy()).to(dev)
    tb = torch.from_numpy(bcl.ravel().copy()).to(dev)
    tu = torch.zeros_like(tf)
    sx.solve(S, tf, tb, tu, iters=False)
    torch.cuda.synchronize()
    ref = tu.clone()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        sx.solve(S, tf, tb, tu, iters=False)
    for _ in range(4):
        tu.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(tu, ref)
        v = torch.zeros_like(tu)
        sx.solve(S, tf, tb, v, iters=False)
        torch.cuda.synchronize()
        assert torch.equal(v, ref)
