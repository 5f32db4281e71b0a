"""Direct solves along the elimination tree on meshes whose parts differ: a
long duct one element wide joined to a square section (many short regions in
one stage with a few long ones), and the same two parts apart.  Three fields
at once, each against the CPU FP64 oracle.  Bar: relative L2 <= 1e-12, that of
every direct solve.
"""
import numpy as np
import pytest

import oracle_lib as O
import semtex_amd as sx
from semtex_amd.workloads import helmholtz_batch
from solve_helpers import oracle_solve, rel, solved

pytestmark = pytest.mark.gpu


def duct_mesh(n, length, gap=0):
    """n x n unit squares and a row of `length` more from its lower right
    corner (gap: that many squares left out between them)."""
    cells = [(i, j) for j in range(n) for i in range(n)]
    cells += [(n + gap + i, 0) for i in range(length)]
    at = {c: e for e, c in enumerate(cells)}
    nel = len(cells)
    vx, vy = np.zeros((nel, 4)), np.zeros((nel, 4))
    nbr = -np.ones((nel, 4), dtype=np.int32)
    skind = np.zeros((nel, 4), dtype=np.int32)
    for e, (i, j) in enumerate(cells):
        for c, (di, dj) in enumerate(((0, 0), (1, 0), (1, 1), (0, 1))):
            vx[e, c], vy[e, c] = i + di, j + dj
        for s, (di, dj, other) in enumerate(((0, -1, 2), (1, 0, 3), (0, 1, 0), (-1, 0, 1))):
            q = at.get((i + di, j + dj), -1)
            if q >= 0:
                nbr[e, s] = 4 * q + other
            else:
                skind[e, s] = 1
    return dict(nel=nel, vx=vx, vy=vy, nbr=nbr, skind=skind)


@pytest.mark.parametrize("np_,n,length,gap", [
    (16, 12, 64, 0), (9, 24, 128, 0), (7, 24, 512, 0), (7, 8, 20, 2)])
def test_duct(cuda, np_, n, length, gap, monkeypatch):
    import torch
    for v in ("SEMX_AUTOTUNE", "SEMX_BAND_COOP", "SEMX_BAND_XCOOP", "SEMX_BAND_PARTS", "SEMX_TREE"):
        monkeypatch.delenv(v, raising=False)
    print(f"[duct] np {np_} {n}x{n} + {length}, gap {gap}", flush=True)
    m = duct_mesh(n, length, gap)
    P, Q = sx.Mesh(np_, m), O.Mesh(np_, m)
    S = sx.ModalMatrixSys(P, 2.0, 1.0, 0, 2, 4, sx.DIRECT)
    ins = [helmholtz_batch(P, 4, 2.0, 1.0, seed=s)[:2] for s in (1, 2, 3)]
    dev = torch.device("cuda:0")
    for nf in (1, 2, 3):
        fs = [torch.from_numpy(f.ravel().copy()).to(dev) for f, _ in ins[:nf]]
        bs = [torch.from_numpy(b.ravel().copy()).to(dev) for _, b in ins[:nf]]
        us = [torch.zeros_like(t) for t in fs]
        sx.solve_fields(S, fs, bs, us)
        torch.cuda.synchronize()
        assert S.sweep_info()["pick"][nf] == 9
        for (f, b), u in zip(ins, us):
            if nf == 3:
                uo, _ = oracle_solve(Q, 4, 2.0, 1.0, f, b)
                assert rel(solved(P, u.cpu().numpy().reshape(f.shape)), solved(P, uo)) <= 1e-12
