"""Element condensation and recovery on the matrix cores against the CPU FP64
oracle, through the C ABI: the smallest and largest np and the edges of the
nodes-per-lane split (np = 8 / 9, 11 / 12, 13 / 14) and of the 16-row tiles,
groups with a remainder, elements that share a geometric set and elements
that do not, essential and natural sides that meet at a corner, a mode
without a second plane, one to three fields, and the right-hand sides of PCG
modes.  Bar: relative L2 <= 1e-12, that of every direct solve; 1e-9 for PCG
solves stopped at 1e-12 of the right-hand side.
"""
import numpy as np
import pytest

import oracle_lib as O
import semtex_amd as sx
from semtex_amd.mesh import rect_mesh
from semtex_amd.workloads import helmholtz_batch
from solve_helpers import gpu_solve, natural_lines, oracle_solve, rel, solved

pytestmark = pytest.mark.gpu

CASES = [
    # kx, ky, np, nz, distort, bc (sides 0-3)
    (1, 1, 3, 1, 0.0, "DDDD"),
    (7, 5, 3, 6, 0.0, "DNDD"),
    (17, 3, 8, 4, 0.0, "DDDN"),
    (17, 3, 9, 4, 0.0, "DNDN"),
    (5, 4, 11, 6, 0.2, "DNDD"),
    (5, 7, 12, 4, 0.0, "DDDD"),
    (3, 2, 13, 2, 0.2, "DNDN"),
    (5, 3, 14, 4, 0.0, "DNDD"),
    (4, 3, 16, 4, 0.1, "DDDN"),
    (33, 1, 16, 2, 0.0, "DNDD"),
]


def _case(kx, ky, np_, nz, dist, bc, seed):
    m = rect_mesh(kx, ky, 0, 1.0 + 0.1 * kx, 0, 1.0 + 0.1 * ky, bc=tuple(bc), distort=dist)
    P, Q = sx.Mesh(np_, m), O.Mesh(np_, m)
    f, bcl, _ = helmholtz_batch(P, nz, 3.0, 1.3, seed=seed)
    if "N" in bc:
        bcl = natural_lines(P, nz, bcl)
    return P, Q, f, bcl


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{c[0]}x{c[1]}-np{c[2]}-{c[5]}")
def test_direct_parity(cuda, case):
    import torch
    print(f"[elem] {case}", flush=True)
    kx, ky, np_, nz, dist, bc = case
    nm = max(nz // 2, 1)
    P, Q, f0, b0 = _case(*case, seed=3)
    S = sx.ModalMatrixSys(P, 3.0, 1.3, 0, nm, nz, sx.DIRECT)
    ins = [(f0, b0)] + [_case(*case, seed=3 + i)[2:] for i in (1, 2)]
    dev = torch.device("cuda:0")
    for nf in (1, 2, 3):
        fs = [torch.from_numpy(f.ravel().copy()).to(dev) for f, _ in ins[:nf]]
        bs = [torch.from_numpy(b.ravel().copy()).to(dev) for _, b in ins[:nf]]
        us = [torch.zeros_like(t) for t in fs]
        sx.solve_fields(S, fs, bs, us)
        torch.cuda.synchronize()
        for (f, b), t, u in zip(ins, fs, us):
            uo, _ = oracle_solve(Q, nz, 3.0, 1.3, f, b)
            r = rel(solved(P, u.cpu().numpy().reshape(f.shape)), solved(P, uo))
            print(f"  fields {nf}: rel L2 {r:.3e}", flush=True)
            assert r <= 1e-12
            assert np.array_equal(t.cpu().numpy(), f.ravel())     # the forcing is only read


@pytest.mark.parametrize("case", [CASES[1], CASES[3], CASES[6]],
                         ids=lambda c: f"{c[0]}x{c[1]}-np{c[2]}")
def test_mixed_parity(cuda, case):
    import torch
    print(f"[elem] mixed {case}", flush=True)
    P, Q, f, bcl = _case(*case, seed=9)
    nz = case[3]
    S = sx.ModalMatrixSys(P, 3.0, 1.3, 0, max(nz // 2, 1), nz, sx.MIXED)
    ug, _ = gpu_solve(torch, P, S, f, bcl)
    uo, _ = oracle_solve(Q, nz, 3.0, 1.3, f, bcl)
    assert rel(solved(P, ug), solved(P, uo)) <= 1e-9


def test_solution_in_place_of_forcing(cuda):
    """u and f may be one buffer: each element is read before it is written."""
    import torch
    P, Q, f, bcl = _case(*CASES[3], seed=5)
    nz = CASES[3][3]
    S = sx.ModalMatrixSys(P, 3.0, 1.3, 0, nz // 2, nz, sx.DIRECT)
    dev = torch.device("cuda:0")
    t = torch.from_numpy(f.ravel().copy()).to(dev)
    b = torch.from_numpy(bcl.ravel().copy()).to(dev)
    sx.solve(S, t, b, t, iters=False)
    torch.cuda.synchronize()
    uo, _ = oracle_solve(Q, nz, 3.0, 1.3, f, bcl)
    assert rel(solved(P, t.cpu().numpy().reshape(f.shape)), solved(P, uo)) <= 1e-12
