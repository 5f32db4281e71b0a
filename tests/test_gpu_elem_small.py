"""Element condensation and recovery of the smallest elements against the CPU
FP64 oracle: np = 3 (a thread per node), np = 4 and 5 of one geometry and of
one each (a wavefront per element; counts that leave a workgroup part empty),
with one to three fields, with and without a second plane, and with the
solution in place of the forcing.  Bar: relative L2 <= 1e-12, that of every
direct solve.
"""
import numpy as np
import pytest

import oracle_lib as O
import semtex_amd as sx
from semtex_amd.mesh import rect_mesh
from semtex_amd.workloads import helmholtz_batch
from solve_helpers import natural_lines, oracle_solve, rel, solved

pytestmark = pytest.mark.gpu

CASES = [(kx, ky, np_, nz, d, bc) for np_ in (3, 4, 5) for kx, ky, nz, d, bc in (
    (1, 1, 4, 0.0, "DNDN"), (7, 5, 6, 0.2, "DNDD"), (9, 7, 1, 0.15, "DDDN"), (6, 4, 2, 0.0, "DDDD"),
    (23, 11, 8, 0.2, "DDDD"))]


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{c[0]}x{c[1]}-np{c[2]}-nz{c[3]}")
def test_small_elements(cuda, case):
    import torch
    print(f"[small elements] {case}", flush=True)
    kx, ky, np_, nz, dist, bc = case
    m = rect_mesh(kx, ky, 0, 1.0 + 0.1 * kx, 0, 1.0 + 0.1 * ky, bc=tuple(bc), distort=dist)
    P, Q = sx.Mesh(np_, m), O.Mesh(np_, m)
    ins = []
    for seed in (1, 2, 3):
        f, b, _ = helmholtz_batch(P, nz, 3.0, 1.3, seed=seed)
        ins.append((f, natural_lines(P, nz, b) if "N" in bc else b))
    ref = [solved(P, oracle_solve(Q, nz, 3.0, 1.3, f, b)[0]) for f, b in ins]
    S = sx.ModalMatrixSys(P, 3.0, 1.3, 0, max(nz // 2, 1), nz, sx.DIRECT)
    dev = torch.device("cuda:0")
    for nf in (1, 2, 3):
        fs = [torch.from_numpy(f.ravel().copy()).to(dev) for f, _ in ins[:nf]]
        bs = [torch.from_numpy(b.ravel().copy()).to(dev) for _, b in ins[:nf]]
        us = [torch.zeros_like(t) for t in fs]
        sx.solve_fields(S, fs, bs, us)
        sx.solve_fields(S, fs, bs, fs)
        torch.cuda.synchronize()
        for r, u, v in zip(ref, us, fs):
            g = u.cpu().numpy().reshape(nz, -1)
            w = v.cpu().numpy().reshape(nz, -1)
            assert rel(solved(P, g), r) <= 1e-12
            assert np.array_equal(solved(P, g), solved(P, w))
