"""JACPCG held on chip against the CPU FP64 oracle, through the C ABI: every
np with a kernel of its own (4 to 12) and one on either side, planes in one
workgroup and in several, elements that share their factors and elements that
do not (in registers up to np = 7, from memory above), FP64 and FP32 refined,
and a batch of all of them.  Bar: relative L2 <= 1e-9 for solves stopped at
1e-12 of the right-hand side (condition numbers below 1e3 here).
"""
import numpy as np
import pytest

import oracle_lib as O
import semtex_amd as sx
from semtex_amd.mesh import rect_mesh
from semtex_amd.workloads import helmholtz_batch
from solve_helpers import gpu_solve, oracle_solve, rel, solved

pytestmark = pytest.mark.gpu

LAM2, BETA = 40.0, 1.2


def _case(kx, ky, np_, nz, dist, seed):
    m = rect_mesh(kx, ky, 0, 0.5 * kx, 0, 0.5 * ky, distort=dist)
    P, Q = sx.Mesh(np_, m), O.Mesh(np_, m)
    f, bcl, _ = helmholtz_batch(P, nz, LAM2, BETA, seed=seed)
    return P, Q, f, bcl


@pytest.mark.parametrize("dist", [0.0, 0.15], ids=["uniform", "distorted"])
@pytest.mark.parametrize("np_", [3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13])
def test_planes(cuda, np_, dist):
    import torch
    for kx, ky, nz in ((3, 2, 1), (17, 9, 4)):
        print(f"[pcg chip] np {np_} distort {dist} {kx}x{ky} nz {nz}", flush=True)
        P, Q, f, bcl = _case(kx, ky, np_, nz, dist, seed=np_)
        uo, _ = oracle_solve(Q, nz, LAM2, BETA, f, bcl)
        for prec in ("FP64", "FP32"):
            S = sx.ModalMatrixSys(P, LAM2, BETA, 0, max(nz // 2, 1), nz, sx.JACPCG)
            if prec == "FP32":
                S.set_pcg(sx.PCG_FP32_REFINED, inner_tol=1e-4, max_outer=40)
            ug, it = gpu_solve(torch, P, S, f, bcl)
            r = rel(solved(P, ug), solved(P, uo))
            print(f"  {prec}: {it} iterations, rel L2 {r:.2e}", flush=True)
            assert r <= 1e-9


def test_batch_of_every_np(cuda):
    import torch
    dev = torch.device("cuda:0")
    sizes = [(3, 2, n) for n in range(4, 13)] + [(13, 8, n) for n in range(4, 13)]
    for prec in ("FP64", "FP32"):
        hs, fs, bs, us, ref, keep = [], [], [], [], [], []
        for i, (kx, ky, np_) in enumerate(sizes):
            P, Q, f, bcl = _case(kx, ky, np_, 1, 0.1 * (i % 2), seed=50 + i)
            S = sx.ModalMatrixSys(P, LAM2, BETA, 0, 1, 1, sx.JACPCG)
            if prec == "FP32":
                S.set_pcg(sx.PCG_FP32_REFINED, inner_tol=1e-4, max_outer=40)
            keep.append(P)
            hs.append(S)
            fs.append(torch.from_numpy(f.ravel().copy()).to(dev))
            bs.append(torch.from_numpy(bcl.ravel().copy()).to(dev))
            us.append(torch.zeros_like(fs[-1]))
            ref.append((P, oracle_solve(Q, 1, LAM2, BETA, f, bcl)[0]))
        B = sx.Batch(hs)
        B.solve(fs, bs, us, tol_rel=1e-12, step_max=10000)
        torch.cuda.synchronize()
        for (P, uo), u in zip(ref, us):
            assert rel(u.cpu().numpy()[:P.nPlane], uo[0, :P.nPlane]) <= 1e-9
