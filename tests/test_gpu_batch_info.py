"""What semx_batch_info says of a batch held on chip (no operator before the
first solve, then the wavefront-level one and no tuner) and of one that is not
(BF16 refinement, tuned on its first solve)."""
import pytest

import semtex_amd as sx
from semtex_amd.mesh import rect_mesh
from semtex_amd.workloads import single_plane_problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [sx.PCG_FP64, sx.PCG_FP32_REFINED, sx.PCG_BF16_REFINED],
                         ids=["fp64", "fp32r", "bf16r"])
def test_batch_info(cuda, prec, monkeypatch):
    import torch
    for v in ("SEMX_BATCH_OP", "SEMX_BATCH_WG", "SEMX_PCG_CHIP"):
        monkeypatch.delenv(v, raising=False)
    print(f"[batch info] precision {prec}", flush=True)
    meshes, hs, fs, bs = [], [], [], []
    for i, (k, np_) in enumerate(((3, 5), (4, 8), (6, 6))):
        P = sx.Mesh(np_, rect_mesh(k, k, 0, 1.0, 0, 1.0))
        f, b, _ = single_plane_problem(P, 3.0, i)
        S = sx.ModalMatrixSys(P, 3.0, 1.0, 0, 1, 1, sx.JACPCG)
        if prec != sx.PCG_FP64:
            S.set_pcg(prec, inner_tol=1e-2, max_outer=80)
        meshes.append(P)
        hs.append(S)
        fs.append(torch.from_numpy(f.ravel().copy()).to("cuda:0"))
        bs.append(torch.from_numpy(b.ravel().copy()).to("cuda:0"))
    B = sx.Batch(hs)
    assert B.info() == ([None] * 3, 0.0)
    B.solve(fs, bs, [torch.zeros_like(f) for f in fs], iters=False)
    ops, ms = B.info()
    if prec == sx.PCG_BF16_REFINED:
        assert set(ops) <= {"wave", "mfma"} and ms > 0.0
    else:
        assert (ops, ms) == (["wave"] * 3, 0.0)
