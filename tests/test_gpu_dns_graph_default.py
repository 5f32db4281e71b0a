"""DNS steps replayed from HIP graphs with the default solvers (direct systems
along the elimination tree, start-up systems on chip) against the same steps
launched kernel by kernel: bit for bit, over two full cycles of the step's
buffer roles, periodic and bounded, in 2D and 3D.  A cycle, and so the graphs
captured, is 2 N_TIME + 1 steps, twice that for the alternating form; with
planes at N_TIME = 3, 88 steps of the skew-symmetric form and 182 of the
alternating one.
"""
import numpy as np
import pytest

import semtex_amd as sx
from semtex_amd.mesh import rect_mesh

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def default_switches(monkeypatch):
    for v in ("SEMX_AUTOTUNE", "SEMX_BAND_COOP", "SEMX_BAND_XCOOP", "SEMX_BAND_PARTS", "SEMX_TREE",
              "SEMX_PCG_CHIP", "SEMX_PCG_WG", "SEMX_PCG_OP"):
        monkeypatch.delenv(v, raising=False)


def _field(P, nz, c):
    a = np.zeros((nz, P.planeSize))
    for k in range(0, min(nz, 6)):
        if k != 1:
            q = np.random.default_rng(10 * c + k).standard_normal(3)
            a[k, :P.nPlane] = 0.3 * q[0] * np.sin(P.x + q[1]) * np.cos(P.y + q[2])
    return a.reshape(-1)


@pytest.mark.parametrize("walls", [False, True], ids=["periodic", "walls"])
@pytest.mark.parametrize("nz,adv,norder,cycle", [
    (8, 0, 3, 88), (8, 1, 3, 182), (8, 2, 3, 7), (8, 0, 2, 5), (8, 1, 1, 6), (8, 3, 2, 5),
    (2, 0, 3, 7), (2, 1, 2, 10), (1, 0, 3, 7), (1, 1, 3, 14), (1, 0, 1, 3)])
def test_replay_equals_eager(cuda, nz, adv, norder, cycle, walls):
    import torch
    steps, nc = 2 * cycle, 3 if nz > 1 else 2
    m = rect_mesh(6, 5, 0, 2 * np.pi, 0, 2 * np.pi, bc=("D",) * 4, periodic_x=True,
                  periodic_y=not walls)
    P = sx.Mesh(5, m)
    kw = {}
    if walls:
        mp = dict(m, skind=np.where(m["skind"] == 1, 2, m["skind"]).astype(np.int32))
        kw["pressure_mesh"] = sx.Mesh(5, mp)
        kw["bc"] = [torch.zeros(nz * P.nline, dtype=torch.float64, device="cuda:0") for _ in range(nc)]
    out = []
    for graphs in (False, True):
        print(f"[dns replay] nz {nz} advection {adv} N_TIME {norder} walls {walls} graphs {graphs}", flush=True)
        D = sx.DNS(P, nz, 1.0, 1e-3, 0.02, norder=norder, advection=adv, tol_rel=1e-12,
                   step_max=500, **kw)
        D.set_graph(graphs)
        f = [torch.from_numpy(_field(P, nz, c) * (c < nc)).to("cuda:0") for c in range(3)]
        f.append(torch.zeros_like(f[0]))
        for n in (norder, steps // 2, steps - steps // 2):
            D.run(n, *f)
        torch.cuda.synchronize()
        ng, rp = D.graph_info()
        print(f"  graphs {ng}, replayed steps {rp}", flush=True)
        assert (ng, rp) == ((cycle, steps) if graphs else (0, 0))
        out.append([t.clone() for t in f])
        del D
    for name, a, b in zip("uvwp", out[0], out[1]):
        assert torch.equal(a, b), name
        assert bool(torch.isfinite(a).all()), name
    assert float(out[0][0].abs().max()) > 0.01
