"""Set-up of a small direct system (no GPU): the elimination tree's dense
matrices cost no more time than the band factor they stand in for.  The best
of several runs each; the bar leaves room for a loaded host (measured 0.75 of
the band's time; 1.9 when a merged region was factorised as one matrix).
"""
import time

import pytest

import semtex_amd as sx
from semtex_amd.mesh import rect_mesh


@pytest.mark.parametrize("kx,ky,np_,nz,distort", [(11, 7, 6, 36, 0.2), (8, 8, 8, 1, 0.0)])
def test_setup_no_slower_than_band(kx, ky, np_, nz, distort, monkeypatch):
    for v in ("SEMX_AUTOTUNE", "SEMX_BAND_COOP", "SEMX_BAND_XCOOP", "SEMX_BAND_PARTS", "SEMX_TREE"):
        monkeypatch.delenv(v, raising=False)
    P = sx.Mesh(np_, rect_mesh(kx, ky, 0, 1.0, 0, 1.0, distort=distort))

    def create():
        t = time.perf_counter()
        S = sx.ModalMatrixSys(P, 3.0, 1.0, 0, max(nz // 2, 1), nz, sx.DIRECT)
        t = time.perf_counter() - t
        del S
        return t

    best = {"tree": 1e9, "band": 1e9}
    for _ in range(8):
        monkeypatch.delenv("SEMX_TREE", raising=False)
        best["tree"] = min(best["tree"], create())
        monkeypatch.setenv("SEMX_TREE", "0")
        best["band"] = min(best["band"], create())
    print({k: f"{1e3 * v:.1f} ms" for k, v in best.items()})
    assert best["tree"] <= 1.4 * best["band"]
