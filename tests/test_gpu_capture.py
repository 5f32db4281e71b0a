"""Solves captured into a HIP graph right after a solve that changed how the
next one is launched: a call under capture allocates nothing, so whatever it
launches from has to be in place by then.  Three replays with eager work
between them equal the eager solve bit for bit.
"""
import numpy as np
import pytest

import semtex_amd as sx
from semtex_amd.mesh import rect_mesh
from semtex_amd.workloads import helmholtz_batch

pytestmark = pytest.mark.gpu

SWITCHES = ("SEMX_AUTOTUNE", "SEMX_BAND_COOP", "SEMX_BAND_XCOOP", "SEMX_BAND_PARTS", "SEMX_TREE",
            "SEMX_PCG_WG", "SEMX_PCG_OP", "SEMX_PCG_CHIP")


@pytest.fixture(autouse=True)
def default_switches(monkeypatch):
    for v in SWITCHES:
        monkeypatch.delenv(v, raising=False)


def _case(kx, ky, np_, nz, seeds, quiet=0):
    """Mesh and per-seed device (f, bc); the first `quiet` planes of f and bc
    are zero, so that their planes take no iterations."""
    import torch
    P = sx.Mesh(np_, rect_mesh(kx, ky, 0, 0.5 * kx, 0, 0.5 * ky, distort=0.1))
    ins = []
    for seed in seeds:
        f, b, _ = helmholtz_batch(P, nz, 2.0, 1.2, seed=seed)
        f[:quiet], b[:quiet] = 0.0, 0.0
        ins.append([torch.from_numpy(a.ravel().copy()).to("cuda:0") for a in (f, b)])
    return P, ins


def _capture_and_replay(torch, call, ref):
    """call(us) captured on its own output buffers, replayed three times."""
    us = [torch.zeros_like(r) for r in ref]
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        for u in us:
            u.zero_()
        call(us)
    for _ in range(3):
        for u in us:
            u.fill_(1.0)
        g.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(u, r) for u, r in zip(us, ref))
        vs = [torch.zeros_like(r) for r in ref]
        call(vs)
        torch.cuda.synchronize()
        assert all(torch.equal(v, r) for v, r in zip(vs, ref))


@pytest.mark.parametrize("kx,ky", [(4, 3), (17, 9)], ids=["one-workgroup", "several"])
def test_pcg_captured_after_reranking(cuda, kx, ky):
    """Iteration counts read back reverse the order the planes are taken in
    (the low modes, listed first, take none); the next solve is captured."""
    import torch
    print(f"[capture] reranked {kx}x{ky}", flush=True)
    P, [(f, b)] = _case(kx, ky, 6, 16, [1], quiet=8)
    S = sx.ModalMatrixSys(P, 2.0, 1.2, 0, 8, 16, sx.JACPCG)
    ref = torch.zeros_like(f)
    sx.solve(S, f, b, ref)                      # counts read back
    it = S.plane_iters()
    assert it[:8].max() == 0 and it[8:].min() > 0
    _capture_and_replay(torch, lambda u: sx.solve(S, f, b, u[0], iters=False), [ref])


def test_batch_reranked_solves_repeat(cuda):
    """A batch whose measured counts change the order its problems are taken
    in gives the same bits in every order."""
    import torch
    sizes = [(3, 3, 5), (9, 8, 6), (2, 2, 9), (17, 9, 6), (5, 4, 7)]
    hs, fs, bs, keep = [], [], [], []
    for i, (kx, ky, np_) in enumerate(sizes):
        # the largest problems take no iterations
        P, [(f, b)] = _case(kx, ky, np_, 1, [i], quiet=int(kx > 6))
        keep.append(P)
        hs.append(sx.ModalMatrixSys(P, 2.0, 1.2, 0, 1, 1, sx.JACPCG))
        fs.append(f)
        bs.append(b)
    B = sx.Batch(hs)
    ref = None
    for r in range(4):
        us = [torch.zeros_like(f) for f in fs]
        B.solve(fs, bs, us, iters=r != 2)
        torch.cuda.synchronize()
        ref = ref or us
        assert all(torch.equal(u, v) for u, v in zip(us, ref)), r


@pytest.mark.parametrize("method", [sx.DIRECT, sx.JACPCG, sx.MIXED], ids=["direct", "jacpcg", "mixed"])
def test_fewer_fields_captured(cuda, method):
    """A system solved with three fields captures a solve of one and of two
    without solving that many before."""
    import torch
    print(f"[capture] fields, method {method}", flush=True)
    P, ins = _case(7, 6, 6, 8, [3, 4, 5])
    S = sx.ModalMatrixSys(P, 2.0, 1.2, 0, 4, 8, method)
    fs, bs = [i[0] for i in ins], [i[1] for i in ins]
    ref = [torch.zeros_like(f) for f in fs]
    sx.solve_fields(S, fs, bs, ref, iters=False)
    torch.cuda.synchronize()
    for nf in (1, 2):
        _capture_and_replay(
            torch, lambda us: sx.solve_fields(S, fs[:nf], bs[:nf], us, iters=False), ref[:nf])


@pytest.mark.parametrize("method", [sx.DIRECT, sx.JACPCG, sx.MIXED], ids=["direct", "jacpcg", "mixed"])
def test_captured_solve_outlives_larger_ones(cuda, method):
    """A solve of one field captured, then solves of two and three fields,
    which need larger scratch: the graph keeps its own."""
    import torch
    print(f"[capture] outgrown scratch, method {method}", flush=True)
    P, ins = _case(17, 9, 6, 8, [3, 4, 5])
    S = sx.ModalMatrixSys(P, 2.0, 1.2, 0, 4, 8, method)
    fs, bs = [i[0] for i in ins], [i[1] for i in ins]
    ref = [torch.zeros_like(f) for f in fs]
    sx.solve(S, fs[0], bs[0], ref[0], iters=False)
    u = torch.zeros_like(fs[0])
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        u.zero_()
        sx.solve(S, fs[0], bs[0], u, iters=False)
    for nf in (2, 3):
        vs = [torch.zeros_like(f) for f in fs[:nf]]
        sx.solve_fields(S, fs[:nf], bs[:nf], vs, iters=False)
        keep = torch.full((1 << 22,), 7.0, dtype=torch.float64, device="cuda:0")   # reuse what was freed
        u.fill_(1.0)
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(u, ref[0]) and torch.equal(vs[0], ref[0])
        assert float(keep.min()) == 7.0 and float(keep.max()) == 7.0


@pytest.mark.parametrize("prec", [sx.PCG_FP64, sx.PCG_BF16_REFINED], ids=["fp64", "bf16r"])
def test_batch_captured(cuda, prec):
    """A batch's solve captured (100 problems: more pointers than one block of
    them), replayed between eager solves into other buffers."""
    import torch
    print(f"[capture] batch, precision {prec}", flush=True)
    hs, fs, bs, keep = [], [], [], []
    for i in range(100):
        P, [(f, b)] = _case(2 + i % 4, 2 + i % 3, 4 + i % 5, 1, [i])
        S = sx.ModalMatrixSys(P, 2.0, 1.2, 0, 1, 1, sx.JACPCG)
        if prec == sx.PCG_BF16_REFINED:
            S.set_pcg(prec, inner_tol=1e-2, max_outer=80)
        keep.append(P)
        hs.append(S)
        fs.append(f)
        bs.append(b)
    B = sx.Batch(hs)
    ref = [torch.zeros_like(f) for f in fs]
    B.solve(fs, bs, ref)
    _capture_and_replay(torch, lambda us: B.solve(fs, bs, us, iters=False), ref)


def test_captured_after_precision_change(cuda):
    """Three fields solved in one kernel, one field in the other after a change
    of precision: a solve of two fields is captured in either."""
    import torch
    print("[capture] precision changes", flush=True)
    P, ins = _case(17, 9, 6, 8, [3, 4, 5])
    fs, bs = [i[0] for i in ins], [i[1] for i in ins]
    bf16 = dict(precision=sx.PCG_BF16_REFINED, inner_tol=1e-2, max_outer=120)
    for first, second in ((bf16, {}), ({}, bf16)):
        S = sx.ModalMatrixSys(P, 2.0, 1.2, 0, 4, 8, sx.JACPCG)
        S.set_pcg(**first)
        sx.solve_fields(S, fs, bs, [torch.zeros_like(f) for f in fs], iters=False)
        S.set_pcg(**second)
        sx.solve(S, fs[0], bs[0], torch.zeros_like(fs[0]), iters=False)
        us = [torch.zeros_like(f) for f in fs[:2]]
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            for u in us:
                u.zero_()
            sx.solve_fields(S, fs[:2], bs[:2], us, iters=False)
        g.replay()
        torch.cuda.synchronize()
        for f, b, u in zip(fs, bs, us):
            v = torch.zeros_like(f)
            sx.solve(S, f, b, v, iters=False)
            torch.cuda.synchronize()
            assert torch.equal(u, v)
