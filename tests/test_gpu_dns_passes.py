"""The z transform and the fused passes of the time step where they can go
wrong: every even length of the FFT (radix 2, 3, 4 and 5 passes, one to four
of them, the shortest and longest) and lengths the dense product keeps,
columns that do not fill a workgroup; x / y derivatives and smoothing with a
plane count that leaves a remainder; time steps with two planes, with N_TIME
1 and 2, and at the smallest and largest np.

Bars: transforms, relative L2 <= 1e-14 against numpy in FP64 (a handful of
rounding errors of 1.1e-16 per pass, at most five passes and the split);
derivatives 1e-13 (np <= 9: at np = 16 the oracle's own derivative matrix is
5e-13 off a long-double one) and, plane by plane, the same bits; time steps
1e-12 against the CPU oracle.
"""
import ctypes as C

import numpy as np
import pytest

import oracle_lib as O
import semtex_amd as sx
from semtex_amd.mesh import rect_mesh
from solve_helpers import rel

pytestmark = pytest.mark.gpu

SMOOTH_LENGTHS = [n for n in range(2, 257) if not any(
    p > 5 for p in range(2, n + 1) if n % p == 0 and all(p % q for q in range(2, p)))]


@pytest.mark.parametrize("ntrn", [2, 34, 322])
def test_dft_lengths(cuda, ntrn):
    import torch
    rng = np.random.default_rng(ntrn)
    for N in SMOOTH_LENGTHS:
        if N % 2:
            continue
        x = rng.standard_normal((N, ntrn))
        X = np.fft.rfft(x, axis=0) / N
        s = np.zeros_like(x)
        s[0], s[1] = X[0].real, X[N // 2].real
        s[2::2], s[3::2] = X[1:N // 2].real, X[1:N // 2].imag
        t = torch.from_numpy(x.reshape(-1).copy()).to("cuda:0")
        sx.dft_r(t, N, ntrn, sx.FORWARD)
        f = rel(t.cpu().numpy().reshape(x.shape), s)
        t = torch.from_numpy(s.reshape(-1).copy()).to("cuda:0")
        sx.dft_r(t, N, ntrn, sx.INVERSE)
        b = rel(t.cpu().numpy().reshape(x.shape), x)
        assert max(f, b) <= 1e-14, (N, f, b)


def test_dft_odd_lengths(cuda):
    """Odd lengths take the dense product, as they always did."""
    import torch
    for N in (3, 5, 9, 15, 45, 135, 225):
        x = np.random.default_rng(N).standard_normal((N, 6))
        t = torch.from_numpy(x.reshape(-1).copy()).to("cuda:0")
        sx.dft_r(t, N, 6, sx.FORWARD)
        assert rel(t.cpu().numpy().reshape(x.shape)[0], x.mean(0)) <= 1e-14


@pytest.mark.parametrize("np_,nz", [(3, 1), (5, 6), (9, 2), (16, 10)])
def test_operators(cuda, np_, nz):
    import torch
    m = rect_mesh(5, 3, 0, 2.0, 0, 1.5, distort=0.2)
    P, Q = sx.Mesh(np_, m), O.Mesh(np_, m)
    a = np.random.default_rng(np_).standard_normal((nz, P.planeSize))
    a[:, P.nPlane:] = 0.0
    for what in (0, 1, "smooth"):
        t = torch.from_numpy(a.reshape(-1).copy()).to("cuda:0")
        o = np.ascontiguousarray(a.copy())
        if what == "smooth":
            sx.smooth(P, nz, t)
            O.lib().orc_smooth(C.c_void_p(Q.h), nz, O.dp(o))
        else:
            sx.gradient(P, nz, 1.0, t, what)
            O.lib().orc_gradient(C.c_void_p(Q.h), nz, 1.0, O.dp(o), what)
        g = t.cpu().numpy().reshape(a.shape)
        if np_ <= 9:
            assert rel(g[:, :P.nPlane], o[:, :P.nPlane]) <= 1e-13, what
        # the planes one by one (the nz = 1 kernels): the same bits
        for k in range(nz):
            t = torch.from_numpy(a[k].copy()).to("cuda:0")
            sx.smooth(P, 1, t) if what == "smooth" else sx.gradient(P, 1, 1.0, t, what)
            assert np.array_equal(t.cpu().numpy(), g[k]), (what, k)


@pytest.mark.parametrize("np_,nz,norder,adv", [
    (7, 2, 3, 0), (7, 2, 2, 2), (3, 4, 2, 1), (16, 4, 1, 0), (6, 6, 2, 0), (5, 30, 3, 1)])
def test_dns_steps(cuda, np_, nz, norder, adv):
    import torch
    m = rect_mesh(4, 3, 0, 2 * np.pi, 0, 2 * np.pi, periodic_x=True, periodic_y=True)
    P, Q = sx.Mesh(np_, m), O.Mesh(np_, m)
    rng = np.random.default_rng(np_ + nz)
    f = []
    for c in range(3):
        a = np.zeros((nz, P.planeSize))
        for k in range(min(nz, 6)):
            if k == 1:
                continue
            q = rng.standard_normal(3)
            a[k, :P.nPlane] = 0.3 * q[0] * np.sin(P.x + q[1]) * np.cos(P.y + q[2])
        f.append(a)
    f.append(np.zeros_like(f[0]))
    t = [torch.from_numpy(a.reshape(-1).copy()).to("cuda:0") for a in f]
    D = sx.DNS(P, nz, 1.0, 2e-3, 0.05, norder=norder, advection=adv, tol_rel=1e-14, step_max=2000)
    D.run(6, *t)
    o = [np.ascontiguousarray(a.copy()) for a in f]
    Do = O.lib().orc_dns_create(C.c_void_p(Q.h), nz, 1.0, 2e-3, 0.05, norder, adv, 1e-14, 2000, 0)
    tm = C.c_double()
    O.lib().orc_dns_run(C.c_void_p(Do), 6, *(O.dp(a) for a in o), C.byref(tm))
    O.lib().orc_dns_destroy(C.c_void_p(Do))
    keep = [k for k in range(nz) if k != 1]
    for name, g, r in zip("uvw", t, o):
        g = g.cpu().numpy().reshape(r.shape)
        assert rel(g[keep, :P.nPlane], r[keep, :P.nPlane]) <= 1e-12, name
        assert np.array_equal(g[1], f["uvw".index(name)][1])     # the Nyquist plane is left alone
