"""The Navier-Stokes step's derivative operators (ssxk_ns_curl, ssxk_ns_div,
ssxk_ns_grad) against numpy at every order they take, n = 2..10, on one
element, on one element past a workgroup's share (512 / n^3 of them, at least
one) and on a few of these shares.

Bar, per value: with absolute values everywhere the same operator bounds the
sum of the magnitudes of its terms; a term passes through at most n additions
of a derivative, 9 of the components and about 6 products, so two correct
evaluations differ by at most 2 (n + 15) eps of that bound."""
import ctypes as C

import numpy as np
import pytest

torch = pytest.importorskip("torch")

import ssenss_amd as S  # noqa: E402
from oracle import pyoracle as P  # noqa: E402

pytestmark = pytest.mark.gpu
X = ["il,ezyl->ezyi", "jl,ezlx->ezjx", "kl,elyx->ekyx"]


def _curl(D, a, ti, w, minus):
    """minus -1.0: the curl; 1.0, on absolute values: its bound"""
    J = [[np.einsum(X[b], D, a[c]) for b in range(3)] for c in range(3)]
    out = []
    for c in range(3):
        k, l = (5 - c) // 2, (2 - c) // 2
        s = minus if c == 1 else 1.0
        out.append(w * sum(s * J[k][i] * ti[3 * l + i]
                           + s * minus * J[l][i] * ti[3 * k + i]
                           for i in range(3)))
    return np.stack(out)


def _div(D, a, ti, w, scale):
    return scale * w * sum(np.einsum(X[b], D, a[c]) * ti[3 * c + b]
                           for c in range(3) for b in range(3))


def _grad(D, p, ti, w, sign):
    return np.stack([sign * sum(np.einsum(X[b], D.T, ti[3 * c + b] * (p * w))
                                for b in range(3)) for c in range(3)])


@pytest.mark.parametrize("shares", [0, 1, 3])
@pytest.mark.parametrize("n", range(2, 11))
def test_operators(n, shares):
    nel = shares * max(512 // n ** 3, 1) + 1
    rng = np.random.default_rng(10 * n + shares)
    D = np.asarray(P.gll_basis(n)[2]).reshape(n, n)
    a = rng.standard_normal((3, nel, n, n, n))
    ti = rng.standard_normal((9, nel, n, n, n))
    w = rng.random((nel, n, n, n)) + 0.1
    L = S.load()
    dev = lambda v: torch.from_numpy(np.ascontiguousarray(v)).cuda()
    ptr = lambda ts: (C.c_void_p * len(ts))(*[t.data_ptr() for t in ts])
    one = lambda t: C.c_void_p(t.data_ptr())
    st = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    dd, dw = dev(D), dev(w)
    da, dt = [dev(v) for v in a], [dev(v) for v in ti]
    guard = 64                      # nothing is written past the elements
    out = [torch.full((w.size + guard,), 7.0, device="cuda",
                      dtype=torch.float64) for _ in range(3)]
    aD, aa, at = np.abs(D), np.abs(a), np.abs(ti)
    bar = 2 * (n + 15) * np.finfo(float).eps

    def check(o, ref, bound):
        torch.cuda.synchronize()
        got = o.cpu().numpy()
        assert (got[w.size:] == 7.0).all()
        err = np.abs(got[:w.size].reshape(w.shape) - ref)
        assert (err <= bar * bound).all()

    for mass in (None, w):
        wv = np.ones_like(w) if mass is None else w
        assert L.ssxk_ns_curl(st, nel, n, one(dd), ptr(da), ptr(dt),
                              None if mass is None else one(dw),
                              ptr(out)) == 0
        ref, bound = _curl(D, a, ti, wv, -1.0), _curl(aD, aa, at, wv, 1.0)
        for c in range(3):
            check(out[c], ref[c], bound[c])
    assert L.ssxk_ns_div(st, nel, n, one(dd), ptr(da), ptr(dt), one(dw),
                         C.c_double(-2.5), one(out[0])) == 0
    check(out[0], _div(D, a, ti, w, -2.5), _div(aD, aa, at, w, 2.5))
    assert L.ssxk_ns_grad(st, nel, n, one(dd), one(da[0]), one(dw), ptr(dt),
                          ptr(out)) == 0
    ref, bound = _grad(D, a[0], ti, w, -1.0), _grad(aD, aa[0], at, w, 1.0)
    for c in range(3):
        check(out[c], ref[c], bound[c])
