"""The convection operator's kernel (ssxk_ns_conv) at every order it takes
against the same operator in numpy: n = 2..10 points interpolated to nc =
3n/2, whose line counts nc^2 fill their last tile of 16 fully (nc = 4, 12),
by one line (nc = 7, 9, 13, 15) or partly, on 1 and 3 elements.

Bar, per value: the operator evaluated with absolute values everywhere
bounds the sum of the magnitudes of all terms a value is summed from; one
term passes through at most n + n + n (interpolation), nc (derivative),
nc + nc + nc (integration) additions and about 20 products, so a correct
evaluation differs from another by at most 2 (3 n + 4 nc + 20) eps of that
bound."""
import ctypes as C

import numpy as np
import pytest

torch = pytest.importorskip("torch")

import ssenss_amd as S  # noqa: E402
from oracle import pyoracle as P  # noqa: E402

pytestmark = pytest.mark.gpu


def _operator(pr, D, u, v, g):
    """pr[p, i] = l_p(xi_i), D[i, l]; u, v [3, nel, n, n, n] (z, y, x); g
    [nel, 9, nc, nc, nc]"""
    up = lambda a: np.einsum("pi,qj,rk,fepqr->feijk", pr, pr, pr, a,
                             optimize=True)
    U, V = up(u), up(v)
    d = [lambda a: np.einsum("il,ezyl->ezyi", D, a),
         lambda a: np.einsum("jl,ezlx->ezjx", D, a),
         lambda a: np.einsum("kl,elyx->ekyx", D, a)]
    out = []
    for c in range(3):
        s = 0.0
        for b in range(3):
            cb = sum(U[a] * g[:, 3 * a + b] for a in range(3))
            tb = sum(g[:, 3 * a + b] for a in range(3))
            s = s + 0.5 * (cb * d[b](V[c]) + tb * d[b](U[b] * V[c]))
        out.append(np.einsum("pi,qj,rk,eijk->epqr", pr, pr, pr, s,
                             optimize=True))
    return np.stack(out)


@pytest.mark.parametrize("nel", [1, 3])
@pytest.mark.parametrize("n", range(2, 11))
def test_convection_every_order(n, nel):
    nc = 3 * n // 2
    rng = np.random.default_rng(10 * n + nel)
    pr = np.asarray(P.interp_matrix(n, nc)).reshape(n, nc)
    D = np.asarray(P.gll_basis(nc)[2]).reshape(nc, nc)
    u, v = rng.standard_normal((2, 3, nel, n, n, n))
    g = rng.standard_normal((nel, 9, nc, nc, nc))
    ref = _operator(pr, D, u, v, g)
    bound = _operator(*(np.abs(a) for a in (pr, D, u, v, g)))
    L = S.load()
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    dp, dd, dg = dev(pr), dev(D), dev(g)
    du, dv = [dev(a) for a in u], [dev(a) for a in v]
    do = [torch.full_like(a, np.nan) for a in du]
    arr = lambda t: (C.c_void_p * 3)(*[a.data_ptr() for a in t])
    torch.cuda.synchronize()
    rc = L.ssxk_ns_conv(None, nel, n, C.c_void_p(dp.data_ptr()),
                        C.c_void_p(dd.data_ptr()), arr(du), arr(dv),
                        C.c_void_p(dg.data_ptr()), arr(do))
    torch.cuda.synchronize()
    assert rc == 0
    got = np.stack([a.cpu().numpy() for a in do])
    err = np.abs(got - ref) / bound
    print(f"[gpu] convection n={n} nel={nel}: {err.max():.2e}")
    assert err.max() <= 2 * (3 * n + 4 * nc + 20) * 2.3e-16


def test_convection_order_refused():
    L = S.load()
    assert L.ssxk_ns_conv(None, 1, 11, None, None, (C.c_void_p * 3)(),
                          (C.c_void_p * 3)(), None, (C.c_void_p * 3)()) == 1
