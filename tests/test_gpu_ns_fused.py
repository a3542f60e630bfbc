"""The Navier-Stokes step's fused vector passes against the same sums in
torch: ssxk_ns_rk_stage for every number of terms with and without the
stage's argument and with one or three components, its result in place of one
of the terms, ssxk_ns_rk_end, and ssxk_ns_dss3 bit for bit against ssxk_dss_all
one field at a time; lengths around one workgroup of 256.

Bar, per value: m terms are m fused multiply-adds here, products and sums
there, and the inverse mass is one product: at most 2 (m + 2) eps of the sum
of the terms' magnitudes."""
import ctypes as C

import numpy as np
import pytest

torch = pytest.importorskip("torch")

import ssenss_amd as S  # noqa: E402

pytestmark = pytest.mark.gpu
EPS = np.finfo(float).eps
LENGTHS = [1, 255, 256, 257, 5000]


def _st():
    return C.c_void_p(torch.cuda.current_stream().cuda_stream)


def _ptrs(ts):
    return (C.c_void_p * len(ts))(*[t.data_ptr() for t in ts])


def _mk(n, k, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return [torch.randn(n, generator=g, device="cuda", dtype=torch.float64)
            for _ in range(k)]


@pytest.mark.parametrize("stage", [False, True])
@pytest.mark.parametrize("terms", range(4))
@pytest.mark.parametrize("n", LENGTHS)
def test_rk_stage(n, terms, stage):
    L = S.load()
    co = [0.375, -1.7, 0.9]
    for nc in (1, 3):
        x, ut, f = _mk(n, 9, n), _mk(n, 3, 1), _mk(n, 3, 2)
        im = _mk(n, 1, 3)[0].abs()
        a, y = [[torch.full((n,), 7.0, device="cuda", dtype=torch.float64)
                 for _ in range(3)] for _ in range(2)]
        a[0] = x[3 * (terms - 1)] if terms else a[0]     # in place
        want, bound = [], []
        for c in range(nc):
            t = [co[k] * x[3 * k + c] for k in range(terms)]
            want.append(sum(t) + 0 * im)
            bound.append(sum(v.abs() for v in t) + 0 * im)
        assert L.ssxk_ns_rk_stage(
            _st(), C.c_size_t(n), nc, terms, _ptrs(x), (C.c_double * 3)(*co),
            _ptrs(ut), _ptrs(f) if stage else None, C.c_void_p(im.data_ptr()),
            C.c_double(-0.3), _ptrs(a), _ptrs(y)) == 0
        torch.cuda.synchronize()
        for c in range(3):
            if terms and c < nc:
                assert ((a[c] - want[c]).abs()
                        <= 2 * (terms + 2) * EPS * bound[c]).all()
            elif c:
                assert (a[c] == 7.0).all()
            if stage and c < nc:
                g = -0.3 * (im * f[c])
                assert ((y[c] - (ut[c] + g)).abs()
                        <= 6 * EPS * (ut[c].abs() + g.abs())).all()
            else:
                assert (y[c] == 7.0).all()


@pytest.mark.parametrize("n", LENGTHS)
def test_rk_end(n):
    L = S.load()
    f, ut, im = _mk(n, 12, n), _mk(n, 3, 1), _mk(n, 1, 3)[0]
    co = [-0.25, 0.7, 0.7, -0.25]
    t = [[co[i] * (im * f[3 * i + c]) for i in range(4)] for c in range(3)]
    want = [ut[c] + sum(t[c]) for c in range(3)]
    bound = [ut[c].abs() + sum(v.abs() for v in t[c]) for c in range(3)]
    assert L.ssxk_ns_rk_end(_st(), C.c_size_t(n), _ptrs(f),
                            C.c_void_p(im.data_ptr()), C.c_double(co[0]),
                            C.c_double(co[1]), _ptrs(ut)) == 0
    torch.cuda.synchronize()
    for c in range(3):
        assert ((ut[c] - want[c]).abs() <= 12 * EPS * bound[c]).all()


@pytest.mark.parametrize("groups", [(0, 0, 0), (300, 0, 1), (0, 257, 0),
                                    (256, 1, 256), (5, 300, 40)])
def test_dss3(groups):
    L = S.load()
    size = [2, 4, 8]
    n = sum(g * m for g, m in zip(groups, size)) + 11
    perm = torch.randperm(n, generator=torch.Generator().manual_seed(n)).int()
    lists, at = [], 0
    for g, m in zip(groups, size):
        lists.append(perm[at:at + g * m].cuda())
        at += g * m
    grp, ng = _ptrs(lists), (C.c_longlong * 3)(*groups)
    u = _mk(n, 3, 5)
    one = [v.clone() for v in u]
    for v in one:
        assert L.ssxk_dss_all(_st(), grp, ng, C.c_void_p(v.data_ptr()), None,
                              None, 0, None) == 0
    assert L.ssxk_ns_dss3(_st(), grp, ng, _ptrs(u)) == 0
    torch.cuda.synchronize()
    assert all(torch.equal(v, w) for v, w in zip(u, one))
