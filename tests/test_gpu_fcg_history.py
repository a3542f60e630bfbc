"""The flexible CG's passes over its history at every length: the inner
products of ssxk_multidot bit for bit those of one vector at a time and near
k_dot's, on lengths below one block, around one round of the grid
(1024 * 256) and around the rounds that go out together (2, 3, 4 and 6 of
them); the scalars of ssxk_fcg_pair.

Bar of an inner product against k_dot's (the same order of additions, but a
product of its own where the other has a fused multiply-add): a term passes
through the rounds of its lane, 8 + 2 + 8 levels of trees and two products,
so they differ by at most 2 (rounds + 20) eps of sum |x s y|."""
import ctypes as C

import numpy as np
import pytest

torch = pytest.importorskip("torch")

import ssenss_amd as S  # noqa: E402

pytestmark = pytest.mark.gpu

NPART, ROUND = 1024, 1024 * 256
PAP0, BETA0 = 100, 120          # slots of this test's own scalars


def _p(t):
    return C.c_void_p(t.data_ptr() if t is not None else 0)


def _ptrs(ts):
    return (C.c_void_p * 10)(*[t.data_ptr() for t in ts])  # rest null


def _dot(L, st, n, x, s, y, part, scal):
    assert L.ssxk_dot(st, C.c_size_t(n), _p(x), _p(s), _p(y), _p(part),
                      0) == 0
    assert L.ssxk_reduce(st, _p(part), 0, _p(scal), 0) == 0
    torch.cuda.synchronize()
    return scal[0].item()


@pytest.mark.parametrize("n", [1, 200, ROUND - 1, ROUND + 77,
                               3 * ROUND + 1, 4 * ROUND, 7 * ROUND - 300])
def test_history_passes(n):
    L = S.load()
    st = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    g = torch.Generator(device="cuda").manual_seed(n)
    mk = lambda *s: torch.randn(*s, generator=g, device="cuda",
                                dtype=torch.float64)
    x, s = mk(n), mk(n).abs()
    ys = [mk(n) for _ in range(10)]
    part = torch.zeros(10 * NPART, device="cuda", dtype=torch.float64)
    scal = torch.zeros(256, device="cuda", dtype=torch.float64)
    eps = np.finfo(float).eps
    one = []
    for y in ys:
        ref = _dot(L, st, n, x, s, y, part, scal)
        scal[PAP0] = 1.0
        assert L.ssxk_multidot(st, C.c_size_t(n), _p(x), _p(s), _ptrs([y]),
                               1, _p(part), _p(scal), 0, PAP0, BETA0) == 0
        torch.cuda.synchronize()
        one.append(scal[0].item())
        bound = (x * s * y).abs().sum().item()
        assert abs(one[-1] - ref) <= 2 * (-(-n // ROUND) + 20) * eps * bound
    for m in range(1, 11):
        scal.zero_()
        scal[PAP0:PAP0 + 10] = torch.arange(1, 11)
        assert L.ssxk_multidot(st, C.c_size_t(n), _p(x), _p(s), _ptrs(ys), m,
                               _p(part), _p(scal), 0, PAP0, BETA0) == 0
        torch.cuda.synchronize()
        assert scal[:m].tolist() == one[:m]
        assert scal[BETA0:BETA0 + m].tolist() == [
            one[k] / (k + 1.0) for k in range(m)]
        assert not scal[m:PAP0].any() and not scal[BETA0 + m:].any()


@pytest.mark.parametrize("shift", [0, 1, 9])
def test_pair_scalars(shift):
    """slots as the solver's enum lays them out: found from the values"""
    L = S.load()
    st = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    n = 2 * ROUND + 5
    g = torch.Generator(device="cuda").manual_seed(shift)
    p, s, ap, r = [torch.randn(n, generator=g, device="cuda",
                               dtype=torch.float64) for _ in range(4)]
    part = torch.zeros(4 * NPART, device="cuda", dtype=torch.float64)
    tmp = torch.zeros(256, device="cuda", dtype=torch.float64)
    tmp[PAP0:PAP0 + 2] = 1.0
    assert L.ssxk_multidot(st, C.c_size_t(n), _p(p), _p(s), _ptrs([ap, r]), 2,
                           _p(part), _p(tmp), 0, PAP0, BETA0) == 0
    torch.cuda.synchronize()
    pap, pr = tmp[:2].tolist()
    before = torch.arange(1000.0, 1256.0, device="cuda", dtype=torch.float64)
    scal = before.clone()
    assert L.ssxk_fcg_pair(st, C.c_size_t(n), _p(p), _p(s), _p(ap), _p(r),
                           _p(part), _p(scal), shift) == 0
    torch.cuda.synchronize()
    a = scal.tolist()
    at = [i for i, v in enumerate(a) if v == pap]
    assert len(at) == 2                       # the history's first, the pair's
    p0, pn = at
    assert a[pn + 1] == pr
    assert a.count(pr / pap) == 1
    assert a[p0 + 1:p0 + 1 + shift] == [1000.0 + p0 + k for k in range(shift)]
    changed = sum(v != w for v, w in zip(a, before.tolist()))
    assert changed == 4 + shift
