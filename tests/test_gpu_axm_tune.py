"""Where the FP64 operator runs the matrix kernel (n = 12; n = 9..11 up to
512 elements) the autotuner reports one time per streaming hint and takes the
faster; the other bits of the shape, which the batched operator takes, are
those of the fastest team kernel.  That kernel, launched for the ranking
alone, computes the masked Poisson operator and its partials at every order
and shape (against the oracle, 1e-12 relative; the shapes bit-identical)."""
import ctypes as C

import numpy as np
import pytest

torch = pytest.importorskip("torch")

import ssenss_amd as S  # noqa: E402
from conftest import rel  # noqa: E402
from oracle import pyoracle as P  # noqa: E402
from ssenss_amd.mesh import box_mesh  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [9, 10, 11, 12])
def test_autotune(n):
    mesh = box_mesh(n, (3, 2, 2), deform=1, amp=0.05)
    ctx = S.Context(mesh)
    try:
        ctx.autotune(1)
        v, us = ctx.ax_variant(0, 0)
        assert 0 <= v < 8 and us[v] == min(us) > 0.0
        assert all(us[k] == us[k & 2] for k in range(8))
        team = (C.c_double * 8)()
        assert S.load().ssx_ax_team_times(ctx.h, 0, team) == 1
        best = min(range(8), key=lambda k: team[k])
        assert min(team) > 0.0 and len(set(team)) > 1
        assert (v & ~2) == (best & ~2)
    finally:
        ctx.close()


@pytest.mark.parametrize("n", [9, 10, 11, 12])
def test_team_kernel(n):
    mesh = box_mesh(n, (5, 1, 1), deform=1, amp=0.05)   # a ragged last team
    rng = np.random.default_rng(n)
    u = rng.standard_normal(mesh.ntot)
    o = P.Oracle(mesh)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    ptr = lambda a: C.c_void_p(a.data_ptr())
    with S.Context(mesh) as ctx:
        ctx.set_stream(torch.cuda.current_stream())
        mask = ctx.level_data(0, S.DATA_MASK)
        m = mask.reshape(mesh.nel, n, n, n) == 0
        h = n // 2
        faces = (m[:, h, h, 0], m[:, h, h, -1], m[:, h, 0, h], m[:, h, -1, h],
                 m[:, 0, h, h], m[:, -1, h, h])
        bc = sum(f.astype(np.int32) << k for k, f in enumerate(faces))
        D = np.asarray(P.gll_basis(n)[2]).T.ravel()     # D[i][l]
        gf, mass = (dev(ctx.level_data(0, w))
                    for w in (S.DATA_GFAC, S.DATA_MASS))
    ref = o.ax(0, P.OP_POISSON, u) * mask
    parts = (u * ref).reshape(mesh.nel, -1).sum(1)
    o.close()
    du, dd, dbc = dev(u), dev(np.concatenate([D, D])), dev(bc)
    first = None
    for v in range(8):
        au = torch.full_like(du, np.nan)
        part = torch.full((mesh.nel,), np.nan, device="cuda",
                          dtype=torch.float64)
        torch.cuda.synchronize()
        assert S.load().ssxk_ax_team(
            None, n, v, mesh.nel, ptr(du), ptr(au), ptr(gf), ptr(mass),
            ptr(dd), C.c_double(1.0), ptr(dbc), ptr(part)) == 0
        torch.cuda.synchronize()
        first = first or (au, part)
        print(f"[gpu] team n={n} shape {v}: "
              f"{rel(au.cpu().numpy(), ref):.1e}", flush=True)
        assert torch.equal(au, first[0]) and torch.equal(part, first[1])
    assert rel(first[0].cpu().numpy(), ref) <= 1e-12
    assert rel(first[1].cpu().numpy(), parts) <= 1e-12
