"""The FP64 operator on the matrix instruction (9 to 12 points a direction)
against the oracle: every order it takes, whose line counts n^2 fill their
last tile of 16 by one line (n = 9, 11), a quarter (10) or fully (12), below
and above the size where orders 9 to 11 go to the team kernel (512 / 513
elements), with and without walls and with the SVV matrix (its own
derivative matrix in three of the six products).

Bars: the operator 1e-12 relative, as everywhere (the contractions are summed
in another order than the oracle's); Jacobi-PCG, which takes the fused
direction update and solution step, the oracle's iteration count within one
and its solution to the tolerance; FCG + p-multigrid the same."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import ssenss_amd as S  # noqa: E402
from conftest import rel  # noqa: E402
from oracle import pyoracle as P  # noqa: E402
from ssenss_amd.mesh import PERIODIC, box_mesh  # noqa: E402

pytestmark = pytest.mark.gpu


def _mesh(n, dims, walls, svva):
    bc = (-1,) * 6 if walls else (PERIODIC,) * 6
    mesh = box_mesh(n, dims, bc=bc, deform=1 if walls else 0, amp=0.1,
                    dt=0.05, visc=0.5)
    mesh.svva = svva
    return mesh


@pytest.mark.parametrize("n,dims,walls,svva", [
    (9, (2, 2, 2), True, 0.0), (9, (3, 3, 3), False, 0.7),
    (10, (1, 1, 1), True, 0.3), (10, (3, 3, 3), False, 0.0),
    (11, (2, 1, 2), True, 0.5), (12, (2, 2, 1), True, 0.4),
    (12, (3, 3, 3), False, 0.0), (9, (8, 8, 8), True, 0.2),
    (9, (3, 9, 19), True, 0.2)])
def test_operator(n, dims, walls, svva):
    mesh = _mesh(n, dims, walls, svva)
    rng = np.random.default_rng(n)
    u = rng.standard_normal(mesh.ntot)
    o = P.Oracle(mesh)
    with S.Context(mesh) as ctx:
        ctx.set_stream(torch.cuda.current_stream())
        du = torch.from_numpy(u).cuda()
        for v in (0, 2):                # without and with streaming hints
            ctx.set_ax_variant(0, S.PREC_FP64, v)
            for op in (S.OP_POISSON, S.OP_HELMHOLTZ):
                au = torch.full_like(du, np.nan)
                ctx.ax(0, op, du, au)
                e1 = rel(au.cpu().numpy(), o.ax(0, op, u))
                p = o.dss_average(0, u)
                ap = torch.full_like(du, np.nan)
                ctx.opeval(0, op, S.X_VELOCITY, torch.from_numpy(p).cuda(),
                           ap)
                e2 = rel(ap.cpu().numpy(), o.opeval(0, op, P.X_VELOCITY, p))
                print(f"[gpu] n={n} {dims} op {op}: {e1:.1e} {e2:.1e}",
                      flush=True)
                assert e1 <= 1e-12 and e2 <= 1e-12
    o.close()


@pytest.mark.parametrize("n", [9, 10, 11, 12])
@pytest.mark.parametrize("walls", [True, False])
def test_solves(n, walls):
    mesh = _mesh(n, (2, 3, 2) if walls else (3, 3, 3), walls, 0.0)
    rng = np.random.default_rng(20 + n)
    o = P.Oracle(mesh)
    f = o.dss(0, rng.standard_normal(mesh.ntot))
    eps = 1e-10 * np.sqrt(o.dot(0, f, f))
    with S.Context(mesh) as ctx:
        ctx.set_stream(torch.cuda.current_stream())
        d = torch.from_numpy(f).cuda()
        x = torch.zeros_like(d)
        st = ctx.cg(0, S.OP_HELMHOLTZ, S.X_VELOCITY, d, x, eps, 3000)
        xo, it, _, _ = o.cg(0, P.OP_HELMHOLTZ, P.X_VELOCITY, f,
                            np.zeros(mesh.ntot), eps, 3000)
        assert abs(st.iterations - it) <= 1
        assert rel(x.cpu().numpy(), xo) <= 1e-8
        d = torch.from_numpy(f).cuda()
        x = torch.zeros_like(d)
        st = ctx.fcg(S.OP_POISSON, S.PRESSURE, S.PC_MG, d, x, eps, 500)
        xo, it, _, _ = o.fcg(P.OP_POISSON, P.PRESSURE, P.PC_MG, f,
                             np.zeros(mesh.ntot), eps, 500)
        print(f"[gpu] n={n} walls={walls}: FCG {st.iterations} / {it}",
              flush=True)
        assert abs(st.iterations - it) <= 1
        assert rel(x.cpu().numpy(), xo) <= 1e-8
    o.close()
