"""CG iterations whose reductions are replayed by the kernels that need them
(two launches an iteration, small levels) against the reductions as launches
of their own (SSX_OPT_GATHER_DSS 0 takes those, with the same sums in the
same order): bit-identical solutions and iteration counts.

The replay sums in the order of a 1024-lane reduction, so its edges are the
numbers of partials: elements below, at and above 1024 (a virtual lane's
second partial), the largest level that replays and the first that does not
(up to n = 11 FP64 1024 and, to n = 10, FP32 4096 elements; fewer above); workgroups smaller than a wavefront
(n = 3, 5, 6, 7 under the one-wave launch shapes) and of several, below and
above the 2048 workgroups up to which every launch reads the done flag late
(a replaying one always does); the pressure's four sums; a solve that stops in the middle of a chunk of
launches and one stopped by its iteration limit."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import ssenss_amd as S  # noqa: E402
from ssenss_amd.mesh import PERIODIC, box_mesh  # noqa: E402

pytestmark = pytest.mark.gpu


def _pair(mesh, run, variant=None):
    """run(ctx) with the reductions as launches and replayed"""
    out = []
    with S.Context(mesh) as ctx:
        ctx.set_stream(torch.cuda.current_stream())
        if variant is not None:
            # the first cycle makes the FP32 copies and picks their shape
            ctx.set_option(S.OPT_SMOOTHER_PRECISION, S.PREC_FP32)
            f = _rhs(ctx, 1)
            ctx.mg_precon(S.OP_POISSON, S.PRESSURE, 1e-3, f,
                          torch.zeros_like(f))
            ctx.set_option(S.OPT_SMOOTHER_PRECISION, S.PREC_FP64)
            for prec in (S.PREC_FP64, S.PREC_FP32):
                ctx.set_ax_variant(0, prec, variant)
        for g in (0, 1):
            ctx.set_option(S.OPT_GATHER_DSS, g)
            out.append(run(ctx))
    return out


def _rhs(ctx, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    f = torch.randn(ctx.ntot(0), generator=gen, device="cuda",
                    dtype=torch.float64)
    ctx.dss(0, f)
    return f


def _same(a, b):
    for x, y in zip(a, b):
        if isinstance(x, torch.Tensor):
            assert torch.equal(x, y)
        else:
            assert x == y


@pytest.mark.parametrize("n,dims", [
    (3, (2, 2, 2)), (3, (16, 8, 8)), (3, (17, 8, 8)), (4, (16, 16, 16)),
    (3, (17, 16, 16)), (12, (3, 2, 2))])
def test_replayed_reductions_by_element_count(n, dims):
    mesh = box_mesh(n, dims, deform=1, amp=0.05, dt=0.1, visc=0.1)

    def run(ctx):
        res = []
        for var, most in ((S.X_VELOCITY, 400), (S.X_VELOCITY, 5)):
            f = _rhs(ctx, 3)
            u = torch.zeros_like(f)
            st = ctx.cg(0, S.OP_HELMHOLTZ, var, f, u, 1e-6, most,
                        allow_notconv=True)
            res += [st.iterations, st.residual, u]
        for prec in (S.PREC_FP32, S.PREC_BF16):
            ctx.set_option(S.OPT_SMOOTHER_PRECISION, prec)
            zs = []
            for eps in (1e-12, 0.05):       # 15 iterations, and fewer
                f = _rhs(ctx, 4)
                z = torch.zeros_like(f)
                ctx.mask(0, S.X_VELOCITY, f)
                norm = float(np.sqrt(ctx.dot(0, f, f)))
                ctx.mg_precon(S.OP_HELMHOLTZ, S.X_VELOCITY, eps * norm, f, z)
                zs.append(z)
            assert not torch.equal(*zs)
            res += zs
        ctx.set_option(S.OPT_SMOOTHER_PRECISION, S.PREC_FP64)
        return res
    print(f"[gpu] replay n={n} {dims}", flush=True)
    _same(*_pair(mesh, run))


@pytest.mark.parametrize("n", [3, 5, 6, 7, 8, 10])
@pytest.mark.parametrize("variant", [1, 4])
def test_replayed_reductions_by_workgroup(n, variant):
    mesh = box_mesh(n, (3, 3, 3), lo=(0,) * 3, hi=(6.0,) * 3,
                    bc=(PERIODIC,) * 6, dt=0.1, visc=0.1)

    def run(ctx):
        res = []
        for prec in (S.PREC_FP64, S.PREC_FP32):
            ctx.set_option(S.OPT_SMOOTHER_PRECISION, prec)
            f = _rhs(ctx, 5)
            u = torch.zeros_like(f)
            eps = 1e-9 * float(np.sqrt(ctx.dot(0, f, f)))
            st = ctx.fcg(S.OP_POISSON, S.PRESSURE, S.PC_MG, f, u, eps, 60,
                         allow_notconv=True)
            res += [st.iterations, u]
        ctx.set_option(S.OPT_SMOOTHER_PRECISION, S.PREC_FP64)
        return res
    print(f"[gpu] replay n={n} variant {variant}", flush=True)
    _same(*_pair(mesh, run, variant))


@pytest.mark.parametrize("dims", [(8, 16, 16), (13, 13, 13)])
def test_replayed_stop_by_grid(dims):
    """One team of two wavefronts a workgroup (n = 9, one-wave shape): 2048
    and 2197 workgroups, stopped before the smoother's last iteration."""
    mesh = box_mesh(9, dims, deform=1, amp=0.05, dt=0.1, visc=0.1)

    def run(ctx):
        res = []
        for prec in (S.PREC_FP32, S.PREC_BF16):
            ctx.set_option(S.OPT_SMOOTHER_PRECISION, prec)
            zs = []
            for eps in (1e-12, 0.05):   # the first call picks a shape
                f = _rhs(ctx, 6)
                z = torch.zeros_like(f)
                ctx.mask(0, S.X_VELOCITY, f)
                norm = float(np.sqrt(ctx.dot(0, f, f)))
                ctx.mg_precon(S.OP_HELMHOLTZ, S.X_VELOCITY, eps * norm, f, z)
                zs.append(z)
                ctx.set_ax_variant(0, prec, 1)
            assert not torch.equal(*zs)         # it did stop early
            res += zs
        ctx.set_option(S.OPT_SMOOTHER_PRECISION, S.PREC_FP64)
        return res
    print(f"[gpu] replayed stop {dims}", flush=True)
    _same(*_pair(mesh, run))


@pytest.mark.parametrize("n,dims", [
    (12, (4, 4, 4)), (12, (2, 3, 11)), (13, (8, 8, 8)), (13, (9, 19, 3)),
    (16, (4, 4, 2)), (16, (4, 3, 3)), (16, (16, 4, 4)), (16, (4, 6, 11))])
def test_replayed_reductions_at_high_order(n, dims):
    """The largest level that replays and one just past it: FP64 n = 12 (64 /
    66 elements), 13 (512 / 513), 16 (32 / 36), FP32 n = 16 (256 / 264)."""
    test_replayed_reductions_by_element_count(n, dims)
