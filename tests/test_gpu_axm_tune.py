"""Where the FP64 operator runs the matrix kernel (n = 12; n = 9..11 up to
512 elements) the autotuner reports one time per streaming hint and takes the
faster."""
import pytest

torch = pytest.importorskip("torch")

import ssenss_amd as S  # noqa: E402
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
    finally:
        ctx.close()
