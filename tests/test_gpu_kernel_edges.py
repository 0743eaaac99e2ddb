"""HIP kernels against the oracle, bit for bit, at the sizes where their tilings can go wrong."""
import pytest

from fast_amd import cases
from tests import helpers as H
from tests.test_gpu_parity import assert_same, ctxmod, orc, run_pair  # noqa: F401  (fixtures)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mesh", ["cart", "full"])
@pytest.mark.parametrize("mode", ["bdf_ss2", "local"])
@pytest.mark.parametrize("n", [(2, 2, 2), (2, 7, 9), (3, 8, 16), (16, 9, 8), (17, 16, 7), (34, 25, 24)])
def test_lu_stream_tiles(ctxmod, orc, mesh, mode, n):  # noqa: F811
    """The streaming LU-SGS on one pencil, on pencils of 1, 7 and 8 lines in j and k, on lines shorter
    than the ring of rows and than the 15 steps without all neighbours, with odd and even numbers of
    steps."""
    nsub = 2 if mode == "bdf_ss2" else 1
    if mesh == "cart":
        mk = lambda: cases.tgv_zone(n, H.numerics("ausmpred", mode), perturb=0.02)
    else:
        mk = lambda: H.jittered_box(n, H.numerics("ausmpred", mode), bcs=H.WALL_J)
    zo, zg, _, _ = run_pair(ctxmod, orc, mk, nsub, nsteps=2)
    assert_same(zo, zg, ghosts=True)
