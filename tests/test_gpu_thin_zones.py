"""Zones of one to three cells in one direction, against the oracle, bit for bit."""
import pytest

from fast_amd import cases
from tests import helpers as H
from tests.test_gpu_kernel_edges import bc_set
from tests.test_gpu_parity import assert_same, ctxmod, orc, run_pair  # noqa: F401  (fixtures)

pytestmark = pytest.mark.gpu

BOTH = [("BCFarfield", "imin", None), ("BCFarfield", "imax", None), ("BCWallViscous", "jmin", None),
        ("BCWallInviscid", "jmax", None), ("BCOutflow", "kmin", None), ("BCFarfield", "kmax", None)]


@pytest.mark.parametrize("kind", ["split", "overlap", "both"])
@pytest.mark.parametrize("mode", ["explicit", "bdf_ss2"])
@pytest.mark.parametrize("n", [(2, 9, 7), (9, 2, 7), (9, 7, 2), (2, 2, 7), (9, 2, 2), (2, 3, 2)])
def test_conditions_of_thin_zones(ctxmod, orc, n, mode, kind):  # noqa: F811
    """Conditions on opposite faces two cells apart share a launch: each reads two cells deep at most."""
    nsub = {"explicit": 3, "bdf_ss2": 2}[mode]
    bcs = BOTH if kind == "both" else bc_set(n, kind)
    mk = lambda: H.jittered_box(n, H.numerics("ausmpred", mode), bcs=bcs)
    zo, zg, _, _ = run_pair(ctxmod, orc, mk, nsub, nsteps=2)
    assert_same(zo, zg, ghosts=True)


@pytest.mark.parametrize("scheme", ["ausmpred", "senseur", "roe_min", "roe_kap"])
@pytest.mark.parametrize("mode", ["explicit", "bdf_ss2"])
@pytest.mark.parametrize("flow", ["lamin", "euler"])
@pytest.mark.parametrize("mesh", ["cart", "full"])
@pytest.mark.parametrize("n", [(9, 1, 7), (66, 1, 5), (66, 2, 5), (130, 3, 4)])
def test_residuals_of_few_rows(ctxmod, orc, n, mesh, flow, mode, scheme):  # noqa: F811
    """One to three rows of cells, where the residual's schedule changes, each mesh, flow and scheme."""
    nsub = {"explicit": 3, "bdf_ss2": 2}[mode]
    bcs = H.WALL_J[:2] + [("BCExtrapolate", "jmin", None), ("BCExtrapolate", "jmax", None)] + H.WALL_J[4:]
    num = H.numerics(scheme, mode)
    if mesh == "cart":
        mk = lambda: cases.tgv_zone(n, num, perturb=0.02, flow=flow, bcs=bcs)
    else:
        mk = lambda: H.jittered_box(n, num, flow=flow, bcs=bcs)
    zo, zg, _, _ = run_pair(ctxmod, orc, mk, nsub, nsteps=2)
    assert_same(zo, zg, ghosts=True)
