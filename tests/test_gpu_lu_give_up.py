"""LU-SGS waits that give up: reported once, and nothing of them is left in what is computed next."""
import numpy as np
import pytest

from fast_amd import cases
from tests import helpers as H
from tests.test_gpu_parity import ctxmod  # noqa: F401  (fixture)

pytestmark = pytest.mark.gpu
FIELDS = ("ro", "ro_m1", "ro_p1", "drodm")


@pytest.mark.parametrize("mesh", ["cart", "full"])
@pytest.mark.parametrize("zones", [1, 3])
@pytest.mark.parametrize("schedule", ["stream", "dataflow"])
def test_steps_after_a_give_up(ctxmod, schedule, zones, mesh):  # noqa: F811
    """The error word of every zone is set from the host, as a wait that gives up sets it, so that the
    sweeps of two steps stop waiting and leave what they like in the exchanges.  One call reports it for
    all zones; from the state as it was before, every field of the next steps is what a context gives
    whose sweeps never gave up."""
    num = H.numerics("ausmpred", "bdf")
    sizes = [(24, 20, 18), (9, 33, 17), (40, 17, 25)][:zones]

    def make():
        if mesh == "cart":
            zs = [cases.tgv_zone(n, num, perturb=0.02, seed=q) for q, n in enumerate(sizes)]
        else:
            zs = [H.jittered_box(n, num, seed=q, bcs=H.WALL_J) for q, n in enumerate(sizes)]
        ctx = ctxmod.Context(0)
        ctx.set_option(ctxmod.OPT_LU_SCHEDULE, ctxmod.LU_STREAM if schedule == "stream" else ctxmod.LU_DATAFLOW)
        for z in zs:
            ctx.add_zone(z)
        return ctx, zs

    def start(ctx, zs):
        for q, z in enumerate(zs):
            for f in (ctxmod.FIELD_RO, ctxmod.FIELD_RO_M1, ctxmod.FIELD_RO_P1):
                ctx.set(q, f, z.ro)
            ctx.apply_bc(q, 0)

    def steps(ctx, zs):
        start(ctx, zs)
        ctx.compute(0, 1, 1, nit_c=5, modulo_verif=0, first_it=0)
        return [{f: ctx.get(q, getattr(ctxmod, "FIELD_" + f.upper()), np.zeros_like(z.ro)) for f in FIELDS}
                for q, z in enumerate(zs)]

    ctx, zs = make()
    want = steps(ctx, zs)
    ctx.close()
    ctx, zs = make()
    start(ctx, zs)
    ctx.compute(0, 1, 1, nit_c=1, modulo_verif=0, first_it=0)
    ctx.sync()
    ctx.set_option(ctxmod.OPT_LU_GIVE_UP, 1)
    ctx.compute(1, 1, 1, nit_c=2, modulo_verif=0, first_it=1)
    buf = np.zeros_like(zs[0].ro)
    with pytest.raises(ctxmod.FastMIError, match="timed out"):
        ctx.get(0, ctxmod.FIELD_RO, buf)
    ctx.get(0, ctxmod.FIELD_RO, buf)
    got = steps(ctx, zs)
    ctx.close()
    for q in range(zones):
        for f in FIELDS:
            assert np.array_equal(got[q][f], want[q][f]), (q, f)
