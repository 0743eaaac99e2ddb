"""HIP kernels against the oracle, bit for bit, at the sizes where their tilings can go wrong."""
import numpy as np
import pytest

from fast_amd import cases, params as P
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


@pytest.mark.parametrize("kcol", [0, 1, 3, 64])
@pytest.mark.parametrize("n", [(2, 2, 2), (3, 5, 4), (56, 4, 2), (57, 3, 5), (61, 9, 7), (126, 6, 3)])
@pytest.mark.parametrize("case", ["ausmpred-lamin-cart", "roe_min-euler-full", "senseur-lamin-full", "roe_kap-lamin-wall"])
def test_residual_planes_tiles(ctxmod, orc, case, n, kcol):  # noqa: F811
    """The residual's planes on rows that end before, at and after a wave's 60 cells, on groups of 1 to 4
    rows, and on columns of one cell, of lengths that do not divide nk and longer than nk."""
    scheme, flow, mesh = case.split("-")
    mode = "bdf_ss2" if mesh == "cart" else "explicit" if flow == "euler" else "local"
    nsub = {"bdf_ss2": 2, "explicit": 3, "local": 1}[mode]
    num = H.numerics(scheme, mode)
    if mesh == "cart":
        mk = lambda: cases.tgv_zone(n, num, perturb=0.02, flow=flow)
    else:
        mk = lambda: H.jittered_box(n, num, flow=flow, bcs=H.WALL_J if mesh == "wall" else None)
    zo, zg, _, _ = run_pair(ctxmod, orc, mk, nsub, options=((ctxmod.OPT_RESIDUAL_SCHEDULE, ctxmod.RES_KCOL),
                                                            (ctxmod.OPT_RES_KCOL_N, kcol)))
    assert_same(zo, zg, ghosts=True)


def bc_set(n, kind):
    """Conditions of a zone of n cells: "split" cuts the j faces into four windows each (10 conditions and
    more than one launch), "overlap" lets two conditions of a face share cells, where the later one wins."""
    ni, nj, nk = n
    a, b = max(1, ni // 2), max(1, nk // 2)
    per = [("BCautoperiod", f, None) for f in ("imin", "imax", "kmin", "kmax")]
    if kind == "overlap":
        return per + [("BCWallViscous", "jmin", None), ("BCFarfield", (3, [1, a, 1, 1, 1, nk]), None),
                      ("BCOutflow", "jmax", None), ("BCWallViscous", (4, [a, ni, nj, nj, 1, b]), None)]
    out = [("BCFarfield", "imin", None), ("BCOutflow", "imax", None)] + per[2:]
    names = ["BCWallViscous", "BCFarfield", "BCExtrapolate", "BCWallInviscid"]
    for idir, j in ((3, 1), (4, nj)):
        names = names[1:] + names[:1]
        q = [[1, a, 1, b], [a + 1, ni, 1, b], [1, a, b + 1, nk], [a + 1, ni, b + 1, nk]]
        out += [(m, (idir, [w[0], w[1], j, j, w[2], w[3]]), None) for m, w in zip(names, q)]
    return out


@pytest.mark.parametrize("mode", ["explicit", "bdf_ss2", "local"])
@pytest.mark.parametrize("kind", ["split", "overlap"])
@pytest.mark.parametrize("n", [(2, 2, 2), (3, 3, 3), (9, 6, 5), (34, 5, 19)])
def test_bc_sets(ctxmod, orc, n, kind, mode):  # noqa: F811
    """Boundary conditions sharing a launch, over more than one launch, and one after another where
    their windows overlap or the zone is two cells wide."""
    nsub = {"explicit": 3, "bdf_ss2": 2, "local": 1}[mode]
    mk = lambda: H.jittered_box(n, H.numerics("ausmpred", mode), bcs=bc_set(n, kind))
    zo, zg, _, _ = run_pair(ctxmod, orc, mk, nsub, nsteps=2)
    assert_same(zo, zg, ghosts=True)


@pytest.mark.parametrize("n", [(3, 4, 5), (46, 46, 37), (46, 46, 38), (80, 80, 55), (80, 80, 56), (90, 90, 90), (90, 90, 91),
                               (130, 97, 81)])
def test_field_copies(ctxmod, n):  # noqa: F811
    """Fields written and read back, at sizes around those where the copy changes its way: 4, 16 and 32 MB,
    and a last chunk that is short."""
    z = cases.tgv_zone(n, H.numerics("ausmpred", "explicit"))
    ctx = ctxmod.Context(0)
    zid = ctx.add_zone(z)
    rng = np.random.default_rng(11)
    for f in (ctxmod.FIELD_RO, ctxmod.FIELD_RO_M1):
        a = rng.random(z.ro.size)
        ctx.set(zid, f, a)
        assert np.array_equal(ctx.get(zid, f, np.zeros_like(a)), a)
    ctx.close()


@pytest.mark.parametrize("mesh", ["cart", "full"])
@pytest.mark.parametrize("n", [(2, 2, 2), (63, 4, 5), (64, 9, 3), (17, 33, 26), (170, 7, 172)])
def test_adjoint_tiles(ctxmod, orc, n, mesh):  # noqa: F811
    """The transposed Jacobian's segments (lines no longer than one, of a cell over, of several) and rows
    ending on a wave; the wall gradients of whole and part faces, beyond one pinned slot on the largest."""
    num = H.numerics("ausmpred", "bdf")
    if mesh == "cart":
        mk = lambda: cases.tgv_zone(n, num, perturb=0.05, seed=3, flow="euler", bcs=H.INVISCID_J)
    else:
        mk = lambda: H.jittered_box(n, num, bcs=H.INVISCID_J, flow="euler")
    zo, zg = mk(), mk()
    orc.init_metric(zo)
    orc.apply_bc(zo, zo.ro)
    ctx = ctxmod.Context(0)
    zid = ctx.add_zone(zg)
    ctx.apply_bc(zid, 0)
    lam = np.random.default_rng(4).standard_normal(5 * zo.nd)
    assert np.array_equal(ctx.residual_vjp(zid, lam), orc.residual_vjp(zo, lam))
    ni, nj, nk = n
    for idir, w in ((3, [1, ni, 1, 1, 1, nk]), (4, [2, ni, nj + 1, nj + 1, 2, nk]), (1, [1, 1, 1, nj, 1, nk]),
                    (2, [ni + 1, ni + 1, 2, nj, 1, nk]), (5, [1, ni, 1, nj, 1, 1]), (6, [1, ni, 1, 1, nk + 1, nk + 1])):
        f = [np.full(5 * zo.nd, v) for v in (7.0, -3.0, 7.0, -3.0)]
        orc.dpj_dpw(zo, idir, np.array(w, dtype=np.int32), 0.9, 0.3, 0.5, dcd=f[0], dcl=f[1])
        ctx.dpj_dpw(zid, idir, w, 0.9, 0.3, 0.5, f[2], f[3])
        assert np.array_equal(f[0], f[2]) and np.array_equal(f[1], f[3]), idir
    ctx.close()


@pytest.mark.parametrize("mode", ["explicit", "bdf_ss2", "local"])
def test_zones_in_one_launch(ctxmod, mode):  # noqa: F811
    """Coefficients and residuals of zones that share launches (two meshes, two flows, three schemes, sizes
    below and above a wave, one with sensors and one with corrected wall fluxes that run alone) give
    what each zone gives alone, eager and from captured steps, with and without residual norms."""
    nsub = {"explicit": 3, "bdf_ss2": 2, "local": 1}[mode]
    num = lambda s: H.numerics(s, mode)
    mks = [lambda: cases.tgv_zone((9, 8, 7), num("ausmpred"), perturb=0.02),
           lambda: cases.tgv_zone((61, 5, 30), num("ausmpred"), perturb=0.03),
           lambda: cases.tgv_zone((2, 3, 2), num("ausmpred"), perturb=0.03),
           lambda: cases.tgv_zone((70, 66, 60), num("ausmpred"), perturb=0.02, flow="euler"),
           lambda: H.jittered_box((10, 9, 6), num("ausmpred"), bcs=H.WALL_J),
           lambda: H.jittered_box((8, 13, 5), num("ausmpred"), flow="euler"),
           lambda: H.jittered_box((12, 9, 9), num("roe_min")),
           lambda: cases.tgv_zone((12, 19, 9), num("roe_kap"), perturb=0.02),
           lambda: H.jittered_box((11, 9, 8), num("senseur")),
           lambda: H.jittered_box((10, 9, 8), num("roe_min"), bcs=H.WALL_J)]

    def run(ms):
        ctx = ctxmod.Context(0)
        zs = [m() for m in ms]
        for n, z in enumerate(zs):
            ctx.add_zone(z)
            ctx.apply_bc(n, 0)
        out = []
        for s in range(8):
            ctx.compute(s, 1, 3 if mode == "explicit" else nsub + 1, modulo_verif=5, first_it=min(s, 1))
            out.append([ctx.get(n, ctxmod.FIELD_RO, np.zeros_like(z.ro)) for n, z in enumerate(zs)])
        ctx.close()
        return out

    # (every step: the explicit step is too long for the finest zone, which overflows after some)
    together = run(mks)
    for n, m in enumerate(mks):
        assert np.isfinite(together[1][n]).all()
        for s, one in enumerate(run([m])):
            assert np.array_equal(one[0], together[s][n], equal_nan=True), (n, s)


@pytest.mark.parametrize("n", [(2, 2, 2), (4, 8, 8), (257, 3, 5), (64, 64, 32), (67, 52, 39)])
def test_norm_blocks(ctxmod, orc, n):  # noqa: F811
    """Residual norms of fewer cells than a block, of one block, of blocks and one cell over, of as many
    blocks as there can be and of more cells than those hold at once."""
    mk = lambda: cases.tgv_zone(n, H.numerics("ausmpred", "bdf"), perturb=0.02)
    zo, zg, rdm, norms = run_pair(ctxmod, orc, mk, 1, stop=2)
    r = rdm.reshape(-1, 2, 5, int(zo.param_int[P.NSSITER]))
    dtc = zo.param_real[P.DTC]
    # (positive terms summed in another order: at most their number times 2^-53 apart, taken at 1e-12)
    np.testing.assert_allclose(norms[:5], np.sqrt(r[:, 0, :, 0].sum(axis=0) / np.prod(n)) / dtc, rtol=1e-12, atol=0)
    assert np.array_equal(norms[5:], r[:, 1, :, 0].max(axis=0) / dtc)


@pytest.mark.parametrize("mode", ["local", "bdf_ss2"])
def test_lu_stream_more_pencils_than_fit(ctxmod, orc, mode):  # noqa: F811
    """A curvilinear zone of 625 pencils, more than the workgroups that are resident at once (some 512): a
    workgroup takes a second pencil with its rows, products and ticket still in LDS from the first."""
    mk = lambda: H.jittered_box((3, 200, 200), H.numerics("ausmpred", mode), bcs=H.WALL_J)
    zo, zg, _, _ = run_pair(ctxmod, orc, mk, 2 if mode == "bdf_ss2" else 1, nsteps=2)
    assert_same(zo, zg, ghosts=True)


def test_lu_stream_list_more_pencils_than_fit(ctxmod):  # noqa: F811
    """The same over two curvilinear zones in one launch, 840 pencils, against each zone alone."""
    num = H.numerics("ausmpred", "local")
    mks = [lambda: H.jittered_box((4, 160, 168), num, seed=1, bcs=H.WALL_J), lambda: H.jittered_box((5, 160, 168), num, seed=2)]

    def run(ms):
        ctx = ctxmod.Context(0)
        zs = [m() for m in ms]
        for n, z in enumerate(zs):
            ctx.add_zone(z)
            ctx.apply_bc(n, 0)
            for f in (ctxmod.FIELD_RO_M1, ctxmod.FIELD_RO_P1):
                ctx.set(n, f, ctx.get(n, ctxmod.FIELD_RO, np.zeros_like(z.ro)))
        ctx.compute(0, 1, 1, nit_c=4, modulo_verif=0, first_it=0)
        out = [[ctx.get(n, f, np.zeros_like(z.ro)) for f in (ctxmod.FIELD_RO, ctxmod.FIELD_DRODM)] for n, z in enumerate(zs)]
        ctx.close()
        return out

    both = run(mks)
    for n, m in enumerate(mks):
        one = run([m])[0]
        assert all(np.isfinite(a).all() for a in one)
        assert all(np.array_equal(a, b) for a, b in zip(one, both[n])), n
