"""Fields to and from host memory of each kind."""
import numpy as np
import pytest
import torch

from fast_amd import cases
from tests import helpers as H
from tests.test_gpu_parity import ctxmod  # noqa: F401  (fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(9, 8, 7), (46, 46, 38), (90, 90, 91)])
def test_pinned_and_pageable_arrays(ctxmod, n):  # noqa: F811
    """Whole pinned arrays, views into one that start and end inside it, and pageable arrays, at sizes
    below and above those where the copy of a pageable array changes its way."""
    z = cases.tgv_zone(n, H.numerics("ausmpred", "explicit"))
    ctx = ctxmod.Context(0)
    ctx.add_zone(z)
    m = z.ro.size
    pin = torch.zeros(m + 7, dtype=torch.float64, pin_memory=True).numpy()
    rng = np.random.default_rng(5)
    for src in (pin[:m], pin[3:3 + m], np.zeros(m)):
        src[:] = rng.random(m)
        ctx.set(0, ctxmod.FIELD_RO, src)
        want = src.copy()
        for dst in (np.zeros(m), pin[:m], pin[5:5 + m]):
            dst[:] = 0.0
            assert np.array_equal(ctx.get(0, ctxmod.FIELD_RO, dst), want)
    ctx.close()


@pytest.mark.parametrize("moved", [0, 48, 80])
def test_copies_before_and_after_the_slots(ctxmod, moved):  # noqa: F811
    """Fields of 4 to 41 MB, and one below, written and read in a context that has moved that many MB
    before: in a process that has moved none, directly, from some copy on through the pinned slots, and
    through them from the start."""
    sizes = [(3, 4, 5), (46, 46, 37), (46, 46, 38), (80, 80, 55), (80, 80, 56), (90, 90, 90), (90, 90, 91), (130, 97, 81)]
    ctx = ctxmod.Context(0)
    zs = [cases.tgv_zone(n, H.numerics("ausmpred", "explicit")) for n in sizes]
    for z in zs:
        ctx.add_zone(z)
    step = zs[2].ro.nbytes
    for _ in range(moved * 10**6 // step):
        ctx.get(2, ctxmod.FIELD_RO, np.zeros_like(zs[2].ro))
    rng = np.random.default_rng(6)
    for q, z in enumerate(zs):
        a = rng.random(z.ro.size)
        ctx.set(q, ctxmod.FIELD_RO_M1, a)
        assert np.array_equal(ctx.get(q, ctxmod.FIELD_RO_M1, np.zeros_like(a)), a), sizes[q]
    ctx.close()


@pytest.mark.parametrize("n", [(33, 8, 17), (257, 8, 33), (400, 8, 39), (410, 8, 39)])
def test_efforts_before_and_after_the_slot(ctxmod, n):  # noqa: F811
    """Wall efforts and wall gradients, again and again: in a process that has computed none, the first
    through arrays of their own, later ones through the pinned slot where the window's faces fit it (the
    last size is above)."""
    z = cases.tgv_zone(n, H.numerics("ausmpred", "bdf"), perturb=0.02, flow="euler", bcs=H.INVISCID_J)
    ctx = ctxmod.Context(0)
    ctx.add_zone(z)
    ctx.apply_bc(0, 0)
    w = [1, n[0], 1, 1, 1, n[2]]

    def both():
        g = np.full(5 * z.nd, 3.0), np.full(5 * z.nd, -2.0)
        ctx.dpj_dpw(0, 3, w, 0.9, 0.3, 0.5, *g)
        return ctx.wall_effort(0, 3, w) + g

    first = both()
    for _ in range(12):
        for a, b in zip(both(), first):
            assert np.array_equal(a, b)
    ctx.close()
