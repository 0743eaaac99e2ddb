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
