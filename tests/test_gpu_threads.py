"""Calls of several host threads on one context and on several: what each would get alone."""
import threading

import numpy as np
import pytest

from fast_amd import cases
from tests import helpers as H
from tests.test_gpu_parity import ctxmod  # noqa: F401  (fixture)

pytestmark = pytest.mark.gpu


def at_once(calls):
    """Runs the calls side by side, each several times; raises what one of them raised."""
    errors, go = [], threading.Barrier(len(calls))

    def work(f):
        try:
            go.wait()
            for _ in range(6):
                f()
        except BaseException as e:
            errors.append(e)

    th = [threading.Thread(target=work, args=(f,)) for f in calls]
    for t in th:
        t.start()
    for t in th:
        t.join()
    if errors:
        raise errors[0]


@pytest.mark.parametrize("n", [(40, 46, 46), (64, 64, 61), (96, 90, 90)])
def test_threads_share_a_context(ctxmod, n):  # noqa: F811
    """Fields of zones of their own written and read, wall efforts, wall gradients and transposed products
    of small and large zones, at once, at sizes on both sides of those where the copies change their way."""
    ctx = ctxmod.Context(0)
    num = H.numerics("ausmpred", "bdf")
    sizes = [n, n, (9, 8, 7), (33, 5, 40)]
    zs = [cases.tgv_zone(m, num, perturb=0.02, seed=q, flow="euler", bcs=H.INVISCID_J) for q, m in enumerate(sizes)]
    for q, z in enumerate(zs):
        ctx.add_zone(z)
        ctx.apply_bc(q, 0)
    # (the copies' pinned slots are made after 64 MB, whoever moved them)
    for _ in range(64 * 2**20 // zs[0].ro.nbytes + 1):
        ctx.get(0, ctxmod.FIELD_RO, np.zeros_like(zs[0].ro))
    lam = [np.random.default_rng(q).standard_normal(5 * z.nd) for q, z in enumerate(zs)]

    def fields(q):
        a = np.random.default_rng(50 + q).random(zs[q].ro.size)

        def call():
            a[:] += 1.0
            ctx.set(q, ctxmod.FIELD_RO_M1, a)
            assert np.array_equal(ctx.get(q, ctxmod.FIELD_RO_M1, np.zeros_like(a)), a), ("field", q)
        return call

    def window(q):
        ni, nj, nk = sizes[q]
        return [1, ni, 1, 1, 1, nk]

    def gradient(q):
        a, b = np.full(5 * zs[q].nd, 3.0), np.full(5 * zs[q].nd, -2.0)
        ctx.dpj_dpw(q, 3, window(q), 0.9, 0.3, 0.5, a, b)
        return a, b

    ref = [(ctx.wall_effort(q, 3, window(q)), gradient(q), ctx.residual_vjp(q, lam[q])) for q in range(len(zs))]

    def adjoint(q):
        def call():
            eff, fl = ctx.wall_effort(q, 3, window(q))
            assert np.array_equal(eff, ref[q][0][0]) and np.array_equal(fl, ref[q][0][1]), ("effort", q)
            for x, y in zip(gradient(q), ref[q][1]):
                assert np.array_equal(x, y), ("gradient", q)
            assert np.array_equal(ctx.residual_vjp(q, lam[q]), ref[q][2]), ("product", q)
        return call

    at_once([fields(q) for q in range(len(zs))] + [adjoint(q) for q in range(len(zs))])
    ctx.close()


@pytest.mark.parametrize("n", [(46, 46, 38), (96, 90, 90)])
def test_contexts_of_several_threads(ctxmod, n):  # noqa: F811
    """Four contexts, a thread each: one copy at a time goes through the device's pinned slots, the others
    directly; contexts closed while others copy."""
    num = H.numerics("ausmpred", "bdf")
    made = []

    def call(q):
        def f():
            z = cases.tgv_zone(n, num, perturb=0.02, seed=q, flow="euler", bcs=H.INVISCID_J)
            ctx = ctxmod.Context(0)
            ctx.add_zone(z)
            a = np.random.default_rng(q).random(z.ro.size)
            for _ in range(5):
                a += 1.0
                ctx.set(0, ctxmod.FIELD_RO_M1, a)
                assert np.array_equal(ctx.get(0, ctxmod.FIELD_RO_M1, np.zeros_like(a)), a), q
            w = [1, n[0], 1, 1, 1, n[2]]
            one, two = ctx.wall_effort(0, 3, w), ctx.wall_effort(0, 3, w)
            assert np.array_equal(one[0], two[0]) and np.array_equal(one[1], two[1]), q
            ctx.close()
            made.append(q)
        return f

    at_once([call(q) for q in range(4)])
    assert len(made) == 24
