"""Solves whose num_iter is not a whole number of launch blocks (16
iterations): the iterations are those of a longer solve, bit for bit, for one
problem, for problems of different num_iter in one batch, and in mixed
precision (the FP64 rebuild at the end of the budget)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from wannier90_amd import capi

    c = capi.Context(0)
    yield c
    c.close()


@pytest.fixture(scope="module")
def prob():
    from wannier90_amd import synth

    p = synth.make_problem(31, kind="fcc", nw=6, mp=(3, 3, 3), decay=2.0)
    u, m = synth.initial_state(p)
    return p, m, u


def control(n, fixed, **kw):
    from wannier90_amd import capi

    return capi.control(num_iter=n, lfixstep=int(fixed), fixed_step=0.5, **kw)


ITERS = [0, 1, 2, 15, 16, 17, 31, 32, 33, 48, 50]


@pytest.mark.parametrize("fixed", [False, True])
def test_short_solves_are_prefixes(ctx, prob, fixed):
    p, m, u = prob

    def solve(n):
        s = ctx.session(p.kmesh, p.num_wann, p.num_kpts, control(n, fixed))
        s.load(m, u)
        r = s.solve()
        h = s.history()
        r2 = s.solve()  # the same session again
        assert r2.omega_total == r.omega_total and r2.iterations == r.iterations
        s.close()
        return r, h

    _, full = solve(64)
    for n in ITERS:
        r, h = solve(n)
        assert r.iterations == n and len(h) == n + 1
        assert np.array_equal(h, full[: n + 1])


@pytest.mark.parametrize("fixed", [False, True])
def test_uneven_num_iter_in_a_batch(ctx, prob, fixed):
    from wannier90_amd import capi

    p, m, u = prob
    s = ctx.session(p.kmesh, p.num_wann, p.num_kpts, control(64, fixed))
    s.load(m, u)
    s.solve()
    full = s.history()
    s.close()
    b = ctx.batch(sum(capi.problem_bytes(p.num_wann, p.num_kpts, p.kmesh.nntot, n) for n in ITERS))
    ids = [b.add(p.kmesh, m, u, control(n, fixed)) for n in ITERS]
    b.run()
    for i, n in zip(ids, ITERS):
        r = b.result(i)
        assert r.iterations == n and r.omega_total == full[n, 0]
    b.close()


def test_mixed_budget_ends_in_fp64(ctx, prob):
    from wannier90_amd import capi

    p, m, u = prob
    for n in (1, 15, 16, 17, 33):
        s = ctx.session(p.kmesh, p.num_wann, p.num_kpts, control(n, True, precision=capi.PREC_MIXED))
        s.load(m, u)
        r = s.solve()
        mf, uf, _, _ = s.fetch()
        s.close()
        assert r.iterations == n
        # M is the FP64 rebuild from the initial overlaps: the same as rotating
        # them by U0^+ U (one product of order 6: 1e-13)
        e = np.einsum("jik,jlk->ilk", u.conj(), uf)
        for b in range(p.kmesh.nntot):
            k2 = p.kmesh.nnlist[:, b] - 1
            ref = np.einsum("jik,jlk,lmk->imk", e.conj(), m[:, :, b, :], e[:, :, k2])
            assert np.abs(mf[:, :, b, :] - ref).max() <= 1e-13
