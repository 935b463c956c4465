"""The FP64 rotation by adjoint pairs: a solve whose overlaps satisfy
M(k+b, -b) = M(k, b)^+ forms one block of each pair, any other solve forms
every block.

Both ways are run with a fixed step (no line search, so rounding is not
amplified) on the same physical problem: as generated, and with the overlaps
of one block off their pair's identity by 1e-9, which the check at load must
notice.  Over 4 iterations of step 1 the two differ by the change of the
inputs, 1e-9 in one of nk nntot nw^2 elements of modulus <= 1, times a few
(each iteration rotates by a bounded gradient of the overlaps): 1e-7 bounds
it at every size here, and a pair stored wrongly (transposed, conjugated, in
another block) changes U by more than 1e-3.  The general path is compared
with the oracle on overlaps far from any pairing (1e-9, as both are FP64
trajectories of 3 fixed steps).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

po = pytest.importorskip("oracle.pyoracle")

# both sides of every tile edge, each kernel, meshes where k + b = k - b
SIZES = [("sc", 17, (3, 3, 3)), ("fcc", 32, (2, 2, 2)), ("sc", 33, (4, 2, 3)), ("bcc", 47, (3, 3, 3)),
         ("hex", 48, (2, 2, 3)), ("triclinic", 49, (2, 3, 2)), ("sc", 63, (3, 2, 2)), ("bcc", 64, (2, 2, 2)),
         ("sc", 65, (2, 2, 2)), ("fcc", 96, (2, 2, 2)), ("hex", 129, (2, 2, 2)), ("sc", 24, (1, 1, 4))]


@pytest.fixture(scope="module")
def ctx():
    from wannier90_amd import capi

    c = capi.Context(0)
    yield c
    c.close()


def solve(ctx, p, m, u, iters):
    from wannier90_amd import capi

    ctl = capi.control(num_iter=iters, lfixstep=1, fixed_step=1.0)
    s = ctx.session(p.kmesh, p.num_wann, p.num_kpts, ctl)
    s.load(m, u)
    s.solve()
    out = s.fetch()
    s.close()
    return out


@pytest.mark.parametrize("case", SIZES, ids=lambda c: f"{c[0]}-nw{c[1]}-{'x'.join(map(str, c[2]))}")
def test_pairs_equal_block_by_block(ctx, case):
    from wannier90_amd import synth

    kind, nw, mp = case
    print(f"[pairs] {case}", flush=True)
    p = synth.make_problem(977 + nw, kind=kind, nw=nw, mp=mp, decay=2.0)
    u0, m0 = synth.initial_state(p)
    m, u, cen, spr = solve(ctx, p, m0, u0, 4)
    m1 = m0.copy(order="F")
    m1[nw - 1, 0, 0, p.num_kpts - 1] += 1e-9
    mg, ug, ceng, sprg = solve(ctx, p, m1, u0, 4)
    assert np.abs(u - ug).max() <= 1e-7
    assert np.abs(m - mg).max() <= 1e-7
    assert np.abs(cen - ceng).max() <= 1e-7
    assert np.abs(spr - sprg).max() <= 1e-7
    assert np.abs(u - u0).max() > 1e-3  # the steps moved U


@pytest.mark.parametrize("nw", [17, 40, 64, 70])
def test_overlaps_without_pairs_match_oracle(ctx, nw):
    from wannier90_amd import synth

    print(f"[no pairs] nw {nw}", flush=True)
    p = synth.make_problem(977 + nw, kind="sc", nw=nw, mp=(3, 2, 2), decay=2.0)
    u0, m0 = synth.initial_state(p)
    rng = np.random.default_rng(nw)
    m1 = np.asfortranarray(m0 + 0.02 / nw * (rng.normal(size=m0.shape) + 1j * rng.normal(size=m0.shape)))
    ctl = dict(num_iter=3, num_cg_steps=5, conv_window=-1, conv_tol=1e-10, trial_step=2.0, lfixstep=1, fixed_step=1.0)
    o = po.wann_main(po.Problem(nw, p.num_kpts, p.kmesh), ctl, m1, u0)
    m, u, cen, spr = solve(ctx, p, m1, u0, 3)
    assert np.abs(u - o["u"]).max() <= 1e-9
    assert np.abs(cen - o["centres"]).max() <= 1e-9
