"""The FP64 rotation by column panels (17-48 bands) where a workgroup takes
several blocks of a k: sets of more than 4096 blocks, rotated by pairs (two
blocks to a workgroup, a remainder of one) and block by block (three each).

The overlaps that a solve returns are compared with the overlaps it was given,
rotated by the U that it returns relative to the U that it was given:
M = V(k)^+ M0 V(k+b), V = U0^+ U.  Both sides round once per product and
iteration: 3 iterations of four products of at most 48 terms each, relative to
blocks of norm 1, are below 3 * 4 * 2 * 48 * 1.1e-16 = 1.3e-13 an element, and
the retraction's departure from unitarity is of the same size; 1e-11 is far above that
and far below any misplaced element (about 1/nw).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from wannier90_amd import capi

    c = capi.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("nw,mp,paired", [(17, (12, 12, 12), True), (31, (12, 12, 12), False),
                                          (33, (12, 12, 12), False), (48, (12, 12, 10), True)])
def test_several_blocks_to_a_workgroup(ctx, nw, mp, paired):
    from wannier90_amd import capi, synth

    print(f"[rot panel] nw {nw} mesh {mp} paired {paired}", flush=True)
    p = synth.make_problem(31 + nw, kind="sc", nw=nw, mp=mp, decay=2.0)
    u0, m0 = synth.initial_state(p)
    if not paired:
        m0[nw - 1, 0, 0, p.num_kpts - 1] += 1e-3
    s = ctx.session(p.kmesh, nw, p.num_kpts, capi.control(num_iter=3, lfixstep=1, fixed_step=1.0))
    s.load(m0, u0)
    s.solve()
    m, u, _, _ = s.fetch()
    s.close()
    v = np.matmul(np.conj(np.transpose(u0, (2, 1, 0))), np.transpose(u, (2, 0, 1)))
    worst = 0.0
    for b in range(p.kmesh.nntot):
        k2 = p.kmesh.nnlist[:, b] - 1
        r = np.matmul(np.conj(np.transpose(v, (0, 2, 1))), np.matmul(np.transpose(m0[:, :, b, :], (2, 0, 1)), v[k2]))
        worst = max(worst, np.abs(np.transpose(m[:, :, b, :], (2, 0, 1)) - r).max())
    assert worst <= 1e-11
    assert np.abs(v - np.eye(nw)).max() > 1e-7  # the steps moved U, far above the bound
