"""Disentanglement of overlaps or eigenvalues that are not finite: the call
returns, with an Omega_I or eigenvalues that are not finite, whether LDS or
global memory holds the eigenvectors of the subspace Hamiltonian."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from wannier90_amd import capi

    c = capi.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("nb,nw", [(6, 4), (72, 66)])
@pytest.mark.parametrize("what", ["m", "eig"])
def test_nan_does_not_reach_an_index(ctx, nb, nw, what):
    from wannier90_amd import synth

    print(f"[dis nan] {nb} -> {nw} {what}", flush=True)
    p, ctl = synth.make_dis_problem(88 + nb, kind="sc", num_bands=nb, num_wann=nw, mp=(2, 1, 1), decay=2.0)
    ctl["num_iter"] = 2
    m, eig = p.m_orig.copy(order="F"), p.eig.copy(order="F")
    if what == "m":
        m[1, 2, 0, 0] = np.nan
    else:
        eig[2, 0] = np.nan
    g = ctx.disentangle(p.kmesh, nb, ctl, eig, p.amat_dis, m)
    bad = g["omega_invariant"] if what == "m" else g["eigval_opt"]
    assert not np.isfinite(bad).all()
