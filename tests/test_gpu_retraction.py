"""The retraction U <- U exp(dW), M <- exp(dW)^+ M exp(dW) at the edges of
its column panels (16, 32, 48, 64 bands) and of its scaling (no squaring to
about ten), against the eigenvector form in FP64 numpy.

Tolerance: the polynomial's products round at nw eps and every squaring
doubles what is there; with ||dW||_2 = r there are log2(r / 0.04) squarings,
so 4 nw eps max(1, 25 r) bounds the error of exp(dW) and U, and M takes two
factors of it: 8 nw eps max(1, 25 r) <= 1e-12 max(1, 25 r) at 64 bands; 1e-12
is the bound of the phase tests at every size.
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


@pytest.mark.parametrize("nw", [1, 2, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64, 65, 81])
def test_retraction_matches_eigenvectors(ctx, nw):
    from wannier90_amd import synth

    print(f"[retraction] nw {nw}", flush=True)
    p = synth.make_problem(55 + nw, kind="sc", nw=nw, mp=(2, 2, 2), decay=2.0)
    u0, m0 = synth.initial_state(p)
    rng = np.random.default_rng(nw)
    w = rng.normal(size=u0.shape) + 1j * rng.normal(size=u0.shape)
    w = w - np.conj(np.transpose(w, (1, 0, 2)))
    w /= max(np.linalg.norm(w[:, :, k], 2) for k in range(w.shape[2]))
    for r in (0.0, 1e-12, 0.041, 0.042, 0.9, 25.0):
        dw = np.asfortranarray(r * w)
        lam, v = np.linalg.eigh(1j * np.transpose(dw, (2, 0, 1)))
        e = (v * np.exp(-1j * lam)[:, None, :]) @ np.conj(np.transpose(v, (0, 2, 1)))
        u, m = np.array(u0, order="F"), np.array(m0, order="F")
        ctx.new_u_and_m(p.kmesh, dw, u, m)
        tol = 1e-12 * max(1.0, 25.0 * r)
        uk = np.transpose(u0, (2, 0, 1)) @ e
        assert np.abs(np.transpose(u, (2, 0, 1)) - uk).max() <= tol
        for b in range(p.kmesh.nntot):
            k2 = p.kmesh.nnlist[:, b] - 1
            mk = np.conj(np.transpose(e, (0, 2, 1))) @ np.transpose(m0[:, :, b, :], (2, 0, 1)) @ e[k2]
            assert np.abs(np.transpose(m[:, :, b, :], (2, 0, 1)) - mk).max() <= tol


@pytest.mark.parametrize("nw", [1, 3, 16, 17, 32, 33, 48, 49, 64, 65, 90])
def test_projection_matches_svd(ctx, nw):
    """overlap_project at the edges of the panels: singular values in [0.3,
    1.3], so the polar factor is known to a few nw eps (1e-12); a singular or
    non-finite A is refused."""
    from wannier90_amd import capi, synth

    print(f"[projection] nw {nw}", flush=True)
    p = synth.make_problem(77 + nw, kind="sc", nw=nw, mp=(2, 2, 2), decay=2.0)
    rng = np.random.default_rng(nw)
    a = rng.normal(size=(8, nw, nw)) + 1j * rng.normal(size=(8, nw, nw))
    z, _, vh = np.linalg.svd(a)
    a = (z * rng.uniform(0.3, 1.3, size=(8, 1, nw))) @ vh
    ref = z @ vh
    af = np.asfortranarray(np.transpose(a, (1, 2, 0)))
    m = np.array(p.m_orig, order="F")
    u = ctx.project(p.kmesh, af, m)
    assert np.abs(np.transpose(u, (2, 0, 1)) - ref).max() <= 1e-12
    k2 = p.kmesh.nnlist[:, 0] - 1
    mk = np.conj(np.transpose(ref, (0, 2, 1))) @ np.transpose(p.m_orig[:, :, 0, :], (2, 0, 1)) @ ref[k2]
    assert np.abs(np.transpose(m[:, :, 0, :], (2, 0, 1)) - mk).max() <= 1e-11
    for bad in (0.0, np.nan, np.inf):
        b = af.copy(order="F")
        b[:, 0, 3] = bad
        with pytest.raises(capi.W90Error):
            ctx.project(p.kmesh, b, np.array(p.m_orig, order="F"))
