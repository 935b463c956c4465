"""An outer window that lies between two bands at some k holds no state there:
the call is refused before any kernel runs (its first state and its size would
lie outside the arrays)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nan", [False, True])
def test_window_in_a_gap_is_refused(nan):
    from wannier90_amd import capi, synth

    nb, nw = 6, 3
    p, ctl = synth.make_dis_problem(4, kind="sc", num_bands=nb, num_wann=nw, mp=(2, 2, 2), decay=2.0)
    eig = np.asfortranarray(np.tile(np.arange(nb, dtype=float)[:, None], (1, p.num_kpts)))
    eig[3:, 1] += 10.0  # a gap from 2 to 13 at the second k
    ctl.update(win_min=2.5, win_max=5.5)
    if nan:
        eig[:, 1] = np.nan
    ctx = capi.Context(0)
    with pytest.raises(capi.W90Error, match=r"fewer states than number of target WFs \(k-point 2, ndimwin=0"):
        ctx.disentangle(p.kmesh, nb, ctl, eig, p.amat_dis, p.m_orig)
    ctx.close()
