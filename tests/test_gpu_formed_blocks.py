"""How many blocks a rotation forms (w90gpu_session_formed_blocks), and the work
that the benchmark's roofline counts from it: half of the blocks by pairs in
FP64 above 16 bands, every block else, whatever the precision of the solve (the
timed rotation is the FP64 one)."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from wannier90_amd import capi

    c = capi.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("nw,paired,half", [(16, True, False), (17, True, True), (17, False, False), (65, True, True),
                                            (65, False, False)])
def test_roofline_counts_the_formed_blocks(ctx, nw, paired, half, mixed):
    import bench
    from wannier90_amd import capi, synth

    p = synth.make_problem(53 + nw, kind="bcc", nw=nw, mp=(2, 2, 2), decay=2.0)
    u, m = synth.initial_state(p)
    if not paired:
        m[0, 1, 3, 2] += 1e-9
    prec = capi.PREC_MIXED if mixed else capi.PREC_FP64
    s = ctx.session(p.kmesh, nw, p.num_kpts, capi.control(num_iter=2, precision=prec))
    with pytest.raises(capi.W90Error):
        s.formed_blocks()
    s.load(m, u)
    s.solve()
    nn, nk = p.kmesh.nntot, p.num_kpts
    formed = nn // 2 if half else nn
    assert s.formed_blocks() == formed
    r = bench.rotation_roofline(s, nw, nk, nn, 2)
    s.close()
    assert r["algorithmic_flops"] == 16 * nk * formed * nw**3
    assert r["algorithmic_bytes"] == 16 * nk * nw**2 * (formed + nn + 1)
    assert r["achieved"] > 0 and r["avg_launch_ms"] > 0
