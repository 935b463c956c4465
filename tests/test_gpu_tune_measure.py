"""What the online tuner (W90GPU_TUNE=1) times.

Up to 48 bands its choice is for the FP32 phase (the FP64 rotation is one
kernel whatever the choice), so it has to time the FP32 kernels: at 24 bands
fused64 works on a padded 64 x 64 tile, four times the area of fused32's, and
2.9 to 3.3 times slower by the FP64 instances of both; 1.5 times is asked for.
Timings of one kernel under two names agree to a few percent.

Above 48 bands it times the FP64 rotation as it will run: for overlaps that
pair, half of the blocks.  At 52 bands 0.8 of the time block by block is asked
for (0.61 at 64 bands, measured as 419 of 690 us).
"""
import pytest

pytestmark = pytest.mark.gpu


def tuned(monkeypatch, path, kmesh, nw, nk, m, u, **kw):
    """The choice and the times (us) that the first solve of the key records."""
    from wannier90_amd import capi

    nn = kmesh.nntot
    capi.tune_set(nw, nn, None)
    monkeypatch.setenv("W90GPU_TUNE", "1")
    monkeypatch.setenv("W90GPU_TUNE_FILE", str(path))
    try:
        c = capi.Context(0)
        s = c.session(kmesh, nw, nk, capi.control(num_iter=1, **kw))
        s.load(m, u)
        s.solve()
        s.close()
        c.close()
    finally:
        monkeypatch.delenv("W90GPU_TUNE")
        monkeypatch.delenv("W90GPU_TUNE_FILE")
        capi.Context(0).close()  # the environment is read when a context is created
        capi.tune_set(nw, nn, None)
    (line,) = [ln.split() for ln in open(path) if ln.split()[:2] == [str(nw), str(nn)]]
    times = {k: float(v) for k, v in (f.split("=") for f in line[3:] if not f.startswith("items"))}
    print(f"[tune] nw {nw} nn {nn}: {line[2]} of {times}", flush=True)
    return line[2], times


def problem(nw):
    from wannier90_amd import synth

    p = synth.make_problem(600 + nw, kind="sc", nw=nw, mp=(4, 4, 4), decay=2.0)
    u, m = synth.initial_state(p)
    return p, u, m


@pytest.mark.parametrize("mixed", [False, True])
def test_up_to_48_bands_the_fp32_kernels_are_timed(monkeypatch, tmp_path, mixed):
    from wannier90_amd import capi

    p, u, m = problem(24)
    prec = capi.PREC_MIXED if mixed else capi.PREC_FP64
    pick, t = tuned(monkeypatch, tmp_path / "t.txt", p.kmesh, 24, p.num_kpts, m, u, precision=prec)
    assert set(t) == {"fused32", "fused64"}
    assert t["fused64"] > 1.5 * t["fused32"]
    assert pick == "fused32"


def test_above_48_bands_the_rotation_by_pairs_is_timed(monkeypatch, tmp_path):
    p, u, m = problem(52)
    _, by_pairs = tuned(monkeypatch, tmp_path / "pairs.txt", p.kmesh, 52, p.num_kpts, m, u)
    m1 = m.copy(order="F")
    m1[51, 0, 0, 0] += 1e-3
    _, by_block = tuned(monkeypatch, tmp_path / "blocks.txt", p.kmesh, 52, p.num_kpts, m1, u)
    assert set(by_pairs) == set(by_block) == {"fused64", "direct64"}
    for k in by_pairs:
        assert by_pairs[k] < 0.8 * by_block[k]
