"""Each rotation kernel on the problems where it is the one that runs, by pairs
and block by block: the FP64 kernels above 48 bands, the FP32 ones in the mixed
bulk phase from 17 bands on, the FP64 rebuild that ends it, and the two ways
next to each other in a batch and one after the other in a session.

The overlaps that a solve returns are compared with the overlaps it was given,
rotated by the U that it returns relative to the U that it was given:
M = V(k)^+ M0 V(k+b), V = U0^+ U, formed by numpy.  Each of the 3 iterations
rounds two products of at most nw terms of blocks of norm 1, 2 nw eps an
element or less, and V's departure from unitarity is of that size too; 3 * 4 *
96 * 1.1e-16 = 1.3e-13 at the largest, and 1e-11 is far above that and far below
any misplaced element (about 1/nw).
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


_cache = {}


def problem(kind, nw, mp, paired):
    """Overlaps that pair, or with one element off by 1e-9 (the check at load
    allows 2 nw eps)."""
    from wannier90_amd import synth

    key = (kind, nw, mp)
    if key not in _cache:
        p = synth.make_problem(811 + nw, kind=kind, nw=nw, mp=mp, decay=2.0)
        _cache[key] = (p, *synth.initial_state(p))
    p, u, m = _cache[key]
    if not paired:
        m = m.copy(order="F")
        m[nw - 1, 0, 0, p.num_kpts - 1] += 1e-9
    return p, u, m


class forced:
    def __init__(self, p, name):
        self.key, self.name = (p.num_wann, p.kmesh.nntot), name

    def __enter__(self):
        from wannier90_amd import capi

        capi.tune_set(*self.key, self.name)

    def __exit__(self, *exc):
        from wannier90_amd import capi

        capi.tune_set(*self.key, None)


def solve(ctx, p, u, m, n=3, lfixstep=1, **kw):
    from wannier90_amd import capi

    s = ctx.session(p.kmesh, p.num_wann, p.num_kpts, capi.control(num_iter=n, lfixstep=lfixstep, fixed_step=1.0, **kw))
    s.load(m, u)
    formed = s.formed_blocks()
    r = s.solve()
    hist = s.history()
    mf, uf, _, _ = s.fetch()
    s.close()
    return r, formed, hist, mf, uf


def check_rotated(p, u0, m0, u, m):
    v = np.matmul(np.conj(np.transpose(u0, (2, 1, 0))), np.transpose(u, (2, 0, 1)))
    assert np.abs(v - np.eye(p.num_wann)).max() > 1e-7  # the steps moved U, far above the bound
    for b in range(p.kmesh.nntot):
        k2 = p.kmesh.nnlist[:, b] - 1
        r = np.matmul(np.conj(np.transpose(v, (0, 2, 1))), np.matmul(np.transpose(m0[:, :, b, :], (2, 0, 1)), v[k2]))
        assert np.abs(np.transpose(m[:, :, b, :], (2, 0, 1)) - r).max() <= 1e-11


def mates(kmesh):
    """(k, b) -> (k', b') with k' = k + b, b' = -b."""
    nk, nn = kmesh.nnlist.shape
    out = {}
    for k in range(nk):
        for b in range(nn):
            k2 = int(kmesh.nnlist[k, b]) - 1
            (b2,) = [c for c in range(nn) if kmesh.nnlist[k2, c] == k + 1
                     and np.allclose(kmesh.bk[:, c, k2], -kmesh.bk[:, b, k], atol=1e-6)]
            out[k, b] = k2, b2
    return out


FP64 = [("sc", 49, (3, 2, 2)), ("bcc", 52, (2, 2, 2)), ("triclinic", 64, (2, 2, 2))]
FP64_PARAMS = [(c, k) for c in FP64 for k in ("fused64", "direct64")]
FP64_PARAMS += [(c, k) for c in [("sc", 65, (2, 2, 3)), ("fcc", 96, (2, 2, 2))] for k in ("gemm64", "gemm32")]
FP64_PARAMS += [(c, None) for c in [("hex", 17, (2, 3, 2)), ("fcc", 32, (2, 2, 2)), ("sc", 33, (3, 3, 2)),
                                    ("bcc", 48, (2, 2, 2))]]


@pytest.mark.parametrize("paired", [True, False])
@pytest.mark.parametrize("case,kernel", FP64_PARAMS, ids=lambda x: "-".join(map(str, x[:2])) if type(x) is tuple else x)
def test_fp64_kernel_rotates(ctx, case, kernel, paired):
    print(f"[forced] {case} {kernel} paired {paired}", flush=True)
    p, u0, m0 = problem(*case, paired)
    with forced(p, kernel):
        _, formed, _, m, u = solve(ctx, p, u0, m0)
    assert formed == (p.kmesh.nntot // 2 if paired else p.kmesh.nntot)
    check_rotated(p, u0, m0, u, m)
    if paired:  # the second block of a pair is the adjoint of the first, to the bit
        for (k, b), (k2, b2) in mates(p.kmesh).items():
            assert np.array_equal(m[:, :, b2, k2], m[:, :, b, k].conj().T)


FP32 = [(("fcc", 24, (3, 3, 3)), ("fused32", "fused64")), (("sc", 40, (3, 3, 3)), ("direct64", "fused64", "fused48")),
        (("bcc", 52, (2, 2, 2)), ("direct64", "fused64")), (("hex", 70, (2, 2, 2)), ("gemm64", "gemm32"))]


@pytest.mark.parametrize("paired", [True, False])
@pytest.mark.parametrize("case,kernel", [(c, k) for c, ks in FP32 for k in ks],
                         ids=lambda x: "-".join(map(str, x[:2])) if type(x) is tuple else x)
def test_fp32_kernel_in_the_bulk_phase(ctx, case, kernel, paired):
    """5 steps in FP32 follow FP64's Omega to 1e-4 relative (five
    rotations of blocks of norm 1 round at nw 2^-24 an element, 2e-5 at 70
    bands; Omega is a sum over such elements), and the M returned is the FP64
    rebuild from the initial overlaps."""
    from wannier90_amd import capi

    print(f"[forced mixed] {case} {kernel} paired {paired}", flush=True)
    p, u0, m0 = problem(*case, paired)
    with forced(p, kernel):
        _, _, h64, _, _ = solve(ctx, p, u0, m0, 5, 0)
        r, _, h, m, u = solve(ctx, p, u0, m0, 5, 0, precision=capi.PREC_MIXED)
    assert r.iterations == 5 and r.bulk_iterations > 0
    nb = r.bulk_iterations
    assert np.abs(h[:nb, 0] - h64[:nb, 0]).max() <= 1e-4 * np.abs(h64[:, 0]).max()
    check_rotated(p, u0, m0, u, m)


SHAPES = [("sc", 20, (3, 3, 2)), ("fcc", 40, (2, 2, 2)), ("sc", 52, (2, 2, 2)), ("hex", 70, (2, 2, 2))]


def test_paired_and_unpaired_members_of_a_batch(ctx):
    """Every result is that of the problem alone, bit for bit, with members of
    both kinds in each launch."""
    from wannier90_amd import capi

    ctl = capi.control(num_iter=3, lfixstep=1, fixed_step=1.0)
    todo = [problem(*c, paired) for c in SHAPES for paired in (True, False, True)]
    b = ctx.batch(sum(capi.problem_bytes(p.num_wann, p.num_kpts, p.kmesh.nntot, 3) for p, _, _ in todo))
    ids = [b.add(p.kmesh, m, u, ctl) for p, u, m in todo]
    b.run()
    for i, (p, u0, m0) in zip(ids, todo):
        m, u = b.fetch(i, want_m=True)[:2]
        _, _, _, ma, ua = solve(ctx, p, u0, m0)
        assert np.array_equal(m, ma) and np.array_equal(u, ua)
    b.close()


@pytest.mark.parametrize("case", SHAPES, ids=lambda c: f"{c[0]}-{c[1]}")
def test_session_loaded_with_paired_and_unpaired_overlaps(ctx, case):
    from wannier90_amd import capi

    p, u0, m0 = problem(*case, True)
    _, _, m1 = problem(*case, False)
    nn = p.kmesh.nntot
    s = ctx.session(p.kmesh, p.num_wann, p.num_kpts, capi.control(num_iter=3, lfixstep=1, fixed_step=1.0))
    for m in (m0, m1, m0):
        s.load(m, u0)
        assert s.formed_blocks() == (nn // 2 if m is m0 else nn)
        s.solve()
        mf, uf, _, _ = s.fetch()
        _, _, _, ma, ua = solve(ctx, p, u0, m)
        assert np.array_equal(mf, ma) and np.array_equal(uf, ua)
    s.close()
