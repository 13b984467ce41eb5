"""The modular (int8) contraction: FP64 setups of all but the smallest bases,
and every EXH_SPLIT modulus count.

A 12-atom cell (lmaxapw 10, K = 2904, 1766 G+k) runs on it.  Truncated to
small and ragged G+k counts (edges of the 32, 128 and 384 tiles) H and O are
compared with the oracle, element by element, relative to the norms of the
columns that meet in it: with K = 2904 the operands' rounding is at most
2 sqrt(2K) 2^-55 = 4.2e-15 of them, and the oracle's own FP64 sums at most
about K 2^-53 = 3.2e-13 (B = aa.A adds as much): 1e-12 covers both.  The
overlap, which has no B, is also held to its rounding bound alone, against
extended precision; the FP64 kernels' sums exceed that bound.
"""
import numpy as np
import pytest

import oracle
from exciting_amd import lapw, synth
from tests import _cases, bruteforce
from tests.test_gpu_edges import truncated
from tests.test_gpu_split import split_expected, rel


def cell(rel_="none", lmaxmat=10, rgkmax=8.0):
    rng = np.random.default_rng(77)
    n = (2, 2, 3)
    pts = [[], []]
    for s in np.ndindex(*n):
        pts[sum(s) % 2].append((np.array(s, float) + rng.normal(0, 0.01, 3)) / np.array(n))
    s = synth.build(synth.CellSpec(
        name="c12", avec=5.13 * np.diag(np.array(n, float)), positions=[np.array(p) for p in pts],
        rmt=[2.0, 2.0], lmaxapw=10, lmaxmat=lmaxmat, apword=2, lo_l=[[0, 1], [0]],
        rgkmax=rgkmax, gmaxvr=12.0, kpoints=np.array([[0.11, 0.23, 0.31]]), seed=5))
    if rel_ != "none":
        synth.add_relativity(s, seed=6, iora=rel_ == "iora")
    op = 16 * s.natmtot * sum(2 * (2 * l + 1) for l in range(lmaxmat + 1)) * s.ngkmax
    assert op > 64 << 20, "the cell has to exceed the line of the rule"
    return s


@pytest.fixture(scope="module")
def ctxs():
    cache = {}

    def get(*key):
        if key not in cache:
            s = cell(*key)
            cache[key] = (s, lapw.Context(0).load(s))
        return cache[key]
    yield get
    for s, c in cache.values():
        c.close()


def operands(s, A, ng):
    X, B = [], []
    for a in range(s.natmtot):
        x = bruteforce.stacked_A(s, A, a, ng)
        X.append(x)
        B.append(s.aa[:x.shape[0], :x.shape[0], a] @ x)
    return np.concatenate(X), np.concatenate(B)


def device_setup(ctx, s, A, flags=0, h=None, o=None, only_o=False):
    """H and O (n x n) of the first k-point from the host array A."""
    import torch
    k, n = s.kpts[0], s.kpts[0].ngk + s.nlotot
    dev = lambda x, dt: torch.from_numpy(np.ascontiguousarray(x.ravel(order="F"))).to("cuda", dt)
    a, ig, vg = dev(A, torch.complex128), dev(k.igpig, torch.int32), dev(k.vgpc, torch.float64)
    mk = lambda x: (torch.full((n, n), float("nan"), dtype=torch.complex128, device="cuda")
                    if x is None else torch.from_numpy(np.ascontiguousarray(x.T)).cuda())
    y = lapw.EvSystem(None if only_o else lapw.HermitianMatrix(n, mk(h)),
                      lapw.HermitianMatrix(n, mk(o)))
    ctx.profile(True)
    ctx.profile_reset()
    (ctx.overlapsetup if only_o else ctx.hamiltonandoverlapsetup)(y, k.ngk, a, ig, vg, flags=flags)
    torch.cuda.synchronize()
    ran = {name for name, v in ctx.profile_read().items() if v[1]}
    ctx.profile(False)
    return (None if only_o else y.hamilton.za.cpu().numpy().T, y.overlap.za.cpu().numpy().T, ran)


def norms(X):
    return np.linalg.norm(X, axis=0)


def check_apw_block(got, want, scale, ng, tol):
    d = np.abs(got[:ng, :ng] - want[:ng, :ng])
    assert (d <= tol * (scale + np.abs(want[:ng, :ng]))).all(), (d / scale).max()
    np.testing.assert_allclose(got[ng:], want[ng:], rtol=1e-12, atol=1e-12)
    assert np.array_equal(np.tril(got, -1), np.tril(got.conj().T, -1))


@pytest.mark.gpu
@pytest.mark.parametrize("ng", [1, 31, 33, 127, 129, 383, 385, 640, 0])
def test_fp64_setup_on_the_modular_path(ctxs, ng):
    s, ctx = ctxs()
    s = truncated(s, ng) if ng else s
    ng = s.kpts[0].ngk
    print(f"[modular] ngk {ng}", flush=True)
    A = oracle.match(oracle.System(s), 0)
    H0, O0 = oracle.setup(oracle.System(s), 0, A)
    H, O, ran = device_setup(ctx, s, A)
    assert "oz_gemm" in ran and "ho" not in ran
    X, B = operands(s, A, ng)
    nx, nb = norms(X), norms(B)
    check_apw_block(H, H0, np.outer(nx, nb) + np.outer(nb, nx), ng, 1e-12)
    check_apw_block(O, O0, np.outer(nx, nx), ng, 1e-12)
    # the overlap against extended precision on up to 40 columns
    c = np.unique(np.linspace(0, ng - 1, 40).astype(int))
    xr, xi = X[:, c].real.astype(np.longdouble), X[:, c].imag.astype(np.longdouble)
    HI, OI = bruteforce.interstitial(s, s.kpts[0])
    re = xr.T @ xr + xi.T @ xi + OI[np.ix_(c, c)].real
    im = xr.T @ xi - xi.T @ xr + OI[np.ix_(c, c)].imag
    up = np.triu(np.ones(re.shape, bool))
    got = O[np.ix_(c, c)]
    err = np.hypot((got.real - re).astype(float), (got.imag - im).astype(float))
    bound = (2 * np.sqrt(2 * X.shape[0]) * 2.0 ** -55 + 2.0 ** -53) * np.outer(nx[c], nx[c]) \
        + 2.0 ** -52 * np.abs(got)
    assert (err <= bound)[up].all(), (err / bound)[up].max()
    # O alone, and accumulation onto a Hermitian matrix
    _, O1, ran = device_setup(ctx, s, A, only_o=True)
    assert "oz_gemm" in ran and np.array_equal(O1, O)
    rng = np.random.default_rng(3)
    P = rng.standard_normal(H.shape) + 1j * rng.standard_normal(H.shape)
    P = P + P.conj().T
    Ha, Oa, _ = device_setup(ctx, s, A, flags=lapw.ACCUMULATE, h=P, o=P)
    iu = np.triu_indices(H.shape[0])
    np.testing.assert_allclose(Ha[iu], (H + P)[iu], rtol=1e-14, atol=1e-14)
    np.testing.assert_allclose(Oa[iu], (O + P)[iu], rtol=1e-14, atol=1e-14)


@pytest.mark.gpu
@pytest.mark.parametrize("key", [("iora", 10, 8.0), ("zora", 10, 8.0), ("none", 8, 8.8)])
def test_fp64_modular_layouts(ctxs, key):
    """iora* (the overlap's own column operand), zora, and a packed A^T
    (lmaxmat < lmaxapw)."""
    s, ctx = ctxs(*key)
    s = truncated(s, 301)
    ng = 301
    A = oracle.match(oracle.System(s), 0)
    H0, O0 = oracle.setup(oracle.System(s), 0, A)
    H, O, ran = device_setup(ctx, s, A)
    assert "oz_gemm" in ran
    X, B = operands(s, A, ng)
    nx, nb = norms(X), norms(B)
    check_apw_block(H, H0, np.outer(nx, nb) + np.outer(nb, nx), ng, 1e-12)
    check_apw_block(O, O0, 1.1 * np.outer(nx, nx), ng, 1e-12)
    _, O1, _ = device_setup(ctx, s, A, only_o=True)
    assert np.array_equal(O1, O)


@pytest.mark.gpu
def test_modular_columns_out_of_range(ctxs):
    """Zero columns, columns scaled far beyond where squares over- or
    underflow, and columns that are not finite."""
    s, ctx = ctxs()
    s = truncated(s, 150)
    ng = 150
    A = oracle.match(oracle.System(s), 0)
    A[3] = 0.0
    A[7] *= 1e-170
    A[11] *= 1e170
    H0, O0 = oracle.setup(oracle.System(s), 0, A)
    H, O, ran = device_setup(ctx, s, A)
    assert "oz_gemm" in ran
    X, B = operands(s, A, ng)
    big = lambda M: np.array([float(np.sqrt((np.abs(c.astype(np.clongdouble)) ** 2).sum()))
                              for c in M.T])
    nx, nb = big(X), big(B)
    with np.errstate(over="ignore"):   # (11, 11) itself overflows FP64
        scale_h, scale_o = np.outer(nx, nb) + np.outer(nb, nx), np.outer(nx, nx)
        ok = np.triu(np.isfinite(scale_h) & np.isfinite(scale_o))
        for got, want, sc in ((H, H0, scale_h), (O, O0, scale_o)):
            d = np.abs(got[:ng, :ng] - want[:ng, :ng])
            assert (d[ok] <= 1e-12 * (sc + np.abs(want[:ng, :ng]))[ok]).all()
    A[20, 0, 5, 2] = np.inf
    A[40, 1, 9, 4] = np.nan
    Hn, On, _ = device_setup(ctx, s, A)
    bad = np.zeros((ng, ng), bool)
    bad[[20, 40]] = True
    bad[:, [20, 40]] = True
    for got, fin in ((Hn, H), (On, O)):
        assert not np.isfinite(got[:ng, :ng][bad]).any()
        keep = ~bad
        assert np.array_equal(got[:ng, :ng][keep], fin[:ng, :ng][keep], equal_nan=True)


@pytest.mark.gpu
@pytest.mark.parametrize("nmod", [8, 10, 11, 12])
def test_split_modulus_counts(nmod):
    """The counts test_gpu_split does not run (12 multiplies 13 moduli): the
    rounded operands' product exactly."""
    s = _cases.system("tiny")
    ctx = lapw.Context(0).load(s)
    try:
        A = oracle.match(oracle.System(s), 0)
        H0, O0 = oracle.setup(oracle.System(s), 0, A)
        He, Oe, _ = split_expected(s, s.kpts[0], A, H0, O0, nmod)
        H, O, _ = device_setup(ctx, s, A, flags=lapw.SPLIT(nmod))
        assert rel(H, He) <= 1e-12 and rel(O, Oe) <= 1e-12
    finally:
        ctx.close()


@pytest.mark.gpu
@pytest.mark.parametrize("name,path", [("tiny_multi", "ho_grouped"), ("fcc2", "oz_gemm"),
                                       ("sc8_4k", "oz_gemm")])
def test_route_by_basis_size(name, path):
    """Bases below 2^15 (K, G+k) pairs stay on the FP64 MFMA tiles."""
    import torch
    s = _cases.system(name)
    ctx = lapw.Context(0).load(s)
    try:
        dk = [lapw.DeviceKPoint(s, i) for i in range(len(s.kpts))]
        ys = [lapw.newsystem(d.rank, device="cuda") for d in dk]
        kp = [lapw.kpoint_struct(d, y.hamilton.za, y.overlap.za) for d, y in zip(dk, ys)]
        ctx.profile(True)
        ctx.profile_reset()
        ctx.setup_batch(kp, flags=lapw.MATCH)
        torch.cuda.synchronize()
        ran = {n for n, v in ctx.profile_read().items() if v[1]}
        assert path in ran and len(ran & {"ho_grouped", "oz_gemm"}) == 1
    finally:
        ctx.close()


@pytest.mark.gpu
def test_grouped_call_mixes_both_contractions(ctxs):
    """One grouped call over a modular and an FP64-MFMA structure, eager and
    replayed from a graph: bitwise the single path."""
    import torch
    small = _cases.system("tiny_multi")
    s, ctx = ctxs()
    s = truncated(s, 257)
    c2 = lapw.Context(0).load(small)
    try:
        sets = [(ctx, lapw.DeviceKPoint(s, 0)), (c2, lapw.DeviceKPoint(small, 0)),
                (ctx, lapw.DeviceKPoint(s, 0)), (c2, lapw.DeviceKPoint(small, 1))]
        ref = []
        for c, d in sets:
            y = lapw.newsystem(d.rank, device="cuda")
            c.match(d.ngk, d.gpc, d.tpgpc, d.sfacgp, d.apwalm)
            c.hamiltonandoverlapsetup(y, d.ngk, d.apwalm, d.igpig, d.vgpc, flags=0)
            ref.append((y.hamilton.za, y.overlap.za))
        out = [lapw.newsystem(d.rank, device="cuda") for _, d in sets]
        kp = [lapw.kpoint_struct(d, y.hamilton.za, y.overlap.za)
              for (_, d), y in zip(sets, out)]
        for rep, flags in enumerate([0] + [lapw.GRAPH] * 3):
            for y in out:
                y.hamilton.za.fill_(rep + 1.0)
                y.overlap.za.fill_(rep + 1.0)
            lapw.setup_multi([c for c, _ in sets], kp, flags=flags | lapw.MATCH)
            torch.cuda.synchronize()
            for y, (h, o) in zip(out, ref):
                assert torch.equal(y.hamilton.za, h) and torch.equal(y.overlap.za, o)
    finally:
        c2.close()
