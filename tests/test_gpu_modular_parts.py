"""The modular products in parts: where the scratch does not hold the residues
of all moduli, they run a few at a time, and H and O are bitwise the same.
Neither the static array's size nor the device's free memory decides which
kernels run.
"""
import dataclasses

import numpy as np
import pytest

from exciting_amd import lapw, synth
from tests import _cases
from tests.test_gpu_edges import truncated
from tests.test_zz_no_alloc import prepared, run

STATIC = 256 << 20   # the static array's part for the modular products


def grid12(lmax, rgkmax):
    rng = np.random.default_rng(78)
    n = (2, 2, 3)
    pts = [[], []]
    for s in np.ndindex(*n):
        pts[sum(s) % 2].append((np.array(s, float) + rng.normal(0, 0.01, 3)) / np.array(n))
    return synth.build(synth.CellSpec(
        name="c12", avec=5.13 * np.diag(np.array(n, float)), positions=[np.array(p) for p in pts],
        rmt=[2.0, 2.0], lmaxapw=lmax, lmaxmat=lmax, apword=2, lo_l=[[0, 1], [0]],
        rgkmax=rgkmax, gmaxvr=12.0, kpoints=np.array([[0.11, 0.23, 0.31]]), seed=5))


def system(name):
    if name == "c12_lmax6_iora":
        return synth.add_relativity(grid12(6, 7.9), seed=6, iora=True)
    return grid12(8, 8.0)


@pytest.mark.gpu
@pytest.mark.parametrize("name,nops", [("c12_lmax6_iora", 3), ("c12_lmax8", 2)])
def test_static_array_that_holds_some_moduli(name, nops):
    import torch
    s = system(name)
    pad = lambda n, m: -(-n // m) * m
    K, G = s.natmtot * s.maxaa, pad(s.ngkmax, 128)
    nt = G // 128
    full = 15 * 2 * nops * pad(K, 128) * G + 60 * nt * (nt + 1) // 2 * 128 * 128
    assert 16 * K * pad(s.ngkmax, 64) * (nops - 1) <= 64 << 20 and full > STATIC
    ctx = lapw.Context(0).load(s)
    try:
        d = prepared(ctx, s)
        print(f"[parts] {name}: K {K} ngk {d.ngk}, residues {full >> 20} MiB", flush=True)
        g = torch.Generator(device="cuda").manual_seed(3)
        pre = [torch.randn(d.rank ** 2, dtype=torch.complex128, device="cuda", generator=g)
               for _ in range(2)]
        for flags, p in ((0, None), (lapw.ACCUMULATE, pre)):
            Hd, Od = run(ctx, d, False, flags, p)
            Hn, On = run(ctx, d, True, flags, p)
            assert torch.equal(Hn, Hd) and torch.equal(On, Od)
    finally:
        ctx.close()


@pytest.mark.gpu
def test_route_and_bits_do_not_depend_on_free_memory():
    """With about 1.1 GiB left on the device, below what the residues and the
    margin for the caller need."""
    import torch
    s = _cases.system("sc8_4k")

    def setups():
        ctx = lapw.Context(0).load(s)
        try:
            ctx.profile(True)
            ctx.profile_reset()
            out = []
            dk = [lapw.DeviceKPoint(s, i) for i in range(2)]
            for d in dk:
                ctx.match(d.ngk, d.gpc, d.tpgpc, d.sfacgp, d.apwalm)
            out += run(ctx, dk[0], False, 0)
            y = lapw.newsystem(dk[1].rank, device="cuda")
            ctx.overlapsetup(lapw.EvSystem(None, y.overlap), dk[1].ngk, dk[1].apwalm,
                             dk[1].igpig, dk[1].vgpc, flags=0)
            out.append(y.overlap.za)
            ys = [lapw.newsystem(d.rank, device="cuda") for d in dk]
            ctx.setup_batch([lapw.kpoint_struct(d, v.hamilton.za, v.overlap.za)
                             for d, v in zip(dk, ys)], flags=0)
            torch.cuda.synchronize()
            ran = {n for n, v in ctx.profile_read().items() if v[1]}
            return out + [m.za for v in ys for m in (v.hamilton, v.overlap)], ran
        finally:
            ctx.close()

    ref, ran = setups()
    assert "oz_gemm" in ran and not ran & {"ho", "ho_grouped"}
    torch.cuda.empty_cache()
    free, _ = torch.cuda.mem_get_info()
    hog = torch.empty(free - (1100 << 20), dtype=torch.uint8, device="cuda")
    try:
        print(f"[parts] {torch.cuda.mem_get_info()[0] >> 20} MiB free", flush=True)
        got, ran = setups()
    finally:
        del hog
        torch.cuda.empty_cache()
    assert "oz_gemm" in ran and not ran & {"ho", "ho_grouped"}
    for a, b in zip(got, ref):
        assert torch.equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("flags", [0, lapw.SPLIT(9)])
@pytest.mark.parametrize("mib", [0, 64, 96, 160, 400])
def test_workspace_limit_bounds_a_grouped_call(mib, flags):
    """Four k-points of 38 MB of arrays and 211 MB (FP64) of residues each: the
    limit is kept, down to what one k-point needs at least (its arrays, and the
    residues of one modulus and one column step, below 60 MB), and the results
    are bitwise the single path's."""
    import torch
    s = _cases.system("sc8_4k")
    warm, ctx = lapw.Context(0).load(s), lapw.Context(0).load(s)
    try:
        dk = [lapw.DeviceKPoint(s, i) for i in range(4)]
        ys, ref = [], []
        for d in dk:
            y = lapw.newsystem(d.rank, device="cuda")
            warm.match(d.ngk, d.gpc, d.tpgpc, d.sfacgp, d.apwalm)
            warm.hamiltonandoverlapsetup(y, d.ngk, d.apwalm, d.igpig, d.vgpc, flags=flags)
            ref.append((y.hamilton.za, y.overlap.za))
            ys.append(lapw.newsystem(d.rank, device="cuda"))
        kp = [lapw.kpoint_struct(d, y.hamilton.za, y.overlap.za) for d, y in zip(dk, ys)]
        for limit in (1, 8 << 30):            # loads every kernel
            warm.set_batch_workspace(limit)
            warm.setup_batch(kp, flags=flags | lapw.MATCH)
        ctx.set_batch_workspace(max(mib << 20, 1))
        torch.cuda.synchronize()
        before = torch.cuda.mem_get_info()[0]
        ctx.setup_batch(kp, flags=flags | lapw.MATCH)
        torch.cuda.synchronize()
        took = before - torch.cuda.mem_get_info()[0]
        print(f"[parts] limit {mib} MiB: took {took >> 20} MiB", flush=True)
        # the allocator's pages of 2 MiB, for each of a dozen buffers
        assert took <= max(mib << 20, 100 << 20) + (24 << 20)
        for y, (h, o) in zip(ys, ref):
            assert torch.equal(y.hamilton.za, h) and torch.equal(y.overlap.za, o)
    finally:
        warm.close()
        ctx.close()


@pytest.mark.gpu
@pytest.mark.parametrize("lmax,edge,route", [(2, 12.3, "ho"), (6, 7.75, "ho"), (8, 6.2, "oz_gemm"),
                                             (8, 9.75, "ho"), (10, 9.75, "oz_gemm"),
                                             (10, 16.0, "ho")])
def test_route_of_short_bases(lmax, edge, route):
    """One atom: K = 18, 98, 162, 162, 242, 242 with 2000, 500, 250, 1000, 1000 and
    4400 G+k.  Few functions stay on the FP64 MFMA tiles, and every entry point
    takes the same kernels: bitwise the same H and O."""
    import torch
    s = synth.build(synth.CellSpec(
        name="one", avec=edge * np.eye(3), positions=[np.array([[0.1, 0.2, 0.3]])], rmt=[2.0],
        lmaxapw=lmax, lmaxmat=lmax, apword=2, lo_l=[[0]], rgkmax=8.0, gmaxvr=9.0,
        kpoints=np.array([[0.1, 0.2, 0.3]]), seed=3))
    ctx = lapw.Context(0).load(s)
    try:
        d = prepared(ctx, s)
        print(f"[parts] K {s.maxaa} ngk {d.ngk}", flush=True)
        ctx.profile(True)
        ctx.profile_reset()
        Hd, Od = run(ctx, d, False, 0)
        ys = [lapw.newsystem(d.rank, device="cuda") for _ in range(3)]
        ctx.overlapsetup(lapw.EvSystem(None, ys[2].overlap), d.ngk, d.apwalm, d.igpig, d.vgpc,
                         flags=0)
        ctx.setup_batch([lapw.kpoint_struct(d, y.hamilton.za, y.overlap.za) for y in ys[:2]],
                        flags=0)
        torch.cuda.synchronize()
        ran = {n for n, v in ctx.profile_read().items() if v[1]}
        want = {"oz_gemm"} if route == "oz_gemm" else {"ho", "ho_grouped"}
        assert ran & {"oz_gemm", "ho", "ho_grouped"} == want
        for y in ys[:2]:
            assert torch.equal(y.hamilton.za.ravel(), Hd)
            assert torch.equal(y.overlap.za.ravel(), Od)
        assert torch.equal(ys[2].overlap.za.ravel(), Od)
        Hn, On = run(ctx, d, True, 0)
        assert torch.equal(Hn, Hd) and torch.equal(On, Od)
    finally:
        ctx.close()


def wide(rel, graded):
    """Four atoms of 162 functions and 7700 G+k: so many that H's and O's
    operands take turns in the scratch."""
    at = np.array([[0.1, 0.2, 0.3], [0.6, 0.5, 0.9], [0.2, 0.7, 0.6], [0.7, 0.9, 0.1]])
    s = synth.build(synth.CellSpec(
        name="wide", avec=19.3 * np.eye(3), positions=[at], rmt=[2.0],
        lmaxapw=8, lmaxmat=8, apword=2, lo_l=[[0]], rgkmax=8.0, gmaxvr=9.0,
        kpoints=np.array([[0.1, 0.2, 0.3]]), seed=3))
    if rel == "iora":
        synth.add_relativity(s, seed=6, iora=True)
    if graded:
        c = np.ldexp(1.0, np.random.default_rng(2).integers(-9, 10, (s.maxaa, s.natmtot)))
        s = dataclasses.replace(s, aa=np.asfortranarray(s.aa * c[:, None] * c[None]))
    return s


def narrow(s):
    """The same k-point in a basis of no more than its own G+k."""
    k, m = s.kpts[0], s.kpts[0].ngk
    k = dataclasses.replace(k, igpig=k.igpig[:m].copy(), vgpc=k.vgpc[:, :m].copy(order="F"),
                            gpc=k.gpc[:m].copy(), tpgpc=k.tpgpc[:, :m].copy(order="F"),
                            sfacgp=k.sfacgp[:m].copy(order="F"))
    return dataclasses.replace(s, ngkmax=m, kpts=[k])


@pytest.mark.gpu
@pytest.mark.parametrize("graded", [False, True])
@pytest.mark.parametrize("rel", ["none", "iora"])
def test_operands_that_take_turns(rel, graded):
    """730 of those G+k, and the same ones in a basis of 730, whose operands are
    all there at once: bitwise the same H and O; also in the smallest parts."""
    import torch
    s = truncated(wide(rel, graded), 730)
    assert s.ngkmax > 7500
    big, small = lapw.Context(0).load(s), lapw.Context(0).load(narrow(s))
    try:
        d, e = lapw.DeviceKPoint(s, 0), lapw.DeviceKPoint(narrow(s), 0)
        for c, x in ((big, d), (small, e)):
            c.match(x.ngk, x.gpc, x.tpgpc, x.sfacgp, x.apwalm)
        big.profile(True)
        big.profile_reset()
        Hs, Os = run(small, e, False, 0)
        Hb, Ob = run(big, d, False, 0)
        assert torch.equal(Hb, Hs) and torch.equal(Ob, Os)
        assert big.profile_read()["oz_gemm"][1] == 2       # H's products, then O's
        print(f"[parts] {rel} graded {graded}", flush=True)
        for limit in (8 << 30, 2050 << 20, 450 << 20, 1):
            big.set_batch_workspace(limit)
            y = lapw.newsystem(d.rank, device="cuda")
            big.setup_batch([lapw.kpoint_struct(d, y.hamilton.za, y.overlap.za)], flags=0)
            torch.cuda.synchronize()
            assert torch.equal(y.hamilton.za.ravel(), Hs) and torch.equal(y.overlap.za.ravel(), Os)
    finally:
        big.close()
        small.close()
