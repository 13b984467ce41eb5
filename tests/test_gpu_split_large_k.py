"""Split precision of a basis whose sums of residue products could leave int32
(natmtot * maxaa above 146000): it runs in FP64, as the same call without it."""
import numpy as np
import pytest

from exciting_amd import lapw, synth


@pytest.mark.gpu
def test_more_functions_than_int32_sums_hold():
    import torch
    rng = np.random.default_rng(9)
    n = 8112                                   # 18 functions each: K = 146016
    s = synth.build(synth.CellSpec(
        name="many", avec=6.0 * np.eye(3), positions=[rng.uniform(0, 1, (n, 3))], rmt=[1.0],
        lmaxapw=2, lmaxmat=2, apword=2, lo_l=[[]], rgkmax=3.0, gmaxvr=7.0,
        kpoints=np.array([[0.1, 0.2, 0.3]]), nrmt=20, seed=9))
    assert s.natmtot * s.maxaa == 146016 and s.ngkmax < 64
    ctx = lapw.Context(0).load(s)
    try:
        d = lapw.DeviceKPoint(s, 0)
        ctx.match(d.ngk, d.gpc, d.tpgpc, d.sfacgp, d.apwalm)
        out = []
        for flags in (0, lapw.SPLIT(7)):
            y, b = lapw.newsystem(d.rank, device="cuda"), lapw.newsystem(d.rank, device="cuda")
            ctx.profile(True)
            ctx.profile_reset()
            ctx.hamiltonandoverlapsetup(y, d.ngk, d.apwalm, d.igpig, d.vgpc, flags=flags)
            ctx.setup_batch([lapw.kpoint_struct(d, b.hamilton.za, b.overlap.za)], flags=flags)
            torch.cuda.synchronize()
            ran = {k for k, v in ctx.profile_read().items() if v[1]}
            assert {"ho", "ho_grouped"} <= ran and "oz_gemm" not in ran
            out += [m.za for v in (y, b) for m in (v.hamilton, v.overlap)]
        for x in (out[2], out[4], out[6]):
            assert torch.equal(x, out[0])
        for x in (out[3], out[5], out[7]):
            assert torch.equal(x, out[1])
    finally:
        ctx.close()
