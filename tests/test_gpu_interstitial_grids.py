"""The interstitial producers (exh_gencfun_device, exh_genveffig_device) on
uneven FFT grids: odd and even lengths along each axis (the half-grid
transform of the real products and the conjugates read for the other half),
lengths that are no multiple of the four rows of a thread, fewer points than
one workgroup, and more atoms (131) than one
block of kernel arguments holds.

Against the oracle; relative error (norm and largest element) <= 1e-12, the
tolerance of the other interstitial tests.
"""
import numpy as np
import pytest

import oracle
from exciting_amd import lapw, synth
from tests.test_gpu_hmlint_many import _cell


def _odd(a, gmax, d):
    return synth.build(synth.CellSpec(
        name="odd", avec=a * np.diag(d) + 0.1 * np.tri(3, k=-1),
        positions=[np.array([[0.02, 0.1, 0.0]]), np.array([[0.5, 0.47, 0.55]])], rmt=[1.0, 0.9],
        lmaxapw=3, lmaxmat=3, apword=1, lo_l=[[0], []], rgkmax=1.2, gmaxvr=gmax,
        kpoints=np.zeros((1, 3)), nrmt=60, seed=3))


CELLS = {"3x4x5": lambda: _odd(4.5, 2.0, (1.0, 1.3, 1.7)),
         "5x8x9": lambda: _odd(5.0, 3.0, (1.0, 1.3, 1.7)),
         "6x8x10": lambda: _odd(5.0, 3.0, (1.1, 1.5, 2.0)),
         "131 atoms": _cell}


@pytest.mark.gpu
@pytest.mark.parametrize("name", list(CELLS))
def test_producers_on_uneven_grids(name):
    import torch
    s = CELLS[name]()
    print(f"[gpu-interstitial-grids] {name}: grid {list(s.ngrid)} atoms {s.natmtot}", flush=True)

    def close(got, want):
        got = got.cpu().numpy()
        assert np.linalg.norm(got - want) <= 1e-12 * np.linalg.norm(want)
        assert np.abs(got - want).max() <= 1e-12 * np.abs(want).max()

    zeros = lambda n, dt=torch.complex128: torch.zeros(n, dtype=dt, device="cuda")
    ctx = lapw.Context(0).load(s)
    try:
        cg0, cr0 = oracle.gencfun(s, cfdamp=0.4, gmaxvr=s.spec.gmaxvr)
        cg, cr = zeros(s.ngrtot), zeros(s.ngrtot, torch.float64)
        ctx.gencfun(s.bvec, s.atposc, cfdamp=0.4, gmaxvr=s.spec.gmaxvr, cfunig=cg, cfunir=cr)
        close(cg, cg0)
        close(cr, cr0)
        v = -0.4 + 0.3 * np.random.default_rng(2).uniform(-1, 1, s.ngrtot)
        outs = {n: zeros(s.ngvec) for n in ("veffig", "meffig", "m2effig")}
        ctx.genveffig_device(torch.from_numpy(v).cuda(), torch.from_numpy(cr0).cuda(), **outs)
        m, m2 = oracle.genmeffig(s, v, cr0, True)
        for n, want in (("veffig", oracle.genveffig(s, v, cr0)), ("meffig", m), ("m2effig", m2)):
            close(outs[n], want)
    finally:
        ctx.close()
