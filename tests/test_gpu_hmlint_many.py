"""Radial integrals of many atoms (exh_hmlint): with at least 256 workgroups
at three channel tiles per wave the radial kernel takes that form.  131 atoms
of two species (chunks of four atoms end in a chunk of two and of one), 13
radial functions (91 pairs: the last of six pair tiles is partly empty), and
channel counts of one tile, two and a quarter, and five and a sixteenth.

Against the oracle; relative error of the largest element <= 1e-12, the
tolerance of the other hmlint tests.
"""
import functools

import numpy as np
import pytest

import oracle
from exciting_amd import lapw, synth


@functools.lru_cache(maxsize=None)
def _cell():
    n = (6, 5, 5)
    pos = np.array(list(np.ndindex(*n)), float)[:131] / n
    return synth.build(synth.CellSpec(
        name="many", avec=4.0 * np.diag(np.array(n, float)), positions=[pos[:70], pos[70:]],
        rmt=[1.8, 1.8], lmaxapw=4, lmaxmat=4, apword=2, lo_l=[[0, 1, 2], [0, 1]], rgkmax=2.0,
        gmaxvr=2.5, kpoints=np.array([[0.13, -0.21, 0.37]]), nrmt=120, seed=31))


@pytest.mark.gpu
@pytest.mark.parametrize("lmaxvr", [3, 5, 8])
def test_hmlint_of_many_atoms(lmaxvr):
    s = synth.add_mt_potential(_cell(), lmaxvr=lmaxvr, seed=9)
    print(f"[gpu-hmlint-many] lmaxvr {lmaxvr} natmtot {s.natmtot}", flush=True)
    want = oracle.hmlint(oracle.System(s))
    ctx = lapw.Context(0).load(s)
    try:
        got = ctx.hmlint(lmaxvr, s.veffmt, s.lofr, True)
        for g, w, what in zip(got, want, ("aa", "loa", "lolo")):
            assert np.abs(g - w).max() <= 1e-12 * np.abs(w).max(), what
    finally:
        ctx.close()
