"""The APW-lo border at the edges of its tiles: local-orbital counts around
its 16-column blocks (one to four of them), species without local orbitals,
f ranges shorter than the four-way split, G+k counts around its 16-row tile,
overwrite, accumulate and O alone; border and lo-lo blocks against the
oracle to 1e-13 of the largest element (sums of at most 48 products in FP64).
"""
import dataclasses

import numpy as np
import pytest

import oracle
from exciting_amd import lapw, synth
from tests.test_gpu_edges import truncated
from tests.test_gpu_modular import device_setup

L16 = [0, 1, 2, 3]
CASES = {  # lo_l per species, lmaxmat, apword
    "1": ([[0], [0]], 3, 2), "16_0": ([L16, []], 3, 2), "17_1": ([L16 + [0], [0]], 3, 1),
    "32_3": ([L16 * 2, [1]], 2, 3), "33_16": ([L16 * 2 + [0], L16], 3, 2),
    "64_48": ([L16 * 4, L16 * 3], 3, 2), "m1": ([[0, 1], [1]], 0, 1),
}


@pytest.mark.gpu
@pytest.mark.parametrize("key", list(CASES))
def test_border_matches_the_oracle(key):
    lo_l, lmaxmat, p = CASES[key]
    spec = dataclasses.replace(synth.tiny(seed=31, lmax=3, lmaxmat=lmaxmat, apword=p,
                                          natoms=(2, 1)), lo_l=lo_l)
    full = synth.build(spec)
    ctx = lapw.Context(0).load(full)
    try:
        for ng in (1, 15, 16, 17, full.kpts[0].ngk):
            s = truncated(full, ng)
            print(f"[lo border] {key} ngk {ng}", flush=True)
            S = oracle.System(s)
            A = oracle.match(S, 0)
            H0, O0 = oracle.setup(S, 0, A)
            n = ng + s.nlotot
            border = np.ones((n, n), bool)
            border[:ng, :ng] = False
            rng = np.random.default_rng(1)
            P = rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))
            P = P + P.conj().T
            H, O, _ = device_setup(ctx, s, A)
            Ha, Oa, _ = device_setup(ctx, s, A, flags=lapw.ACCUMULATE, h=P, o=P)
            _, O1, _ = device_setup(ctx, s, A, only_o=True)
            for got, want in ((H, H0), (O, O0), (Ha, H0 + P), (Oa, O0 + P), (O1, O0)):
                tol = 1e-13 * max(1.0, np.abs(want[border]).max())
                assert np.abs(got - want)[border].max() <= tol
    finally:
        ctx.close()
