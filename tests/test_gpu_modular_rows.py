"""FP64 setups on the modular products do not depend on how the radial
functions are normalised: a function scaled by 2^-p (its matching coefficients
by 2^p, its rows and columns of the muffin-tin tables by 2^-p) leaves H as it
is, and every FP64 sum over it bitwise; the modular products scale the rows of
their operands by the tables' own exponents, so they keep the bits too."""
import dataclasses

import numpy as np
import pytest

import oracle
from exciting_amd import lapw
from tests.test_gpu_edges import truncated
from tests.test_gpu_modular import cell, check_apw_block, device_setup, norms, operands

CELL = ("none", 8, 8.8)   # 8 of lmaxapw 10: a packed operand


def functions(s):
    """(lm, io) of each function of an atom, in the tables' order."""
    return [(l * l + m, io) for l in range(s.spec.lmaxmat + 1) for m in range(2 * l + 1)
            for io in range(s.apwordmax)]


def rescaled(s, A, p):
    """s and A with function f of atom a scaled by 2^-p[a, f]."""
    aa, loa, A = s.aa.copy(order="F"), s.loa.copy(order="F"), A.copy(order="F")
    for a in range(s.natmtot):
        c = np.ldexp(1.0, -p[a])
        aa[:, :, a] *= np.outer(c, c)
        loa[:, :, a] *= c[None, :]
        for f, (lm, io) in enumerate(functions(s)):
            A[:, io, lm, a] *= np.ldexp(1.0, p[a, f])
    return dataclasses.replace(s, aa=aa, loa=loa), A


def h_of(s, A):
    ctx = lapw.Context(0).load(s)
    try:
        H, _, ran = device_setup(ctx, s, A)
        assert "oz_gemm" in ran
        return H
    finally:
        ctx.close()


@pytest.fixture(scope="module")
def base():
    s = truncated(cell(*CELL), 200)
    A = oracle.match(oracle.System(s), 0)
    return s, A, h_of(s, A)


@pytest.mark.gpu
@pytest.mark.parametrize("p", [1, 2, 5, 20, 60, "atoms", "random"])
def test_h_does_not_depend_on_normalisation(base, p):
    s, A, H = base
    n = len(functions(s))
    shift = np.zeros((s.natmtot, n), int)
    if p == "atoms":
        shift[:] = (np.arange(s.natmtot) % 3 * 15)[:, None]
    elif p == "random":
        shift[:] = np.random.default_rng(4).integers(-20, 21, shift.shape)
    else:
        shift[:, 1::2] = p             # the second function of every l
    print(f"[rows] {p}", flush=True)
    s2, A2 = rescaled(s, A, shift)
    H2 = h_of(s2, A2)
    # a factor of two is not worth a scale
    assert p == 1 or np.array_equal(H2, H)
    # and within the oracle's FP64 sums (2 K 2^-53 = 4e-13) of sum |x| |b|, which is
    # at least a hundredth of the norms' product here (its rounding: 4e-15)
    H0, _ = oracle.setup(oracle.System(s2), 0, A2)
    X, B = operands(s2, A2, 200)
    S = np.abs(X).T @ np.abs(B)
    X, B = operands(s, A, 200)
    assert (100 * S >= np.outer(norms(X), norms(B))).all()
    d = np.abs(H2[:200, :200] - H0[:200, :200])
    assert (d <= 1e-12 * (S + S.T + np.abs(H0[:200, :200]))).all(), (d / S).max()


@pytest.mark.gpu
def test_tables_without_a_diagonal(base):
    """Zero rows, a zero diagonal with and without couplings to functions that
    have one, and a table of zeros: within the bound of the ordinary tables
    (the oracle's FP64 sums), relative to the norms."""
    s, A, _ = base
    aa = s.aa.copy(order="F")
    aa[5, :, 0] = aa[:, 5, 0] = 0.0
    aa[7, 7, 0] = aa[8, 8, 0] = aa[9, 9, 1] = 0.0
    keep = aa[20, 21, 2]
    aa[20:22, :, 2] = aa[:, 20:22, 2] = 0.0
    aa[20, 21, 2], aa[21, 20, 2] = keep, np.conj(keep)
    aa[:, :, 3] = 0.0
    s = dataclasses.replace(s, aa=aa)
    H0, _ = oracle.setup(oracle.System(s), 0, A)
    X, B = operands(s, A, 200)
    nx, nb = norms(X), norms(B)
    check_apw_block(h_of(s, A), H0, np.outer(nx, nb) + np.outer(nb, nx), 200, 1e-12)
