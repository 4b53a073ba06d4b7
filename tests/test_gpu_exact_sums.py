"""Exact sums on the GPU against the oracle's ExactSum, bit for bit, at the edges of the
reduction: one block and its neighbours, the full grid of 512 blocks of 256 rows, values
that spread over all bins, totals below zero, zeros and non-finite values.

The identity matrix makes the solve's prologue expose its sums: Σ|b| is residualSum for
x = 0, and for b = 0 normFactor is Σ|x − x̄| + |x̄| with x̄ = Σx/n.
"""
import numpy as np
import pytest

import voluma_amd as va
from oracle import oracle as O
from voluma_amd import workloads as W

pytestmark = pytest.mark.gpu


def _values(n, spread, seed):
    u = 2.0 * W.splitmix_uniform(n, seed) - 1.0
    e = np.floor(W.splitmix_uniform(n, seed + 1) * (2 * spread + 1)) - spread
    return np.ldexp(u, e.astype(np.int64))


@pytest.fixture(scope="module")
def ctx():
    c = va.Context(0)
    yield c
    c.close()


def _prologue(ctx, b, x):
    n = b.size
    lm = va.LduMesh(ctx, n, np.arange(n - 1), np.arange(1, n))
    A = va.LduMatrix(lm, np.ones(n), np.zeros(n - 1))
    return va.solve_ldu(A, b, x.copy(), va.SolverControls("PCG", "diagonal", 1e300, maxIter=2, sums=va.SUMS_EXACT))


@pytest.mark.parametrize("spread", [0, 20, 1000])
@pytest.mark.parametrize("n", [2, 255, 256, 257, 256 * 8 + 1, 256 * 512 - 1, 256 * 512 + 1])
def test_exact_sums(ctx, n, spread):
    v = _values(n, spread, 17 * n + spread)
    assert _prologue(ctx, v, np.zeros(n)).residualSum == O.exact_sum(np.abs(v))
    for x in (v, -np.abs(v)):  # a total of either sign, and one below zero
        xb = O.exact_sum(x) / n
        want = O.exact_sum(np.abs(x - xb) + np.abs(0.0 - xb)) + 1e-20
        assert _prologue(ctx, np.zeros(n), x).normFactor == want


def test_exact_sums_of_zeros_and_non_finite(ctx):
    n = 1000
    assert _prologue(ctx, np.zeros(n), np.zeros(n)).residualSum == 0.0
    v = _values(n, 5, 3)
    v[777] = np.inf
    # Σ|b| is infinite and so is the norm factor: their quotient ends the solve as NaN would
    p = _prologue(ctx, v, np.zeros(n))
    assert np.isinf(p.residualSum)
    v[3] = np.nan
    assert np.isnan(_prologue(ctx, v, np.zeros(n)).residualSum)


@pytest.mark.parametrize("pre", ["none", "diagonal"])
@pytest.mark.parametrize("n", [2, 257, 5000, 256 * 512 + 1])
def test_pcg_with_diagonal_against_oracle(ctx, n, pre):
    """Both sums of an iteration's end in one reduction: bits of the oracle's recurrence with
    exact sums, a stop at every count included; fast sums within their rounding of it."""
    own, nei = np.arange(n - 1), np.arange(1, n)
    u = -1.0 - W.splitmix_uniform(n - 1, 5)
    d = 1.0 + np.bincount(own, -u, n) + np.bincount(nei, -u, n)
    b = 2.0 * W.splitmix_uniform(n, 7) - 1.0
    om, lm = O.LduMesh(n, own, nei), va.LduMesh(ctx, n, own, nei)
    A = va.LduMatrix(lm, d, u)
    for most, least in ((1, 0), (2, 0), (3, 0), (60, 0), (60, 9)):
        xo, po = om.solve(d, u, None, b, x0=np.zeros(n), solver="PCG", preconditioner=pre, tolerance=1e-9,
                          max_iter=most, min_iter=least, mode=O.MODE_EXACT)
        x = np.zeros(n)
        p = va.solve_ldu(A, b, x, va.SolverControls("PCG", pre, 1e-9, 0.0, most, least, sums=va.SUMS_EXACT))
        assert p.iterations == po["iterations"] and p.finalResidual == po["finalResidual"]
        assert np.array_equal(x, xo)
        xf = np.zeros(n)
        va.solve_ldu(A, b, xf, va.SolverControls("PCG", pre, 1e-9, 0.0, most, least))
        # α and β differ by the sums' rounding, n·2^-53 at most, over 60 steps of a system
        # whose condition number is below 10; x is of order 1
        assert np.abs(xf - xo).max() <= 60 * 10 * n * 2.0**-53 + 1e-9
