"""Triangular sweeps over one and several chunks against the oracle's sequential loops, bit
for bit (exact sums), on the graphs of ``helpers.sweep_graph`` and with more sweeps than one
launch takes.
"""
import numpy as np
import pytest

import voluma_amd as va
from helpers import band, sweep_graph
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = va.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("name", ["chain", "one", "two", "wide", "far", "hub", "box"])
def test_sweeps_bit_exact_vs_oracle(ctx, name):
    n, own, nei = sweep_graph(name)
    rng = np.random.default_rng(9)
    nf = own.size
    u = -rng.uniform(0.5, 1.5, nf)
    lo = u * rng.uniform(0.7, 1.3, nf)
    d = 0.1 + np.bincount(own, np.maximum(-u, -lo), n) + np.bincount(nei, np.maximum(-u, -lo), n)
    b = rng.uniform(-1, 1, n)
    x0 = rng.uniform(-1, 1, n)
    lm = va.LduMesh(ctx, n, own, nei)
    om = O.LduMesh(n, own, nei)
    A, N = va.LduMatrix(lm, d, u), va.LduMatrix(lm, d, u, lo)
    for solver, pre, sym, sweeps, mx in (("GaussSeidel", "none", True, 1, 2), ("GaussSeidel", "none", False, 2, 4),
                                         ("GaussSeidel", "none", True, 5, 5), ("symGaussSeidel", "none", False, 1, 2),
                                         ("PCG", "DIC", True, 1, 3), ("PBiCGStab", "DILU", False, 1, 3)):
        xo, po = om.solve(d, u, None if sym else lo, b, x0=x0, solver=solver, preconditioner=pre, tolerance=1e-30,
                          max_iter=mx, n_sweeps=sweeps, mode=O.MODE_EXACT)
        x = x0.copy()
        p = va.solve_ldu(A if sym else N, b, x, va.SolverControls(solver, pre, 1e-30, 0.0, mx, nSweeps=sweeps,
                                                                  sums=va.SUMS_EXACT))
        assert p.iterations == po["iterations"] and p.finalResidual == po["finalResidual"], (solver, sweeps)
        assert np.array_equal(x, xo), (solver, sweeps)


def test_values_before_the_sweep_past_the_halo(ctx, monkeypatch):
    """Enough chunks of long scattered rows that a chunk's neighbours do not fit its LDS:
    what is left of them is read where it lies, from x (at the start of every four sweeps)
    and, in the GAMG smoother's first sweeps, from the zero that x is taken as."""
    n, own, nei = sweep_graph("scattered")
    rng = np.random.default_rng(10)
    u = -rng.uniform(0.5, 1.5, own.size)
    d = 0.1 + np.bincount(own, -u, n) + np.bincount(nei, -u, n)
    rhs, x0 = rng.uniform(-1, 1, n), rng.uniform(-1, 1, n)
    w = rng.uniform(0.5, 1.5, own.size)
    monkeypatch.setenv("VOLUMA_AGGLOMERATION", "host")  # the same hierarchy; its hubs take the device 19 s
    lm, om = va.LduMesh(ctx, n, own, nei, w, 20), O.LduMesh(n, own, nei, w, 20)  # the graph, then the coarsest
    A = va.LduMatrix(lm, d, u)
    for solver, pre, sweeps, mx in (("GaussSeidel", "none", 2, 4), ("GaussSeidel", "none", 5, 5),
                                    ("symGaussSeidel", "none", 1, 2), ("PCG", "GAMG", 1, 2)):
        xo, po = om.solve(d, u, None, rhs, x0=x0, solver=solver, preconditioner=pre, tolerance=1e-30, max_iter=mx,
                          n_sweeps=sweeps, mode=O.MODE_EXACT, smoother=O.SMOOTHER_GS)
        x = x0.copy()
        p = va.solve_ldu(A, rhs, x, va.SolverControls(solver, pre, 1e-30, 0.0, mx, nSweeps=sweeps,
                                                      sums=va.SUMS_EXACT, gamgSmoother=va.GAMG_GAUSS_SEIDEL))
        assert p.iterations == po["iterations"] and p.finalResidual == po["finalResidual"], (solver, sweeps)
        assert np.array_equal(x, xo), (solver, sweeps)


@pytest.mark.parametrize("name", ["one", "two"])
@pytest.mark.parametrize("powers", [(0,), (-398, -402, 0, 398, 402), (-800, 0, 180)])
def test_row_division_over_the_exponent_range(ctx, name, powers):
    """Rows scaled by powers of two on both sides of the range in which a step divides with
    the reciprocal, and zero numerators of both signs: the oracle's quotients bit for bit."""
    n, own, nei = sweep_graph(name)
    rng = np.random.default_rng(11)
    s = 2.0 ** rng.choice(powers, n)
    u, lo = -rng.uniform(0.5, 1.5, own.size), -rng.uniform(0.5, 1.5, own.size)
    d = (0.1 + np.bincount(own, -u, n) + np.bincount(nei, -lo, n)) * rng.choice([-1.0, 1.0], n)
    d, u, lo = d * s, u * s[own], lo * s[nei]
    b = rng.uniform(-1, 1, n) * s
    b[: n // 2] = 0.0
    b[: n // 4] = -0.0
    lm = va.LduMesh(ctx, n, own, nei)
    om = O.LduMesh(n, own, nei)
    for sweeps in (1, 3):
        xo, _ = om.solve(d, u, lo, b, x0=np.zeros(n), solver="GaussSeidel", preconditioner="none", tolerance=1e-300,
                         max_iter=sweeps, n_sweeps=sweeps, mode=O.MODE_EXACT)
        x = np.zeros(n)
        va.solve_ldu(va.LduMatrix(lm, d, u, lo), b, x, va.SolverControls("GaussSeidel", "none", 1e-300, 0.0, sweeps,
                                                                        nSweeps=sweeps, sums=va.SUMS_EXACT))
        assert np.array_equal(x, xo) and np.array_equal(np.signbit(x), np.signbit(xo)), sweeps


@pytest.mark.parametrize("name", ["one", "two", "wide"])
def test_infinite_coefficients_keep_the_loops_signs(ctx, name):
    """Infinite coefficients on faces of a chunk whose rows also read other chunks' values:
    every infinity and every NaN of the sequential loop, and its bits elsewhere."""
    n, own, nei = sweep_graph(name)
    rng = np.random.default_rng(12)
    u, lo = -rng.uniform(0.5, 1.5, own.size), -rng.uniform(0.5, 1.5, own.size)
    d = 0.1 + np.bincount(own, -u, n) + np.bincount(nei, -lo, n)
    b, x0 = rng.uniform(-1, 1, n), rng.uniform(-1, 1, n)
    near = np.flatnonzero((np.minimum(own, nei) > n // 2) & (np.maximum(own, nei) < n // 2 + 400))
    for at, side in zip(rng.choice(near, 6, replace=False), (u, lo) * 3):
        side[at] = rng.choice([-np.inf, np.inf])
    lm, om = va.LduMesh(ctx, n, own, nei), O.LduMesh(n, own, nei)
    A = va.LduMatrix(lm, d, u, lo)
    for sweeps in (1, 2):
        xo, _ = om.solve(d, u, lo, b, x0=x0, solver="GaussSeidel", preconditioner="none", tolerance=1e-30,
                         max_iter=1, n_sweeps=sweeps, mode=O.MODE_EXACT)
        assert np.isinf(xo).any()
        x = x0.copy()
        va.solve_ldu(A, b, x, va.SolverControls("GaussSeidel", "none", 1e-30, 0.0, 1, nSweeps=sweeps,
                                                sums=va.SUMS_EXACT))
        assert np.array_equal(x, xo, equal_nan=True), sweeps


def test_long_chain_is_no_timeout(ctx):
    """Two million cells in a row, one row per level: a chunk's wait lasts as long as all the
    chunks before it take (most of a second), which is no failure."""
    n = 2_000_000
    own, nei = np.arange(n - 1, dtype=np.int32), np.arange(1, n, dtype=np.int32)
    rng = np.random.default_rng(13)
    u = -rng.uniform(0.5, 1.5, n - 1)
    d = 0.1 + np.bincount(own, -u, n) + np.bincount(nei, -u, n)
    b = rng.uniform(-1, 1, n)
    lm, om = va.LduMesh(ctx, n, own, nei), O.LduMesh(n, own, nei)
    A = va.LduMatrix(lm, d, u)
    for solver, pre in (("GaussSeidel", "none"), ("PCG", "DIC")):
        xo, _ = om.solve(d, u, None, b, x0=np.zeros(n), solver=solver, preconditioner=pre, tolerance=1e-30, max_iter=1,
                         mode=O.MODE_EXACT)
        x = np.zeros(n)
        va.solve_ldu(A, b, x, va.SolverControls(solver, pre, 1e-30, 0.0, 1, sums=va.SUMS_EXACT))
        assert np.array_equal(x, xo), solver


@pytest.mark.parametrize("solver,pre,prec", [("PCG", "DIC", va.FP64), ("PBiCGStab", "DILU", va.FP64),
                                             ("PCG", "DIC", va.MIXED), ("GaussSeidel", "none", va.FP64)])
def test_a_timed_out_solve_leaves_nothing_behind(ctx, monkeypatch, solver, pre, prec):
    """A solve whose waits run past their limit (here one of a single poll) ends in an error,
    and the next solve of the same matrix is a fresh one's bit for bit: no factor that the
    failed one left half done."""
    n, own, nei = sweep_graph("chain")
    rng = np.random.default_rng(14)
    u = -rng.uniform(0.5, 1.5, own.size)
    d = 0.1 + np.bincount(own, -u, n) + np.bincount(nei, -u, n)
    b = rng.uniform(-1, 1, n)
    lm = va.LduMesh(ctx, n, own, nei)
    A, fresh = va.LduMatrix(lm, d, u), va.LduMatrix(lm, d, u)
    ctl = va.SolverControls(solver, pre, 1e-30, 0.0, 2, precision=prec)
    monkeypatch.setenv("VOLUMA_SWEEP_POLLS", "1")
    with pytest.raises(va.VolumaError, match="timed out"):
        va.solve_ldu(A, b, np.zeros(n), ctl)
    monkeypatch.delenv("VOLUMA_SWEEP_POLLS")
    x, want = np.zeros(n), np.zeros(n)
    p, pw = va.solve_ldu(A, b, x, ctl), va.solve_ldu(fresh, b, want, ctl)
    assert p.iterations == pw.iterations and p.finalResidual == pw.finalResidual
    assert np.isfinite(want).all() and np.array_equal(x, want)


def test_any_number_of_sweeps_over_one_chunk(ctx):
    """More sweeps than a one-chunk schedule holds go in several launches: the oracle's bits
    after 20, and 20,000 (as one schedule over 2^31 entries) are taken and converge."""
    n, (a, b) = 8192, band(8192, 14, 900, 15)
    keep = (a < b) & (b < n - 1)
    e = np.unique(a[keep].astype(np.int64) * n + b[keep])
    own, nei = (e // n).astype(np.int32), (e % n).astype(np.int32)
    rng = np.random.default_rng(16)
    u = -rng.uniform(0.5, 1.5, own.size)
    d = 0.1 + np.bincount(own, -u, n) + np.bincount(nei, -u, n)
    rhs = rng.uniform(-1, 1, n)
    lm, om = va.LduMesh(ctx, n, own, nei), O.LduMesh(n, own, nei)
    A = va.LduMatrix(lm, d, u)
    xo, _ = om.solve(d, u, None, rhs, x0=np.zeros(n), solver="GaussSeidel", preconditioner="none", tolerance=1e-30,
                     max_iter=1, n_sweeps=20, mode=O.MODE_EXACT)
    x = np.zeros(n)
    va.solve_ldu(A, rhs, x, va.SolverControls("GaussSeidel", "none", 1e-30, 0.0, 1, nSweeps=20, sums=va.SUMS_EXACT))
    assert np.array_equal(x, xo)
    p = va.solve_ldu(A, rhs, x, va.SolverControls("GaussSeidel", "none", 1e-12, 0.0, 1, nSweeps=20000))
    assert p.converged
