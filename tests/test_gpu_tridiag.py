"""The tridiagonal eigensolve and the Gaussian envelope at the edges of their
kernels' tiles: sizes around a chunk of rows, a wave, the grid of shared
Sturm counts and the widths of the multisection; decoupled and repeated
blocks; solutions that outgrow the reference's overflow guard."""
import numpy as np
import pytest

from nadvibs_amd.engine import Engine
from nadvibs_amd.synth import make_problem
from oracle.oracle import givens

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng():
    with Engine(make_problem(2, [3, 3], 2, (500, 3000), 100.0, 20.0, 10.0, seed=3)) as e:
        yield e


def _check(eng, a, b):
    n = a.size
    ev, it, bj, _ = eng.ritz(a, b)
    ev0, it0, bj0, _ = givens(a, b)
    norm = np.sqrt(np.sum(a * a) + 2 * np.sum(b[1:n] ** 2))
    # a Sturm count is that of a matrix within a few roundings of T in every entry
    assert np.max(np.abs(ev - ev0)) <= 16 * np.finfo(float).eps * norm
    # first and last components of separated roots: inverse iteration leaves a relative
    # residual of a few roundings, divided by the relative gap
    gap = np.minimum(np.r_[np.inf, np.diff(ev0)], np.r_[np.diff(ev0), np.inf])
    sep = gap > 1e-7 * norm
    assert sep.any() or n == 1
    tol = 1e3 * np.finfo(float).eps * norm / np.maximum(gap[sep], 1e-7 * norm)
    assert np.all(np.abs(it[sep] - it0[sep]) <= tol)
    assert np.all(np.abs(bj[sep] - bj0[sep]) <= tol * max(abs(b[n]), 1e-300))


@pytest.mark.parametrize("n", [1, 2, 3, 7, 8, 9, 15, 16, 17, 18, 33, 63, 64, 65, 255, 256, 257, 1024, 1025, 1100])
def test_sizes(eng, n):
    rng = np.random.default_rng(n)
    a = 0.1 + 0.05 * rng.standard_normal(n)
    b = 0.03 * (1 + 0.2 * rng.standard_normal(n + 1))
    _check(eng, a, b)


def test_more_roots_than_one_wave_per_simd_takes(eng):
    """n > 2048: sixteen lanes per root."""
    n = 2051
    rng = np.random.default_rng(5)
    a, b = rng.uniform(-1, 1, n), 0.3 * np.ones(n + 1)
    ev, it, _, _ = eng.ritz(a, b)
    w = np.linalg.eigvalsh(np.diag(a) + np.diag(b[1:n], 1) + np.diag(b[1:n], -1))
    norm = np.sqrt(np.sum(a * a) + 2 * np.sum(b[1:n] ** 2))
    assert np.max(np.abs(ev - w)) <= 32 * np.finfo(float).eps * norm
    assert abs(np.sum(it) - 1.0) < 1e-9


def test_decoupled_and_repeated_blocks(eng):
    """Zero off-diagonals and equal diagonal entries: exactly zero pivots, and
    clusters whose members share the first component's weight."""
    a = np.array([0.5, 0.25, 0.25, 0.25, -0.5, 0.125, 0.25, 0.0])
    b = np.array([1.0, 0.0, 0.0, 0.0, 0.3, 0.0, 0.0, 0.2, 0.1])
    ev, it, _, _ = eng.ritz(a, b)
    n = a.size
    w = np.linalg.eigvalsh(np.diag(a) + np.diag(b[1:n], 1) + np.diag(b[1:n], -1))
    assert np.max(np.abs(ev - w)) <= 16 * np.finfo(float).eps * np.sqrt(np.sum(a * a) + 2 * np.sum(b[1:n] ** 2))
    assert abs(np.sum(it) - 1.0) < 1e-12


def test_zero_matrix_and_constant_diagonal(eng):
    ev, it, _, _ = eng.ritz(np.zeros(5), np.zeros(6))
    assert np.all(ev == 0.0) and it[0] == 1.0
    ev, it, _, _ = eng.ritz(np.full(40, 0.3), np.zeros(41))
    np.testing.assert_allclose(ev, 0.3, rtol=1e-14)


@pytest.mark.parametrize("n", [90, 200, 331])
def test_overflow_guard(eng, n):
    """Off-diagonals of 1e-4: the back substitution grows by about 1e4 a row
    away from a root's own row, past the guard's 1e275."""
    rng = np.random.default_rng(n)
    a = rng.permutation(np.linspace(-1.0, 1.0, n))
    b = np.full(n + 1, 1e-4)
    _check(eng, a, b)


@pytest.mark.parametrize("ng,n", [(1, 1), (15, 3), (16, 255), (17, 256), (4096, 257), (65536, 5), (65537, 5)])
def test_envelope_sizes(eng, ng, n):
    rng = np.random.default_rng(ng + n)
    x, y = rng.uniform(0, 100, n), rng.uniform(0.1, 1, n)
    grid = np.linspace(0.0, 100.0, ng) if ng > 1 else np.array([50.0])
    env = eng.convolve(x, y, grid, 20.0)
    ref = np.zeros(ng)
    for xi, yi in zip(x, y):
        ref += yi * np.exp(-0.5 * ((grid - xi) / 20.0) ** 2)
    # n products and sums, an exponential of an argument below 13 in magnitude
    np.testing.assert_allclose(env, ref / ref.max(), rtol=(n + 40) * np.finfo(float).eps)


@pytest.mark.parametrize("ng", [3, 65537])
def test_envelopes_of_the_narrowest_width(eng, ng):
    """A width whose reciprocal overflows: the sticks on grid points alone, in full."""
    rng = np.random.default_rng(2)
    a, b = 0.1 + 0.05 * rng.standard_normal(20), 0.03 * np.ones(21)
    _, it, _, _ = eng.ritz(a, b)
    grid = np.linspace(0.0, 1e-3, ng)
    for sigma in (1e-310, 5e-324, 1e-300):
        want = np.zeros(ng)
        want[0] = it[0]
        assert np.array_equal(eng.spectrum(a, b, grid, sigma), want)
        env = eng.convolve(np.array([0.0, 50.0]), np.array([2.0, 1.0]), grid, sigma)
        assert np.array_equal(env, want != 0.0)
