"""GPU: H*v with the terms of a row shared over the waves of a workgroup,
against the step-table kernels, which the oracle holds: ragged and full last
workgroups, fewer terms than waves, one to ten states, every order, states
coupled through the diagonal part, and the row counts on both sides of the lines
between which the terms are shared; FP32 with the many terms that it takes there."""
import numpy as np
import pytest

from nadvibs_amd.engine import Engine
from nadvibs_amd.synth import make_problem

pytestmark = pytest.mark.gpu

# states, basis, order, inter-state diagonal couplings, quirks
CASES = [
    (2, [7, 73], 1, 0.0, 3),
    (1, [64, 8], 1, 0.0, 3),
    (3, [8, 8, 8], 2, 0.0, 3),
    (2, [13, 41], 3, 20.0, 0),
    (4, [9, 9, 7], 3, 0.0, 3),
    (5, [5, 1, 11, 10], 3, 10.0, 3),
    (10, [13, 8, 5], 2, 5.0, 3),
    (3, [11, 9, 7, 5], 3, 30.0, 3),
    (1, [64, 64, 64], 2, 0.0, 3),
    (1, [64, 17, 241], 2, 0.0, 3),
    (1, [61, 63, 69], 2, 0.0, 3),
    (2, [64, 64, 128], 3, 10.0, 3),
    (1, [74, 85, 84], 2, 0.0, 3),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{c[0]}x{'-'.join(map(str, c[1]))}o{c[2]}")
def test_shared_terms_match_the_step_tables(case, monkeypatch):
    """Bounds: a row sums at most about 1,500 products, so H*v stays within 1e-13 of the largest
    element, and the coefficients of 12 steps within 1e-11."""
    for v in ("NV_HV_KERNEL", "NV_HV_FB"):
        monkeypatch.delenv(v, raising=False)
    ns, nf, ordr, offe, quirks = case
    p = make_problem(ns, nf, ordr, (400, 2500), 200.0, 60.0, 40.0, cubic=10.0, seed=len(nf), quirks=quirks,
                     offdiag_even=offe)
    print(f"case {case} n={p.n}", flush=True)
    x = np.random.default_rng(3).standard_normal(p.n)

    def coefficients(eng):
        eng.lanczos_init(niter=12, reorthog=0, prec="f64")
        eng.run(1, 12)
        a, b, _ = eng.coefficients()
        return np.array(a), np.array(b)

    with Engine(p) as eng:
        y = eng.hv(x, "f64")
        ab = coefficients(eng)
        eng.select_hv_kernel("steps")
        ref = eng.hv(x, "f64")
        assert np.max(np.abs(y - ref)) <= 1e-13 * np.max(np.abs(ref))
        for got, want in zip(ab, coefficients(eng)):
            assert np.max(np.abs(got - want)) <= 1e-11 * np.max(np.abs(want))


# cubic operators of 219 and 285 terms
MANY = [
    (2, [2] * 9, 0.0, 3),
    (4, [2] * 9 + [3], 10.0, 3),
    (3, [3] * 9, 5.0, 0),
    (1, [5, 4] + [3] * 7, 0.0, 3),
    (2, [4] * 4 + [2] * 10, 0.0, 3),
]


@pytest.mark.parametrize("case", MANY, ids=lambda c: f"{c[0]}x{'-'.join(map(str, c[1]))}")
def test_shared_terms_fp32(case, monkeypatch):
    """Bounds: a row sums at most about 2,000 products in FP32, within 2e-6 of the largest element,
    and the coefficients of 12 steps within 5e-6, against FP64 step tables."""
    for v in ("NV_HV_KERNEL", "NV_HV_FB"):
        monkeypatch.delenv(v, raising=False)
    ns, nf, offe, quirks = case
    p = make_problem(ns, nf, 3, (400, 2500), 200.0, 60.0, 40.0, cubic=10.0, seed=len(nf), quirks=quirks,
                     offdiag_even=offe)
    print(f"case {case} n={p.n}", flush=True)
    x = np.random.default_rng(3).standard_normal(p.n)

    def results(eng, prec):
        y = eng.hv(x, prec)
        eng.lanczos_init(niter=12, reorthog=0, prec=prec)
        eng.run(1, 12)
        a, b, _ = eng.coefficients()
        return y, np.array(a), np.array(b)

    with Engine(p) as eng:
        eng.select_hv_kernel("steps")
        ref = results(eng, "f64")
        eng.select_hv_kernel(True)
        got = results(eng, "f32")
    for tol, g, r in zip((2e-6, 5e-6, 5e-6), got, ref):
        assert np.max(np.abs(g - r)) <= tol * np.max(np.abs(r))


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{c[0]}x{'-'.join(map(str, c[1]))}o{c[2]}")
def test_shared_terms_are_reported(case, monkeypatch):
    """Which of the FP64 operators above share a row's terms in their iterations: 512 to 262,144 rows."""
    for v in ("NV_HV_KERNEL", "NV_HV_FB"):
        monkeypatch.delenv(v, raising=False)
    ns, nf, ordr, offe, quirks = case
    p = make_problem(ns, nf, ordr, (400, 2500), 200.0, 60.0, 40.0, cubic=10.0, seed=len(nf), quirks=quirks,
                     offdiag_even=offe)
    rows = int(np.prod(nf))
    with Engine(p) as eng:
        info = eng.hv_kernel("f64")
        assert info.startswith("generic shaped"), info
        assert ("terms shared over 4 waves" in info) == (512 <= rows <= 262144), info


@pytest.mark.parametrize("case", MANY, ids=lambda c: f"{c[0]}x{'-'.join(map(str, c[1]))}")
def test_shared_terms_fp32_are_reported(case):
    ns, nf, offe, quirks = case
    p = make_problem(ns, nf, 3, (400, 2500), 200.0, 60.0, 40.0, cubic=10.0, seed=len(nf), quirks=quirks,
                     offdiag_even=offe)
    with Engine(p) as eng:
        eng.select_hv_kernel(True)
        assert "terms shared over 4 waves" in eng.hv_kernel("f32")
    few = make_problem(3, [8, 8, 8], 2, (400, 2500), 200.0, 60.0, 40.0, seed=1)
    with Engine(few) as eng:
        eng.select_hv_kernel(True)
        assert "waves" not in eng.hv_kernel("f32")
