"""GPU: H*v with the degree-three slow terms in the slab and leading passes
(forced on small operators) against the step-list kernels, which the oracle
holds: one to three modes in LDS, none
to four leading modes, basis sizes of one and two, one to four states, one and
two rows per thread, the last workgroup of an XCD's share empty or not."""
import numpy as np
import pytest

from nadvibs_amd.engine import Engine
from nadvibs_amd.synth import make_problem
from test_slab_tables import CASES

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("case", CASES,
                         ids=lambda c: f"{c[0]}x{'-'.join(map(str, c[1]))}")
def test_slab_hv_matches_the_step_lists(case, monkeypatch):
    """Bounds: a row sums at most about 1,500 products, so FP64 stays within 1e-13 and FP32 within
    2e-6 of the largest element; the coefficients of 12 steps within 1e-11 and 5e-6."""
    monkeypatch.delenv("NV_HV_KERNEL", raising=False)
    ns, nf, offe, quirks = case
    p = make_problem(ns, nf, 3, (400, 2500), 200.0, 60.0, 40.0, cubic=10.0, seed=len(nf), quirks=quirks,
                     offdiag_even=offe)
    print(f"case {case} n={p.n}", flush=True)
    x = np.random.default_rng(3).standard_normal(p.n)

    def coefficients(eng, prec):
        eng.lanczos_init(niter=12, reorthog=0, prec=prec)
        eng.run(1, 12)
        a, b, _ = eng.coefficients()
        return np.array(a), np.array(b)

    monkeypatch.setenv("NV_HV_FB", "0")
    with Engine(p) as eng:
        assert "fast-block" not in eng.hv_kernel("f64")
        ref = eng.hv(x, "f64")
        ra, rb = coefficients(eng, "f64")
    monkeypatch.setenv("NV_HV_FB", "1")
    with Engine(p) as eng:
        for prec, tol_hv, tol_ab in (("f64", 1e-13, 1e-11), ("f32", 2e-6, 5e-6)):
            info = eng.hv_kernel(prec)
            assert info.startswith("generic fast-block"), info
            err = np.max(np.abs(eng.hv(x, prec) - ref)) / np.max(np.abs(ref))
            assert err <= tol_hv, (prec, err)
            a, b = coefficients(eng, prec)
            assert np.max(np.abs(a - ra) / np.abs(ra)) <= tol_ab, prec
            assert np.max(np.abs(b - rb) / np.abs(rb)) <= tol_ab, prec
