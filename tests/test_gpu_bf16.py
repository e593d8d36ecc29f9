"""GPU: the BF16 input copy for state counts whose interleaved rows are no
multiple of four bytes (one and three states) and for those whose rows are."""
import numpy as np
import pytest

from nadvibs_amd.engine import Engine
from nadvibs_amd.synth import make_problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ns", [1, 2, 3, 4, 5])
def test_bf16_coefficients_by_states(ns):
    """Bound: the input is rounded to 2^-9 relative, so alpha of the first steps stays within 2e-2 of
    the largest (ten times the rounding of one element)."""
    p = make_problem(ns, [8, 7, 9], 2, (400, 2500), 200.0, 60.0, 40.0, seed=ns)
    print(f"case {ns} states", flush=True)
    out = {}
    for prec in ("f64", "bf16"):
        with Engine(p) as eng:
            eng.lanczos_init(niter=5, prec=prec)
            eng.run(1, 5)
            out[prec] = np.array(eng.coefficients()[0])
    assert np.max(np.abs(out["bf16"] - out["f64"])) <= 2e-2 * np.max(np.abs(out["f64"]))
