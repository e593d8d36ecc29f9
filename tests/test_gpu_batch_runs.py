"""GPU: runs of one batch that follow each other.  A run of the shape of the
one before keeps its buffers and captured iterations, another shape replaces
them, and coefficients read between the parts of a run are those of the
iterations so far: always the numbers of a batch that runs once."""
import numpy as np
import pytest

from nadvibs_amd.batch import Batch
from nadvibs_amd.synth import make_problem

pytestmark = pytest.mark.gpu

# 1, 500 and 1,100 tiles of rows: one and two rows per thread in FP32
SHAPES = {"one tile": [(2, [6, 6, 5])], "ragged": [(1, [9, 7]), (3, [31, 32, 33]), (2, [40, 50, 49])],
          "two rows": [(2, [66, 64, 66]), (3, [4, 3, 5])]}


def _probs(shapes):
    return [make_problem(ns, nf, 2, (500, 3000), 250.0, 60.0, 40.0, seed=70 + i) for i, (ns, nf) in enumerate(shapes)]


def _all(bt, count, n):
    return np.concatenate([np.concatenate(bt.coefficients(p, n)) for p in range(count)])


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("shapes", list(SHAPES))
def test_repeated_runs(shapes, prec):
    probs = _probs(SHAPES[shapes])
    print(f"case {shapes} {prec}", flush=True)
    want = {}
    for n in (18, 5):
        with Batch(probs) as bt:
            bt.init(n, prec)
            bt.run()
            want[n] = _all(bt, len(probs), n)
            assert np.all(np.isfinite(want[n]))
    other = "f32" if prec == "f64" else "f64"
    with Batch(probs) as bt:
        for n in (18, 18, 5, 5, 18):
            bt.init(n, prec)
            bt.run(1, 3)
            early = [bt.coefficients(p, 3) for p in range(len(probs))]
            bt.run(4, n)
            got = _all(bt, len(probs), n)
            assert np.array_equal(got, want[n])
            for p, (a, b) in enumerate(early):
                late = bt.coefficients(p, n)
                assert np.array_equal(a, late[0][:3]) and np.array_equal(b, late[1][:4])
        bt.init(5, other)
        bt.run()
        bt.init(18, prec)
        bt.run()
        assert np.array_equal(_all(bt, len(probs), 18), want[18])
