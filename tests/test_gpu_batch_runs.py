"""GPU: runs of one batch that follow each other.  A run of the shape of the
one before keeps its buffers and captured iterations, another shape replaces
them, and coefficients read between the parts of a run are those of the
iterations so far: always the numbers of a batch that runs once."""
import time

import numpy as np
import pytest
import torch

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


def test_watching_one_problem_of_a_long_run():
    """Reading one problem between the parts of a run costs what it holds, not what the batch does
    (64 problems of 20,000 iterations: 20 MB): at most five times the same read from a batch of one,
    where a copy of the batch would take more than fifty; and every problem read after the same part
    has the same numbers whether it came alone or with the others."""
    p = make_problem(2, [6, 6, 5], 2, (500, 3000), 250.0, 60.0, 40.0, seed=70)
    times = {}
    for count in (1, 64):
        with Batch([p] * count) as bt:
            bt.init(20000, "f64")
            bt.run(1, 8)
            n, best = 8, np.inf
            for _ in range(12):
                bt.run(n + 1, n + 1)
                n += 1
                torch.cuda.synchronize()
                t0 = time.perf_counter()
                one = bt.coefficients(count - 1, n)
                best = min(best, time.perf_counter() - t0)
            times[count] = best
            # the iterations of one problem are those of every other
            for k in list(range(count)) + list(range(count)):
                for got, want in zip(bt.coefficients(k, n), one):
                    assert np.array_equal(got, want)
    print(f"one read: {times[1] * 1e6:.0f} us of one problem, {times[64] * 1e6:.0f} us of 64", flush=True)
    assert times[64] <= 5.0 * times[1]


def test_reads_on_both_sides_of_the_copy_of_all():
    """Forty problems of 2,000 iterations are 1.3 MB: the first reads come one by one, the rest from
    one copy, in any order and again."""
    probs = [make_problem(2, [5 + k % 3, 6, 4], 2, (500, 3000), 250.0, 60.0, 40.0, seed=k) for k in range(40)]
    with Batch(probs) as bt:
        bt.init(2000, "f64")
        bt.run(1, 20)
        order = np.random.default_rng(1).permutation(40)
        got = {int(k): bt.coefficients(int(k), 20) for k in order}
        again = {k: bt.coefficients(k, 20) for k in range(40)}
    for k, prob in enumerate(probs):
        with Batch([prob]) as bt:
            bt.init(2000, "f64")
            bt.run(1, 20)
            want = bt.coefficients(0, 20)
        for g in (got[k], again[k]):
            assert np.array_equal(g[0], want[0]) and np.array_equal(g[1], want[1])


def test_tuning_holds_for_the_precision_it_was_made_in():
    """A run takes the form that was tuned in its own precision, or the default one: the sums of its
    workgroups, and so the last bits, are those of a batch that knew no other precision."""
    probs = _probs(SHAPES["two rows"])
    n = 18

    def run(bt, prec):
        bt.init(n, prec)
        bt.run()
        return _all(bt, len(probs), n)

    fresh = {}
    for prec in ("f64", "f32"):
        with Batch(probs) as bt:
            fresh[prec] = run(bt, prec)
    for first, other in (("f64", "f32"), ("f32", "f64")):
        with Batch(probs) as bt:
            bt.init(n, first)
            print(bt.tune(), flush=True)
            bt.run()
            tuned = _all(bt, len(probs), n)
            assert np.array_equal(run(bt, other), fresh[other])
            assert np.array_equal(run(bt, first), tuned)
