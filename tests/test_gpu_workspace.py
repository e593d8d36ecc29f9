"""GPU: the eigensolve's workspace, which the contexts of a device share: what
many contexts hold after their solves, and solves that run at once."""
import threading

import numpy as np
import pytest
import torch

from nadvibs_amd.batch import Batch
from nadvibs_amd.engine import Engine
from nadvibs_amd.synth import make_problem

pytestmark = pytest.mark.gpu

KEPT = 512 << 20  # bytes a device may keep between solves


def _prob(seed=3):
    return make_problem(2, [3, 3], 2, (500, 3000), 100.0, 20.0, 10.0, seed=seed)


def _tridiagonal(n, seed):
    rng = np.random.default_rng(seed)
    return 0.1 + 0.05 * rng.standard_normal(n), 0.03 * (1 + 0.2 * rng.standard_normal(n + 1))


def test_contexts_of_a_batch_share_the_workspace():
    """A solve of 1,600 rows takes 102 MB: the twelve problems of a batch keep one workspace, not twelve."""
    a, b = _tridiagonal(1600, 5)
    with Batch([_prob(k) for k in range(12)]) as bt:
        torch.cuda.synchronize()
        free0 = torch.cuda.mem_get_info()[0]
        first = bt.ritz(0, a, b)
        for p in range(1, 12):
            for got, want in zip(bt.ritz(p, a, b), first):
                assert np.array_equal(got, want)
        held = free0 - torch.cuda.mem_get_info()[0]
        print(f"held after twelve solves: {held >> 20} MB", flush=True)
        assert held <= KEPT + (64 << 20)


def test_solves_at_once_on_one_context():
    """Several threads solve different problems on one context and on a second one: the numbers of
    solves one after the other."""
    sizes = [300, 511, 777, 40, 1030]
    grid = np.linspace(0.0, 6000.0, 500)
    jobs = [_tridiagonal(n, n) for n in sizes]
    with Engine(_prob(1)) as e1, Engine(_prob(2)) as e2:
        want = [(e1.ritz(a, b), e1.spectrum(a, b, grid, 30.0)) for a, b in jobs]
        wrong = []

        def work(eng, k):
            a, b = jobs[k]
            for _ in range(6):
                ev, sp = eng.ritz(a, b), eng.spectrum(a, b, grid, 30.0)
                if not all(np.array_equal(g, w) for g, w in zip(ev, want[k][0])) or not np.array_equal(sp, want[k][1]):
                    wrong.append((sizes[k], eng is e1))

        threads = [threading.Thread(target=work, args=(eng, k)) for k in range(len(sizes)) for eng in (e1, e2)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
    assert not wrong, wrong
