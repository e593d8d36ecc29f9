"""GPU: the eigensolve's workspace, which the contexts of a device share: what
many contexts hold after their solves, and solves that run at once."""
import threading

import numpy as np
import pytest
import torch

from nadvibs_amd._lib import NvError
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


def test_a_failed_allocation_takes_back_the_workspace():
    """What is kept for the next solve goes before a call fails for want of memory, and the context
    works on."""
    a, b = _tridiagonal(1600, 5)
    # 1.4e6 elements: a basis of 10^6 of them is 11 TB
    with Engine(make_problem(3, [12, 10, 10, 8, 8, 6], 2, (500, 3000), 200.0, 40.0, 20.0, seed=4)) as eng:
        want = eng.ritz(a, b)
        torch.cuda.synchronize()
        free0 = torch.cuda.mem_get_info()[0]
        with pytest.raises(NvError):
            eng.lanczos_init(niter=1000000, savevecs=True)
        gained = torch.cuda.mem_get_info()[0] - free0
        print(f"given back: {gained >> 20} MB", flush=True)
        assert gained >= 40 * 1600 * 1600 - (8 << 20)
        for got, ref in zip(eng.ritz(a, b), want):
            assert np.array_equal(got, ref)
        eng.lanczos_init(niter=10)
        eng.run(1, 10)
        assert np.all(np.isfinite(eng.coefficients()[0]))


@pytest.mark.parametrize("prec,tol", [("f64", 1e-11), ("f32", 5e-6)])
def test_a_failed_allocation_takes_back_the_slab_buffer(prec, tol, monkeypatch):
    """A run goes on without the slab buffer of its H*v when another call on its context needs the
    memory.  Both forms sum the same at most 1,500 products a row: bounds as for the coefficients of
    the slab pass against the step lists."""
    for v in ("NV_HV_KERNEL", "NV_HV_FB"):
        monkeypatch.delenv(v, raising=False)
    p = make_problem(4, [8] * 7, 3, (400, 2500), 200.0, 60.0, 40.0, cubic=10.0, seed=7)
    buffer = p.n * (8 if prec == "f64" else 4)
    with Engine(p) as eng:
        eng.lanczos_init(niter=12, prec=prec)
        eng.run(1, 12)
        want = eng.coefficients()[:2]
        eng.lanczos_init(niter=12, prec=prec)
        eng.run(1, 5)
        eng.coefficients()
        free0 = torch.cuda.mem_get_info()[0]
        n = 400000  # 40 n^2 bytes: 6.4 TB
        with pytest.raises(NvError):
            eng.ritz(np.ones(n), np.ones(n + 1))
        gained = torch.cuda.mem_get_info()[0] - free0
        print(f"given back: {gained >> 20} MB of {buffer >> 20}", flush=True)
        assert gained >= buffer - (8 << 20)
        eng.run(6, 12)
        for got, ref in zip(eng.coefficients()[:2], want):
            assert np.max(np.abs(got - ref)) <= tol * np.max(np.abs(ref))


def test_a_run_keeps_its_slab_buffer_while_another_thread_lacks_memory(monkeypatch):
    """One thread runs iterations, another fails again and again for want of memory: the run's launches
    never lose the buffer they name.  Bounds as above."""
    for v in ("NV_HV_KERNEL", "NV_HV_FB"):
        monkeypatch.delenv(v, raising=False)
    p = make_problem(4, [8] * 7, 3, (400, 2500), 200.0, 60.0, 40.0, cubic=10.0, seed=7)
    n = 400000
    diag, off = np.ones(n), np.ones(n + 1)
    with Engine(p) as eng:
        eng.lanczos_init(niter=12)
        eng.run(1, 12)
        want = eng.coefficients()[:2]
        stop, failed = threading.Event(), []

        def short():
            while not stop.is_set():
                try:
                    eng.ritz(diag, off)
                except NvError:
                    failed.append(1)

        t = threading.Thread(target=short)
        t.start()
        try:
            for _ in range(6):
                eng.lanczos_init(niter=12)
                for i in range(1, 13, 3):
                    eng.run(i, i + 2)
                for got, ref in zip(eng.coefficients()[:2], want):
                    assert np.max(np.abs(got - ref)) <= 1e-11 * np.max(np.abs(ref))
        finally:
            stop.set()
            t.join()
        assert failed
