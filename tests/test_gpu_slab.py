"""GPU: H*v with the degree-three slow terms in the slab and leading passes
(forced on small operators) against the step-list kernels, which the oracle
holds: one to three modes in LDS, none
to four leading modes, basis sizes of one and two, one to four states, one and
two rows per thread, the last workgroup of an XCD's share empty or not."""
import numpy as np
import pytest
import torch

from nadvibs_amd import torch_ops
from nadvibs_amd.engine import Engine
from nadvibs_amd.synth import make_problem, workload
from oracle.oracle import Oracle
from test_gpu_parity import FAST_BLOCK
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


def _run_of_12(eng, prec):
    eng.lanczos_init(niter=12, reorthog=0, prec=prec)
    eng.run(1, 12)
    a, b, _ = eng.coefficients()
    return np.array(a), np.array(b)


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{c[0]}x{'-'.join(map(str, c[1]))}")
def test_slab_pass_is_reported(case, monkeypatch):
    """The operators above do take the slab pass, with its buffer, standalone and in a run."""
    monkeypatch.delenv("NV_HV_KERNEL", raising=False)
    monkeypatch.delenv("NV_HV_SLAB", raising=False)
    monkeypatch.setenv("NV_HV_FB", "1")
    ns, nf, offe, quirks = case
    p = make_problem(ns, nf, 3, (400, 2500), 200.0, 60.0, 40.0, cubic=10.0, seed=len(nf), quirks=quirks,
                     offdiag_even=offe)
    with Engine(p) as eng:
        for prec in ("f64", "f32"):
            eng.hv(np.ones(p.n), prec)
            _run_of_12(eng, prec)
            info = eng.hv_kernel(prec)
            assert "slab pass (modes " in info and "no memory" not in info, info


CUBIC = [c for c in FAST_BLOCK if c[2] == 3] + [
    # five and seven states, which have no slab pass
    (5, [3, 2, 4, 4, 4], 3, 10.0, 10.0, 3),
    (7, [4, 3, 6, 7], 3, 10.0, 0.0, 0),
]


@pytest.mark.parametrize("slab", ["0", "1"])
@pytest.mark.parametrize("case", CUBIC, ids=lambda c: f"{c[0]}x{'-'.join(map(str, c[1]))}")
def test_cubic_fast_block_with_and_without_the_slab_pass(case, slab, monkeypatch):
    """Cubic operators with the degree-three slow steps in the sweep and in the slab pass, against the
    oracle: bounds as for every fast-block operator."""
    monkeypatch.setenv("NV_HV_FB", "1")
    monkeypatch.setenv("NV_HV_SLAB", slab)
    monkeypatch.delenv("NV_HV_KERNEL", raising=False)
    ns, nf, ordr, cub, offe, quirks = case
    p = make_problem(ns, nf, ordr, (400, 3000), 250.0, 60.0, 40.0, cubic=cub, seed=5, quirks=quirks,
                     offdiag_even=offe)
    print(f"case {case} slab={slab} n={p.n}", flush=True)
    orc = Oracle(p)
    x = np.random.default_rng(3).standard_normal(p.n)
    ref = orc.hv(x)
    r = orc.lanczos(12)
    with Engine(p) as eng:
        for prec, tol_hv, tol_ab in (("f64", 1e-13, 1e-11), ("f32", 2e-6, 5e-6)):
            info = eng.hv_kernel(prec)
            assert info.startswith("generic fast-block"), info
            assert ("slab pass" in info) == (slab == "1" and ns <= 4), info
            assert ("all slow steps in the sweep" in info) == (slab == "0" and ns <= 4), info
            err = np.max(np.abs(eng.hv(x, prec) - ref)) / np.max(np.abs(ref))
            assert err <= tol_hv, (prec, err)
            a, b = _run_of_12(eng, prec)
            assert np.max(np.abs(a - r["alpha"]) / np.abs(r["alpha"])) <= tol_ab, prec
            assert np.max(np.abs(b - r["beta"]) / np.abs(r["beta"])) <= tol_ab, prec


def test_slab_pass_by_size(monkeypatch):
    """Without a switch the slab pass serves from 200 degree-three slow steps: the ten-mode operator has
    560, one of four slow modes at most 120."""
    for v in ("NV_HV_KERNEL", "NV_HV_FB", "NV_HV_SLAB"):
        monkeypatch.delenv(v, raising=False)
    with Engine(workload("cfg3")) as eng:
        for prec in ("f32", "f64"):
            info = eng.hv_kernel(prec)
            assert "slab pass (modes 4..6 in LDS) and a leading pass (modes 0..3)" in info, info
    p = make_problem(4, [12, 11, 13, 12, 8, 8], 3, (400, 2500), 200.0, 60.0, 40.0, cubic=10.0, seed=2)
    with Engine(p) as eng:
        for prec in ("f32", "f64"):
            info = eng.hv_kernel(prec)
            assert info.startswith("generic fast-block") and "slab pass" not in info, info
            assert "all slow steps in the sweep" in info, info


def test_captured_hv_with_the_slab_pass(monkeypatch):
    """A captured standalone H*v replays with new inputs, between the program's own work, to the bits of
    the eager call."""
    monkeypatch.delenv("NV_HV_KERNEL", raising=False)
    monkeypatch.delenv("NV_HV_SLAB", raising=False)
    monkeypatch.setenv("NV_HV_FB", "1")
    p = make_problem(4, [3, 5, 4, 4, 4, 4], 3, (400, 2500), 200.0, 60.0, 40.0, cubic=10.0, seed=6)
    gen = torch.Generator(device="cuda").manual_seed(3)
    with Engine(p) as eng:
        for prec in ("f64", "f32"):
            xs = [torch.randn(p.n, generator=gen, device="cuda", dtype=torch.float64) for _ in range(4)]
            want = [torch_ops.hv(eng, x, prec).clone() for x in xs]
            x, y = xs[0].clone(), torch.empty_like(xs[0])
            torch.cuda.synchronize()
            g = torch.cuda.CUDAGraph()
            with torch.cuda.graph(g):
                torch_ops.hv(eng, x, prec, out=y)
            for xi, w in list(zip(xs, want)) * 2:
                x.copy_(xi)
                y.zero_()
                g.replay()
                torch.cuda.synchronize()
                assert torch.equal(y, w), prec
                assert torch.equal(torch_ops.hv(eng, xi, prec), w)
