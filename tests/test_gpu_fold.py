"""GPU: captured iterations with and without their finishing sums folded into
the kernels after them (NV_FOLD_MAX; by default up to 4,096 partials a sum, about
a million rows), in one call and cut into several: the bits of the reference's
loop, launch by launch (Source/main.f90:63-76)."""
import numpy as np
import pytest

from nadvibs_amd.engine import Engine
from nadvibs_amd.synth import workload

pytestmark = pytest.mark.gpu

N, PERIOD = 160, 50


def _loop(eng, reorthog, prec, omega=True):
    """The loop's results after every iteration, and the iterations that listed vectors."""
    eng.lanczos_init(niter=N, reorthog=reorthog, prec=prec, chkorthog=PERIOD)
    stats, listed = [(0, 0)], []
    for i in range(1, N + 1):
        eng.update_lanczos(i)
        eng.Hv(i)
        eng.lanczos_step(i)
        if reorthog and i > 1:
            eng.set_omega(i)
            eng.partial_orthog(i)
        if reorthog:
            stats.append(eng.pro_stats())
            if stats[i] != stats[i - 1]:
                listed.append(i)
    return eng.coefficients(omega=bool(reorthog)), stats, listed


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("reorthog", [1, 2])
@pytest.mark.parametrize("fold", ["on", "off"])
def test_reorthogonalised_runs_cut_anywhere(fold, reorthog, prec, monkeypatch):
    """Cuts right after an iteration that listed vectors, after the one behind it, after an exact
    check, and runs of a single iteration; beta, omega and the counts at every cut and at the end."""
    if fold == "off":
        monkeypatch.setenv("NV_FOLD_MAX", "0")
    else:
        monkeypatch.delenv("NV_FOLD_MAX", raising=False)
    with Engine(workload("cfg1")) as eng:
        (a0, b0, w0), stats, listed = _loop(eng, reorthog, prec)
        print(f"listed at {listed[:6]}... of {len(listed)}", flush=True)
        inner = [i for i in listed if 3 < i < N - 3]
        assert inner
        f, m = inner[0], inner[len(inner) // 2]
        for ends in ([N], [17, 50, N], [f, N], [f + 1, N], [PERIOD, PERIOD + 1, 2 * PERIOD, N],
                     sorted({1, 2, f, m, m + 1, 100, N - 1, N})):
            eng.lanczos_init(niter=N, reorthog=reorthog, prec=prec, chkorthog=PERIOD)
            at = 0
            for end in ends:
                eng.run(at + 1, end)
                at = end
                a, b, _ = eng.coefficients()
                assert np.array_equal(a[:end], a0[:end]) and np.array_equal(b[:end + 1], b0[:end + 1]), (ends, end)
                assert eng.pro_stats() == stats[end], (ends, end)
            assert np.array_equal(eng.coefficients(omega=True)[2], w0), ends


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("fold", ["on", "off"])
def test_plain_runs_cut_anywhere(fold, prec, monkeypatch):
    """Without re-orthogonalisation: graphs of 16 iterations, single ones, and the per-call path."""
    if fold == "off":
        monkeypatch.setenv("NV_FOLD_MAX", "0")
    else:
        monkeypatch.delenv("NV_FOLD_MAX", raising=False)
    with Engine(workload("cfg1")) as eng:
        (a0, b0, _), _, _ = _loop(eng, 0, prec)
        for ends in ([N], [1, 17, 34, N], [16, 33, 40, 41, N]):
            eng.lanczos_init(niter=N, reorthog=0, prec=prec)
            at = 0
            for end in ends:
                eng.run(at + 1, end)
                at = end
                a, b, _ = eng.coefficients()
                assert np.array_equal(a[:end], a0[:end]) and np.array_equal(b[:end + 1], b0[:end + 1]), (ends, end)
