"""The gradient's bilinear forms and the projected vectors on the matrix cores:
against the dense restatement at the sizes where tiles, chunks of rows and
states per tile end, and against the term-by-term kernel's operators."""
import numpy as np
import pytest

from nadvibs_amd.engine import Engine
from nadvibs_amd.synth import make_problem
from oracle.adjoint import krylov_gradient, parameter_matrices

pytestmark = pytest.mark.gpu


def _prob(ns, nf, ordr, quirks=3, offe=0.0):
    return make_problem(ns, list(nf), ordr, (600, 2800), 250.0, 60.0, 40.0, cubic=15.0 if ordr > 2 else 0.0,
                        gap=1500.0, seed=7 * ns + len(nf), quirks=quirks, offdiag_even=offe)


def _flat(g, p):
    out = list(np.asarray(g["omega"])) + list(np.asarray(g["concoef"]))
    from nadvibs_amd.inputs import noterms
    for b in range(p.nstblks):
        for q in range(1, p.ordr + 1):
            out += list(np.asarray(g["potterms"])[b, q - 1, :noterms(p.nmodes, q)])
    return np.array(out)


# columns: (modes + 1) * states over tiles of 16 (5 modes of three states, 4 of four a tile); rows: a
# multiple of 32 and not; functions: one, two and more; weights: more than seven modes take two tiles
@pytest.mark.parametrize("ns,nf,ordr", [
    (1, (33,), 2), (1, (3, 2, 2, 2, 2, 2, 1, 2, 2), 2), (2, (4, 4, 2), 2), (2, (5, 1, 4, 3), 2),
    (2, (3, 2, 2, 2, 2, 2, 2, 2), 2), (3, (4, 3, 5), 2), (3, (3, 3, 2, 2), 2), (3, (2,) * 5, 2), (3, (2,) * 7, 2),
    (4, (3, 4, 3), 2), (4, (2, 3, 2, 2), 2), (4, (2,) * 8, 2), (3, (5, 4, 3), 1),
    (5, (3, 4), 2), (2, (4, 3, 3), 3)])
def test_gradient_of_edge_shapes(ns, nf, ordr):
    p = _prob(ns, nf, ordr, quirks=0, offe=10.0)
    n = min(6, p.n - 1)
    rng = np.random.default_rng(1)
    t = rng.standard_normal((n, n))
    t = t + t.T
    with Engine(p) as eng:
        eng.select_hv_kernel(True)
        eng.lanczos_init(n, savevecs=True)
        eng.run(1, n)
        q = np.array([eng.lanczos_vector(j) for j in range(1, n + 1)])
        g = eng.krylov_gradient(t)
    ref = krylov_gradient(q, t, [m for m in parameter_matrices(p) if m is not None])
    got = _flat(g, p)
    # sums of n^2 N products of order one in FP64, in two orders
    assert np.max(np.abs(got - ref)) <= 1e-12 * np.max(np.abs(ref))


@pytest.mark.parametrize("n", [1, 3, 4, 5, 16, 17, 33, 49, 63, 64, 65, 70])
def test_projected_vectors(n):
    """Ritz vectors of every root: n outputs of n vectors, below and above the 64 of one pass and of one stage."""
    p = _prob(2, (7, 7, 3), 2)
    with Engine(p) as eng:
        eng.lanczos_init(n, savevecs=True, reorthog=1)
        eng.run(1, n)
        a, b, _ = eng.coefficients()
        q = np.array([eng.lanczos_vector(j) for j in range(1, n + 1)])
        res = eng.identify_roots(a, b, n, vectors=True)
    t = np.diag(a) + np.diag(b[1:n], 1) + np.diag(b[1:n], -1)
    w, s = np.linalg.eigh(t)
    y = s.T @ q
    gap = np.minimum(np.r_[np.inf, np.diff(w)], np.r_[np.diff(w), np.inf])
    for i in range(n):
        if gap[i] < 1e-6:
            continue
        v = res["vectors"][i]
        sg = 1.0 if np.dot(v, y[i]) > 0 else -1.0
        # the eigenvectors' own accuracy, eps |T| / gap, dominates
        assert np.max(np.abs(sg * v - y[i])) <= 1e-13 + 1e-14 / gap[i], (i, gap[i])
