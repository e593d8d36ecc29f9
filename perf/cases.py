"""The workloads whose speed this framework is judged by, from the smallest
operator to the largest, through the public entry points.

A case is a dict of plain values.  Its "kind" names what a program does:

    hv        y = H x on device tensors (nadvibs_amd.torch_ops.hv)
    lanczos   a Lanczos run: init, the iterations, the coefficients
    job       a run with partial re-orthogonalisation, then its broadened
              spectrum
    batch     many operators of uneven size advanced together
    fit       one step of a fit: a broadened spectrum and the gradient of a
              loss with respect to the frequencies and couplings
    ritz      the tridiagonal eigenproblem of a finished run and the envelope
              of its sticks

Operators are seeded: frequencies and couplings are drawn with the
distributions of nadvibs_amd/synth.py (cm^-1), so another seed is another
Hamiltonian.  With prec "f32" the couplings are applied in FP32 while the
recurrence stays FP64; the results then carry FP32 accuracy, and the program
keeps them as FP32 numbers.

listed(), draw(rng), prepare(case, seed), run(state), work(case) and
exact(case, seed) are the interface; exact() restates the mathematics in
64-bit torch, mode by mode on the product tensor, and shares no code with
the framework.
"""
import dataclasses
import itertools
import math

import numpy as np
import torch

AU2WAVE = 219474.6313705

# Shapes used throughout the repository: the small quadratic model, the
# six-mode three-state model, the ten-mode four-state cubic model.
SMALL = dict(nstates=2, basis="10,10,10", ordr=2)
SIX = dict(nstates=3, basis="12,10,10,8,8,6", ordr=2)
TEN = dict(nstates=4, basis="8,8,6,6,6,5,5,4,4,4", ordr=3)
# odd sizes in every mode, cubic
ODD = dict(nstates=3, basis="11,9,7,7,5,3", ordr=3)


def listed():
    return [
        # a two-state, three-mode model: what a user starts with; a call is all launch latency
        dict(name="hv_2k_f64", kind="hv", prec="f64", **SMALL),
        # one H*v of the six-mode model inside a user's own FP32 propagator or eigensolver
        dict(name="hv_1m4_f32", kind="hv", prec="f32", **SIX),
        # a short run of the small model: launches and gaps
        dict(name="lanczos_2k_f64", kind="lanczos", prec="f64", niter=33, **SMALL),
        # a cubic model with odd basis sizes, all in FP64
        dict(name="lanczos_218k_odd_f64", kind="lanczos", prec="f64", niter=33, **ODD),
        # the six-mode model in mixed precision, the vectors resident in the caches
        dict(name="lanczos_1m4_f32", kind="lanczos", prec="f32", niter=17, **SIX),
        # the ten-mode cubic model: the largest job, FP32 couplings
        dict(name="lanczos_88m_f32", kind="lanczos", prec="f32", niter=17, **TEN),
        # the same all in FP64
        dict(name="lanczos_88m_f64", kind="lanczos", prec="f64", niter=17, **TEN),
        # the usual production job: partial re-orthogonalisation, then the spectrum from 0 to 6000 cm^-1
        dict(name="job_1m4_f64", kind="job", prec="f64", niter=500, points=4096, sigma=15.0, top=6000.0, **SIX),
        # the same with FP32 couplings, which re-orthogonalises more
        dict(name="job_1m4_f32", kind="job", prec="f32", niter=300, points=4096, sigma=15.0, top=1500.0, **SIX),
        # a scan: 64 operators of 4 to 6 modes and 2 or 3 states
        dict(name="batch_64_f32", kind="batch", prec="f32", niter=17, count=64, mmin=4, mmax=6, fmin=4, fmax=12),
        # one gradient step of fitting the couplings to a spectrum
        dict(name="fit_1m4_f64", kind="fit", prec="f64", niter=120, points=4096, sigma=60.0, top=6000.0, **SIX),
        # after the iterations: eigenvalues, intensities and the convolved spectrum
        dict(name="ritz_2000", kind="ritz", n=2000, points=4096, sigma=15.0, top=6000.0),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_operator(rng, lo, hi):
    """States, basis sizes and order of an operator with about exp(U(log lo, log hi)) elements."""
    target = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    ns = rng.choice([2, 3, 3, 4])
    ordr = rng.choice([2, 2, 3])
    for _ in range(1000):
        m = rng.randint(3, 10)
        base = (target / ns) ** (1.0 / m)
        nf = [max(3, min(13, int(round(base * math.exp(rng.uniform(-0.35, 0.35)))))) for _ in range(m)]
        nf.sort(reverse=True)
        n = ns * math.prod(nf)
        if max(lo, 0.6 * target) <= n <= min(hi, 1.6 * target):
            return dict(nstates=ns, basis=",".join(map(str, nf)), ordr=ordr)
    return dict(SMALL)


def draw(rng):
    kind = rng.choice(["hv", "hv", "lanczos", "lanczos", "lanczos", "job", "batch", "fit", "ritz"])
    prec = rng.choice(["f32", "f64"])
    if kind == "hv":
        return dict(kind=kind, prec=prec, **_draw_operator(rng, 2e3, 6e7))
    if kind == "lanczos":
        # short runs: the sizes vary, not the length (1 + 16 or 1 + 2 * 16 iterations and a remainder)
        c = _draw_operator(rng, 2e3, 6e7)
        n = _elements(c)
        return dict(kind=kind, prec=prec, niter=rng.randint(9, 24 if prec == "f64" and n > 5e4 else 17), **c)
    if kind == "job":
        ns, m = rng.choice([2, 3]), rng.choice([5, 6])
        nf = sorted((rng.randint(6, 11) for _ in range(m)), reverse=True)
        return dict(kind=kind, prec=prec, niter=rng.randint(240, 400), points=rng.randint(500, 4096), sigma=15.0,
                    top=1500.0, nstates=ns, basis=",".join(map(str, nf)), ordr=2)
    if kind == "batch":
        return dict(kind=kind, prec=prec, niter=rng.randint(9, 17), count=_log_int(rng, 3, 64), mmin=4, mmax=6,
                    fmin=4, fmax=rng.randint(7, 12))
    if kind == "fit":
        c = _draw_operator(rng, 2e4, 1.4e6)
        c["ordr"] = 2
        return dict(kind=kind, prec="f64", niter=rng.randint(24, 48), points=rng.randint(500, 4096), sigma=200.0,
                    top=6000.0, **c)
    return dict(kind="ritz", n=_log_int(rng, 100, 2500), points=rng.randint(500, 4096), sigma=15.0, top=6000.0)


# ---------------------------------------------------------------------------
# seeded operators
# ---------------------------------------------------------------------------
def _basis(case):
    return [int(v) for v in case["basis"].split(",")]


def _elements(case):
    return case["nstates"] * math.prod(_basis(case))


@dataclasses.dataclass
class _Model:
    """Frequencies (hartree), state constants and, per monomial (a non-decreasing
    tuple of modes), the symmetric state-coupling matrix in dimensionless coordinates."""
    ns: int
    nf: list
    ordr: int
    omega: np.ndarray
    const: np.ndarray
    coup: dict


def _model(ns, nf, ordr, seed):
    """Frequencies U(300, 3200), linear N(0, 300), quadratic N(0, 80), bilinear
    N(0, 40), cubic N(0, 10) cm^-1, states 2000 cm^-1 apart; between different
    states no constant and no all-even monomials."""
    rng = np.random.default_rng([seed, ns, ordr] + list(nf))
    omega = rng.uniform(300.0, 3200.0, size=len(nf)) / AU2WAVE
    coup = {}
    for p in range(1, ordr + 1):
        for mon in itertools.combinations_with_replacement(range(len(nf)), p):
            even = all(mon.count(k) % 2 == 0 for k in mon)
            sig = (300.0, 80.0 if len(set(mon)) == 1 else 40.0, 10.0)[p - 1]
            c = rng.normal(0.0, sig, size=(ns, ns))
            c = np.tril(c) + np.tril(c, -1).T
            if even:
                c = np.diag(np.diag(c))
            coup[mon] = c / AU2WAVE
    return _Model(ns, list(nf), ordr, omega, np.arange(ns) * 2000.0 / AU2WAVE, coup)


def _case_model(case, seed):
    return _model(case["nstates"], _basis(case), case["ordr"], seed)


def _potterms(m):
    """The raw nadvibs.in coefficients [block, order, monomial]: a monomial's
    coupling times prod_k omega_k^(p_k / 2)."""
    from nadvibs_amd.inputs import monomials, noterms
    nm = len(m.nf)
    blocks = [(i, j) for i in range(m.ns) for j in range(i + 1)]
    pot = np.zeros((len(blocks), m.ordr, noterms(nm, m.ordr)))
    for p in range(1, m.ordr + 1):
        for k, mon in enumerate(monomials(nm, p)):
            c = m.coup[tuple(sorted(mon))]
            scale = math.prod(math.sqrt(m.omega[v]) for v in mon)
            for b, (i, j) in enumerate(blocks):
                pot[b, p - 1, k] = c[i, j] * scale
    concoef = np.array([m.const[i] if i == j else 0.0 for i, j in blocks])
    return concoef, pot


def _problem(m):
    from nadvibs_amd.inputs import Problem
    concoef, pot = _potterms(m)
    return Problem(nstates=m.ns, nmodes=len(m.nf), ordr=m.ordr, nfunc=list(m.nf), aomega=m.omega, concoef=concoef,
                   potterms=pot, statew=np.ones(m.ns), npirrep=[len(m.nf)], initstate=[0] * len(m.nf))


def _batch_models(case, seed):
    rng = np.random.default_rng(seed)
    out = []
    for _ in range(case["count"]):
        ns = int(rng.integers(2, 4))
        nm = int(rng.integers(case["mmin"], case["mmax"] + 1))
        nf = [int(v) for v in rng.integers(case["fmin"], case["fmax"] + 1, size=nm)]
        out.append(_model(ns, nf, 2, int(rng.integers(1 << 30))))
    return out


def _wave(n, seed, dtype, device="cuda"):
    """A normalised random vector, in the precision the program holds its vectors in."""
    g = torch.Generator(device=device).manual_seed(int(seed) + 17)
    x = torch.randn(n, generator=g, device=device, dtype=torch.float64)
    return (x / torch.linalg.vector_norm(x)).to(dtype)


def _tridiagonal(n, seed):
    """alpha(1:n), beta(0:n) (hartree) as a run from a low vibrational state
    leaves them: both rise towards the middle and a quarter of the band."""
    rng = np.random.default_rng(seed)
    rise = np.sqrt((np.arange(n) + 1.0) / n)
    alpha = 0.03 + 0.18 * rise * (1.0 + 0.02 * rng.standard_normal(n))
    beta = np.empty(n + 1)
    beta[0] = 1.0
    beta[1:] = 0.095 * rise * (1.0 + 0.02 * rng.standard_normal(n))
    return alpha, beta


# ---------------------------------------------------------------------------
# the program
# ---------------------------------------------------------------------------
def _kept(a, prec):
    """What the program keeps of a result computed with couplings in `prec`."""
    return a.astype(np.float32) if prec == "f32" else a


def prepare(case, seed):
    kind = case["kind"]
    if kind == "batch":
        from nadvibs_amd.batch import Batch
        bt = Batch([_problem(m) for m in _batch_models(case, seed)])
        return dict(case=case, batch=bt)
    if kind == "ritz":
        from nadvibs_amd.engine import Engine
        alpha, beta = _tridiagonal(case["n"], seed)
        return dict(case=case, eng=Engine(_problem(_model(2, [4, 4], 2, 1))), alpha=alpha, beta=beta,
                    grid=np.linspace(0.0, case["top"], case["points"]))
    m = _case_model(case, seed)
    if kind == "fit":
        target = np.random.default_rng(seed + 5).uniform(0.0, 1.0, size=case["points"])
        concoef, pot = _potterms(m)
        par = [torch.from_numpy(v).requires_grad_(True) for v in (m.omega.copy(), concoef, pot)]
        return dict(case=case, prob=_problem(m), par=par, target=torch.from_numpy(target),
                    grid=torch.linspace(0.0, case["top"], case["points"], dtype=torch.float64))
    from nadvibs_amd.engine import Engine
    st = dict(case=case, eng=Engine(_problem(m)))
    if kind == "hv":
        # the program's own stream: its conversions and H*v follow each other there
        st["stream"] = torch.cuda.Stream()
        st["x"] = _wave(_elements(case), seed, torch.float32 if case["prec"] == "f32" else torch.float64)
    if kind == "job":
        st["grid"] = np.linspace(0.0, case["top"], case["points"])
    return st


def run(st):
    case = st["case"]
    kind, prec = case["kind"], case.get("prec", "f64")
    if kind == "hv":
        from nadvibs_amd import torch_ops
        with torch.cuda.stream(st["stream"]):
            y = torch_ops.hv(st["eng"], st["x"].double(), prec)
            return y.float() if prec == "f32" else y
    if kind == "lanczos":
        eng = st["eng"]
        eng.lanczos_init(case["niter"], prec=prec)
        eng.run(1, case["niter"])
        a, b, _ = eng.coefficients()
        return dict(alpha=_kept(a, prec), beta=_kept(b, prec))
    if kind == "job":
        eng = st["eng"]
        eng.lanczos_init(case["niter"], reorthog=1, prec=prec)
        eng.run(1, case["niter"])
        a, b, _ = eng.coefficients()
        return _kept(eng.spectrum(a, b, st["grid"], case["sigma"]), prec)
    if kind == "batch":
        bt = st["batch"]
        bt.init(case["niter"], prec)
        bt.run()
        ab = [bt.coefficients(p) for p in range(case["count"])]
        return dict(alpha=_kept(np.concatenate([a for a, _ in ab]), prec),
                    beta=_kept(np.concatenate([b for _, b in ab]), prec))
    if kind == "fit":
        from nadvibs_amd.adjoint import spectrum_of_parameters
        for p in st["par"]:
            p.grad = None
        env = spectrum_of_parameters(st["prob"], *st["par"], case["niter"], st["grid"], case["sigma"], prec=prec,
                                     reorthog=1)
        loss = torch.sum((env - st["target"]) ** 2)
        loss.backward()
        return dict(spectrum=env.detach(), omega=st["par"][0].grad, concoef=st["par"][1].grad,
                    potterms=st["par"][2].grad)
    ev, inten, bji, _ = st["eng"].ritz(st["alpha"], st["beta"])
    env = st["eng"].convolve((ev - ev[0]) * AU2WAVE, inten, st["grid"], case["sigma"])
    return dict(eigenvalues=ev, intensities=inten, residuals=bji, envelope=env)


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _hv_flops(ns, nf, ordr):
    """Mixing the states of every monomial (ns^2 multiply-adds) and forming each
    monomial's vector from a shorter one (two neighbours per row and state)."""
    t = sum(math.comb(len(nf) + p - 1, p) for p in range(1, ordr + 1))
    return 2.0 * math.prod(nf) * t * (ns * ns + 2 * ns)


def _iteration(ns, nf, ordr, prec):
    """(bytes, flops) of one iteration: q_i and its H*v input read, H q_i
    written, then q_i, q_{i-1}, the diagonal and H q_i read and r written; the
    residual normalised in place and copied for the next H*v."""
    n = ns * math.prod(nf)
    el = 4 if prec == "f32" else 8
    return n * ((8 + 8 + el + el) + (8 + 8 + 8 + el + 8) + (8 + 8 + el)), _hv_flops(ns, nf, ordr) + 20.0 * n


def work(case):
    kind = case["kind"]
    if kind == "ritz":
        n, g = case["n"], case["points"]
        # 53 halvings of every root with a Sturm count of three operations a row, two solves with the
        # factored matrix; a Gaussian of every stick at every grid point
        return dict(bytes=16.0 * n + 16.0 * g + 24.0 * n, flops=53 * 3.0 * n * n + 20.0 * n * n + 25.0 * n * g)
    prec = case["prec"]
    if kind == "batch":
        by = fl = 0.0
        for m in _batch_models(case, 1):
            b, f = _iteration(m.ns, m.nf, 2, prec)
            by += case["niter"] * b
            fl += case["niter"] * f
        return dict(bytes=by, flops=fl)
    ns, nf, ordr = case["nstates"], _basis(case), case["ordr"]
    n = ns * math.prod(nf)
    if kind == "hv":
        return dict(bytes=2.0 * n * (4 if prec == "f32" else 8), flops=_hv_flops(ns, nf, ordr))
    b, f = _iteration(ns, nf, ordr, prec)
    b, f = b * case["niter"], f * case["niter"]
    if kind == "fit":
        # the basis read once for the projected vectors (niter^2 multiply-adds a row), once for the
        # derivatives of every monomial
        k = case["niter"]
        b += 3.0 * 8 * n * k
        f += 2.0 * k * k * n + k * _hv_flops(ns, nf, ordr)
    return dict(bytes=b, flops=f)


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------
def _position(nf, p):
    """<m| q^p |n> over nf oscillator functions.  As in the framework's default
    conventions, q^3 couples neighbouring functions with sqrt((m + 1)^3 / 8)."""
    big = np.zeros((nf + p + 2, nf + p + 2))
    for m in range(nf + p + 1):
        big[m, m + 1] = big[m + 1, m] = math.sqrt((m + 1) / 2.0)
    q = np.linalg.matrix_power(big, p)[:nf, :nf].copy()
    if p == 3:
        for m in range(nf - 1):
            q[m, m + 1] = q[m + 1, m] = math.sqrt((m + 1) ** 3 / 8.0)
    return q


class _Exact:
    """H on the product tensor [states, n_1, ..., n_M], one mode at a time."""

    def __init__(self, m, device):
        self.m, self.dev = m, device
        self.nm = len(m.nf)
        self.D = math.prod(m.nf)
        self.q = {(k, p): torch.from_numpy(_position(m.nf[k], p)).to(device) for k in range(self.nm)
                  for p in range(1, m.ordr + 1)}
        e = torch.zeros(m.nf, dtype=torch.float64, device=device)
        for k in range(self.nm):
            shape = [1] * self.nm
            shape[k] = m.nf[k]
            lev = (torch.arange(m.nf[k], dtype=torch.float64, device=device) + 0.5) * float(m.omega[k])
            e += lev.reshape(shape)
        self.energy = e.reshape(-1)
        # monomials by their powers, ((mode, power), ...) with increasing modes
        self.terms = {}
        for mon, c in m.coup.items():
            key = tuple((k, mon.count(k)) for k in sorted(set(mon)))
            self.terms[key] = torch.from_numpy(np.ascontiguousarray(c)).to(device)

    def along(self, k, p, x):
        """q_k^p x for x of shape [rows, D]."""
        nf = self.m.nf[k]
        r = math.prod(self.m.nf[k + 1:])
        v = x.reshape(-1, nf, r)
        q = self.q[(k, p)]
        out = torch.zeros_like(v)
        for d in range(-p, p + 1, 2):  # the bands of q^p
            if abs(d) >= nf:
                continue
            lo, hi = max(0, -d), min(nf, nf - d)
            band = torch.diagonal(q, d)
            out[:, lo:hi].addcmul_(v[:, lo + d:hi + d], band.reshape(1, -1, 1))
        return out.reshape(x.shape)

    def monomials(self, x, key=(), left=None, start=0):
        """(key, monomial applied to x) for every term, each from a shorter one."""
        left = self.m.ordr if left is None else left
        for k in range(start, self.nm):
            for p in range(1, left + 1):
                u = self.along(k, p, x)
                kk = key + ((k, p),)
                if kk in self.terms:
                    yield kk, u
                if left > p:
                    yield from self.monomials(u, kk, left - p, k + 1)

    def hv(self, x):
        x = x.reshape(self.m.ns, self.D)
        y = x * (self.energy[None, :] + torch.from_numpy(self.m.const).to(self.dev)[:, None])
        for key, u in self.monomials(x):
            y.addmm_(self.terms[key], u)
        return y.reshape(-1)

    def start(self):
        v = torch.zeros(self.m.ns, self.D, dtype=torch.float64, device=self.dev)
        v[:, 0] = 1.0 / math.sqrt(self.m.ns)
        return v.reshape(-1)

    def lanczos(self, n, full=False):
        """alpha(1:n), beta(0:n) and, when full, the basis kept orthogonal by
        two passes of Gram-Schmidt."""
        r = self.start()
        a, b = np.zeros(n), np.zeros(n + 1)
        b[0] = 1.0
        basis = torch.empty(n, r.numel(), dtype=torch.float64, device=self.dev) if full else None
        prev = None
        for j in range(n):
            q = r / b[j]
            if full:
                basis[j] = q
            r = self.hv(q)
            a[j] = float(torch.dot(q, r))
            r.add_(q, alpha=-a[j])
            if prev is not None:
                r.add_(prev, alpha=-b[j])
            if full:
                for _ in range(2):
                    r.sub_(basis[:j + 1].T.mv(basis[:j + 1].mv(r)))
            b[j + 1] = float(torch.linalg.vector_norm(r))
            prev = q
        return a, b, basis

    def cost(self):
        """Seconds of one H*v, roughly: a dozen memory passes a term at 5 TB/s, and launches."""
        t = len(self.terms)
        return 12 * t * 8.0 * self.D * self.m.ns / 5e12 + t * 10 * 1.2e-5


def _eigen(a, b):
    t = torch.from_numpy(np.diag(a) + np.diag(b[1:-1], 1) + np.diag(b[1:-1], -1))
    w, s = torch.linalg.eigh(t)
    return w, s


def _envelope(theta, weight, grid, sigma):
    """sum_i w_i exp(-((x - x_i) / sigma)^2 / 2), sticks in cm^-1 above the lowest."""
    x = (theta - theta[0]) * AU2WAVE
    return torch.exp(-0.5 * ((grid[:, None] - x[None, :]) / sigma) ** 2) @ weight


def _exact_fit(case, seed, ex):
    """The spectrum and the gradient of the squared distance to the target,
    projected on the Krylov space: sum_jk Tbar_jk q_j . (dH / dparameter) q_k."""
    m, n, sigma = ex.m, case["niter"], case["sigma"]
    a, b, basis = ex.lanczos(n, full=True)
    theta, s = _eigen(a, b)
    grid = torch.linspace(0.0, case["top"], case["points"], dtype=torch.float64)
    target = torch.from_numpy(np.random.default_rng(seed + 5).uniform(0.0, 1.0, size=case["points"]))
    w = s[0]
    env = _envelope(theta, w * w, grid, sigma)
    gbar = 2.0 * (env - target)
    # divided differences of W(t) = sum_x gbar_x G(x - t) and the origin's share
    u = (grid[:, None] - ((theta - theta[0]) * AU2WAVE)[None, :]) / sigma
    g = torch.exp(-0.5 * u * u)
    big = gbar @ g
    der = (gbar @ (u * g)) * (AU2WAVE / sigma)
    dt = theta[:, None] - theta[None, :]
    near = dt.abs() <= 1e-7 * sigma / AU2WAVE
    d = torch.where(near, 0.5 * (der[:, None] + der[None, :]),
                    (big[:, None] - big[None, :]) / torch.where(near, torch.ones_like(dt), dt))
    mm = d * w[:, None] * w[None, :]
    mm[0, 0] -= float((w * w * der).sum())
    tbar = (s @ mm @ s.T).to(ex.dev)
    lvec = tbar @ basis  # rows sum_k Tbar_jk q_k
    blocks = [(i, j) for i in range(m.ns) for j in range(i + 1)]
    dev = ex.dev

    def bilinear(x, y):
        """sum over the basis of x_a . y_c, [states, states]."""
        out = torch.zeros(m.ns, m.ns, dtype=torch.float64, device=dev)
        for i in range(m.ns):
            for j in range(m.ns):
                out[i, j] = torch.sum(x[:, i] * y[:, j])
        return out

    g_om = np.zeros(ex.nm)
    g_con = np.zeros(len(blocks))
    acc = {}
    diag = {}
    chunk = max(1, int(2e8 / (m.ns * ex.D)))
    for j0 in range(0, n, chunk):
        q = basis[j0:j0 + chunk].reshape(-1, m.ns, ex.D)
        l = lvec[j0:j0 + chunk].reshape(-1, m.ns, ex.D)
        prod = (l * q).sum(dim=(0, 1)).reshape(m.nf)
        for k in range(ex.nm):
            v = prod.sum(dim=[i for i in range(ex.nm) if i != k])
            g_om[k] += float((v * (torch.arange(m.nf[k], device=dev, dtype=torch.float64) + 0.5)).sum())
        c0 = bilinear(l, q).cpu().numpy()
        g_con += np.array([c0[i, j] for i, j in blocks])
        for key, uq in ex.monomials(q.reshape(-1, ex.D)):
            uq = uq.reshape(q.shape)
            acc[key] = acc.get(key, 0.0) + bilinear(l, uq).cpu().numpy()
            if all(p % 2 == 0 for _, p in key):
                h = torch.ones(m.nf, dtype=torch.float64, device=dev)
                for k, p in key:
                    shape = [1] * ex.nm
                    shape[k] = m.nf[k]
                    h = h * torch.diagonal(ex.q[(k, p)]).reshape(shape)
                diag[key] = diag.get(key, 0.0) + bilinear(l, q * h.reshape(1, 1, -1)).cpu().numpy()
    # monomials in file order: non-increasing tuples, first entry fastest
    ntm = math.comb(ex.nm + m.ordr - 1, m.ordr)
    g_pot = np.zeros((len(blocks), m.ordr, ntm))
    for p in range(1, m.ordr + 1):
        for k, mon in enumerate(itertools.combinations_with_replacement(range(ex.nm), p)):
            key = tuple((v, mon.count(v)) for v in sorted(set(mon)))
            scale = math.prod(1.0 / math.sqrt(m.omega[v]) for v in mon)
            dd = diag.get(key)
            for bi, (i, j) in enumerate(blocks):
                v = acc[key][i, j]
                if i != j:
                    # both off-diagonal blocks; the part diagonal in the vibrations acts below the state diagonal only
                    v += acc[key][j, i] - (dd[j, i] if dd is not None else 0.0)
                g_pot[bi, p - 1, k] = v * scale
                c = m.coup[mon][i, j]
                if c != 0.0:
                    for kk, pw in key:
                        g_om[kk] -= 0.5 * pw / m.omega[kk] * c * v
    return dict(spectrum=env, omega=torch.from_numpy(g_om), concoef=torch.from_numpy(g_con),
                potterms=torch.from_numpy(g_pot))


def exact(case, seed):
    kind = case["kind"]
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    if kind == "ritz":
        alpha, beta = _tridiagonal(case["n"], seed)
        w, s = _eigen(alpha, beta)
        inten = s[0] ** 2
        env = _envelope(w, inten, torch.linspace(0.0, case["top"], case["points"], dtype=torch.float64),
                        case["sigma"])
        return dict(eigenvalues=w, intensities=inten, residuals=(beta[-1] * s[-1]).abs(), envelope=env / env.max())
    if kind == "batch":
        models = [_Exact(m, dev) for m in _batch_models(case, seed)]
        if sum(x.cost() for x in models) * case["niter"] > 15.0:
            return None
        ab = [x.lanczos(case["niter"]) for x in models]
        return dict(alpha=np.concatenate([a for a, _, _ in ab]), beta=np.concatenate([b for _, b, _ in ab]))
    ex = _Exact(_case_model(case, seed), dev)
    if kind == "hv":
        dtype = torch.float32 if case["prec"] == "f32" else torch.float64
        return ex.hv(_wave(_elements(case), seed, dtype, dev).double())
    if ex.cost() * case["niter"] > 15.0:
        return None
    if kind == "lanczos":
        a, b, _ = ex.lanczos(case["niter"])
        return dict(alpha=a, beta=b)
    if kind == "job":
        a, b, _ = ex.lanczos(case["niter"], full=True)
        theta, s = _eigen(a, b)
        return _envelope(theta, s[0] ** 2, torch.linspace(0.0, case["top"], case["points"], dtype=torch.float64),
                         case["sigma"])
    return _exact_fit(case, seed, ex)
