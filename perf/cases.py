"""Performance cases: what a user of the framework has it do, through its public entry points.

Each case is a dict of plain values.  ``kind`` says which entry point it goes through:

  step      one accepted step of a drop-in solver (``ETD35(...).step``)
  single    one trajectory, a drop-in solver's ``evolve`` with a built-in nonlinear term
  ensemble  many trajectories of uneven grids, ``BatchSolver.evolve``
  ac2d      a batch of 2-D Allen-Cahn problems (rfft2 grids), ``BatchSolver.evolve``
  radial    a batch of radial NLS beams (Hankel transform), ``BatchSolver.evolve``
  hankel    batched Hankel transforms, ``HankelTransform.ht`` / ``iht``
  callable  a drop-in solver's ``evolve`` with the user's own ``nl_func``
  cheb      a drop-in solver's ``evolve`` with a dense (Chebyshev) ``lin_op``

Intervals are short enough that a pass takes at most some tenths of a second and that rounding is
not amplified by the chaotic families; the step sizes and tolerances are the workloads' own.
IF45DP appears in single steps only: its error estimate drives whole runs to steps of ~1e-5.
"""
import math

import numpy as np
import torch

import rkstiff_amd
from rkstiff_amd import grids, models
from rkstiff_amd.batch import BatchSolver
from rkstiff_amd.config import ETDConfig, SolverConfig
from rkstiff_amd.nonlinear import AdvectiveNL, AllenCahnNL, CubicNL
from rkstiff_amd.transforms import HankelTransform

KS_SIZES = (256, 512, 1024, 2048, 4096)
NLS_SIZES = (1024, 2048, 4096, 8192)
ADAPTIVE = ("ETD35", "ETD34", "IF34")
CONSTANT = ("ETD5", "ETD4", "IF4")
CHECKED = 5  # trajectories of a batch that exact() computes


def listed():
    return [
        # one step in the smallest grid used in earnest: a user's own time loop around step()
        dict(name="step_nls256_etd35_f64", kind="step", problem="nls", method="ETD35", n=256, precision="f64", h=0.01),
        # the README's quickstart: KS, n = 1024, IF34, snapshots every 20 steps, tf = 50
        dict(name="ks1024_if34_f64", kind="single", problem="ks", method="IF34", n=1024, precision="f64", eps=1e-4,
             tf=50.0, store=20),
        # one large trajectory: two colliding solitons, n = 8192, ETD35
        dict(name="nls8192_etd35_f64", kind="single", problem="nls", method="ETD35", n=8192, precision="f64", eps=1e-6,
             tf=2.0, store=0),
        # the KS ensemble of uneven grids, single precision
        dict(name="ks_ensemble2048_if34_f32", kind="ensemble", problem="ks", method="IF34", count=2048, precision="f32",
             eps=1e-5, tf=10.0),
        # a smaller one in the parity precision with the other main method
        dict(name="ks_ensemble512_etd35_f64", kind="ensemble", problem="ks", method="ETD35", count=512, precision="f64",
             eps=1e-5, tf=10.0),
        # the multi-soliton NLS ensemble in the benchmark's headline precision
        dict(name="nls_ensemble1024_etd35_mixed", kind="ensemble", problem="nls", method="ETD35", count=1024,
             precision="mixed", eps=1e-6, tf=1.0),
        # the 2-D Allen-Cahn batch: the largest working set
        dict(name="ac2d_64x512_etd35_f32", kind="ac2d", n=512, count=64, method="ETD35", precision="f32", eps=1e-5, tf=4.0),
        # a few small 2-D problems, where launches count
        dict(name="ac2d_8x128_etd35_f64", kind="ac2d", n=128, count=8, method="ETD35", precision="f64", eps=1e-5, tf=4.0),
        # radial beams on the demo's 100-point Hankel grid (not a power of two)
        dict(name="radial1024_nr100_etd35_f64", kind="radial", n=100, count=1024, method="ETD35", precision="f64",
             eps=1e-5, tf=0.4),
        # Hankel transforms of a batch of complex profiles, an odd number of radial points
        dict(name="hankel_nr251_b1024", kind="hankel", n=251, count=1024, inverse=False, complex=True),
        # the reference's main use: an nl_func of the user's own (torch.fft), KS
        dict(name="callable_ks1024_if34_f64", kind="callable", method="IF34", n=1024, eps=1e-4, tf=10.0),
        # the Chebyshev Allen-Cahn demo with a dense lin_op
        dict(name="cheb20_etd35_dense", kind="cheb", method="ETD35", n=20, eps=1e-4, tf=2.0),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("step", "single", "single", "ensemble", "ensemble", "ensemble", "ac2d", "ac2d", "radial", "hankel",
                       "callable", "cheb"))
    if kind == "step":
        return dict(kind=kind, problem=rng.choice(("nls", "ks", "burgers")), n=1 << rng.randint(5, 13), precision="f64",
                    method=rng.choice(ADAPTIVE + CONSTANT + ("IF45DP",)), h=round(rng.uniform(0.002, 0.01), 6))
    if kind == "single":
        method = rng.choice(("ETD35", "IF34") + ADAPTIVE + CONSTANT)
        problem = rng.choice(("ks", "nls", "kdv", "burgers"))
        n = 1 << (rng.randint(7, 10) if problem == "kdv" else rng.randint(8, 13))
        if method in CONSTANT:  # grids that the fixed steps are stable on
            problem, n = rng.choice((("ks", 512), ("ks", 1024), ("nls", 512), ("nls", 1024), ("kdv", 256)))
        f32 = problem in ("ks", "nls") and method in ADAPTIVE and rng.random() < 0.4
        span = {"ks": 20.0, "nls": 1.0, "kdv": 0.5, "burgers": 0.5}[problem]
        return dict(kind=kind, problem=problem, method=method, n=n, precision="f32" if f32 else "f64",
                    eps=1e-6 if f32 else 10.0 ** -rng.randint(4, 6), tf=round(span * rng.uniform(0.5, 1.0), 4),
                    store=0 if f32 or problem == "burgers" else rng.choice((0, 5, 20)))
    if kind == "ensemble":
        problem = rng.choice(("ks", "nls"))
        return dict(kind=kind, problem=problem, method=rng.choice(("ETD35", "IF34")), count=_log_int(rng, 16, 1500),
                    precision=rng.choice(("f64", "f32", "mixed")), eps=1e-5 if problem == "ks" else 1e-6,
                    tf=round(rng.uniform(3.0, 8.0) if problem == "ks" else rng.uniform(0.2, 0.6), 3))
    if kind == "ac2d":
        n = 1 << rng.randint(5, 9)
        return dict(kind=kind, n=n, count=_log_int(rng, 1, 48), method=rng.choice(("ETD35", "IF34")),
                    precision=rng.choice(("f64", "f32", "mixed")), eps=1e-5, tf=round(rng.uniform(1.0, 3.0), 3))
    if kind == "radial":
        return dict(kind=kind, n=rng.randint(24, 200), count=_log_int(rng, 1, 1024), method=rng.choice(("ETD35", "IF34")),
                    precision=rng.choice(("f64", "mixed")), eps=1e-5, tf=round(rng.uniform(0.1, 0.3), 3))
    if kind == "hankel":
        return dict(kind=kind, n=_log_int(rng, 16, 1024), count=_log_int(rng, 1, 4096), inverse=rng.random() < 0.5,
                    complex=rng.random() < 0.7)
    if kind == "callable":
        return dict(kind=kind, method=rng.choice(("IF34", "ETD35")), n=2 * _log_int(rng, 32, 2048), eps=1e-4,
                    tf=round(rng.uniform(3.0, 10.0), 3))
    return dict(kind=kind, method=rng.choice(("ETD35", "IF34")), n=rng.randint(16, 40), eps=1e-4,
                tf=round(rng.uniform(0.5, 2.0), 3))


# ---------------------------------------------------------------------------
# inputs (NumPy, made from the seed)
# ---------------------------------------------------------------------------
def _rfft_grid(n, a, b):
    x = a + np.arange(n) * ((b - a) / n)
    return x, 2 * np.pi * np.fft.rfftfreq(n, d=(b - a) / n)


def _problem(problem, n, rng):
    """One trajectory: (term, kx, coefficient, L, u0_hat); term is "advect" or "cubic".  The seed
    moves the profile along the (periodic) axis and turns its phase, so the number of stored
    snapshots does not depend on it."""
    if problem == "nls":
        x = -64.0 + np.arange(n) * (128.0 / n)
        kx = 2 * np.pi * np.fft.fftfreq(n, d=128.0 / n)
        u = 2.0 / np.cosh(2.0 * (x + 10)) * np.exp(1j * x) + 1.5 / np.cosh(1.5 * (x - 10)) * np.exp(-0.5j * x)
        return "cubic", kx, 1.0, -0.5j * kx**2, np.fft.fft(u) * np.exp(1j * (kx * rng.uniform(-4, 4) + rng.uniform(0, 6)))
    if problem == "ks":
        return ("advect",) + _ks_field(n, rng)
    if problem == "kdv":
        x, kx = _rfft_grid(n, -30.0, 30.0)
        return "advect", kx, -6.0, 1j * kx**3, np.fft.rfft(0.5 / np.cosh((x + rng.uniform(-5, 5)) / 2) ** 2)
    x, kx = _rfft_grid(n, -np.pi, np.pi)
    return "advect", kx, -1.0, -0.0005 * kx**2, np.fft.rfft(np.exp(-10 * np.sin((x - rng.uniform(-3, 3)) / 2) ** 2))


def _ks_field(n, rng):
    x, kx = _rfft_grid(n, 0.0, 32 * np.pi)
    x = x - rng.uniform(0.0, 32 * np.pi)
    return kx, -1.0, kx**2 * (1 - kx**2), np.fft.rfft(np.cos(x / 16) * (1 + np.sin(x / 16)))


def _member(problem, rng, i):
    """Trajectory i of an ensemble, the grids taken in turn: KS on a random domain, or NLS with 1-3
    solitons."""
    if problem == "ks":
        n, dom = KS_SIZES[i % len(KS_SIZES)], rng.uniform(22.0, 200.0)
        _, kx = _rfft_grid(n, 0.0, dom)
        amp, th = rng.normal(0.0, 0.1, 8), rng.uniform(0.0, 2 * np.pi, 8)
        # the sum of the eight modes, written into its spectrum
        u = np.zeros(n // 2 + 1, dtype=np.complex128)
        u[1:9] = 0.5 * n * amp * np.exp(1j * th)
        return "advect", kx, -1.0, kx**2 * (1 - kx**2), u
    n, m = NLS_SIZES[i % len(NLS_SIZES)], int(rng.integers(1, 4))
    x = -64.0 + np.arange(n) * (128.0 / n)
    kx = 2 * np.pi * np.fft.fftfreq(n, d=128.0 / n)
    u = np.zeros(n, dtype=np.complex128)
    for _ in range(m):
        eta, v, x0, ph = rng.uniform(1.0, 2.5), rng.uniform(-2.0, 2.0), rng.uniform(-40.0, 40.0), rng.uniform(0, 2 * np.pi)
        u += eta / np.cosh(eta * (x - x0)) * np.exp(1j * (v * x + ph))
    return "cubic", kx, 1.0, -0.5j * kx**2, np.fft.fft(u)


def _ac2d_field(n, seed, i):
    return np.random.default_rng((seed, i)).uniform(-0.05, 0.05, (n, n))


def _ac2d_op(n):
    ky, kx = np.fft.fftfreq(n, d=1.0 / n), np.fft.rfftfreq(n, d=1.0 / n)
    k2 = ky[:, None] ** 2 + kx[None, :] ** 2
    return -0.01 * k2, np.sqrt(k2) <= min(32, n // 4)


def _beams(r, count, seed):
    rng = np.random.default_rng(seed)
    return [rng.uniform(1.8, 2.0) * np.exp(-(r / rng.uniform(0.9, 1.1)) ** 2) + 0j for _ in range(count)]


def _profiles(case, seed):
    rng = np.random.default_rng(seed)
    f = rng.standard_normal((case["count"], case["n"]))
    return f + 1j * rng.standard_normal(f.shape) if case["complex"] else f


def _cheb_state(x, rng):
    u = 0.53 * x + 0.47 * rng.uniform(0.95, 1.05) * np.sin(-1.5 * np.pi * x)
    u[np.abs(x) == 1.0] = x[np.abs(x) == 1.0]
    return (u - x)[1:-1].astype(np.complex128)


# ---------------------------------------------------------------------------
# the framework's side
# ---------------------------------------------------------------------------
def _dtype(precision):
    return torch.complex64 if precision == "f32" else torch.complex128


def _dev(a, dtype=torch.complex128):
    return torch.as_tensor(np.ascontiguousarray(a)).to(dtype).cuda()


def _term(term, kx, coef):
    return AdvectiveNL(kx, coef) if term == "advect" else CubicNL(len(kx), coef)


def _solver(method, L, nl, eps, **kw):
    cls = getattr(rkstiff_amd, method)
    if method in CONSTANT:
        return cls(L, nl, **kw)
    return cls(L, nl, config=SolverConfig(epsilon=eps), **kw)


def _fixed_step(case):
    """The step of a constant-step run: 64 steps."""
    return case["tf"] / 64


def prepare(case, seed):
    kind, rng = case["kind"], np.random.default_rng(seed)
    st = dict(case=case)
    if kind in ("step", "single"):
        term, kx, coef, L, u0 = _problem(case["problem"], case["n"], rng)
        st["solver"] = _solver(case["method"], torch.as_tensor(L), _term(term, kx, coef), case.get("eps", 1e-4))
        st["u0"] = _dev(u0, _dtype(case["precision"]))
    elif kind == "ensemble":
        ens = [_member(case["problem"], rng, i) for i in range(case["count"])]
        st["batch"] = BatchSolver(case["method"], [(torch.as_tensor(L), _term(t, kx, c)) for t, kx, c, L, _ in ens],
                                  precision=case["precision"], config=SolverConfig(epsilon=case["eps"]))
        st["u0"] = [_dev(e[4], _dtype(case["precision"])) for e in ens]
    elif kind == "ac2d":
        n = case["n"]
        L, keep = _ac2d_op(n)
        nl, mask = AllenCahnNL(n), torch.as_tensor(keep).cuda()
        st["batch"] = BatchSolver(case["method"], [(torch.as_tensor(L.reshape(-1)), nl)] * case["count"],
                                  precision=case["precision"], config=SolverConfig(epsilon=case["eps"]))
        w = [torch.as_tensor(_ac2d_field(n, seed, i)).cuda() for i in range(case["count"])]
        st["u0"] = [(torch.fft.rfft2(f) * mask).reshape(-1).to(_dtype(case["precision"])) for f in w]
    elif kind == "radial":
        ht = HankelTransform(nr=case["n"], rmax=5.0)
        st["batch"] = BatchSolver(case["method"], [(-1j * ht.kr**2, ht.cubic_nl(2.0))] * case["count"],
                                  precision=case["precision"], config=SolverConfig(epsilon=case["eps"]))
        st["u0"] = list(ht.ht(_dev(np.stack(_beams(ht.r.cpu().numpy(), case["count"], seed)))).unbind(0))
    elif kind == "hankel":
        st["ht"] = HankelTransform(nr=case["n"], rmax=5.0)
        st["f"] = torch.as_tensor(_profiles(case, seed)).cuda()
    elif kind == "callable":
        n = case["n"]
        kx, _, L, u0 = _ks_field(n, rng)
        ik = _dev(1j * kx)

        def nl(u):
            return -torch.fft.rfft(torch.fft.irfft(u, n=n) * torch.fft.irfft(ik * u, n=n))
        st["solver"], st["u0"] = _solver(case["method"], torch.as_tensor(L), nl, case["eps"]), _dev(u0)
    else:
        x, D = grids.construct_x_dx_cheb(case["n"], -1, 1)
        L, nl = models.allen_cahn_ops(x, D, 0.01)
        kw = {} if case["method"] == "IF34" else dict(etd_config=ETDConfig(contour_points=64, contour_radius=20))
        st["solver"] = _solver(case["method"], L, nl, case["eps"], **kw)
        st["u0"] = _dev(_cheb_state(x.cpu().numpy(), rng))
    return st


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "step":
        out = state["solver"].step(state["u0"], case["h"])
        # (u_new, h_used): the next step's size hangs on the error estimate's rounding
        return list(out[:2]) if isinstance(out, tuple) else [out]
    if kind in ("single", "callable", "cheb"):
        s, store = state["solver"], case.get("store", 0)
        if case["method"] in CONSTANT:
            u = s.evolve(state["u0"], 0.0, case["tf"], _fixed_step(case), store_data=store > 0, store_freq=max(store, 1))
        else:
            u = s.evolve(state["u0"], 0.0, case["tf"], store_data=store > 0, store_freq=max(store, 1))
        return {"u": u, "t": np.array(s.t), "snapshots": torch.stack(s.u)} if store else {"u": u}
    if kind == "hankel":
        return (state["ht"].iht if case["inverse"] else state["ht"].ht)(state["f"])
    uf = state["batch"].evolve(state["u0"], 0.0, case["tf"])
    k = min(CHECKED if kind != "ac2d" else 1, len(uf))
    return {"first": torch.cat(uf[:k]), "rest": torch.cat(uf[k:]) if len(uf) > k else None}


# ---------------------------------------------------------------------------
# work: each input read and each output written once; the transforms and stage sums of the
# attempts that the error control takes on these inputs (typical counts per unit of time)
# ---------------------------------------------------------------------------
STAGES = {"ETD35": 6, "ETD34": 4, "IF34": 4, "IF45DP": 7, "ETD5": 6, "ETD4": 4, "IF4": 4}
TERMS = {"ETD35": 25, "ETD34": 15, "IF34": 14, "IF45DP": 34, "ETD5": 25, "ETD4": 15, "IF4": 14}
RATE = {"ks": 10.0, "nls": 60.0, "kdv": 25.0, "burgers": 50.0, "ac2d": 10.0, "radial": 70.0, "cheb": 9.0}


def _attempts(case, problem):
    if case["kind"] == "step":
        return 1
    if case["method"] in CONSTANT:
        return 64
    return max(4, int(RATE[problem] * case["tf"]))


def _attempt_flops(method, term, n):
    modes = n // 2 + 1 if term == "advect" else n
    fft = (7.5 if term == "advect" else 10.0) * n * math.log2(n)
    return STAGES[method] * fft + 8.0 * TERMS[method] * modes


def work(case):
    kind = case["kind"]
    e = 8 if case.get("precision") == "f32" else 16
    if kind in ("step", "single", "callable"):
        problem = case.get("problem", "ks")
        term = "cubic" if problem == "nls" else "advect"
        m = case["n"] if term == "cubic" else case["n"] // 2 + 1
        snaps = _attempts(case, problem) // case["store"] if case.get("store") else 0
        return dict(bytes=m * (2 * e + 16 + snaps * e),
                    flops=_attempts(case, problem) * _attempt_flops(case["method"], term, case["n"]))
    if kind == "ensemble":
        sizes, term = (KS_SIZES, "advect") if case["problem"] == "ks" else (NLS_SIZES, "cubic")
        modes = [n if term == "cubic" else n // 2 + 1 for n in sizes]
        return dict(bytes=case["count"] * sum(modes) / len(modes) * (2 * e + 16),
                    flops=case["count"] * _attempts(case, case["problem"])
                    * sum(_attempt_flops(case["method"], term, n) for n in sizes) / len(sizes))
    if kind == "ac2d":
        n, m = case["n"], case["n"] * (case["n"] // 2 + 1)
        f = STAGES[case["method"]] * 10.0 * n * n * math.log2(n) + 8.0 * TERMS[case["method"]] * m
        return dict(bytes=m * (case["count"] * 2 * e + 8), flops=case["count"] * _attempts(case, "ac2d") * f)
    if kind == "radial":
        n = case["n"]
        f = STAGES[case["method"]] * 8.0 * n * n + 8.0 * TERMS[case["method"]] * n
        return dict(bytes=16 * n * 3 * case["count"] + 8 * n * n, flops=case["count"] * _attempts(case, "radial") * f)
    if kind == "hankel":
        n, w = case["n"], 2 if case["complex"] else 1
        return dict(bytes=8 * n * n + 16 * w * n * case["count"], flops=2.0 * w * n * n * case["count"])
    n = case["n"] - 1
    return dict(bytes=16 * n * n + 32 * n, flops=_attempts(case, "cheb") * TERMS[case["method"]] * 8.0 * n * n)


# ---------------------------------------------------------------------------
# exact: the same schemes and step control in plain NumPy, 64 bits
# ---------------------------------------------------------------------------
def _psi(z):
    e = np.exp(z)
    return (e - 1) / z, 2 * (e - 1 - z) / z**2, 6 * (e - 1 - z - z**2 / 2) / z**3


def _psi_of(z, f, h):
    """h psi_1..3 of f z for a vector z: closed forms, contour means where |z| < 0.01."""
    out = [np.zeros(z.shape, dtype=np.complex128) for _ in range(3)]
    small = np.abs(z) < 0.01
    for o, v in zip(out, _psi(f * z[~small])):
        o[~small] = h * v
    nodes = np.exp(2j * np.pi * (np.arange(32) + 0.5) / 32)
    for o, v in zip(out, _psi(f * (z[small][:, None] + nodes))):
        o[small] = h * v.mean(axis=1)
    return out


def _psi_dense(z, f, h, points=64, radius=20.0):
    """h psi_1..3 of f z for a matrix z, by the contour integral."""
    r = radius * np.exp(2j * np.pi * (np.arange(points) + 0.5) / points)
    inv = np.linalg.inv(r[:, None, None] * np.eye(z.shape[0]) - f * z)
    return [h * np.tensordot(r * p, inv, axes=1) / points for p in _psi(r)]


class _Scheme:
    """One method on a diagonal (1-D) or dense (2-D) L: attempt(u, h, NL1) -> (u_new, err, NL_last)."""

    def __init__(self, method, L, nl):
        self.method, self.nl, self.L = method, nl, np.asarray(L, dtype=np.complex128)
        self.dense = self.L.ndim == 2
        self.h = None

    def _coef(self, h):
        z = h * self.L
        if self.dense:
            exp, psi, self.mul = (lambda f: torch.linalg.matrix_exp(torch.as_tensor(f * z)).numpy(),
                                  lambda f: _psi_dense(z, f, h), np.matmul)
        else:
            exp, psi, self.mul = lambda f: np.exp(f * z), lambda f: _psi_of(z, f, h), np.multiply
        if self.method in ("IF34", "IF4"):
            self.c = exp(0.5), exp(1.0)
        elif self.method in ("ETD34", "ETD4"):
            (p, q, _), (a, b, c) = psi(0.5), psi(1.0)
            self.c = (exp(0.5), exp(1.0), 0.5 * p, 0.5 * (p - q), 0.5 * q, a - b, b,
                      a - 1.5 * b + 2 / 3 * c, b - 2 / 3 * c, -0.5 * b + 2 / 3 * c)
        else:
            (p1, p2, _), (q1, q2, _), (r1, r2, _), (a, b, c) = psi(0.25), psi(0.5), psi(0.75), psi(1.0)
            self.c = (exp(0.25), exp(0.5), exp(0.75), exp(1.0), p1 / 4, (p1 - p2 / 2) / 4, p2 / 8, (q1 - q2) / 2, q2 / 2,
                      0.75 * (r1 - 0.75 * r2), -0.375 * r1, 9 / 16 * r2, (-77 * a + 59 * b) / 42, 8 / 7 * a,
                      (111 * a - 87 * b) / 28, (-47 * a + 143 * b) / 84, 7 * (257 * a - 497 * b + 270 * c) / 2700,
                      (1097 * a - 467 * b - 150 * c) / 1350, 2 * (-49 * a + 199 * b - 135 * c) / 225,
                      (-313 * a + 883 * b - 90 * c) / 1350, (509 * a - 2129 * b + 1830 * c) / 2700)

    def attempt(self, u, h, N1):
        if h != self.h:
            self._coef(h)
            self.h = h
        m, nl = self.mul, self.nl
        if self.method in ("IF34", "IF4"):
            E2, E = self.c
            N2 = nl(m(E2, u + h / 2 * N1))
            N3 = nl(m(E2, u) + h / 2 * N2)
            N4 = nl(m(E, u) + h * m(E2, N3))
            k = m(E, u + h / 6 * N1) + h / 3 * m(E2, N2 + N3) + h / 6 * N4
            N5 = nl(k)
            return k, h * (N4 - N5) / 6, N5
        if self.method in ("ETD34", "ETD4"):
            E2, E, a21, a31, a32, a41, a43, a51, a52, a54 = self.c
            N2 = nl(m(E2, u) + m(a21, N1))
            N3 = nl(m(E2, u) + m(a31, N1) + m(a32, N2))
            N4 = nl(m(E, u) + m(a41, N1) + m(a43, N3))
            k = m(E, u) + m(a51, N1) + m(a52, N2 + N3) + m(a54, N4)
            N5 = nl(k)
            return k, m(a54, N4 - N5), N5
        (E14, E12, E34, E, a21, a31, a32, a41, a43, a51, a52, a54, a61, a62, a63, a65, a71, a73, a74, a75, a76) = self.c
        N2 = nl(m(E14, u) + m(a21, N1))
        N3 = nl(m(E14, u) + m(a31, N1) + m(a32, N2))
        N4 = nl(m(E12, u) + m(a41, N1) + m(a43, N3))
        N5 = nl(m(E34, u) + m(a51, N1) + m(a52, N2 - N3) + m(a54, N4))
        N6 = nl(m(E, u) + m(a61, N1) + m(a62, N2 - 1.5 * N4) + m(a63, N3) + m(a65, N5))
        k = m(E, u) + m(a71, N1) + m(a73, N3) + m(a74, N4) + m(a75, N5) + m(a76, N6)
        return k, m(a75, -N1 + 4 * N3 - 6 * N4 + 4 * N5 - N6), None

    def accepted(self, u, h, N1, eps):
        """The attempts from h down to the first accepted one: (u_new, h, h_next, NL1 of the next step)."""
        while True:
            k, err, last = self.attempt(u, h, N1)
            on = np.abs(k) > 0.01 * np.abs(k).max()
            s = 0.8 * (eps * np.linalg.norm(k[on]) / np.linalg.norm(err[on])) ** 0.25
            if np.isfinite(s) and s >= 1.0:
                return k, h, min(s, 4.0) * h if min(s, 4.0) > 1.25 else h, self.nl(k) if last is None else last
            h *= min(max(s, 0.25), 0.85) if np.isfinite(s) else 0.25

    def evolve(self, u, tf, eps, store=0):
        ts, us, t, steps, N1 = [0.0], [u], 0.0, 0, self.nl(u)
        h = _fixed_step(dict(tf=tf)) if self.method in CONSTANT else tf / 100
        while t < tf:
            if self.method in CONSTANT:
                u, _, last = self.attempt(u, h, N1)
                hn, N1 = h, self.nl(u) if last is None else last
            else:
                u, h, hn, N1 = self.accepted(u, h, N1, eps)
            t, steps = t + h, steps + 1
            if self.method not in CONSTANT:
                h = tf - t if t + hn > tf else hn
            if store and steps % store == 0:
                ts.append(t)
                us.append(u)
        return u, np.array(ts), np.stack(us)


def _nl64(term, kx, coef):
    if term == "cubic":
        def nl(u):
            v = np.fft.ifft(u)
            return 1j * coef * np.fft.fft((v.real**2 + v.imag**2) * v)
    else:
        n = 2 * (len(kx) - 1)

        def nl(u):
            return coef * np.fft.rfft(np.fft.irfft(u, n=n) * np.fft.irfft(1j * kx * u, n=n))
    return nl


def _bessel(x):
    """J0 and J1: Bessel's integral below 20 (the trapezoid rule is exact to rounding), torch's above."""
    t = torch.as_tensor(x)
    j0, j1 = torch.special.bessel_j0(t).numpy(), torch.special.bessel_j1(t).numpy()
    low = x < 20.0
    th = 2 * np.pi * np.arange(80) / 80
    arg = np.sin(th) * x[low][:, None]
    j0[low], j1[low] = np.cos(arg).mean(axis=1), np.cos(th - arg).mean(axis=1)
    return j0, j1


def _hankel64(n, rmax=5.0):
    """r, kr, Y and S of the order-zero quasi-discrete Hankel transform."""
    z = np.pi * (np.arange(1, n + 2) - 0.25)
    z = z + 1 / (8 * z)
    for _ in range(4):
        j0, j1 = _bessel(z)
        z = z + j0 / j1
    z, top = z[:-1], z[-1]
    Y = 2 * _bessel(np.outer(z, z) / top)[0] / (top * _bessel(z)[1] ** 2)
    return rmax * z / top, z / rmax, Y, rmax**2 / top


def exact(case, seed):
    kind, rng = case["kind"], np.random.default_rng(seed)
    if kind in ("step", "single"):
        if case["method"] == "IF45DP":
            return None
        term, kx, coef, L, u0 = _problem(case["problem"], case["n"], rng)
        s = _Scheme(case["method"], L, _nl64(term, kx, coef))
        if kind == "step":
            if case["method"] in CONSTANT:
                return [s.attempt(u0, case["h"], s.nl(u0))[0]]
            return list(s.accepted(u0, case["h"], s.nl(u0), 1e-4)[:2])
        u, t, us = s.evolve(u0, case["tf"], case["eps"], case["store"])
        return {"u": u, "t": t, "snapshots": us} if case["store"] else {"u": u}
    if kind == "hankel":
        _, _, Y, S = _hankel64(case["n"])
        return _profiles(case, seed) @ (Y.T / S if case["inverse"] else S * Y.T)
    if kind == "callable":
        kx, _, L, u0 = _ks_field(case["n"], rng)
        return {"u": _Scheme(case["method"], L, _nl64("advect", kx, -1.0)).evolve(u0, case["tf"], case["eps"])[0]}
    if kind == "cheb":
        n = case["n"]
        x = -np.cos(np.pi * np.arange(n + 1) / n)
        c = np.where((np.arange(n + 1) % n) == 0, 2.0, 1.0) * (-1.0) ** np.arange(n + 1)
        dx = x[:, None] - x[None, :] + np.eye(n + 1)
        D = np.outer(c, 1 / c) / dx
        D -= np.diag(D.sum(axis=1))
        L, xi = (0.01 * D @ D + np.eye(n + 1))[1:-1, 1:-1], x[1:-1]
        s = _Scheme(case["method"], L, lambda w: xi - (w + xi) ** 3)
        return {"u": s.evolve(_cheb_state(x, rng), case["tf"], case["eps"])[0]}
    if kind == "ac2d":
        n = case["n"]
        L, keep = _ac2d_op(n)

        def nl(u):
            w = np.fft.irfft2(u.reshape(keep.shape), s=(n, n))
            return np.fft.rfft2(w - w**3).reshape(-1)
        u0s, make = [(np.fft.rfft2(_ac2d_field(n, seed, 0)) * keep).reshape(-1)], lambda: (L.reshape(-1), nl)
        ops = [make()]
    elif kind == "radial":
        r, kr, Y, S = _hankel64(case["n"])

        def nl(u):
            f = Y @ u / S
            return 2j * (S * (Y @ ((f.real**2 + f.imag**2) * f)))
        u0s = [S * (Y @ b) for b in _beams(r, min(CHECKED, case["count"]), seed)]
        ops = [(-1j * kr**2, nl)] * len(u0s)
    else:
        ens = [_member(case["problem"], rng, i) for i in range(min(CHECKED, case["count"]))]
        u0s, ops = [e[4] for e in ens], [(e[3], _nl64(*e[:3])) for e in ens]
    done = [_Scheme(case["method"], L, nl).evolve(u0, case["tf"], case["eps"])[0] for (L, nl), u0 in zip(ops, u0s)]
    return {"first": np.concatenate(done), "rest": None}
