"""Batches whose trajectories have real and complex lin_ops: each reads its own kind.  The bound
is the suite's for two runs of one trajectory by different FP64 kernels (test_gpu_engine.py)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def rel(a, b):
    return float(torch.linalg.norm(a - b) / torch.linalg.norm(b))


def _problems(kind):
    """(lin_op, term, u0) of two or three trajectories, the real lin_op last."""
    from rkstiff_amd.nonlinear import AdvectiveNL, CubicNL
    from rkstiff_amd.transforms import HankelTransform
    out = []
    if kind == "hankel":
        ht = HankelTransform(nr=60, rmax=4.0)
        u0 = ht.ht(torch.exp(-(ht.r / 0.9) ** 2).to(torch.complex128))
        for L in (-1j * ht.kr**2, -0.5 * ht.kr**2):
            out.append((L, ht.cubic_nl(2.0), u0))
        return out
    for n in (64, 512, 64):
        x = -16.0 + np.arange(n) * (32.0 / n)
        if kind == "cubic":
            k = 2 * np.pi * np.fft.fftfreq(n, d=32.0 / n)
            nl, u0 = CubicNL(n, 1.0), np.fft.fft(1.2 / np.cosh(1.2 * x) * np.exp(0.3j * x))
            L = -0.5j * k**2
        else:
            k = 2 * np.pi * np.fft.rfftfreq(n, d=32.0 / n)
            nl, u0 = AdvectiveNL(torch.as_tensor(k), -6.0), np.fft.rfft(0.5 / np.cosh(x / 2) ** 2)
            L = 1j * k**3
        out.append((torch.as_tensor(L), nl, torch.as_tensor(u0).cuda()))
    L, nl, u0 = out[-1]
    out[-1] = (torch.as_tensor(-0.1 * k**2), nl, u0)
    return out


@pytest.mark.parametrize("kind", ["cubic", "hankel", "advect"])
@pytest.mark.parametrize("method", ["ETD35", "IF34"])
def test_real_and_complex_lin_ops_in_one_batch(kind, method):
    from rkstiff_amd.batch import BatchSolver
    from rkstiff_amd.config import SolverConfig
    probs = _problems(kind)

    def run(ps):
        bs = BatchSolver(method, [(L, nl) for L, nl, _ in ps], config=SolverConfig(epsilon=1e-5))
        out = bs.evolve([u0 for *_, u0 in ps], 0.0, 0.2)
        assert not bs.failures()
        return out, [s["attempts"] for s in bs.stats()]

    print(kind, method, flush=True)
    together, attempts = run(probs)
    for i, p in enumerate(probs):
        alone, (a,) = run([p])
        assert attempts[i] == a
        assert rel(together[i], alone[0]) < 1e-11
