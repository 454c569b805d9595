"""Whole runs on every FFT tile against the oracle: the compiled and the general kernels, with
rejected attempts, kept and changed steps.  Bound: a run on another tile (test_gpu_tiles.py)."""
import numpy as np
import pytest

from oracle import problems, solvers
from test_gpu_tile_choice import WIDEST

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _problem(kind, n):
    if kind == "advect":
        x, kx = np.arange(n) * (32 * np.pi / n), 2 * np.pi * np.fft.rfftfreq(n, d=32 * np.pi / n)
        return kx, kx**2 * (1 - kx**2), problems.rfft_advect_nl(kx, -1.0), np.fft.rfft(np.cos(x / 16) * (1 + np.sin(x / 16)))
    x, k = -16.0 + np.arange(n) * (32.0 / n), 2 * np.pi * np.fft.fftfreq(n, d=32.0 / n)
    u = 1.5 / np.cosh(1.5 * x) * np.exp(1j * x) + 1.2 / np.cosh(1.2 * (x - 6))
    return k, -0.5j * k**2, problems.nls_nl(1.0), np.fft.fft(u)


@pytest.mark.parametrize("method", ["ETD35", "IF34", "ETD34", "ETD5", "IF4"])
@pytest.mark.parametrize("kind,n", sorted(k for k in WIDEST if k[1] >= 512))
def test_runs_on_every_tile_match_the_oracle(kind, n, method):
    from rkstiff_amd import _lib
    from rkstiff_amd.config import SolverConfig
    from rkstiff_amd.engine import Plan
    from rkstiff_amd.nonlinear import AdvectiveNL, CubicNL
    k, L, f, u0 = _problem(kind, n)
    nl = AdvectiveNL(torch.as_tensor(k), -1.0) if kind == "advect" else CubicNL(n, 1.0)
    drv = solvers.make_solver(method, L, f, solvers.SolverConfig(epsilon=1e-5))
    adaptive = method in ("ETD35", "IF34", "ETD34")
    tf, h = (3.0, 1.5) if kind == "advect" else (0.6, 0.3)
    if not adaptive:
        tf, h = 16 * 2.0**-9, 2.0**-9
    ref = drv.evolve(u0, 0.0, tf, h, store_data=False)
    plan = Plan(method, nl, _lib.F64, SolverConfig(epsilon=1e-5), None, [nl.descriptor(torch.as_tensor(L))])
    ut = torch.as_tensor(u0).cuda()
    uf = torch.empty_like(ut)
    for tile in range(WIDEST[kind, n][0] + 1):
        print(kind, n, method, "tile", tile, flush=True)
        plan.set_launch(True, None, [tile])
        plan.evolve([ut], [uf], [0.0], [tf], [h])
        st = plan.stats()[0]
        assert st["status"] == _lib.RKS_OK
        if adaptive:
            assert st["attempts"] == len(drv.log) and st["rejects"] > 0
        else:
            assert st["steps"] == 16
        assert np.linalg.norm(uf.cpu().numpy() - ref) < 1e-10 * np.linalg.norm(ref)
