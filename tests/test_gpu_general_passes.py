"""One step of every method and precision by the kernels that read their tableau, at the sizes
where their chunks, workgroups and mode pairs change.  FP64 against the oracle; FP32 and MIXED
against it too: a stage sums at most 34 products of numbers rounded to FP32, in at most 7 stages,
each rounding 2^-24 of its term."""
import numpy as np
import pytest

from oracle import problems, solvers

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu
BOUND = {"f64": 1e-12, "f32": 7 * 34 * 2.0**-24, "mixed": 7 * 34 * 2.0**-24}


@pytest.mark.parametrize("method", ["ETD34", "ETD4", "ETD5", "IF4", "IF45DP"])
@pytest.mark.parametrize("n", [16, 64, 512, 1024, 2048, 8192])
@pytest.mark.parametrize("kind", ["cubic", "drift", "advect"])
def test_one_step_of_the_general_kernels(kind, n, method):
    from rkstiff_amd import _lib
    from rkstiff_amd.engine import Plan
    from rkstiff_amd.nonlinear import AdvectiveNL, CubicNL
    if kind == "advect":
        k = np.arange(n // 2 + 1) / 16.0
        x = np.arange(n) * (32 * np.pi / n)
        nl, L, f = AdvectiveNL(torch.as_tensor(k), -1.0), k**2 * (1 - k**2), problems.rfft_advect_nl(k, -1.0)
        u0 = np.fft.rfft(np.cos(x / 16) * (1 + np.sin(x / 16)))
    else:
        x, k = -16.0 + np.arange(n) * (32.0 / n), 2 * np.pi * np.fft.fftfreq(n, d=32.0 / n)
        nl, f = CubicNL(n, 1.0), problems.nls_nl(1.0)
        L = -0.5j * k**2 + (0.3j * k if kind == "drift" else 0)  # drift: mirror modes differ
        u0 = np.fft.fft(0.8 / np.cosh(0.8 * x) * np.exp(0.3j * x))
    h = 2.0**-10
    drv = solvers.make_solver(method, L, f)
    out = drv.step(u0, h)
    ref = out[0] if isinstance(out, tuple) else out
    for prec, bound in BOUND.items():
        P, dt = {"f64": (_lib.F64, torch.complex128), "f32": (_lib.F32, torch.complex64),
                 "mixed": (_lib.MIXED, torch.complex128)}[prec]
        plan = Plan(method, nl, P, None, None, [nl.descriptor(torch.as_tensor(L))])
        ut = torch.as_tensor(u0).to(dt).cuda()
        for tile in (0, None):
            print(kind, n, method, prec, "tile", tile, flush=True)
            plan.set_launch(True, None, None if tile is None else [tile])
            plan.reset()
            un = torch.empty_like(ut)
            plan.step([ut], [un], [h])
            st = plan.stats()[0]
            assert st["status"] == _lib.RKS_OK and st["rejects"] == 0
            assert np.linalg.norm(un.cpu().numpy() - ref) < bound * np.linalg.norm(ref)
