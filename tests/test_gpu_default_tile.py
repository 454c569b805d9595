"""The FFT tile that a plan chooses by itself: the nonlinear terms of every size at few and many
trajectories, the rule, and whole runs against the base tile (bounds of test_gpu_tiles.py)."""
import numpy as np
import pytest

from oracle import problems

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def rel(a, b):
    return float(np.linalg.norm(np.asarray(a) - np.asarray(b)) / np.linalg.norm(np.asarray(b)))


def _plan(kind, n, prec, count=1, damped=True):
    from rkstiff_amd import _lib
    from rkstiff_amd.engine import Plan
    from rkstiff_amd.nonlinear import AdvectiveNL, CubicNL
    if kind == "advect":
        kx = 2 * np.pi * np.fft.rfftfreq(n, d=32 * np.pi / n)
        nl, L = AdvectiveNL(torch.as_tensor(kx), -1.0), kx**2 * (1 - kx**2) if damped else -0.0005 * kx**2
        ref = problems.rfft_advect_nl(kx, -1.0)
    else:
        nl, L, ref = CubicNL(n, 1.0), -0.5j * np.fft.fftfreq(n, d=1.0 / n) ** 2, problems.nls_nl(1.0)
    P = {"f64": _lib.F64, "f32": _lib.F32, "mixed": _lib.MIXED}[prec]
    return Plan("ETD35", nl, P, None, None, [nl.descriptor(torch.as_tensor(L))] * count), ref


@pytest.mark.parametrize("count", [1, 300])
@pytest.mark.parametrize("kind,n", [(k, 1 << l) for k in ("advect", "cubic") for l in range(8, 14)])
def test_default_tile_nl_matches_oracle(kind, n, count):
    plan, ref = _plan(kind, n, "f64", count)
    print(kind, n, count, "tiles", plan.tiles(), flush=True)
    rng = np.random.default_rng(n)
    m = n // 2 + 1 if kind == "advect" else n
    env = np.exp(-np.minimum(np.arange(m), n - np.arange(m)) / 30.0)
    u = (rng.standard_normal((2, m)) + 1j * rng.standard_normal((2, m))) * env
    if kind == "advect":
        u[:, [0, -1]] = u[:, [0, -1]].real
    ut = [torch.as_tensor(u[i % 2]).cuda() for i in range(count)]
    out = [torch.empty_like(x) for x in ut]
    plan.nl_eval(ut, out)
    for i in {0, 1 % count, count - 1}:
        assert rel(out[i].cpu().numpy(), ref(u[i % 2])) < 1e-13


def test_default_tile_rule():
    """Another tile rounds differently: precisions and runs that show it keep the base tile."""
    for kind, n in (("advect", 1024), ("cubic", 1024), ("cubic", 4096)):
        assert _plan(kind, n, "f64")[0].tiles()[0] > 0
        for prec in ("f32", "mixed"):
            assert _plan(kind, n, prec)[0].tiles() == [0]
    assert _plan("advect", 1024, "f64", damped=False)[0].tiles() == [0]
    plan, _ = _plan("cubic", 1024, "f64")
    plan.set_launch(True, None, [1])
    assert plan.tiles() == [1]
    plan.set_launch(True, None, None)
    plan.set_storage(0, 0, 16)
    assert plan.tiles() == [0]
    plan.set_storage(0, 0, 0)
    plan.set_records(4)
    assert plan.tiles() == [0]
    with pytest.raises(ValueError):
        plan.set_launch(True, None, [2])


@pytest.mark.parametrize("n", [512, 1024, 2048, 4096, 8192])
def test_default_tile_evolve_agrees_with_base_tile(n):
    """A resolved soliton for half a time unit: rounding-level differences only."""
    plan, _ = _plan("cubic", n, "f64", 200)
    x = -16.0 + np.arange(n) * (32.0 / n)
    u0 = [torch.as_tensor(np.fft.fft(1.5 / np.cosh(1.5 * (x - 0.01 * i)))).cuda() for i in range(200)]
    res = []
    for tile in (None, [0]):
        plan.set_launch(True, None, tile)
        uf = [torch.empty_like(u) for u in u0]
        plan.evolve(u0, uf, [0.0] * 200, [1e-3] * 200, [1e-5] * 200)
        res.append(torch.stack(uf).cpu().numpy())
    assert rel(res[0], res[1]) < 1e-11
