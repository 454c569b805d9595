"""Every tile that a plan runs on can be chosen by its caller, and tuning starts from the plan's own."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _plan(kind, n, prec="f64", count=1, method="ETD35"):
    from rkstiff_amd import _lib
    from rkstiff_amd.engine import Plan
    from rkstiff_amd.nonlinear import AdvectiveNL, CubicNL
    if kind == "advect":
        kx = 2 * np.pi * np.fft.rfftfreq(n, d=32 * np.pi / n)
        nl, L = AdvectiveNL(torch.as_tensor(kx), -1.0), kx**2 * (1 - kx**2)
    else:
        nl, L = CubicNL(n, 1.0), -0.5j * (2 * np.pi * np.fft.fftfreq(n, d=32.0 / n)) ** 2
    P = {"f64": _lib.F64, "f32": _lib.F32, "mixed": _lib.MIXED}[prec]
    return Plan(method, nl, P, None, None, [nl.descriptor(torch.as_tensor(L))] * count)


# widest tile of a plan without / with the proposer variant
WIDEST = {("cubic", 256): (0, 0), ("cubic", 512): (1, 1), ("cubic", 1024): (2, 1), ("cubic", 2048): (2, 1),
          ("cubic", 4096): (1, 1), ("cubic", 8192): (1, 0), ("advect", 256): (0, 0), ("advect", 512): (1, 1),
          ("advect", 1024): (2, 1), ("advect", 2048): (1, 1), ("advect", 4096): (1, 1), ("advect", 8192): (0, 0)}


@pytest.mark.parametrize("kind,n", sorted(WIDEST))
@pytest.mark.parametrize("prec", ["f64", "f32"])
def test_set_launch_takes_every_tile_of_the_plan(kind, n, prec):
    plan = _plan(kind, n, prec)
    own = plan.tiles()
    plan.set_launch(True, None, own)
    plan.set_launch(True, None, [-1])
    assert plan.tiles() == own
    for records, widest in zip((0, 4), WIDEST[kind, n]):
        plan.set_records(records)
        for tile in range(widest + 1):
            plan.set_launch(True, None, [tile])
            assert plan.tiles() == [tile]
        for tile in (-2, widest + 1):
            with pytest.raises(ValueError):
                plan.set_launch(True, None, [tile])
    # a chosen tile without a proposer variant gives way to the base tile while records are on
    plan.set_records(0)
    plan.set_launch(True, None, [WIDEST[kind, n][0]])
    plan.set_records(4)
    assert plan.tiles() == [WIDEST[kind, n][0] if WIDEST[kind, n][0] == WIDEST[kind, n][1] else 0]


def test_tuning_starts_from_the_plans_own_tiles():
    from rkstiff_amd.autotune import tune_launch, tune_together
    plan = _plan("cubic", 1024, count=8)
    own = plan.tiles()
    assert own == [2]
    x = -16.0 + np.arange(1024) * (32.0 / 1024)
    u0 = [torch.as_tensor(np.fft.fft(1.5 / np.cosh(1.5 * (x - 0.1 * i)))).cuda() for i in range(8)]
    info = tune_launch(plan, u0, 0.0, 0.05, 0.001)
    plan.set_launch(info["concurrent"], info["wg_per_cu"], info["tile"])
    plan.set_launch(True, None, info["trials"][0]["tile"])
    assert plan.tiles() == own
    joint = tune_together([(plan, u0, 0.0, 0.05, 0.001, torch.cuda.current_stream())], uniform=True)
    shapes = []
    for t in joint["trials"]:
        plan.set_launch(True, None, t["tiles"][0])
        shapes.append(plan.tiles())
    assert shapes[0] == own and [0] in shapes and [1] in shapes
    plan.set_launch(True, None, joint["tiles"][0])


@pytest.mark.parametrize("kind,n", [("advect", 1024), ("cubic", 8192)])
def test_result_does_not_depend_on_the_rest_of_the_plan(kind, n):
    """A trajectory alone, among 299 like it, and beside one whose last modes are not damped (and
    that one alone): the same bits, in any order of the bucket."""
    from rkstiff_amd import _lib
    from rkstiff_amd.engine import Plan
    from rkstiff_amd.nonlinear import AdvectiveNL, CubicNL
    if kind == "advect":
        x, k = np.arange(n) * (32 * np.pi / n), 2 * np.pi * np.fft.rfftfreq(n, d=32 * np.pi / n)
        nl, u, tf = AdvectiveNL(torch.as_tensor(k), -1.0), np.fft.rfft(np.cos(x / 16) * (1 + np.sin(x / 16))), 2.0
        ops = [k**2 * (1 - k**2), -0.05 * k**2]
    else:
        x, k = -16.0 + np.arange(n) * (32.0 / n), 2 * np.pi * np.fft.fftfreq(n, d=32.0 / n)
        nl, u, tf = CubicNL(n, 1.0), np.fft.fft(1.5 / np.cosh(1.5 * x)), 0.05
        ops = [-0.5j * k**2, -0.4j * k**2]
    ut = torch.as_tensor(u).cuda()

    def run(which, cost=None):
        plan = Plan("ETD35", nl, _lib.F64, None, None, [nl.descriptor(torch.as_tensor(ops[w])) for w in which])
        if cost is not None:
            plan.set_priority(cost)
        uf, m = [torch.empty_like(ut) for _ in which], len(which)
        plan.evolve([ut] * m, uf, [0.0] * m, [tf] * m, [tf / 50] * m)
        assert all(s["status"] == _lib.RKS_OK for s in plan.stats())
        return uf, plan.tiles()

    (a,), own = run([0])
    (b,), other = run([1])
    print(kind, n, "tiles", own, other, flush=True)
    many, tiles = run([0] * 300)
    assert tiles == own and all(torch.equal(x, a) for x in many)
    which = [0, 1] * 150
    for cost in (None, np.arange(300.0)):
        mixed, tiles = run(which, cost)
        assert tiles == own
        assert all(torch.equal(x, b if w else a) for x, w in zip(mixed, which))


@pytest.mark.parametrize("kind,n", [("advect", 1024), ("cubic", 2048)])
def test_logged_run_on_the_same_tile_has_the_same_bits(kind, n):
    from rkstiff_amd import _lib
    plan = _plan(kind, n)
    x = np.arange(n) / n
    u = np.fft.fft(np.exp(-200 * (x - 0.5) ** 2)) if kind == "cubic" else np.fft.rfft(np.cos(2 * np.pi * x))
    ut = torch.as_tensor(u).cuda()
    uf = [torch.empty_like(ut) for _ in range(2)]
    own = plan.tiles()
    for out, log in zip(uf, (0, 64)):
        if log:
            plan.set_launch(tile=own)
            plan.set_storage(0, 0, log)
        assert plan.tiles() == own
        plan.evolve([ut], [out], [0.0], [0.2], [0.02])
        assert plan.stats()[0]["status"] == _lib.RKS_OK
    assert torch.equal(uf[0], uf[1])
