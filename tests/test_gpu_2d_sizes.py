"""Short evolves of the 2-D engine at every grid size, for a method of each kind: compiled in
with a recomputed NL1 (ETD35), compiled in with NL1 from a slot (IF34), tableau from memory
(ETD34).  Bounds of test_gpu_2d.py (FP64), and of its single evaluation times the attempts
(FP32)."""
import numpy as np
import pytest

from oracle import problems, solvers

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("method", ["ETD35", "IF34", "ETD34"])
@pytest.mark.parametrize("n", [32, 64, 128, 256, 512])
def test_ac2d_evolve_every_size(method, n):
    import rkstiff_amd as rk
    print(f"ac2d evolve {method} n={n}", flush=True)
    p = problems.allen_cahn_2d(n, n, eps=0.01, kcut=n / 8, seed=n, batch=2)
    u0 = [p["u0"][i] * 20.0 for i in range(2)]
    L, nl = rk.allen_cahn_ops(n)
    tfs = [0.2, 0.3]
    for prec, dtype, tol in (("f64", torch.complex128, 1e-11), ("f32", torch.complex64, 1e-4)):
        b = rk.batch.BatchSolver(method, [(L, nl)] * 2, precision=prec, config=rk.SolverConfig(epsilon=1e-5))
        uf = b.evolve([torch.as_tensor(u).to(dtype).cuda() for u in u0], 0.0, tfs, h=[0.02, 0.05])
        for i in range(2):
            drv = solvers.make_solver(method, p["L"], p["nl"], solvers.SolverConfig(epsilon=1e-5))
            ref = drv.evolve(u0[i], t0=0.0, tf=tfs[i], h_init=[0.02, 0.05][i], store_data=False)
            assert solvers.rel_l2(uf[i].cpu().numpy().astype(np.complex128), ref) < tol
            if prec == "f64":
                assert b.stats()[i]["attempts"] == len(drv.log)
