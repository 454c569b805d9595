"""Coefficient updates of small and large dense systems from two threads at once."""
import threading

import numpy as np
import pytest

from oracle import solvers

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def test_dense_coefficients_of_two_sizes_from_two_threads():
    from rkstiff_amd import dense
    etd, hs = solvers.ETDConfig(), [0.03, 0.2]
    ops = {}
    for n in (4, 40):
        L = -(np.diag(np.arange(1.0, n + 1.0)) + 0.3 * np.random.default_rng(n).standard_normal((n, n)))
        ops[n] = torch.as_tensor(np.stack([L, 0.5 * L]).astype(np.complex128)).cuda()
    alone = {n: dense.coefficients("ETD35", L, hs, etd).cpu() for n, L in ops.items()}
    wrong = []

    def run(n):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                for _ in range(20):
                    if not torch.equal(dense.coefficients("ETD35", ops[n], hs, etd).cpu(), alone[n]):
                        wrong.append(n)
        except Exception as e:
            wrong.append((n, str(e)))
    torch.cuda.synchronize()
    threads = [threading.Thread(target=run, args=(n,)) for n in ops]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
