"""Dense systems on both sides of the size whose matrices fit LDS, and stage sums of every number
of terms.  Tolerances: coefficients as in test_gpu_dense.py; a sum of n products rounds to at
most about n eps of the sum of their absolute values."""
import numpy as np
import pytest

from oracle import solvers

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu
EPS = np.finfo(np.float64).eps


@pytest.mark.parametrize("n", [1, 2, 16, 39, 40, 41])
@pytest.mark.parametrize("method", ["ETD35", "IF34"])
def test_dense_coefficients_at_the_lds_limit(n, method):
    from tableau_interp import dense_coefficients
    from rkstiff_amd import _lib, dense
    rng = np.random.default_rng(n)
    L = -(np.diag(np.arange(1.0, n + 1.0)) + 0.3 * rng.standard_normal((n, n))).astype(np.complex128)
    etd = solvers.ETDConfig()
    t = _lib.tableau(method)
    hs = [0.03, 0.2]
    got = dense.coefficients(method, torch.as_tensor(np.stack([L, 0.5 * L])).cuda(), hs, etd).cpu().numpy()
    for b, (A, h) in enumerate(zip((L, 0.5 * L), hs)):
        ref = dense_coefficients(t, A, h, etd)
        top = max(np.max(np.abs(r)) for r in ref)
        for c in range(t.ncoef):
            err = np.max(np.abs(got[b, c] - ref[c])) / (np.max(np.abs(ref[c])) + 1e-2 * top)
            assert err < 1e-12, (c, err)


@pytest.mark.parametrize("n", [1, 19, 256])
def test_dense_combine_all_terms(n):
    from rkstiff_amd import dense
    rng = np.random.default_rng(n)

    def rc(*s):
        return rng.standard_normal(s) + 1j * rng.standard_normal(s)
    B = 2
    host = [(rc(B, n, n) if k % 3 else None, rc(B, n), rc(B, n) if k % 2 else None, 0.5 - k, 0.25 * k - 1) for k in range(8)]
    dev = [tuple(torch.as_tensor(v).cuda() if isinstance(v, np.ndarray) else v for v in t) for t in host]
    got = dense.combine(dev, torch.empty((B, n), dtype=torch.complex128, device="cuda")).cpu().numpy()
    want, size = np.zeros((B, n), complex), np.zeros((B, n))
    for m, x, x2, s2, a in host:
        v = x + (s2 * x2 if x2 is not None else 0)
        av = np.abs(x) + (abs(s2) * np.abs(x2) if x2 is not None else 0)
        want += a * (v if m is None else np.einsum("bij,bj->bi", m, v))
        size += abs(a) * (av if m is None else np.einsum("bij,bj->bi", np.abs(m), av))
    assert np.all(np.abs(got - want) <= 8 * (n + 16) * EPS * size)
