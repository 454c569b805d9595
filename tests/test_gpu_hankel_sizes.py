"""Hankel products at the edges of the kernels' row, column and vector tiles.  Tolerance: a sum
of n products rounds to at most about n eps of the sum of their absolute values, in any
order."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu
EPS = np.finfo(np.float64).eps


def rel(a, b):
    return float(np.linalg.norm(np.asarray(a) - np.asarray(b)) / np.linalg.norm(np.asarray(b)))


@pytest.mark.parametrize("nr", [4, 15, 16, 17, 63, 65, 251])
@pytest.mark.parametrize("batch", [1, 16, 17, 33, 1100])
@pytest.mark.parametrize("cplx", [False, True])
def test_hankel_products_at_tile_edges(nr, batch, cplx):
    from rkstiff_amd.transforms import HankelTransform
    ht = HankelTransform(nr, 5.0)
    Y = ht.hankel_matrix().numpy()
    rng = np.random.default_rng(nr + batch)
    f = rng.standard_normal((batch, nr))
    if cplx:
        f = f + 1j * rng.standard_normal((batch, nr))
    ft = torch.as_tensor(f).cuda()
    S = float(ht._scalefactor())
    for got, c in ((ht.ht(ft), S), (ht.iht(ft), 1.0 / S)):
        bound = 4 * (nr + 8) * EPS * abs(c) * (np.abs(f) @ np.abs(Y).T)
        assert np.all(np.abs(got.cpu().numpy() - c * (f @ Y.T)) <= bound)


@pytest.mark.parametrize("nr", [17, 100, 251])
@pytest.mark.parametrize("cplx", [False, True])
def test_hankel_products_do_not_depend_on_the_batch(nr, cplx):
    """A profile transformed alone and among others: the same bits, whichever row tile runs."""
    from rkstiff_amd.transforms import HankelTransform
    ht = HankelTransform(nr, 5.0)
    rng = np.random.default_rng(nr)
    f = rng.standard_normal((6000, nr))
    if cplx:
        f = f + 1j * rng.standard_normal(f.shape)
    ft = torch.as_tensor(f).cuda()
    for op in (ht.ht, ht.iht) + ((ht.cubic_nl(2.0),) if cplx else ()):
        many = op(ft) if op in (ht.ht, ht.iht) else torch.stack([op(x) for x in ft[:40]])
        for i in (0, 15, 16, 39):
            assert torch.equal(op(ft[i]), many[i])
