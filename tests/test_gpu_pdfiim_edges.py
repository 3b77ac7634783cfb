"""PDFIIM construction on the GPU where its device transposes could go wrong:
one row, two rows, a column and a row that every row shares, and columns that
must be refused before anything is indexed by them.  The host producer's
factors bit for bit."""
import numpy as np
import pytest

import cmamd

pytestmark = pytest.mark.gpu


def _same(a, b):
    for m, k in ((a.G, b.G), (a.H, b.H)):
        assert np.array_equal(m.ptr, k.ptr) and np.array_equal(m.idx, k.idx)
        assert m.val.tobytes() == k.val.tobytes()
    assert a.idv.tobytes() == b.idv.tobytes()


def _arrow(n, seed):
    """Tridiagonal plus a full last column and row."""
    import scipy.sparse as sp
    rng = np.random.default_rng(seed)
    m = sp.diags([rng.uniform(-1, 0, n - 1), np.full(n, 6.0), rng.uniform(-1, 0, n - 1)], [-1, 0, 1]).tolil()
    m[:, n - 1] = rng.uniform(-0.1, 0.1, (n, 1))
    m[n - 1, :] = rng.uniform(-0.1, 0.1, (1, n))
    m[n - 1, n - 1] = 6.0
    return cmamd.Csr.from_scipy(m.tocsr())


@pytest.mark.parametrize("n", [1, 2, 3])
def test_tiny(n):
    import scipy.sparse as sp
    A = cmamd.Csr.from_scipy(sp.csr_matrix(np.tri(n, n, 1) * np.triu(np.ones((n, n)), -1) + 3 * np.eye(n)))
    Fd, _ = cmamd.pdfiim_device(A, 1, 1, 1, 0.0)
    _same(Fd, cmamd.pdfiim(A, 1, 1, 1, 0.0))


def test_arrow():
    A = _arrow(200, 3)
    Fd, _ = cmamd.pdfiim_device(A, 1, 1, 1, 0.0)
    _same(Fd, cmamd.pdfiim(A, 1, 1, 1, 0.0))


@pytest.mark.parametrize("col", [-1, 50, 2 ** 30])
def test_columns_out_of_range_are_refused(col):
    A = cmamd.gen_convdiff(2, 7, 1.0, seed=1)
    idx = A.idx.copy()
    idx[len(idx) // 2] = col
    with pytest.raises(cmamd.EngineError, match="out of range"):
        cmamd.pdfiim_device(cmamd.Csr(A.n, A.ptr, idx, A.val), 1, 1, 1, 0.0)
