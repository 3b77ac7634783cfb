"""Triangular solves by the rows of a level: few of them (chunks of two rows up
to chunks of 64).  Against the oracle's sequential
solves, each row a sum of four products with diagonals that dominate: 1e-12
normwise."""
import numpy as np
import pytest
import scipy.sparse as sp

import cmamd
import oracle

pytestmark = pytest.mark.gpu


def _levels(n, w, lower, rng):
    """Levels of w rows: a row reads the one above it and two others of the
    level before."""
    i = np.arange(n)
    deep = i >= w
    rows, cols = [i], [i]
    for k in range(3):
        c = i - w if k == 0 else (i // w - 1) * w + rng.integers(0, w, n)
        rows.append(i[deep])
        cols.append(c[deep])
    r, c = np.concatenate(rows), np.concatenate(cols)
    v = np.where(r == c, 1.0 + (r % 7) / 8, rng.uniform(-0.2, 0.2, len(r)))
    m = sp.csr_matrix((v, (r, c)), shape=(n, n))
    if not lower:
        m = m[::-1, ::-1].tocsr()
    m.sort_indices()
    return cmamd.Csr.from_scipy(m)


def _check(n, w):
    rng = np.random.default_rng(n + w)
    L, U = _levels(n, w, True, rng), _levels(n, w, False, rng)
    I = cmamd.Csr(n, np.arange(n + 1, dtype=np.int32), np.arange(n, dtype=np.int32), np.ones(n))
    d, v = rng.uniform(0.5, 2.0, n), rng.uniform(-1, 1, n)
    for mode in "IJ":
        print(f"levels of {w} rows, n={n}, mode {mode}", flush=True)
        s = cmamd.System("acifim", I, cmamd.Factors(I, d, I, L, U), mode=mode)
        z = oracle.trsv(L, v, lower=True)
        z = oracle.trsv(U, z * d if mode == "I" else z, lower=False)
        for _ in range(2):
            assert np.linalg.norm(s.apply(v) - z) <= 1e-12 * np.linalg.norm(z)
        s.close()


@pytest.mark.parametrize("n,w", [(20000, 1), (3000, 2), (3001, 3), (3000, 5), (3000, 9), (4000, 17), (5000, 40)])
def test_levels_of_few_rows(n, w):
    _check(n, w)
