"""The batched solve at the edges of its kernels: one workgroup with 2, 4 or 8
rows per thread (512 threads), the last size the LDS kernel takes (4096 rows)
and the first beyond it, together in one launch; products whose entries fill
several tiles; and more bytes of vectors than the pinned staging takes.  Bars
are the FP64 path's: info equal, pass counts within 2%, x within 1e-7 of the
oracle's (at most 60 passes, over which rounding grows to 1e-10)."""
import numpy as np
import pytest

import cmamd
import oracle

pytestmark = pytest.mark.gpu


def _item(A, F, seed, variant="afiim", tol=1e-8, nmax=500):
    b = cmamd.csr_mv_host(A, cmamd.gen_uniform(seed, A.n))
    xo, rvo, ito, info_o, _ = oracle.bicgstab(variant, A, b, F, tol=tol, nmax=nmax)
    return (cmamd.System(variant, A, F), b, None, tol, nmax), (xo, ito, info_o)


def _check(items, want, **kw):
    print("batch n =", [it[0].n for it in items], flush=True)
    for r, (xo, ito, info_o) in zip(cmamd.batch_solve(items, **kw), want):
        assert r.info == info_o
        assert abs(r.iter - ito) <= max(1, int(np.ceil(0.02 * ito)))
        assert np.linalg.norm(r.x - xo) <= 1e-7 * max(np.linalg.norm(xo), 1e-300)


def test_batch_edges_in_one_launch():
    pairs = []
    for k, N in enumerate((2, 16, 22, 23, 32, 33, 45, 46, 64, 65)):  # 4 .. 4225 rows
        A = cmamd.gen_convdiff(2, N, 1.0, seed=20 + k)
        pairs.append(_item(A, cmamd.afiim(A, 0.1), 40 + k))
    for N in (8, 15, 16, 17):  # 512, 3375, 4096, 4913 rows
        A = cmamd.gen_convdiff(3, N, 2.0, seed=60 + N)
        pairs.append(_item(A, cmamd.acifim(A, 0.01, 0.1), 70 + N, "acifim"))
    _check([p[0] for p in pairs], [p[1] for p in pairs])


def test_batch_long_rows_and_empty_rows():
    import scipy.sparse as sp
    n = 4096
    rng = np.random.default_rng(5)
    m = sp.random(n, n, density=3.0 / n, random_state=np.random.RandomState(5), format="lil")
    for r in (0, 1777, n - 1):  # three rows of 4000 entries: more than one tile
        c = rng.choice(n, size=4000, replace=False)
        m[r, c] = rng.uniform(-1, 1, 4000) / 4000
    m.setdiag(4.0 + rng.uniform(0, 1, n))
    A = cmamd.Csr.from_scipy(m.tocsr())
    I = cmamd.Csr(n, np.arange(n + 1, dtype=np.int32), np.arange(n, dtype=np.int32), np.ones(n))
    none = cmamd.Csr(n, np.r_[np.zeros(n, np.int32), np.int32(1)], np.array([n - 1], np.int32), np.ones(1))
    d = 1.0 / m.tocsr().diagonal()
    a, wa = _item(A, cmamd.Factors(I, d, I), 3)
    # M = e e^T: everything but one component is out of reach, NMAX ends it
    b, wb = _item(A, cmamd.Factors(I, d, none), 3, nmax=7)
    res = cmamd.batch_solve([a, b])
    assert res[0].info == wa[2] == 0 and abs(res[0].iter - wa[1]) <= 1
    assert np.linalg.norm(res[0].x - wa[0]) <= 1e-7 * np.linalg.norm(wa[0])
    assert res[1].info == wb[2] and res[1].iter == wb[1]


def test_batch_beyond_the_staging():
    """70 columns of 40^3 rows (72 MB of vectors) and a small system among them."""
    A = cmamd.gen_convdiff(3, 40, 2.0, seed=1)
    big, want = _item(A, cmamd.afiim(A, 0.1), 2)
    S = cmamd.gen_convdiff(2, 20, 1.0, seed=3)
    small, wsmall = _item(S, cmamd.afiim(S, 0.1), 4)
    _check([big] * 65 + [small] + [big] * 5, [want] * 65 + [wsmall] + [want] * 5)
