"""The triangular solves of ACIFIM's apply modes I and J on shapes that stress
their chunks and waits: one row per level, one level for all rows, levels just
around a wave's rows, rows longer than the entries loaded ahead, rows without
a stored diagonal, and few rows.  Against the oracle's sequential solves, each
row a sum of at most 300 products: 1e-12 normwise, with diagonals that dominate
(so that the recursions do not amplify rounding)."""
import numpy as np
import pytest

import cmamd
import oracle

pytestmark = pytest.mark.gpu


def _tri(n, kind, lower, rng):
    """A triangle (in full CSR) of the named shape, diagonal 1 or absent."""
    rows, cols, vals = [], [], []
    for i in range(n):
        if kind == "chain":
            c = [i - 1] if i else []
        elif kind == "diag":
            c = []
        elif kind == "steps":  # 63 to 66 rows per level
            w = 63 + (i // 260) % 4
            c = [i - w] if i >= w else []
        elif kind == "long":
            c = list(rng.choice(i, size=min(i, 300), replace=False)) if i % 97 == 96 else ([i - 5] if i >= 5 else [])
        else:  # grid: the neighbours of a 3D grid of 12^2 planes
            c = [j for j in (i - 144, i - 12, i - 1) if j >= 0]
        v = list(rng.uniform(-1, 1, len(c)) / max(4, 2 * len(c)))
        if not (kind == "nodiag" and i % 3 == 0):
            c, v = c + [i], v + [1.0 + (i % 7) / 8]
        o = np.argsort(c)
        rows += [i] * len(c)
        cols += [c[k] for k in o]
        vals += [v[k] for k in o]
    import scipy.sparse as sp
    m = sp.csr_matrix((vals, (rows, cols)), shape=(n, n))
    if not lower:
        m = m[::-1, ::-1]  # the same graph backwards
    return cmamd.Csr.from_scipy(m.tocsr())


def _with_diag(T):
    m = T.to_scipy().tolil()
    for i in np.flatnonzero(m.diagonal() == 0.0):
        m[i, i] = 1.0
    return cmamd.Csr.from_scipy(m.tocsr())


@pytest.mark.parametrize("kind,n", [("chain", 700), ("diag", 5000), ("steps", 2000), ("long", 3001), ("grid", 1729),
                                    ("nodiag", 1000), ("grid", 1), ("chain", 2), ("grid", 63), ("grid", 257)])
def test_triangular_shapes(kind, n):
    rng = np.random.default_rng(n)
    L, U = _tri(n, kind, True, rng), _tri(n, kind, False, rng)
    I = cmamd.Csr(n, np.arange(n + 1, dtype=np.int32), np.arange(n, dtype=np.int32), np.ones(n))
    d = rng.uniform(0.5, 2.0, n)
    v = rng.uniform(-1, 1, n)
    for mode in "IJ":
        print(f"triangles {kind} n={n} mode {mode}", flush=True)
        s = cmamd.System("acifim", I, cmamd.Factors(I, d, I, L, U), mode=mode)
        # the oracle divides by the stored diagonal: give it the 1 a missing one stands for
        z = oracle.trsv(_with_diag(L), v, lower=True)
        z = oracle.trsv(_with_diag(U), z * d if mode == "I" else z, lower=False)
        for _ in range(2):  # the buffers of the first are the second's
            y = s.apply(v)
            assert np.linalg.norm(y - z) <= 1e-12 * np.linalg.norm(z)
        s.close()


def test_triangular_mixed_and_nan():
    """FP32 and FP16 factors in the inner solves, and a right-hand side with a
    NaN, which every wait has to get past."""
    A = cmamd.gen_convdiff(3, 17, 5.0, seed=4)
    F = cmamd.acifim(A, 0.01, 0.1)
    xs = cmamd.gen_uniform(5, A.n)
    b = cmamd.csr_mv_host(A, xs)
    s = cmamd.System("acifim", A, F, mode="I")
    s.set_rhs(b)
    for bits in (32, 16):
        s.enable_mixed(bits)
        s.set_x(None)
        rv, outer, inner, info = s.solve_mixed(bits, tol=1e-10)
        assert info == 0 and rv <= 1e-10 and np.linalg.norm(s.get_x() - xs) <= 1e-7 * np.linalg.norm(xs)
    v = cmamd.gen_uniform(6, A.n)
    v[100] = np.nan
    z = oracle.trsv(F.U, oracle.trsv(F.L, v, lower=True) * F.idv, lower=False)
    y = s.apply(v)
    assert np.array_equal(np.isnan(y), np.isnan(z)) and np.isnan(y).any() and not np.isnan(y).all()
    s.close()
