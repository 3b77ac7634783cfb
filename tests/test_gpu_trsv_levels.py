"""Triangular solves by the rows of a level: few of them (chunks of two rows up
to chunks of 64), and so many that each level is a launch of its own (a mean of
more than 6000), on both sides of that line.  Against the oracle's sequential
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


def _check(n, w, wu=None):
    rng = np.random.default_rng(n + w)
    L, U = _levels(n, w, True, rng), _levels(n, wu or w, False, rng)
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


@pytest.mark.parametrize("n,w,wu", [(12000, 6000, None), (12002, 6001, None), (60000, 12000, None), (50001, 25000, None),
                                    (6001, 6001, None), (42000, 7000, 40), (42000, 40, 7000)])
def test_wide_levels(n, w, wu):
    _check(n, w, wu)


def test_wide_levels_in_solves():
    """A five-point system in red-black order, L = I + lower(A) / D and U = I +
    D^-1 upper(A) (two levels each): FP64 against the oracle, FP32 and FP16
    inner solves, and the captured passes with the launches among them against
    passes launched one by one."""
    N = 250
    i = np.arange(N * N)
    p = np.argsort((i // N + i % N) % 2, kind="stable")
    m = cmamd.gen_convdiff(2, N, 1.0, seed=3).to_scipy()[p][:, p].tocsr()
    m.sort_indices()
    A = cmamd.Csr.from_scipy(m)
    D = sp.diags(1.0 / m.diagonal())
    L, U = (sp.tril(m, -1) @ D + sp.identity(A.n)).tocsr(), (D @ sp.triu(m, 1) + sp.identity(A.n)).tocsr()
    I = cmamd.Csr(A.n, np.arange(A.n + 1, dtype=np.int32), np.arange(A.n, dtype=np.int32), np.ones(A.n))
    F = cmamd.Factors(I, 1.0 / m.diagonal(), I, cmamd.Csr.from_scipy(L), cmamd.Csr.from_scipy(U))
    xs = cmamd.gen_uniform(5, A.n)
    b = cmamd.csr_mv_host(A, xs)
    for mode in "IJ":
        s = cmamd.System("acifim", A, F, mode=mode)
        s.set_rhs(b)
        out = []
        for graphs in (True, False, True):
            s.graphs(graphs)
            s.set_x(None)
            rv, it, info, _ = s.solve(tol=1e-8, nmax=30)
            out.append((s.get_x(), it, info))
        xo, rvo, ito, info_o, _ = oracle.bicgstab("acifim", A, b, F, tol=1e-8, nmax=30, mode=mode)
        assert all(np.array_equal(o[0], out[0][0]) and o[1:] == out[0][1:] for o in out)
        assert out[0][1:] == (ito, info_o)  # 30 passes: NMAX
        assert np.linalg.norm(out[0][0] - xo) <= 1e-7 * np.linalg.norm(xo)
        v = cmamd.gen_uniform(6, A.n)
        z = oracle.trsv(F.L, v, lower=True)
        z = oracle.trsv(F.U, z * F.idv if mode == "I" else z, lower=False)
        assert np.linalg.norm(s.apply(v) - z) <= 1e-12 * np.linalg.norm(z)
        if mode == "I":
            for bits in (32, 16):
                s.enable_mixed(bits)
                s.set_x(None)
                rv, outer, inner, info = s.solve_mixed(bits, tol=1e-10, nmax=500)
                assert info == 0 and rv <= 1e-10, (bits, rv, outer, inner, info)
        s.close()
