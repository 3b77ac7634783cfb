"""Blocks of right-hand sides solved in resident launches (every column on
workgroups of its own) against the oracle.

Sizes sit at the edges of the launch shapes for a block (one workgroup per
column, a last workgroup with few rows, 512 threads with 1, 2 and 4 rows each,
all CUs taken) and beyond them (two halves in FP32, launched passes).  Bars
are the FP64 path's: info equal, pass counts within 2%, x within 1e-7 of the
oracle's where both leave on the same pass; refinement reaches its tolerance."""
import threading

import numpy as np
import pytest

import cmamd
import oracle

pytestmark = pytest.mark.gpu


def _system(dim, N, prec, seed):
    A = cmamd.gen_convdiff(dim, N, 2.0, seed=seed)
    F = cmamd.afiim(A, 0.05) if prec == "afiim" else cmamd.pdfiim(A, 2, 2, 1, 0.05)
    return A, F


def _rhs(A, k, seed):
    return np.stack([cmamd.csr_mv_host(A, cmamd.gen_uniform(seed + j, A.n)) for j in range(k)], axis=1)


def _check(A, F, B, prec, bits=(64, 32, 16), X0=None):
    k = B.shape[1]
    s = cmamd.System(prec, A, F)
    for q in bits:
        if q != 64:
            s.enable_mixed(q)
    for q in bits:
        print(f"block resident n={A.n} k={k} bits={q}", flush=True)
        s.block_set(B, X0)
        if q == 64:
            rv, it, info = s.block_solve(tol=1e-8, nmax=500)
            X = s.block_get()
            for j in range(k):
                x0 = None if X0 is None else X0[:, j]
                xo, rvo, ito, info_o = oracle.bicgstab(prec, A, B[:, j], F, tol=1e-8, nmax=500, x0=x0)[:4]
                assert info[j] == info_o, j
                assert abs(it[j] - ito) <= max(1, int(np.ceil(0.02 * ito))), (j, it[j], ito)
                if it[j] == ito:
                    assert np.linalg.norm(X[:, j] - xo) <= 1e-7 * np.linalg.norm(xo), j
        else:
            rv, outer, inner, info = s.block_solve_mixed(q, tol=1e-10, inner_tol=1e-4, nmax=500)
            X = s.block_get()
            assert np.all(info == 0) and inner >= outer >= 1
            for j in range(k):
                r0 = B[:, j] if X0 is None else B[:, j] - cmamd.csr_mv_host(A, X0[:, j])
                r = B[:, j] - cmamd.csr_mv_host(A, X[:, j])
                assert np.linalg.norm(r) <= 1.01e-10 * np.linalg.norm(r0), (q, j)
    s.close()


@pytest.mark.parametrize("dim,N,prec,k", [
    (2, 4, "afiim", 16),    # 16 rows
    (2, 16, "pdfiim", 16),  # a full workgroup of 256 rows, 16 columns
    (2, 33, "afiim", 3),    # 1089 rows: last workgroup of one with 65
    (3, 16, "pdfiim", 16),  # 4096 rows: 16 x 16 workgroups, all CUs
    (3, 36, "pdfiim", 5),   # 1024 (FP64) and 2048 rows per workgroup
    (3, 36, "afiim", 14),   # FP32 in two halves, FP64 launched
    (3, 50, "pdfiim", 4),   # 125000 rows: 62 x 4 workgroups of 2048
])
def test_block_resident(dim, N, prec, k):
    A, F = _system(dim, N, prec, 7)
    _check(A, F, _rhs(A, k, 100), prec)


@pytest.mark.parametrize("N,k", [(64, 2), (64, 3), (79, 2)])
def test_block_resident_large(N, k):
    """The most rows: all CUs for two columns, halves, a launch per column."""
    A, F = _system(3, N, "pdfiim", 3)
    _check(A, F, _rhs(A, k, 40), "pdfiim", bits=(32,))


def test_block_resident_start_and_columns():
    """A start vector; columns equal their solves in another company to
    rounding; no pass and one pass."""
    A, F = _system(3, 20, "pdfiim", 9)
    B = _rhs(A, 4, 10)
    X0 = np.stack([cmamd.gen_uniform(j, A.n) for j in range(4)], axis=1)
    _check(A, F, B, "pdfiim", X0=X0)
    s = cmamd.System("pdfiim", A, F)
    s.block_set(B, None)
    s.block_solve(tol=1e-8, nmax=500)
    X = s.block_get()
    for cols in ([0], [2, 1], [3, 3, 3, 0, 1]):
        s.block_set(np.ascontiguousarray(B[:, cols]), None)
        s.block_solve(tol=1e-8, nmax=500)
        Y = s.block_get()
        for q, j in enumerate(cols):
            assert np.linalg.norm(Y[:, q] - X[:, j]) <= 1e-9 * np.linalg.norm(X[:, j])
    for nmax in (0, 1):
        s.block_set(B, X0)
        _, it, info = s.block_solve(tol=1e-8, nmax=nmax)
        want = oracle.bicgstab("pdfiim", A, B[:, 0], F, tol=1e-8, nmax=nmax, x0=X0[:, 0])
        assert it[0] == want[2] and info[0] == want[3]
        assert np.linalg.norm(s.block_get()[:, 0] - want[0]) <= 1e-9 * np.linalg.norm(want[0])
    s.close()


def test_block_long_rows_stay_launched():
    """Matrices whose rows' CSR entries would be summed serially."""
    A = cmamd.gen_stencil27(14, 0.05, 200, 600, seed=9)
    F = cmamd.afiim(A, 0.1)
    _check(A, F, _rhs(A, 3, 60), "afiim", bits=(64, 32))
    s = cmamd.System("afiim", A, F)
    s.autotune(2)
    b = _rhs(A, 1, 61)[:, 0]
    s.set_rhs(b)
    s.set_x(None)
    _, it, info, _ = s.solve(tol=1e-8, nmax=500)
    xo, _, ito, info_o = oracle.bicgstab("afiim", A, b, F, tol=1e-8, nmax=500)[:4]
    assert info == info_o and abs(it - ito) <= 1
    if it == ito:
        assert np.linalg.norm(s.get_x() - xo) <= 1e-7 * np.linalg.norm(xo)
    s.close()


def test_block_resident_from_threads():
    """Blocks of several systems at the same time: the grids share the CUs,
    and the columns are those found alone to rounding."""
    work = []
    for N, k, seed in ((36, 5, 1), (30, 8, 2), (19, 14, 3), (45, 2, 4)):
        A, F = _system(3, N, "pdfiim", seed)
        s = cmamd.System("pdfiim", A, F)
        s.enable_mixed(32)
        B = _rhs(A, k, 10 * seed)
        s.block_set(B, None)
        s.block_solve_mixed(32, tol=1e-11, inner_tol=1e-4, nmax=500)
        work.append((s, B, s.block_get()))
    bad = []

    def loop(s, B, X):
        for rep in range(6):
            s.block_set(B, None)
            info = (s.block_solve(tol=1e-11, nmax=500)[2] if rep % 2 else
                    s.block_solve_mixed(32, tol=1e-11, inner_tol=1e-4, nmax=500)[3])
            e = np.linalg.norm(s.block_get() - X) / np.linalg.norm(X)
            if np.any(info != 0) or not e <= 1e-8:
                bad.append((s.n, rep, info, e))
    th = [threading.Thread(target=loop, args=w) for w in work]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not bad, bad
    for s, _, _ in work:
        s.close()
