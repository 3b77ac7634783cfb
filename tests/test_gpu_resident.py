"""The resident solve (one launch per solve, taken by tuned systems of at most
524288 rows) against the oracle.

Sizes sit at the edges of its launch shapes (256 or 512 threads, 1, 2 or 4
rows per thread, one workgroup, a last workgroup with one row, the most rows);
matrices in diagonals, in diagonals with a remainder, and in CSR with rows
longer than a staged tile.  Bars are the FP64 path's: info equal, pass counts
within 2%, residual norms of the first 20 passes within 1e-8 (over a floor of
1e-12 ||r_0||), and x within 1e-7 of the oracle's where the oracle's own x is
determinate: both leave the loop on the same pass, where their difference is
rounding amplified over the passes, which the oracle shows by its answers for
two summation orders (thread counts) -- 3e-7 on the 72 passes of the weakly
preconditioned 51^3 system, 1e-11 and less on the others."""
import threading

import numpy as np
import pytest

import cmamd
import exit_cases
import oracle
from cmamd.workloads import upper_triangle

pytestmark = pytest.mark.gpu


def _check(name, variant, A, F, b, sym=False, tol=1e-8, nmax=500):
    s = cmamd.System(variant, A, F, a_symmetric=sym)
    s.enable_mixed(32)
    s.enable_mixed(16)
    s.autotune(3)
    s.set_rhs(b)
    s.set_x(None)
    print(f"resident {name} {variant} n={A.n} {s.spmv_formats()[64]}", flush=True)
    rv, it, info, tr = s.solve(tol=tol, nmax=nmax, trace_cap=64)
    x = s.get_x()
    oracle.set_threads(3)
    x3 = oracle.bicgstab(variant, A, b, F, tol=tol, nmax=nmax, issym=sym)[0]
    oracle.set_threads(4)
    xo, rvo, ito, info_o, tro = oracle.bicgstab(variant, A, b, F, tol=tol, nmax=nmax, trace_cap=64, issym=sym)
    determinate = np.linalg.norm(x3 - xo) <= 1e-8 * np.linalg.norm(xo)
    assert info == info_o
    assert abs(it - ito) <= max(1, int(np.ceil(0.02 * ito)))
    m = min(len(tr), len(tro), 20)
    assert m > 0 and np.all(np.abs(tr[:m] - tro[:m]) <= 1e-8 * tro[:m] + 1e-12 * tro[0])
    if it == ito and determinate:
        assert np.linalg.norm(x - xo) <= 1e-7 * np.linalg.norm(xo)
    # a second solve, from the solution: stops at once on the recursive residual
    rv2, it2, info2, _ = s.solve(tol=1e-3, nmax=nmax)
    assert info2 in (0, 2) and it2 <= max(it, 1)
    for bits in (32, 16):
        s.set_x(None)
        rvm, outer, inner, infom = s.solve_mixed(bits, tol=1e-10, nmax=nmax)
        assert infom == 0 and rvm <= 1e-10 and inner >= outer >= 1, (bits, rvm, outer, inner)
    s.close()


@pytest.mark.parametrize("dim,N,prec", [
    (2, 4, "afiim"),     # 16 rows
    (2, 16, "pdfiim"),   # one workgroup, full
    (2, 17, "afiim"),    # 289 rows
    (2, 101, "afiim"),   # remainders in G and H
    (3, 40, "acifim"),   # 64000 rows, 250 workgroups of 256
    (3, 41, "pdfiim"),   # 68921 rows, 512 threads
    (3, 51, "acifim"),   # 132651 rows, two rows per thread in FP64
    (3, 64, "pdfiim"),   # 262144 rows, 256 full workgroups
    (3, 65, "acifim"),   # 274625 rows, four rows per thread
])
def test_resident_matches_oracle(dim, N, prec):
    A = cmamd.gen_convdiff(dim, N, 1.0, seed=3)
    F = {"afiim": lambda: cmamd.afiim(A, 0.1), "pdfiim": lambda: cmamd.pdfiim(A, 2, 2, 1, 0.05),
         "acifim": lambda: cmamd.acifim(A, 0.01, 0.1)}[prec]()
    _check(f"{dim}d{N}", prec, A, F, cmamd.csr_mv_host(A, cmamd.gen_uniform(4, A.n)))


def test_resident_symmetric():
    A = cmamd.gen_convdiff(3, 13, 0.0, seed=3)
    b = cmamd.csr_mv_host(A, cmamd.gen_uniform(4, A.n))
    U = upper_triangle(A)
    F = cmamd.pdfiim(U, 2, 2, 1, 0.05)
    _check("sym", "pdfiim", U, cmamd.Factors(F.G, F.idv, None), b, sym=True)


@pytest.mark.parametrize("n,long_rows", [(257, (0,)), (5000, (0, 17, 4999))])
def test_resident_irregular_csr(n, long_rows):
    """Random sparse rows, some with more entries than a staged tile holds."""
    import scipy.sparse as sp
    rng = np.random.default_rng(n)
    m = sp.random(n, n, density=4.0 / n, random_state=np.random.RandomState(n), format="lil")
    for r in long_rows:
        c = rng.choice(n, size=min(n, 4500), replace=False)
        m[r, c] = rng.uniform(-1, 1, len(c)) / len(c)
    m.setdiag(4.0 + rng.uniform(0, 1, n))
    A = cmamd.Csr.from_scipy(m.tocsr())
    _check("irregular", "afiim", A, cmamd.afiim(A, 0.01), cmamd.csr_mv_host(A, cmamd.gen_uniform(4, A.n)))


@pytest.mark.parametrize("variant", ["afiim", "acifim"])
def test_resident_exits(variant):
    for name in sorted(exit_cases.DIVERGING):
        A, b, F, _ = exit_cases.diverging(name)
        s = cmamd.System(variant, A, F)
        s.autotune(3)
        s.set_rhs(b)
        s.set_x(None)
        rv, it, info, tr = s.solve(tol=1e-8, nmax=200, trace_cap=128)
        limit = exit_cases.maxmsteps("afiim", A.n)
        if variant == "afiim":
            assert (it, info) == (limit, 1)
        else:
            assert it > limit
        for nmax, want in ((0, 3), (-1, 77)):  # NMAX < 0 leaves info
            s.set_x(np.full(A.n, 2.0))
            rv, it, info, _ = s.solve(tol=1e-8, nmax=nmax, info_in=77)
            assert (it, info) == (0, want) and np.all(s.get_x() == 2.0)
        s.close()
    # s = 0, omega = 0/0: AFIIM runs on NaNs to NMAX, ACIFIM's guard stops on pass 2
    n = 300
    I = exit_cases.identity(n)
    A = cmamd.Csr(n, I.ptr, I.idx, np.full(n, 2.0))
    s = cmamd.System(variant, A, cmamd.Factors(I, np.full(n, 0.5), I, I, I))
    s.autotune(3)
    s.set_rhs(np.ones(n))
    s.set_x(None)
    rv, it, info, tr = s.solve(tol=1e-8, nmax=9, trace_cap=16)
    _, rvo, ito, info_o, tro = oracle.bicgstab(variant, A, np.ones(n), cmamd.Factors(I, np.full(n, 0.5), I, I, I),
                                               tol=1e-8, nmax=9, trace_cap=16)
    assert (it, info, len(tr)) == (ito, info_o, len(tro))
    s.close()


def test_resident_from_threads():
    """Solves of different systems at the same time give what they give alone."""
    work = []
    for N, seed in ((30, 1), (45, 2), (64, 3)):
        A = cmamd.gen_convdiff(3, N, 2.0, seed=seed)
        s = cmamd.System("pdfiim", A, cmamd.pdfiim(A, 2, 2, 1, 0.05))
        s.autotune(3)
        s.set_rhs(cmamd.csr_mv_host(A, cmamd.gen_uniform(seed, A.n)))
        s.set_x(None)
        s.solve(tol=1e-8)
        work.append((s, s.get_x()))
    bad = []

    def loop(s, x0):
        for _ in range(6):
            s.set_x(None)
            _, _, info, _ = s.solve(tol=1e-8)
            x = s.get_x()
            # a grid that cannot be resident takes the launched passes: same solution to rounding
            if info != 0 or np.linalg.norm(x - x0) > 1e-9 * np.linalg.norm(x0):
                bad.append((s.n, info, np.linalg.norm(x - x0)))
    th = [threading.Thread(target=loop, args=w) for w in work]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not bad, bad
    for s, _ in work:
        s.close()
