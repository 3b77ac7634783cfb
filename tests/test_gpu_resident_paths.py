"""Which solves run in a resident launch, and the kernel's CSR tiles.

The sizes are those at the edges of the launch shapes; what each call took is
read from the system's counts.  Matrices without diagonals have more entries
per workgroup than the kernel's first tile (1024) and several later ones, up
to the most it takes (four steps of the three products; rows of 256 entries in
all), with one to four rows per thread; beyond that the launched passes run.
Bars are the FP64 path's: info equal, pass counts within 2%, x within 1e-7 of
the oracle's on the same pass (15 passes and fewer); refinement reaches its
tolerance."""
import numpy as np
import pytest
import scipy.sparse as sp

import cmamd
import oracle

pytestmark = pytest.mark.gpu


def _delta(s, f):
    a = s.resident(True)
    out = f()
    b = s.resident(True)
    assert b[1:] == a[1:]
    return out, b[0] - a[0]


@pytest.mark.parametrize("dim,N,prec,taken", [
    (2, 4, "afiim", True), (2, 16, "pdfiim", True), (2, 17, "afiim", True), (2, 101, "afiim", True),
    (3, 40, "acifim", True), (3, 41, "pdfiim", True), (3, 46, "pdfiim", True), (3, 47, "afiim", True),
    (3, 58, "pdfiim", True), (3, 59, "pdfiim", True), (3, 66, "pdfiim", True), (3, 67, "acifim", True),
    (3, 73, "pdfiim", True), (3, 74, "pdfiim", False)])
def test_tuned_solves_are_resident(dim, N, prec, taken):
    A = cmamd.gen_convdiff(dim, N, 1.0, seed=3)
    F = {"afiim": lambda: cmamd.afiim(A, 0.1), "pdfiim": lambda: cmamd.pdfiim(A, 2, 2, 1, 0.05),
         "acifim": lambda: cmamd.acifim(A, 0.01, 0.1)}[prec]()
    s = cmamd.System(prec, A, F)
    for q in (32, 16):
        s.enable_mixed(q)
    xs = cmamd.gen_uniform(4, A.n)
    s.set_rhs(cmamd.csr_mv_host(A, xs))

    def solve(bits):
        s.set_x(None)
        r = s.solve(tol=1e-8)[2] if bits == 64 else s.solve_mixed(bits, tol=1e-10)[3]
        assert r == 0

    assert _delta(s, lambda: solve(64))[1] == 0  # not tuned
    s.autotune(2)
    for bits in (64, 32, 16):
        n = _delta(s, lambda: solve(bits))[1]
        assert n >= 1 if taken else n == 0, (bits, n)
        assert np.linalg.norm(s.get_x() - xs) <= 1e-4 * np.linalg.norm(xs)
    s.profile(True)
    assert _delta(s, lambda: solve(64))[1] == 0
    s.profile(False)
    s.close()


@pytest.mark.parametrize("N,k,bits,taken", [
    (16, 16, 64, True), (16, 16, 32, True), (36, 5, 64, True), (36, 4, 64, True), (36, 14, 64, False),
    (36, 14, 32, True), (50, 4, 32, True), (73, 1, 32, True), (64, 3, 32, False)])
def test_blocks_by_width(N, k, bits, taken):
    """A block is resident by its system and width (1, 2, 4, 8, 16)."""
    A = cmamd.gen_convdiff(3, N, 2.0, seed=7)
    s = cmamd.System("pdfiim", A, cmamd.pdfiim(A, 2, 2, 1, 0.05))
    B = np.stack([cmamd.csr_mv_host(A, cmamd.gen_uniform(j, A.n)) for j in range(k)], axis=1)
    if bits != 64:
        s.enable_mixed(bits)

    def solve():
        s.block_set(B)
        r = s.block_solve(tol=1e-8)[2] if bits == 64 else s.block_solve_mixed(bits, tol=1e-10)[3]
        assert np.all(r == 0)

    n = _delta(s, solve)[1]
    assert n >= k if taken else n == 0, n
    s.close()


def _random(n, m, long_every, long_len, seed):
    """m random entries per row, long_len in every long_every-th, a diagonal
    that dominates; Jacobi as preconditioner."""
    rng = np.random.default_rng(seed)
    per = np.full(n, m)
    if long_every:
        per[long_every // 2::long_every] = long_len
    r = np.repeat(np.arange(n), per)
    c = rng.integers(0, n, len(r))
    v = rng.uniform(-1, 1, len(r)) / np.repeat(per, per)
    A = sp.csr_matrix((v, (r, c)), shape=(n, n)) + sp.diags(3.0 + np.arange(n) % 13)
    A = A.tocsr()
    A.sort_indices()
    I = cmamd.Csr(n, np.arange(n + 1, dtype=np.int32), np.arange(n, dtype=np.int32), np.ones(n))
    return cmamd.Csr.from_scipy(A), cmamd.Factors(I, 1.0 / A.diagonal(), I)


@pytest.mark.parametrize("n,m,long_every,long_len,taken", [
    (1500, 20, 0, 0, True),       # 256 threads, a row each: three tiles
    (3001, 6, 40, 220, True),     # rows over several tiles
    (70001, 18, 0, 0, True),      # 512 threads, a row each
    (120001, 13, 0, 0, True),     # two rows each
    (250001, 9, 0, 0, True),      # three
    (350001, 8, 0, 0, True),      # four
    (3001, 6, 300, 300, False),   # rows that one thread would sum for too long
    (3000, 40, 0, 0, False)])     # too many steps
def test_resident_csr(n, m, long_every, long_len, taken):
    A, F = _random(n, m, long_every, long_len, n)
    xs = cmamd.gen_uniform(4, n)
    b = cmamd.csr_mv_host(A, xs)
    s = cmamd.System("afiim", A, F)
    s.enable_mixed(32)
    s.enable_mixed(16)
    s.autotune(2)
    s.set_rhs(b)
    s.set_x(None)
    print(f"resident csr n={n} m={m} {s.spmv_formats()[64]}", flush=True)
    (rv, it, info, _), took = _delta(s, lambda: s.solve(tol=1e-8))
    assert took == int(taken)
    xo, rvo, ito, info_o, _ = oracle.bicgstab("afiim", A, b, F, tol=1e-8)
    assert info == info_o and abs(it - ito) <= max(1, int(np.ceil(0.02 * ito)))
    if it == ito:
        assert np.linalg.norm(s.get_x() - xo) <= 1e-7 * np.linalg.norm(xo)
    for bits in (32, 16):
        s.set_x(None)
        (rvm, outer, inner, infom), took = _delta(s, lambda: s.solve_mixed(bits, tol=1e-10))
        assert infom == 0 and rvm <= 1e-10 and (took == outer if taken else took == 0), (bits, took, outer)
    s.close()
