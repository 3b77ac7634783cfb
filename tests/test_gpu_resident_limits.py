"""Resident solves whose waits are given up.

The limit of a wait is lowered from the host until waits do end early, at any
place of a solve (a reduction that some workgroups get through and others do
not among them).  Every solve must then be one of two: solved by the resident
launch, or by the launched passes from the starting x, each bit for bit what
it is without the limit."""
import numpy as np
import pytest

import cmamd

pytestmark = pytest.mark.gpu

SPINS = list(range(1, 33)) + [40, 48, 64, 80, 96, 128, 192, 256, 512, 1024]


def _tuned(dim, N, prec="afiim"):
    A = cmamd.gen_convdiff(dim, N, 1.0, seed=2)
    F = cmamd.afiim(A, 0.1) if prec == "afiim" else cmamd.pdfiim(A, 2, 2, 1, 0.05)
    s = cmamd.System(prec, A, F)
    s.autotune(2)
    return A, s


@pytest.mark.parametrize("dim,N,prec", [(2, 40, "afiim"), (3, 30, "pdfiim")])
def test_given_up_solves_start_again(dim, N, prec):
    A, s = _tuned(dim, N, prec)
    s.set_rhs(cmamd.csr_mv_host(A, cmamd.gen_uniform(3, A.n)))
    x0 = cmamd.gen_uniform(4, A.n)

    def solve():
        s.set_x(x0)
        rv, it, info, _ = s.solve(tol=1e-8, nmax=500)
        return s.get_x(), it, info

    before = s.resident(False)
    launched = solve()
    assert s.resident(True) == before  # none of it in a resident launch
    resident = solve()
    assert s.resident(True) == (before[0] + 1, before[1], before[2])
    seen = set()
    for spins in SPINS:
        print(f"spins {spins}", flush=True)
        a = s.resident(True, spins=spins)
        x, it, info = solve()
        b = s.resident(True)
        d = tuple(q - p for p, q in zip(a, b))
        assert d in ((1, 0, 0), (0, 0, 1)), (spins, d)
        want = resident if d[0] else launched
        assert np.array_equal(x, want[0]) and (it, info) == want[1:], (spins, d)
        seen.add(d)
    assert (0, 0, 1) in seen
    x, it, info = solve()
    assert np.array_equal(x, resident[0])
    s.close()


def test_given_up_columns_of_a_block():
    """Columns that finished keep their x, the others start again."""
    A, s = _tuned(3, 12, "pdfiim")
    k = 4
    B = np.stack([cmamd.csr_mv_host(A, cmamd.gen_uniform(10 + j, A.n)) for j in range(k)], axis=1)
    X0 = np.stack([cmamd.gen_uniform(20 + j, A.n) for j in range(k)], axis=1)

    def solve():
        s.block_set(B, X0)
        _, it, info = s.block_solve(tol=1e-8, nmax=500)
        return s.block_get(), it, info

    s.resident(False)
    launched = solve()
    s.resident(True)
    resident = solve()
    given_up = 0
    for spins in SPINS:
        print(f"block spins {spins}", flush=True)
        a = s.resident(True, spins=spins)
        x, it, info = solve()
        b = s.resident(True)
        assert b[0] - a[0] + b[2] - a[2] == k and b[1] == a[1], (spins, a, b)
        given_up += b[2] - a[2]
        left = 0
        for j in range(k):
            same = np.array_equal(x[:, j], resident[0][:, j]) and it[j] == resident[1][j]
            again = np.array_equal(x[:, j], launched[0][:, j]) and it[j] == launched[1][j]
            assert same or again, (spins, j)
            left += not same
        assert left == b[2] - a[2], (spins, left)
    assert given_up
    s.enable_mixed(32)
    for spins in SPINS[::4]:
        s.resident(True, spins=spins)
        s.block_set(B, None)
        rv, outer, inner, info = s.block_solve_mixed(32, tol=1e-11, inner_tol=1e-4, nmax=500)
        assert np.all(info == 0) and np.all(rv <= 1e-11), spins
    s.close()
