"""Resident solves that cannot start, wait for each other, or give up.

The limit of a wait is lowered from the host until waits do end early, at any
place of a solve (a reduction that some workgroups get through and others do
not among them).  Every solve must then be one of two: solved by the resident
launch, or by the launched passes from the starting x, each bit for bit what
it is without the limit.  Solves from several threads wait for their turn and
give bit for bit what they give alone."""
import threading
import time

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

    def solve(nmax):
        s.set_x(x0)
        rv, it, info, _ = s.solve(tol=1e-8, nmax=nmax)
        return s.get_x(), it, info

    # short solves often, at the limits where some waits of a reduction end
    # early and some do not; whole ones at every limit
    plan = [(500, q) for q in SPINS] + [(m, q) for m in (1, 2, 3) for q in range(2, 9) for _ in range(60)]
    before = s.resident(False)
    launched = {m: solve(m) for m in (500, 1, 2, 3)}
    assert s.resident(True) == before  # none of it in a resident launch
    resident = {m: solve(m) for m in (500, 1, 2, 3)}
    assert s.resident(True) == (before[0] + 4, before[1], before[2])
    seen = set()
    for nmax, spins in plan:
        if nmax == 500:
            print(f"spins {spins}", flush=True)
        a = s.resident(True, spins=spins)
        x, it, info = solve(nmax)
        b = s.resident(True)
        d = tuple(q - p for p, q in zip(a, b))
        assert d in ((1, 0, 0), (0, 0, 1)), (nmax, spins, d)
        want = (resident if d[0] else launched)[nmax]
        assert np.array_equal(x, want[0]) and (it, info) == want[1:], (nmax, spins, d)
        seen.add(d)
    assert (0, 0, 1) in seen
    x, it, info = solve(500)
    assert np.array_equal(x, resident[500][0])
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


def test_grid_that_does_not_arrive():
    """No time to arrive: the launched passes from the starting x, and so for
    the solves after it, until the limit is lifted."""
    A, s = _tuned(3, 40, "pdfiim")  # 250 workgroups
    s.set_rhs(cmamd.csr_mv_host(A, cmamd.gen_uniform(3, A.n)))
    x0 = cmamd.gen_uniform(4, A.n)

    def solve():
        s.set_x(x0)
        rv, it, info, _ = s.solve(tol=1e-8, nmax=500)
        return s.get_x(), it, info

    s.resident(False)
    launched = solve()
    a = s.resident(True, join_us=0)
    for _ in range(3):
        x, it, info = solve()
        assert np.array_equal(x, launched[0]) and (it, info) == launched[1:]
    b = s.resident(True)
    assert tuple(q - p for p, q in zip(a, b)) == (0, 1, 0)  # the second and third did not try
    x, it, info = solve()
    assert s.resident(True)[0] == b[0] + 1
    assert np.linalg.norm(x - launched[0]) <= 1e-6 * np.linalg.norm(launched[0])
    s.close()


def test_threads_give_what_they_give_alone():
    """Grids that together exceed the CUs, from four threads: every solve and
    block stays resident and keeps its bits."""
    work = []
    for N, k in ((45, 0), (50, 0), (58, 0), (22, 8)):
        A, s = _tuned(3, N, "pdfiim")
        B = np.stack([cmamd.csr_mv_host(A, cmamd.gen_uniform(10 * N + j, A.n)) for j in range(max(k, 1))], axis=1)
        s.enable_mixed(32)
        if not k:
            s.set_rhs(B[:, 0])

        def solve(s=s, B=B, k=k):
            if k:
                s.block_set(B)
                out = s.block_solve_mixed(32, tol=1e-10)
                return s.block_get(), out[3].tolist()
            s.set_x(None)
            out = s.solve(tol=1e-8)
            return s.get_x(), out[1:3]

        solve()
        c = s.resident(True)
        x, rest = solve()
        each = s.resident(True)[0] - c[0]
        assert each >= 1
        work.append((s, solve, x, rest, each))
    bad = []

    def loop(s, solve, x, rest, each):
        c = s.resident(True)
        for rep in range(8):
            y, r = solve()
            if not np.array_equal(x, y) or r != rest:
                bad.append((s.n, rep, r, rest))
        d = s.resident(True)
        if (d[0] - c[0], d[1] - c[1], d[2] - c[2]) != (8 * each, 0, 0):
            bad.append((s.n, c, d))

    th = [threading.Thread(target=loop, args=w) for w in work]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not bad, bad
    for w in work:
        w[0].close()


@pytest.mark.parametrize("N,bits", [(58, 64), (64, 64), (63, 32), (64, 32), (73, 32)])
def test_launched_solves_go_on_beside_resident_ones(N, bits):
    """A launched solve beside a loop of resident ones finds CUs of its own.
    Next to a grid on all CUs each of its 500 kernels waited for a solve to
    end, 60 times its time alone (12 in FP32)."""
    A, s = _tuned(3, N, "pdfiim")
    s.set_rhs(cmamd.csr_mv_host(A, cmamd.gen_uniform(3, A.n)))
    # three of them: streams share a few hardware queues, and one that shares
    # the resident solves' waits for those whatever CUs are free
    smalls = []
    for _ in range(3):
        C, small = _tuned(2, 100)
        small.resident(False)
        small.set_rhs(cmamd.csr_mv_host(C, cmamd.gen_uniform(5, C.n)))
        smalls.append(small)

    if bits != 64:
        s.enable_mixed(bits)
        s.autotune(2)

    def once(q):
        q.set_x(None)
        t = time.perf_counter()
        q.solve_mixed(bits, tol=1e-11) if q is s and bits != 64 else q.solve(tol=1e-8)
        return time.perf_counter() - t

    alone = min(np.median([once(q) for _ in range(5)]) for q in smalls)
    once(s)
    c = s.resident(True)
    stop = threading.Event()

    def loop():
        while not stop.is_set():
            once(s)

    th = threading.Thread(target=loop)
    th.start()
    time.sleep(0.02)
    beside = min(np.median([once(q) for _ in range(5)]) for q in smalls)
    stop.set()
    th.join()
    assert s.resident(True)[0] > c[0]
    assert beside <= 5 * alone, (beside, alone)
    s.close()
    for q in smalls:
        q.close()
