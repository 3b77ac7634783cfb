"""Batched solves of small systems with many entries per row, on both sides of
the line (80 on the mean, 170 beyond 1024 rows) where they change kernels, in one call with sparse
and with large systems.  Bars are the FP64 path's: info equal, pass counts
within 2%, x within 1e-7 of the oracle's (a dozen passes)."""
import threading

import numpy as np
import pytest
import scipy.sparse as sp

import cmamd
import oracle

pytestmark = pytest.mark.gpu


def _dense(n, nnz, seed):
    """n rows, nnz entries in all: a dominant diagonal and random others."""
    rng = np.random.default_rng(seed)
    m = sp.lil_matrix((n, n))
    per = np.full(n, nnz // n)
    per[: nnz % n] += 1
    for i in range(n):
        c = rng.choice(np.delete(np.arange(n), i), size=per[i] - 1, replace=False)
        m[i, c] = rng.uniform(-1, 1, len(c)) / len(c)
        m[i, i] = 2.0 + i / n
    A = cmamd.Csr.from_scipy(m.tocsr())
    assert A.nnz == nnz
    return A, 1.0 / m.diagonal()


def test_batch_by_entries_per_row():
    items, want = [], []
    for k, (n, nnz) in enumerate(((400, 400 * 80), (400, 400 * 80 + 1), (257, 257 * 257), (1024, 1024 * 80 + 1),
                                  (1025, 1025 * 170), (1025, 1025 * 170 + 1), (97, 97 * 96))):
        A, d = _dense(n, nnz, k)
        I = cmamd.Csr(n, np.arange(n + 1, dtype=np.int32), np.arange(n, dtype=np.int32), np.ones(n))
        F = cmamd.Factors(I, d, I)
        items.append((cmamd.System("afiim", A, F), A, F))
    for dim, N in ((2, 20), (3, 17), (2, 60)):  # 400, 4913 and 3600 rows
        A = cmamd.gen_convdiff(dim, N, 1.0, seed=N)
        F = cmamd.afiim(A, 0.1)
        items.append((cmamd.System("afiim", A, F), A, F))
    batch = []
    for q, (s, A, F) in enumerate(items * 2):
        b = cmamd.csr_mv_host(A, cmamd.gen_uniform(30 + q, A.n))
        batch.append((s, b, None, 1e-8, 500))
        want.append(oracle.bicgstab("afiim", A, b, F, tol=1e-8, nmax=500))
    print("batch n =", [it[0].n for it in batch], flush=True)
    for r, (xo, rvo, ito, info_o, _) in zip(cmamd.batch_solve(batch), want):
        assert r.info == info_o and abs(r.iter - ito) <= max(1, int(np.ceil(0.02 * ito)))
        assert np.linalg.norm(r.x - xo) <= 1e-7 * np.linalg.norm(xo)


def test_mixed_sizes_from_threads():
    """Small items run beside the large ones of their call: from two threads,
    call after call, each item's bits are those of a call of its kind alone."""
    kinds = []
    for dim, N, k in ((3, 18, 6), (2, 40, 30)):  # 5832 and 1600 rows
        A = cmamd.gen_convdiff(dim, N, 1.0, seed=N)
        s = cmamd.System("afiim", A, cmamd.afiim(A, 0.1))
        kinds.append([(s, cmamd.csr_mv_host(A, cmamd.gen_uniform(j, A.n)), None, 1e-8, 500) for j in range(k)])
    want = [r.x for it in kinds for r in cmamd.batch_solve(it)]
    mixed = kinds[0] + kinds[1]
    bad = []

    def loop():
        for rep in range(6):
            for q, r in enumerate(cmamd.batch_solve(mixed)):
                if r.info != 0 or not np.array_equal(r.x, want[q]):
                    bad.append((rep, q, r.info))

    th = [threading.Thread(target=loop) for _ in range(2)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not bad, bad
