"""Served blocks (4 MB and more) from several workers at once: each batch is
what the block solve of its columns gives alone, bit for bit."""
import numpy as np
import pytest

import cmamd

pytestmark = pytest.mark.gpu


def test_served_blocks_equal_block_solves():
    systems, B, want = [], [], []
    for q, N in enumerate((48, 50, 53)):
        A = cmamd.gen_convdiff(3, N, 2.0, seed=q)
        s = cmamd.System("pdfiim", A, cmamd.pdfiim(A, 2, 2, 1, 0.05))
        s.enable_mixed(32)
        b = np.asfortranarray(np.stack([cmamd.csr_mv_host(A, cmamd.gen_uniform(10 * q + j, A.n)) for j in range(5)], axis=1))
        assert b.nbytes > 4 << 20
        s.block_set(b)
        assert np.all(s.block_solve_mixed(32, tol=1e-10, inner_tol=1e-4, nmax=500)[3] == 0)
        systems.append(s)
        B.append(b)
        want.append(s.block_get())
    srv = cmamd.Server(slots=3, precision=32, max_cols=5)
    ids = [srv.add_system(s) for s in systems]
    for rep in range(4):
        rids = [srv.submit(i, b, 1e-10, 500) for i, b in zip(ids, B)]
        for q, rid in enumerate(rids):
            r = srv.wait(rid)
            assert np.all(r.info == 0) and np.array_equal(r.X, want[q]), (rep, q)
    srv.close()
    for s in systems:
        s.close()
