"""Staged transfers (4 MB and more) around systems that come and go: no
event of a transfer is left on a stream that is captured or destroyed."""
import threading

import numpy as np
import pytest

import cmamd

pytestmark = pytest.mark.gpu


def _cycle(A, F, b, want, reps, bad):
    for rep in range(reps):
        s = cmamd.System("pdfiim", A, F)
        s.set_rhs(b)
        s.set_x(None)
        s.solve(tol=1e-8, nmax=20)  # captured passes
        x = s.get_x()
        if want is not None and not np.array_equal(x, want):
            bad.append(rep)
        s.close()
    return x


def test_staged_transfers_of_short_lived_systems():
    """n x 8 B = 4.1 MB: b, x and the matrices are staged.  One thread, then
    two at a time."""
    A = cmamd.gen_convdiff(3, 80, 1.0, seed=4)
    F = cmamd.pdfiim(A, 1, 2, 1, 0.1)
    b = cmamd.csr_mv_host(A, cmamd.gen_uniform(5, A.n))
    bad = []
    x = _cycle(A, F, b, None, 3, bad)
    th = [threading.Thread(target=_cycle, args=(A, F, b, x, 3, bad)) for _ in range(2)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not bad
    r = cmamd.pdfiim_epbicgstab(A, b, F, tol=1e-8, nmax=20)
    assert np.linalg.norm(r.x - x) <= 1e-6 * np.linalg.norm(x)
