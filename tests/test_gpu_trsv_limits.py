"""Triangular solves whose waits are given up (the limit of a wait lowered from
the host): an error from apply, solve and solve_mixed, and the usual results
afterwards."""
import numpy as np
import pytest

import cmamd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["I", "J"])
def test_given_up_triangular_solves_are_errors(mode):
    A = cmamd.gen_convdiff(3, 16, 5.0, seed=4)
    s = cmamd.System("acifim", A, cmamd.acifim(A, 0.01, 0.1), mode=mode)
    s.enable_mixed(32)
    v = cmamd.gen_uniform(6, A.n)
    s.set_rhs(cmamd.csr_mv_host(A, cmamd.gen_uniform(5, A.n)))

    def solve():
        s.set_x(None)
        return (s.apply(v),) + s.solve(tol=1e-8)[:3] + (s.get_x(),)

    want = solve()
    for spins in (1, 2):
        s.resident(True, spins=spins)
        s.set_x(None)
        for call in (lambda: s.apply(v), lambda: s.solve(tol=1e-8), lambda: s.solve_mixed(32, tol=1e-8)):
            with pytest.raises(cmamd.EngineError, match="gave up"):
                call()
    s.resident(True)
    got = solve()
    assert np.array_equal(got[0], want[0]) and got[1:4] == want[1:4] and np.array_equal(got[4], want[4])
    s.close()
