"""The server's account of device bytes holds what resident block solves keep:
for every column five sets of four sums of 256 workgroups (40 KB)."""
import numpy as np
import pytest

import cmamd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [64, 32, 16])
def test_resident_workspaces_are_accounted(precision):
    k, added = 16, {}
    for resident in (False, True):
        A = cmamd.gen_convdiff(3, 12, 1.0, seed=1)
        s = cmamd.System("pdfiim", A, cmamd.pdfiim(A, 2, 2, 1, 0.05))
        if precision != 64:
            s.enable_mixed(precision)
        s.resident(resident)
        srv = cmamd.Server(slots=1, precision=precision)
        sid = srv.add_system(s)
        before = srv.stats()["bytes"]
        B = np.stack([cmamd.csr_mv_host(A, cmamd.gen_uniform(j, A.n)) for j in range(k)], axis=1)
        assert np.all(srv.wait(srv.submit(sid, B, 1e-8, 500)).info == 0)
        added[resident] = srv.stats()["bytes"] - before
        srv.close()
        assert s.resident(resident)[0] >= (k if resident else 0)
        s.close()
    extra = added[True] - added[False]
    assert k * 5 * 4 * 256 * 8 <= extra <= k * 5 * 4 * 256 * 8 + 65536, extra
