"""Factor arrays are read by an exit handler that runs after cmamd's own exit
work (registered before cmamd is imported): the memory behind them is still
theirs."""
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROG = """
import atexit, sys
import numpy as np

held, kept = [], []

def late():
    # fresh blocks of the same sizes, so that freed memory would be taken again
    junk = [np.full(a.size, 77, a.dtype) for a in held for _ in range(4)]
    ok = all(np.array_equal(a, k) for a, k in zip(held, kept))
    sys.stdout.write("same\\n" if ok else "changed\\n")

atexit.register(late)
sys.path.insert(0, sys.argv[1])
import cmamd

A = cmamd.gen_convdiff(3, int(sys.argv[2]), 1.0, seed=1)
F = cmamd.afiim(A, 0.1)
held += [F.G.ptr, F.G.idx, F.G.val, F.idv, F.H.ptr, F.H.idx, F.H.val]
kept += [a.copy() for a in held]
view = F.G.val[3:9]
del A, F
"""


def test_factors_outlive_exit_handlers():
    for n in ("6", "30"):  # from the allocator's bins, and in mappings of their own
        r = subprocess.run([sys.executable, "-c", PROG, os.path.join(ROOT, "computational-mathematics_amd"), n],
                           capture_output=True, text=True, timeout=300)
        assert r.returncode == 0 and r.stdout == "same\n", (n, r.returncode, r.stdout, r.stderr)
