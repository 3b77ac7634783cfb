"""Device memory of a large PDFIIM construction: what is held at the peak is
what the construction asks for (1.2 to 1.5 KB per row at this filter), not
twice that."""
import ctypes
import threading

import pytest

import cmamd

pytestmark = pytest.mark.gpu


def _free(hip):
    a, b = ctypes.c_size_t(), ctypes.c_size_t()
    assert hip.hipMemGetInfo(ctypes.byref(a), ctypes.byref(b)) == 0
    return a.value


def test_peak_memory_of_a_construction():
    cmamd.solve_lib()
    hip = ctypes.CDLL("libamdhip64.so")
    A = cmamd.gen_convdiff(3, 128, 1.0, seed=1)
    cmamd.pdfiim_device(cmamd.gen_convdiff(3, 10, 1.0, seed=1), 2, 2, 1, 0.05)  # library and device set up
    start = _free(hip)
    low, stop = [start], threading.Event()

    def watch():
        while not stop.is_set():
            low[0] = min(low[0], _free(hip))

    th = threading.Thread(target=watch)
    th.start()
    cmamd.pdfiim_device(A, 2, 2, 1, 0.05)
    stop.set()
    th.join()
    held = start - low[0]
    assert 256 * A.n < held < 2048 * A.n, held / A.n
