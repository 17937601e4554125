"""CPU check of the reductions' host side: a thread's results stay its own when
another thread queues a reduction of the same grid before they are read."""
import threading

import numpy as np

import cubismnova_amd as cnv


class Buffer:
    """Host stand-in of a device buffer; a reduction writes through .ptr."""

    def __init__(self, nbytes):
        self.v = np.zeros(nbytes // 8)
        self.ptr = self

    def download(self, dtype, count=None, stream=None):
        if threading.current_thread() is not threading.main_thread():
            queued.set()
            assert other.wait(20)
        return self.v[:count].copy()


queued, other = threading.Event(), threading.Event()


def test_a_threads_results_are_its_own(monkeypatch):
    def call(name, *args):
        out = [a for a in args if isinstance(a, Buffer)]
        if not out:
            return
        out = out[0]
        out.v[:] = [1.0, 2.0, 0.0] if name == "cnv_grid_sums" else [5.0, 6.0, 7.0]

    monkeypatch.setattr(cnv, "DeviceBuffer", Buffer)
    monkeypatch.setattr(cnv, "call", lambda *a: None)
    g = cnv.Cartesian((1, 1, 1), (8, 8, 8))
    monkeypatch.setattr(cnv, "call", call)
    got = []
    t = threading.Thread(target=lambda: got.append(cnv.grid_sums(g)))
    t.start()
    assert queued.wait(20)
    assert cnv.grid_compare(g, g) == (5.0, 6.0, 7.0)
    other.set()
    t.join()
    assert got == [(1.0, 2.0)]
