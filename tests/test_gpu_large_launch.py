"""Launches of 2^32 threads and more: 65535 blocks of 257x257x1 cells (17 GB) step
as columns of one thread per cell and assemble labs in 261 workgroups each."""
import ctypes

import numpy as np
import pytest

import cubismnova_amd as cnv

pytestmark = pytest.mark.gpu


def test_more_threads_than_one_dimension_holds(gpu):
    nb, n, dt = (257, 255, 1), (257, 257, 1), np.float32
    cells = nb[0] * nb[1] * n[0] * n[1]
    assert nb[0] * nb[1] == 65535 and cells >= 1 << 32
    u = cnv.Cartesian(nb, n, dtype=dt)
    out = cnv.Cartesian(nb, n, dtype=dt)
    elems = u.component_bytes // 4
    for g, v in ((u, 0.5), (out, 3.0)):
        cnv.call("cnv_fill", g.data_ptr(0), 0, v, ctypes.c_size_t(elems), None)
    s = cnv.DeviceBuffer(8)
    cnv.diffusion_step(u, out, 1e-3, sumsq=s)  # a constant field stays one, every partial of the norm counted
    assert s.download(np.float64, 1)[0] == 0.25 * cells
    total, square = cnv.grid_sums(out)
    assert total == 0.5 * cells and square == 0.25 * cells
    # labs into out's memory: 257x257 cells and a ghost in x on either side
    st = cnv.Stencil([-1, 0, 0], [2, 1, 1], False)
    p, _ = u.lab_geometry(st, 0)
    assert p == [259, 257, 1]
    lab = cnv.DeviceBuffer(4 * int(np.prod(p)) * 65535)
    lab.fill(np.float32, 3.0)
    u.lab_all(st, 0, lab)
    for b in (0, 1, 32768, 65534):
        part = np.empty(int(np.prod(p)), np.float32)
        cnv.call("cnv_memcpy_d2h", part.ctypes.data_as(ctypes.c_void_p), lab.at(4 * part.size * b), part.nbytes, None)
        assert np.all(part == 0.5), b
