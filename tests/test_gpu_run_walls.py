"""Runs between walls on grids that step two at a time on block tiles."""
import numpy as np
import pytest

import cubismnova_amd as cnv
from tests.helpers import assert_same
from tests.test_gpu_cols import build

pytestmark = pytest.mark.gpu


def run_and_singles(nb, n, dtype, lists, steps, seed=101):
    """Fields and norms of diffusion_run and of as many single steps, compared:
    fields bit for bit, norms to 1e-13 (another summation order)."""
    u, t, a, b = (build(nb, n, dtype, seed, lists)[0] for _ in range(4))
    dt = 0.1 / max(nb[d] * n[d] for d in range(3)) ** 2
    norms, want = cnv.DeviceBuffer(8 * steps), cnv.DeviceBuffer(8 * steps)
    res = cnv.diffusion_run(u, t, steps, dt, norms)
    for k in range(steps):
        cnv.diffusion_step(a, b, dt, sumsq=want.at(8 * k))
        a, b = b, a
    for c in range(len(lists)):
        assert_same(res.download(c), a.download(c), "component %d" % c)
    gn, wn = norms.download(np.float64, steps), want.download(np.float64, steps)
    assert np.max(np.abs(gn - wn) / wn) <= 1e-13


@pytest.mark.parametrize("axis", [0, 1, 2])
def test_symmetry_factor_below_single_precision(gpu, axis):
    """A Symmetry factor that is not zero in the list and zero in the grid's type
    mirrors to a ghost of zero, in both steps of a launch."""
    run_and_singles((4, 4, 4), (32, 32, 32), np.float32, [[(3, axis, 0, 1e-60), (3, axis, 1, -1e-60)]], 4)
