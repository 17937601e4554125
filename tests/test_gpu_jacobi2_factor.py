"""Two sweeps per launch past a Symmetry wall whose factor is not zero in the list
and zero in the grid's type: a ghost of zero in both sweeps."""
import numpy as np
import pytest

import cubismnova_amd as cnv
from tests.helpers import assert_same, random_slab
from tests.test_gpu_jacobi2 import bgrid

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("nb,edge", [((8, 8, 8), 16), ((4, 4, 4), 32), ((3, 3, 2), 64)])
def test_symmetry_factor_below_single_precision(gpu, nb, edge, axis):
    n, dt = (edge,) * 3, np.float32
    bcs = [(3, axis, 0, 1e-60), (3, axis, 1, -1e-60)]
    zf = np.linspace(0.0, 1.0, nb[2] * edge + 1)
    u, v, w, f, o = (bgrid(nb, n, dt, bcs, zf) for _ in range(5))
    u.upload(0, random_slab(3, nb, n, dt))
    f.upload(0, random_slab(5, nb, n, dt))
    cnv.jacobi_sweep(u, f, v)
    cnv.jacobi_sweep(v, f, w)
    cnv.jacobi_sweep2(u, f, o)
    assert_same(o.download(0), w.download(0))
