"""grid_sums and grid_compare over the chunk edges of their kernels: blocks
smaller than a vector, of a whole number of chunks (1024 16-byte vectors), one
cell more or less, several chunks, more chunks than workgroups; every pairing
of precisions.  The FP64 sums are taken in another order than numpy's
extended-precision ones: each of the n additions is within 2^-53 of the
partial sum, and a thread adds at most a few hundred terms, so 1e-13 of the sum
of magnitudes bounds them; maxima are exact."""
import numpy as np
import pytest

import cubismnova_amd as cnv
from tests.helpers import cells_of, random_slab

pytestmark = pytest.mark.gpu

SHAPES = [((2, 1, 1), (1, 1, 1)), ((3, 2, 1), (3, 1, 1)), ((2, 2, 1), (16, 16, 16)), ((2, 1, 1), (17, 241, 1)),
          ((1, 2, 1), (5, 19, 43)), ((1, 1, 2), (40, 41, 42)), ((9, 16, 16), (4, 4, 4))]


def grid(nb, n, dtype, seed):
    g = cnv.Cartesian(nb, n, dtype=dtype)
    slab = random_slab(seed, nb, n, dtype, g.block_stride)
    pad = slab.reshape(g.nblocks_total, g.block_stride)
    pad[:, n[0] * n[1] * n[2]:] = np.nan          # padding is never read
    g.upload(0, pad.reshape(-1))
    return g, cells_of(slab, nb, n, g.block_stride).astype(np.longdouble)


@pytest.mark.parametrize("nb,n", SHAPES)
@pytest.mark.parametrize("da", [np.float32, np.float64])
@pytest.mark.parametrize("db", [np.float32, np.float64])
def test_sums_and_compare(gpu, nb, n, da, db):
    a, x = grid(nb, n, da, 3)
    b, y = grid(nb, n, db, 4)
    s, q = cnv.grid_sums(a)
    assert abs(s - x.sum()) <= 1e-13 * np.abs(x).sum()
    assert abs(q - (x * x).sum()) <= 1e-13 * (x * x).sum()
    d2, b2, mx = cnv.grid_compare(a, b)
    d = (x.astype(np.float64) - y.astype(np.float64)).astype(np.longdouble)
    assert abs(d2 - (d * d).sum()) <= 1e-13 * (d * d).sum()
    assert abs(b2 - (y * y).sum()) <= 1e-13 * (y * y).sum()
    assert mx == float(np.abs(d).max())
