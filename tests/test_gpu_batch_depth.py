"""Planes per work unit of a small batch's single launch: 8 for 16^3 blocks, for
other shapes what 64 KB of tile allow by halving; outputs of the single-grid calls
(WENO5 within 1e-6 of the largest state: its FP32 arithmetic is contracted)."""
import numpy as np
import pytest

import cubismnova_amd as cnv
from tests.helpers import cells_of
from tests.test_gpu_cols import MIXED, build

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nb,n,op,units", [((2, 1, 1), (32, 32, 20), "weno5", 8),       # 5 planes
                                           ((1, 1, 1), (32, 32, 20), "diffusion", 2),   # 10 planes
                                           ((2, 2, 1), (16, 16, 16), "diffusion", 2),   # 8 planes, four items per unit
                                           ((2, 1, 1), (32, 32, 32), "diffusion", 2),   # whole blocks
                                           ((2, 1, 1), (32, 32, 32), "weno5", 8)])      # 8 planes
def test_units_of_a_small_batch(gpu, nb, n, op, units):
    g, _, _ = build(nb, n, np.float32, 31, [MIXED])
    k = 6 if op == "weno5" else 1
    out, ref = (cnv.Cartesian(nb, n, dtype=np.float32, ncomp=k) for _ in range(2))
    b = cnv.Batch([(g, out, op, 3 if op == "weno5" else 1, 1e-6)])
    assert b.form() == (cnv.Batch.SINGLE, units)
    b.run()
    if op == "weno5":
        cnv.weno5(g, ref)
    else:
        cnv.diffusion_step(g, ref, 1e-6)
    for c in range(k):
        got, want = (cells_of(x.download(c), nb, n, g.block_stride) for x in (out, ref))
        if op == "weno5":
            assert np.max(np.abs(got - want)) <= 1e-6 * np.max(np.abs(want))
        else:
            assert np.array_equal(got, want)


def test_16_cubed_diffusion_beside_longer_items(gpu):
    """Whole blocks where another item takes longer than they do."""
    made = [build(nb, n, np.float32, 37, [MIXED])[0] for nb, n in (((2, 2, 1), (16,) * 3), ((1, 2, 1), (32,) * 3))]
    outs, refs = ([cnv.Cartesian(g.nblocks, g.block_cells, dtype=np.float32) for g in made] for _ in range(2))
    b = cnv.Batch([(g, o, "diffusion", 1, 1e-6) for g, o in zip(made, outs)])
    assert b.form() == (cnv.Batch.SINGLE, 1 + 2)
    b.run()
    for g, o, r in zip(made, outs, refs):
        cnv.diffusion_step(g, r, 1e-6)
        assert np.array_equal(o.download(0), r.download(0))
