"""Solver cycles whose sweeps run four per launch on LDS tiles of the domain
(small grids): bit-identical to single sweeps for every split of the sweep count
into fours and pairs, on every face rule, on grids smaller than a tile's halo,
with tiles that end past the grid, and with a stretched z."""
import numpy as np
import pytest

import cubismnova_amd as cnv
from cubismnova_amd import stretch
from tests.helpers import assert_same
from tests.test_gpu_jacobi2 import BC2, bgrid, clear

pytestmark = pytest.mark.gpu

SHAPES = [((1, 1, 1), (16, 16, 2)), ((1, 1, 2), (16, 16, 11)), ((3, 2, 2), (16, 16, 16)), ((1, 2, 2), (32, 32, 20)),
          ((1, 1, 1), (64, 64, 13))]
OMEGA = 2.0 / 3.0


@pytest.mark.parametrize("refine,dtype", [(False, np.float64), (False, np.float32), (True, np.float64)],
                         ids=["fp64", "fp32", "refined"])
@pytest.mark.parametrize("nb,n", SHAPES, ids=str)
@pytest.mark.parametrize("bcs", list(BC2))
def test_cycles_equal_single_sweeps(gpu, refine, dtype, nb, n, bcs):
    N = [nb[d] * n[d] for d in range(3)]
    zf = stretch.tanh_faces(N[2], 2.0)
    rng = np.random.Generator(np.random.PCG64(17))
    u0 = rng.standard_normal((N[2], N[1], N[0])).astype(dtype)
    f0 = rng.standard_normal((N[2], N[1], N[0])).astype(dtype)
    hom = [(k, d, s, 0.0 if k == 2 else v) for (k, d, s, v) in BC2[bcs]]
    u, f, uref = (bgrid(nb, n, dtype, BC2[bcs], zf) for _ in range(3))
    f.upload_global(0, f0)
    work = cnv.Cartesian(nb, n, dtype=np.float32 if refine else dtype, ncomp=3 if refine else 2)
    cnv.set_zfaces(work, zf)
    if refine:
        wref = bgrid(nb, n, np.float32, hom, zf)
        e = [bgrid(nb, n, np.float32, hom, zf) for _ in range(2)]
    else:
        w = bgrid(nb, n, dtype, BC2[bcs], zf)
    for S in (2, 4, 6, 8, 10, 14):
        u.upload_global(0, u0)
        uref.upload_global(0, u0)
        if refine:
            cnv.jacobi_defect(uref, f, wref)
            clear(e[0])
            for k in range(S):
                cnv.jacobi_sweep(e[k % 2], wref, e[1 - k % 2], OMEGA)
            cnv.add_correction(uref, e[S % 2])
        else:
            for k in range(S):
                a, b = (uref, w) if k % 2 == 0 else (w, uref)
                cnv.jacobi_sweep(a, f, b, OMEGA)
        cnv.jacobi_solve(u, f, work, refine=refine, sweeps_per_cycle=S, max_cycles=1, tol=0.0)
        assert_same(u.download(0), uref.download(0), "a cycle of %d sweeps" % S)
