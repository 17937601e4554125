"""Runs on grids too large for LDS tiles, two steps per launch on domain tiles
that march through z (any block shape but FP64 16^3 and 32^3): fields equal to
single steps bit for bit, norms to 1e-13 (another summation order), at shapes with
partly filled tiles on every axis, domains thinner than a vector, a halo or a
chunk, rows that no vector divides, and walls of every rule."""
import numpy as np
import pytest

import cubismnova_amd as cnv
from tests.helpers import assert_same, cells_of
from tests.test_gpu_cols import MIXED, PARTLY, WALLS, build

pytestmark = pytest.mark.gpu

SHAPES = [((5, 6, 5), (24, 24, 24)), ((8, 8, 8), (16, 16, 16)), ((6, 8, 6), (21, 17, 30)), ((1, 60, 20), (3, 5, 50)),
          ((1, 40, 30), (4, 24, 24)), ((30, 31, 1), (20, 20, 1)), ((31, 30, 1), (20, 20, 2)), ((60, 1, 20), (12, 3, 15)),
          ((2, 3, 2), (64, 64, 64))]


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("shape", SHAPES, ids=str)
@pytest.mark.parametrize("walls", ["periodic", "two components"] + sorted(WALLS))
def test_run_matches_single_steps(gpu, dtype, shape, walls):
    nb, n = shape
    lists = {"periodic": [[]], "two components": [MIXED, PARTLY]}.get(walls) or [WALLS[walls]]
    u, _, _ = build(nb, n, dtype, 67, lists)
    v, _, _ = build(nb, n, dtype, 67, lists)
    t, _, _ = build(nb, n, dtype, 67, lists)
    w, _, _ = build(nb, n, dtype, 67, lists)
    dt = 0.1 / max(nb[d] * n[d] for d in range(3)) ** 2
    steps = 7
    norms, want = cnv.DeviceBuffer(8 * steps), cnv.DeviceBuffer(8 * steps)
    norms.fill(np.float64, np.nan)
    assert cnv.diffusion_run(u, t, steps, dt, norms) is t
    a, b = v, w
    for k in range(steps):
        cnv.diffusion_step(a, b, dt, sumsq=want.at(8 * k))
        a, b = b, a
    for c in range(len(lists)):
        assert_same(cells_of(t.download(c), nb, n, t.block_stride), cells_of(a.download(c), nb, n, a.block_stride),
                    "component %d" % c)
    gn, wn = norms.download(np.float64, steps), want.download(np.float64, steps)
    assert np.max(np.abs(gn - wn) / wn) <= 1e-13
    # without norms
    assert cnv.diffusion_run(t, u, 4, dt) is t
    for k in range(4):
        cnv.diffusion_step(a, b, dt)
        a, b = b, a
    assert_same(cells_of(t.download(0), nb, n, t.block_stride), cells_of(a.download(0), nb, n, a.block_stride))


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("nb,n", [((6, 6, 6), (64, 64, 64)), ((24, 24, 24), (16, 16, 16)), ((19, 19, 19), (20, 20, 20))],
                         ids=str)
@pytest.mark.parametrize("walls", ["periodic", "mixed"])
def test_several_rounds_of_workgroups(gpu, dtype, nb, n, walls):
    """Grids whose tiles do not fit the GPU at once: equal to single steps in
    every cell (compared on the device)."""
    N = [nb[d] * n[d] for d in range(3)]
    x = np.random.default_rng(71).standard_normal((N[2], N[1], N[0]), dtype=np.float32).astype(dtype)
    grids = [cnv.Cartesian(nb, n, dtype=dtype) for _ in range(4)]
    for g in grids:
        for (k, d, s, v) in (WALLS[walls] if walls != "periodic" else []):
            g.addFaceBC({1: cnv.Absorbing(d, s), 2: cnv.Dirichlet(d, s, v), 3: cnv.Symmetry(d, s, v)}[k])
    u, t, a, b = grids
    u.upload_global(0, x)
    a.upload_global(0, x)
    dt = 0.1 / max(N) ** 2
    for rep in range(3):
        assert cnv.diffusion_run(u, t, 8, dt) is u
        for k in range(8):
            cnv.diffusion_step(a, b, dt)
            a, b = b, a
        diff = cnv.grid_compare(u, a)
        assert diff[0] == 0.0 and diff[2] == 0.0, diff
