"""Runs of several steps per launch on LDS tiles of the domain (block shapes
outside 16^3 and 32^3): fields equal to single steps bit for bit, norms to 1e-13
(another summation order), for every remainder of the step count, at shapes
where tiles end inside blocks, blocks inside tiles, the domain inside a tile or
its halo, and rows that no vector divides; components with walls of their own."""
import numpy as np
import pytest

import cubismnova_amd as cnv
from tests.helpers import assert_same, cells_of
from tests.test_gpu_cols import MIXED, PARTLY, WALLS, build

pytestmark = pytest.mark.gpu

SHAPES = [((1, 1, 1), (5, 7, 3)), ((2, 3, 1), (6, 5, 33)), ((3, 3, 3), (8, 8, 8)), ((1, 2, 2), (24, 24, 24)),
          ((2, 1, 2), (40, 13, 6)), ((1, 1, 3), (1, 1, 1)), ((2, 1, 1), (65, 64, 5)), ((17, 2, 2), (1, 3, 2)),
          ((1, 2, 1), (64, 64, 64)), ((2, 2, 2), (16, 16, 12)), ((8, 7, 6), (8, 12, 16)), ((9, 10, 9), (12, 12, 12))]


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("shape", SHAPES, ids=str)
@pytest.mark.parametrize("walls", ["periodic", "three components"] + sorted(WALLS))
def test_run_matches_single_steps(gpu, dtype, shape, walls):
    nb, n = shape
    lists = {"periodic": [[]], "three components": [MIXED, [], PARTLY]}.get(walls) or [WALLS[walls]]
    u, _, _ = build(nb, n, dtype, 61, lists)
    v, _, _ = build(nb, n, dtype, 61, lists)
    t, _, _ = build(nb, n, dtype, 61, lists)
    w, _, _ = build(nb, n, dtype, 61, lists)
    dt = 0.1 / max(nb[d] * n[d] for d in range(3)) ** 2
    a, b = v, w
    for steps in (4, 5, 6, 7, 9):
        norms, want = cnv.DeviceBuffer(8 * steps), cnv.DeviceBuffer(8 * steps)
        norms.fill(np.float64, np.nan)
        res = cnv.diffusion_run(u, t, steps, dt, norms)
        assert res is (u if steps % 2 == 0 else t)
        u, t = res, (t if res is u else u)
        for k in range(steps):
            cnv.diffusion_step(a, b, dt, sumsq=want.at(8 * k))
            a, b = b, a
        for c in range(len(lists)):
            assert_same(cells_of(u.download(c), nb, n, u.block_stride), cells_of(a.download(c), nb, n, a.block_stride),
                        "%d steps, component %d" % (steps, c))
        gn, wn = norms.download(np.float64, steps), want.download(np.float64, steps)
        assert np.max(np.abs(gn - wn) / wn) <= 1e-13
    # without norms
    u2 = cnv.diffusion_run(u, t, 4, dt)
    for k in range(4):
        cnv.diffusion_step(a, b, dt)
        a, b = b, a
    assert_same(cells_of(u2.download(0), nb, n, u.block_stride), cells_of(a.download(0), nb, n, a.block_stride))


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("walls", [False, True])
@pytest.mark.parametrize("nb,n", [((2, 2, 2), (20, 20, 20)), ((5, 5, 5), (24, 24, 24)), ((6, 5, 4), (32, 32, 32))],
                         ids=str)
def test_run_with_a_wider_second_grid(gpu, dtype, walls, nb, n):
    """tmp may have more components than u: only u's are stepped, in the launches
    that read tmp too."""
    lists = [MIXED if walls else []]
    u, _, _ = build(nb, n, dtype, 73, lists)
    a, _, _ = build(nb, n, dtype, 73, lists)
    b, _, _ = build(nb, n, dtype, 73, lists)
    t, _, _ = build(nb, n, dtype, 79, lists * 3)
    before = [t.download(c) for c in (1, 2)]
    dt = 0.1 / max(nb[d] * n[d] for d in range(3)) ** 2
    norms, want = cnv.DeviceBuffer(8 * 8), cnv.DeviceBuffer(8 * 8)
    assert cnv.diffusion_run(u, t, 8, dt, norms) is u
    for k in range(8):
        cnv.diffusion_step(a, b, dt, sumsq=want.at(8 * k))
        a, b = b, a
    assert_same(cells_of(u.download(0), nb, n, u.block_stride), cells_of(a.download(0), nb, n, a.block_stride))
    gn, wn = norms.download(np.float64, 8), want.download(np.float64, 8)
    assert np.max(np.abs(gn - wn) / wn) <= 1e-13
    for c in (1, 2):
        assert_same(t.download(c), before[c - 1], "component %d of tmp" % c)


@pytest.mark.parametrize("nb,n", [((2, 2, 2), (32, 32, 32)), ((5, 5, 5), (24, 24, 24))], ids=str)
def test_captured_run(gpu, nb, n):
    """A recorded run replays to the eager run's field and norms."""
    u, _, _ = build(nb, n, np.float32, 83, [MIXED])
    v, _, _ = build(nb, n, np.float32, 83, [MIXED])
    t, _, _ = build(nb, n, np.float32, 83, [MIXED])
    r, _, _ = build(nb, n, np.float32, 83, [MIXED])  # v's own second grid: the first two runs overlap
    dt = 0.1 / max(nb[d] * n[d] for d in range(3)) ** 2
    norms, want = cnv.DeviceBuffer(8 * 12), cnv.DeviceBuffer(8 * 12)
    s = cnv.Stream()
    cnv.diffusion_run(u, t, 12, dt, norms, stream=s)
    cnv.diffusion_run(v, r, 12, dt, want)
    s.synchronize()
    g = cnv.Graph(s).capture()
    cnv.diffusion_run(u, t, 12, dt, norms, stream=s)
    g.end()
    for rep in range(3):
        g.launch()
        s.synchronize()
        cnv.diffusion_run(v, r, 12, dt, want)
        assert_same(cells_of(u.download(0), nb, n, u.block_stride), cells_of(v.download(0), nb, n, v.block_stride))
        assert np.array_equal(norms.download(np.float64, 12), want.download(np.float64, 12))


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("edge,wg,zchunk", [(32, 256, 8), (32, 512, 16), (32, 256, 32), (16, 128, 8), (16, 128, 16)])
@pytest.mark.parametrize("walls", ["periodic", "mixed"])
def test_run_with_a_pinned_block_tile(gpu, dtype, edge, wg, zchunk, walls):
    """The two-step kernel on block tiles at every pinned z depth: each of ten runs
    from the same field gives the single steps' field (a workgroup's last plane
    was stored wrong in some of them)."""
    nb, n = tuple(np.array((6, 5, 4)) * (32 // edge)), (edge,) * 3
    lists = [MIXED if walls == "mixed" else []]
    u, slabs, _ = build(nb, n, dtype, 89, lists)
    t, _, _ = build(nb, n, dtype, 89, lists)
    a, _, _ = build(nb, n, dtype, 89, lists)
    b, _, _ = build(nb, n, dtype, 89, lists)
    dt = 0.1 / 192 ** 2
    for k in range(4):
        cnv.diffusion_step(a, b, dt)
        a, b = b, a
    base = cnv.tune_diffusion_run(dtype, edge)
    try:
        cnv.set_tune_diffusion_run(dtype, edge, wg, zchunk)
        for rep in range(10):
            u.upload(0, slabs[0])
            assert cnv.diffusion_run(u, t, 4, dt) is u
            diff = cnv.grid_compare(u, a)
            assert diff[0] == 0.0 and diff[2] == 0.0, (rep, diff)
    finally:
        cnv.set_tune_diffusion_run(dtype, edge, *base)
