"""Runs between walls on grids that step two at a time on block tiles."""
import numpy as np
import pytest

import cubismnova_amd as cnv
from tests.helpers import assert_same, cells_of, face_bc_lists
from tests.test_gpu_cols import KIND, MIXED, PARTLY, build

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


THREE = [MIXED, [], PARTLY]


@pytest.mark.parametrize("nb,edge,dtype,lists", [
    ((4, 4, 4), 32, np.float32, [[]]),           # two planes per tile
    ((4, 4, 4), 32, np.float32, [MIXED]),
    ((2, 3, 2), 32, np.float64, [MIXED]),        # two planes
    ((6, 5, 4), 32, np.float32, THREE),          # a component without lists among walled ones
    ((6, 5, 4), 32, np.float64, THREE),
    ((5, 5, 5), 16, np.float64, THREE),
    ((5, 5, 5), 16, np.float64, [[], [], []]),
    ((1, 6, 8), 32, np.float32, [MIXED]),        # one block between two walls
    ((8, 1, 6), 32, np.float64, [MIXED]),
    ((8, 6, 1), 32, np.float32, [MIXED, PARTLY]),
])
def test_block_tiles(gpu, nb, edge, dtype, lists):
    """Grids larger than the LDS tiles take: the kernel on block tiles, at its
    shallowest, with several components and with walls a block apart."""
    run_and_singles(nb, (edge,) * 3, dtype, lists, 7)


@pytest.mark.parametrize("edge,dtype", [(16, np.float32), (16, np.float64), (32, np.float32)])
@pytest.mark.parametrize("lists", [[[], [], []], THREE], ids=["periodic", "walls"])
def test_block_tiles_pinned_on_a_small_grid(gpu, edge, dtype, lists):
    saved = cnv.tune_diffusion_run(dtype, edge)
    cnv.set_tune_diffusion_run(dtype, edge, saved[0], 8)
    try:
        run_and_singles((2, 3, 2), (edge,) * 3, dtype, lists, 7)
    finally:
        cnv.set_tune_diffusion_run(dtype, edge, *saved)


@pytest.mark.parametrize("axis", [0, 1, 2])
def test_symmetry_factor_below_single_precision(gpu, axis):
    """A Symmetry factor that is not zero in the list and zero in the grid's type
    mirrors to a ghost of zero, in both steps of a launch."""
    run_and_singles((4, 4, 4), (32, 32, 32), np.float32, [[(3, axis, 0, 1e-60), (3, axis, 1, -1e-60)]], 4)


def relist(g, lists):
    """The grid's lists replaced, a list of faces per component."""
    for c, faces in enumerate(lists):
        for b, lst in face_bc_lists(g.nblocks, faces).items():
            bi = (b % g.nblocks[0], (b // g.nblocks[0]) % g.nblocks[1], b // (g.nblocks[0] * g.nblocks[1]))
            g.setBC(bi, [KIND[k](d, s, v) if k in (2, 3) else KIND[k](d, s) for k, d, s, v in lst], comp=c)


CHANGED = [[(k, d, s, v - 0.375) if k == 2 else (k, d, s, v) for k, d, s, v in MIXED],  # other constants
           [(1, 0, 0, 0.0), (2, 0, 1, 0.25), (3, 1, 0, 0.5), (1, 1, 1, 0.0), (3, 2, 0, -1.0), (2, 2, 1, 2.0)]]  # other rules


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("nb,n", [((2, 2, 2), (20, 20, 20)), ((5, 5, 5), (24, 24, 24)), ((6, 5, 4), (32, 32, 32))],
                         ids=["lds tiles", "domain tiles", "block tiles"])
def test_recorded_run_follows_the_lists(gpu, dtype, nb, n):
    """Lists changed after a run was recorded (as long as before, one rule per
    domain face): a replay takes them from the grids, prepared or run meanwhile, in
    its launches of several steps as in its single ones.  A face of two rules turns it into NaN."""
    first, steps = [MIXED, [], PARTLY], 7
    u, t, v, w = (build(nb, n, dtype, 107, first)[0] for _ in range(4))
    start = [u.download(c) for c in range(3)]
    dt = 0.1 / max(nb[d] * n[d] for d in range(3)) ** 2
    norms, want = cnv.DeviceBuffer(8 * steps), cnv.DeviceBuffer(8 * steps)
    s = cnv.Stream()
    cnv.diffusion_run(u, t, steps, dt, norms, stream=s)
    s.synchronize()
    g = cnv.Graph(s).capture()
    cnv.diffusion_run(u, t, steps, dt, norms, stream=s)
    g.end()

    def replay():
        for x in (u, v):
            for c in range(3):
                x.upload(c, start[c])
        g.launch()
        s.synchronize()

    for k, lists in enumerate([first] + [[x, [], PARTLY] for x in CHANGED + [MIXED]]):
        for x in (u, t, v, w):
            relist(x, lists)
            if k % 2 == 0:
                x.prepare()
        if k % 2 == 1:  # a run of these grids does it too, here one of fused launches alone
            cnv.diffusion_run(u, t, 4, dt, stream=s)
            s.synchronize()
        replay()
        assert cnv.diffusion_run(v, w, steps, dt, want) is w
        for c in range(3):
            assert_same(cells_of(t.download(c), nb, n, t.block_stride), cells_of(w.download(c), nb, n, w.block_stride),
                        "component %d" % c)
        assert np.array_equal(norms.download(np.float64, steps), want.download(np.float64, steps))
    for x in (u, t):
        lst = x.getBC((0, 0, 0))
        x.setBC((0, 0, 0), [cnv.Dirichlet(0, 0, 9.0)] + lst[1:])
        x.prepare()
    replay()
    assert np.any(np.isnan(t.download(0)))
