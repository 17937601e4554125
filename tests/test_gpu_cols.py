"""GPU parity of the column kernels (block shapes outside 16, 32 and 64 cells
per x/y edge, and small grids of those) against the oracle, bit for bit, at the shapes where a lane
numbering can go wrong: rows of one vector, rows that no vector divides,
planes smaller and larger than a workgroup, one-cell and one-block directions,
chunks with a remainder, components with different BC lists."""
import numpy as np
import pytest

import cubismnova_amd as cnv
import oracle
from tests.helpers import assert_same, cells_of, face_bc_lists, random_slab

pytestmark = pytest.mark.gpu

KIND = {0: cnv.Base, 1: cnv.Absorbing, 2: cnv.Dirichlet, 3: cnv.Symmetry}
MIXED = [(2, 0, 0, 0.75), (3, 0, 1, -1.0), (1, 1, 0, 0.0), (3, 1, 1, 1.0), (2, 2, 0, -0.5), (1, 2, 1, 0.0)]
PARTLY = [(1, 2, 0, 0.0), (3, 2, 1, -0.5)]
SHAPES = [((2, 2, 2), (8, 8, 8)), ((3, 2, 2), (4, 12, 9)), ((1, 1, 1), (5, 7, 3)), ((2, 3, 1), (6, 5, 33)),
          ((1, 2, 2), (24, 24, 24)), ((2, 1, 2), (40, 13, 6)), ((1, 1, 3), (1, 1, 1)), ((2, 1, 1), (65, 64, 5)),
          ((7, 5, 3), (8, 8, 8)), ((2, 1, 2), (16, 16, 16)), ((1, 2, 1), (32, 32, 32)), ((1, 1, 2), (64, 64, 6))]


def build(nb, n, dtype, seed, lists):
    """Grid of one component per BC list, its slabs and per-component lists."""
    g = cnv.Cartesian(nb, n, dtype=dtype, ncomp=len(lists))
    slabs, bcs = [], []
    for c, faces in enumerate(lists):
        slab = random_slab(seed + c, nb, n, dtype, g.block_stride)
        g.upload(c, slab)
        bcl = face_bc_lists(nb, faces)
        for b, lst in bcl.items():
            bi = (b % nb[0], (b // nb[0]) % nb[1], b // (nb[0] * nb[1]))
            g.setBC(bi, [KIND[k](d, s, v) if k in (2, 3) else KIND[k](d, s) for k, d, s, v in lst], comp=c)
        slabs.append(slab)
        bcs.append(bcl)
    return g, slabs, bcs


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("shape", SHAPES, ids=str)
@pytest.mark.parametrize("lists", [[[]], [MIXED, [], PARTLY]], ids=["periodic", "walls"])
def test_diffusion_columns(gpu, dtype, shape, lists):
    nb, n = shape
    g, slabs, bcs = build(nb, n, dtype, 7, lists)
    out = cnv.Cartesian(nb, n, dtype=dtype, ncomp=len(lists))
    lap = cnv.Cartesian(nb, n, dtype=dtype, ncomp=len(lists))
    h = [1.0 / (nb[d] * n[d]) for d in range(3)]
    dt = 0.1 * min(h) ** 2
    s = cnv.DeviceBuffer(8)
    cnv.diffusion_step(g, out, dt, lap=lap, sumsq=s)
    tot = 0.0
    for c, slab in enumerate(slabs):
        f = oracle.Field(slab, nb, n, g.block_stride, bcs=bcs[c])
        un, sref, lref = oracle.diffusion_step(f, h, dt, want_lap=True)
        tot += sref
        assert_same(cells_of(out.download(c), nb, n, g.block_stride), cells_of(un, nb, n, g.block_stride), "euler")
        assert_same(cells_of(lap.download(c), nb, n, g.block_stride), cells_of(lref, nb, n, g.block_stride), "lap")
    # the FP64 sum in another order: 1e-13 of it, as everywhere
    assert abs(s.download(np.float64, 1)[0] - tot) <= 1e-13 * tot


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("edge,tile", [(16, (128, 4)), (32, (256, 16)), (64, (512, 8))])
def test_pinned_tile_on_a_small_grid(gpu, dtype, edge, tile):
    """A tile pinned to something else than the built-in one keeps the marching
    kernel where the columns would run."""
    nb, n = (2, 1, 2), (edge, edge, edge)
    g, slabs, bcs = build(nb, n, dtype, 11, [MIXED])
    out = cnv.Cartesian(nb, n, dtype=dtype)
    saved = cnv.tune_stencil7(dtype, edge)
    cnv.set_tune_stencil7(dtype, edge, *tile)
    try:
        cnv.diffusion_step(g, out, 1e-6)
    finally:
        cnv.set_tune_stencil7(dtype, edge, *saved)
    h = [1.0 / (nb[d] * n[d]) for d in range(3)]
    un, _ = oracle.diffusion_step(oracle.Field(slabs[0], nb, n, bcs=bcs[0]), h, 1e-6)
    assert_same(out.download(0), un)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("nb,edge", [((1, 1, 1), 16), ((3, 2, 1), 16), ((9, 8, 7), 16), ((2, 1, 3), 32),
                                     ((6, 5, 3), 32)])
def test_run_depth_by_grid_size(gpu, dtype, nb, edge):
    """diffusion_run picks the two-step kernel's z chunk (2, 4 or 8 planes
    here) from the grid's tile count: fields equal to single steps bit for
    bit, norms to 1e-13 (another summation order)."""
    n = (edge,) * 3
    slab = random_slab(17, nb, n, dtype)
    u, t, v, w = (cnv.Cartesian(nb, n, dtype=dtype) for _ in range(4))
    u.upload(0, slab)
    v.upload(0, slab)
    dt = 0.1 / (edge * max(nb)) ** 2
    norms, want = cnv.DeviceBuffer(8 * 6), cnv.DeviceBuffer(8 * 6)
    res = cnv.diffusion_run(u, t, 6, dt, norms)
    a, b = v, w
    for k in range(6):
        cnv.diffusion_step(a, b, dt, sumsq=want.at(8 * k))
        a, b = b, a
    assert_same(res.download(0), a.download(0))
    gn, wn = norms.download(np.float64, 6), want.download(np.float64, 6)
    assert np.max(np.abs(gn - wn) / wn) <= 1e-13


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("shape", [x for x in SHAPES if min(x[1]) >= 2] + [((2, 1, 1), (2, 3, 2)), ((1, 2, 1), (3, 2, 17))],
                         ids=str)
@pytest.mark.parametrize("lists", [[[]], [MIXED, [], PARTLY]], ids=["periodic", "walls"])
def test_weno5_columns(gpu, dtype, shape, lists):
    """FP64: the oracle's bits.  FP32: the oracle's FP32 evaluation divides where
    the kernel multiplies by hardware reciprocals (1 ulp each, three per
    state), so a few ulp of the stencil's largest value."""
    nb, n = shape
    g, slabs, bcs = build(nb, n, dtype, 23, lists)
    out = cnv.Cartesian(nb, n, dtype=dtype, ncomp=6 * len(lists))
    cnv.weno5(g, out)
    for c, slab in enumerate(slabs):
        f = oracle.Field(slab.astype(np.float64), nb, n, g.block_stride, bcs=bcs[c])
        want = oracle.weno5(f, prec=1)
        for k in range(6):
            got = cells_of(out.download(6 * c + k), nb, n, g.block_stride)
            ref = cells_of(want[k], nb, n, g.block_stride)
            if dtype is np.float64:
                assert_same(got, ref, "comp %d state %d" % (c, k))
            else:
                assert np.max(np.abs(got - ref)) <= 1e-5 * np.max(np.abs(slab))
                assert np.linalg.norm(got - ref) <= 1e-6 * np.linalg.norm(ref)


WALLS = {
    "dirichlet": [(2, d, s, 0.5 - 0.25 * d + 0.125 * s) for d in range(3) for s in (0, 1)],
    "mirror": [(3, d, s, (1.0, -1.0, 0.5)[d]) for d in range(3) for s in (0, 1)],
    "edge": [(1, d, s, 0.0) for d in range(3) for s in (0, 1)],
    "mixed": MIXED,
    "z only": PARTLY,
    "x only": [(3, 0, 0, -1.0), (2, 0, 1, 0.3)],
    "y only": [(1, 1, 0, 0.0), (3, 1, 1, 2.0)],
}


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("nb,edge,walls", [(nb, e, w) for w in sorted(WALLS) for nb, e in
                                           [((1, 1, 1), 16), ((2, 3, 2), 16), ((9, 8, 7), 16), ((1, 1, 1), 32),
                                            ((2, 1, 3), 32), ((6, 5, 3), 32)]] + [((12, 11, 13), 16, "mixed")])
def test_run_between_walls(gpu, dtype, nb, edge, walls):
    """Two steps per launch on grids with walls, at every z chunk the grid size
    picks: the fields of single steps bit for bit, norms to 1e-13 (another
    summation order)."""
    n = (edge,) * 3
    lists = [WALLS[walls], [], PARTLY] if nb == (2, 3, 2) else [WALLS[walls]]
    u, slabs, _ = build(nb, n, dtype, 41, lists)
    v, _, _ = build(nb, n, dtype, 41, lists)
    t, _, _ = build(nb, n, dtype, 41, lists)
    w, _, _ = build(nb, n, dtype, 41, lists)
    dt = 0.1 / (edge * max(nb)) ** 2
    norms, want = cnv.DeviceBuffer(8 * 7), cnv.DeviceBuffer(8 * 7)
    res = cnv.diffusion_run(u, t, 7, dt, norms)
    assert res is t
    a, b = v, w
    for k in range(7):
        cnv.diffusion_step(a, b, dt, sumsq=want.at(8 * k))
        a, b = b, a
    for c in range(len(lists)):
        assert_same(res.download(c), a.download(c), "component %d" % c)
    gn, wn = norms.download(np.float64, 7), want.download(np.float64, 7)
    assert np.max(np.abs(gn - wn) / wn) <= 1e-13
