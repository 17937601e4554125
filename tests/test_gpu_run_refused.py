"""A run that a single step would refuse is refused before its first launch, with
u and tmp untouched, whether or not its launches of several steps would take the
grid; periodic grids of 16^3 and 32^3 blocks whose steps all pair up do run."""
import numpy as np
import pytest

import cubismnova_amd as cnv
from tests.helpers import assert_same, random_slab

pytestmark = pytest.mark.gpu


def grids(nb, n, ncomp=1, bcs=()):
    u, t = (cnv.Cartesian(nb, n, dtype=np.float32, ncomp=ncomp) for _ in range(2))
    slab = random_slab(7, nb, n, np.float32, u.block_stride)
    for c in range(ncomp):
        u.upload(c, slab)
        t.upload(c, -slab)
    for g in (u, t):
        for b in range(nb[1] * nb[2] if bcs else 0):
            g.setBC((0, b % nb[1], b // nb[1]), bcs)
    return u, t, slab


@pytest.mark.parametrize("steps", [1, 4, 5, 8])
@pytest.mark.parametrize("case", ["blocks", "list", "list on 16^3", "components"])
def test_refused_untouched(gpu, case, steps):
    long_list = [cnv.Absorbing(0, 0)] * 64 + [cnv.Absorbing(0, 1)]  # one rule per face
    u, t, slab = {"blocks": lambda: grids((41, 40, 40), (8, 8, 8)),
                  "list": lambda: grids((1, 2, 2), (8, 8, 8), bcs=long_list),
                  "list on 16^3": lambda: grids((1, 1, 2), (16, 16, 16), bcs=long_list),
                  "components": lambda: grids((2, 2, 2), (12, 12, 12), ncomp=9)}[case]()
    norms = cnv.DeviceBuffer(8 * steps)
    norms.fill(np.float64, -1.0)
    with pytest.raises(cnv.CnvError):
        cnv.diffusion_run(u, t, steps, 1e-6, norms)
    assert_same(u.download(0), slab)
    assert_same(t.download(0), -slab)
    assert np.all(norms.download(np.float64, steps) == -1.0)


@pytest.mark.parametrize("edge", [16, 32])
def test_nine_components_in_pairs(gpu, edge):
    nb, n = (2, 1, 2), (edge,) * 3
    u, t, slab = grids(nb, n, ncomp=9)
    a, b, _ = grids(nb, n)
    dt = 0.1 / (2 * edge) ** 2
    with pytest.raises(cnv.CnvError):
        cnv.diffusion_run(u, t, 5, dt)
    assert_same(u.download(8), slab)
    assert cnv.diffusion_run(u, t, 8, dt) is u
    for _ in range(8):
        cnv.diffusion_step(a, b, dt)
        a, b = b, a
    for c in (0, 8):
        assert_same(u.download(c), a.download(0), "component %d" % c)
