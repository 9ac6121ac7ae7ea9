"""Batches whose instances of different sizes share launches: every axis length with a
merged kernel, boxes, 2D and 3D, both precisions, with and without gauge, against the
same contexts alone (bit for bit), and batches that mix them with others."""
import numpy as np
import pytest

import gpue_amd as G
from tests.conftest import seeded_psi

pytestmark = pytest.mark.gpu


def make(shape, prec, gauge, seed, **kw):
    dims = dict(zip(("xDim", "yDim", "zDim"), shape))
    c = G.Context(dimnum=len(shape), xMax=6.0, yMax=7.0, zMax=5.0, g=60.0 + seed, gpe=1, corotating=gauge,
                  omega=0.1 * seed, gdt=1e-3, dt=5e-4, precision=prec, **dims, **kw)
    c.upload(seeded_psi(c.shape, [c.grid(a) for a in range(c.dimnum)], seed=seed, phase=True))
    c.parsum()
    c.set_graph_steps(0)
    return c


GRIDS = {
    # all seven lengths on both axes; blocks that fill a workgroup and ones that do not
    "2d": [(64, 96), (96, 64), (128, 512), (512, 128), (192, 384), (384, 192), (256, 256)],
    "3d": [(64, 64, 64), (64, 128, 96), (96, 64, 64)],
    # an unmerged shape (48), one with other variants (2048) and a 1D line among them
    "mixed": [(64, 64), (48, 64), (128, 64), (2048, 64), (128,)],
}


@pytest.mark.parametrize("prec", [64, 32])
@pytest.mark.parametrize("gauge", [0, 1])
@pytest.mark.parametrize("grids", sorted(GRIDS))
def test_merged_equals_alone(grids, gauge, prec):
    shapes = GRIDS[grids]
    batch = [make(s, prec, gauge, k + 1) for k, s in enumerate(shapes)]
    alone = [make(s, prec, gauge, k + 1) for k, s in enumerate(shapes)]
    for c in (batch[1], alone[1]):   # mixed step parities
        c.evolve(1, 0)
    first = [1 if k == 1 else 0 for k in range(len(shapes))]
    b = G.Batch(batch)
    b.set_active(2, False)
    active = [k != 2 for k in range(len(shapes))]

    def check(steps, gstate):
        b.evolve(steps, gstate)
        for k, c in enumerate(alone):
            if active[k]:
                c.evolve(steps, gstate, first_step=first[k])
                first[k] += steps
            assert np.array_equal(batch[k].download(), c.download()), (shapes[k], steps, gstate)

    check(1, 0)
    check(2, 0)
    b.set_active(2, True)
    active[2] = True
    check(21, 0)   # single steps, a block of 16, pairs and a tail
    check(19, 1)
    check(3, 0)
    e, m = b.energy()
    for k, c in enumerate(alone):
        assert (e[k], m[k]) == c.energy()
    b.close()
    for c in batch + alone:
        c.close()
