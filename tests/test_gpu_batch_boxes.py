"""Boxes of enough shapes to share merged launches in FP64 too, against the same contexts
alone (bit for bit)."""
import numpy as np
import pytest

import gpue_amd as G
from tests.conftest import seeded_psi

pytestmark = pytest.mark.gpu
SHAPES = [(64, 64, 64), (64, 128, 96), (96, 64, 64), (64, 64, 128), (64, 96, 64)]


@pytest.mark.parametrize("prec", [64, 32])
@pytest.mark.parametrize("gauge", [0, 1])
def test_five_shapes_equal_alone(gauge, prec):
    def make(shape, seed):
        c = G.Context(dimnum=3, xDim=shape[0], yDim=shape[1], zDim=shape[2], xMax=6.0, yMax=7.0, zMax=5.0, g=60.0 + seed,
                      gpe=1, corotating=gauge, omega=0.1 * seed, gdt=1e-3, dt=5e-4, precision=prec)
        c.upload(seeded_psi(c.shape, [c.grid(a) for a in range(3)], seed=seed, phase=True))
        c.parsum()
        c.set_graph_steps(0)
        return c

    batch = [make(s, k + 1) for k, s in enumerate(SHAPES)]
    alone = [make(s, k + 1) for k, s in enumerate(SHAPES)]
    b = G.Batch(batch)
    first = 0
    for steps, gstate in ((19, 0), (4, 1), (2, 0)):
        b.evolve(steps, gstate)
        for c in alone:
            c.evolve(steps, gstate, first_step=first)
        first += steps
        for x, y in zip(batch, alone):
            assert np.array_equal(x.download(), y.download()), (x.shape, steps, gstate)
    b.close()
    for c in batch + alone:
        c.close()
