"""Batches of instances with axes of 16 and 32 points, whose narrow strided tiles are less
than a wave, in every kernel variant and after the batch's tuner, against lone contexts.

The two sides round differently (other plans): a step is some 60 roundings a point, 24
of them on two sides stay below 1e-12 in FP64 (1.1e-16 each, all aligned: 3.2e-13) and,
as a random walk of 6e-8, far below 1e-5 in FP32; a norm with a lane's share left out is
off by parts in a hundred."""
import numpy as np
import pytest

import gpue_amd as G
from tests.conftest import rel_l2, seeded_psi

pytestmark = pytest.mark.gpu
TOL = {64: 1e-12, 32: 1e-5}


def make(shape, prec, seed):
    dims = dict(zip(("xDim", "yDim", "zDim"), shape))
    c = G.Context(dimnum=len(shape), xMax=6.0, yMax=7.0, zMax=5.0, g=60.0 + seed, gpe=1, corotating=1, omega=0.2 * seed,
                  gdt=1e-3, dt=5e-4, precision=prec, **dims)
    c.upload(seeded_psi(c.shape, [c.grid(a) for a in range(c.dimnum)], seed=seed, phase=True))
    c.parsum()
    return c


@pytest.mark.parametrize("prec", [64, 32])
@pytest.mark.parametrize("shape", [(64, 16), (64, 32), (48, 16), (16, 32, 48)], ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("variant", ["tuned", 0, 1, 2, 3, 4, 5])
def test_small_axes_equal_alone(shape, prec, variant):
    batch = [make(shape, prec, k + 1) for k in range(3)]
    alone = [make(shape, prec, k + 1) for k in range(3)]
    if variant != "tuned":
        for c in batch:
            c.set_variants([variant] * 3)
    b = G.Batch(batch)
    steps = 0
    for n in (3, 21):
        b.evolve(n, 0)
        for c in alone:
            c.evolve(n, 0, first_step=steps)
        steps += n
        if variant == "tuned" and n == 3:
            b.autotune(0, 4)
    for x, y in zip(batch, alone):
        assert rel_l2(x.download(), y.download()) <= TOL[prec]
    b.close()
    for c in batch + alone:
        c.close()
