"""Rows of 4096 points in small FP64 grids: the default variant, which loads late, gives
the bits of the one with operands up front."""
import numpy as np
import pytest

import gpue_amd as G
from tests.conftest import seeded_psi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(4096, 16), (4096, 64), (4096, 16, 16)], ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("gauge", [0, 1])
def test_late_loads_keep_the_bits(shape, gauge):
    got = []
    for variants in (None, (3, 5, 5)):
        with G.Context(dimnum=len(shape), xDim=4096, yDim=16 if len(shape) == 3 else shape[1], zDim=shape[-1], xMax=6.0,
                       yMax=6.0, zMax=6.0, g=20.0, gpe=1, gdt=1e-3, dt=1e-3, corotating=gauge, omega=0.4) as c:
            assert c.variants()[0] == 1
            if variants:
                c.set_variants(variants)
            c.upload(seeded_psi(c.shape, [c.grid(a) for a in range(len(shape))], seed=2, phase=True))
            c.evolve(4, 0)
            c.evolve(4, 1)
            got.append(c.download())
    assert np.array_equal(got[0], got[1])
