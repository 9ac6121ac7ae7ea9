"""A 1D call that takes several launches gives the bits of calls of single launches."""
import numpy as np
import pytest

import gpue_amd as G
from tests.conftest import seeded_psi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [64, 32])
@pytest.mark.parametrize("n,steps", [(64, 1500), (4096, 600)])
def test_split_runs_keep_their_bits(n, steps, prec):
    got = []
    for calls in ([steps], [100] * (steps // 100)):
        with G.Context(dimnum=1, xDim=n, xMax=8.0, g=30.0, gpe=1, gdt=1e-3, dt=1e-3, precision=prec) as c:
            c.upload(seeded_psi(c.shape, [c.grid(0)], seed=8, phase=True))
            c.parsum()
            first = 0
            for k in calls:
                c.evolve(k, 0, first_step=first)
                first += k
            for k in calls:
                c.evolve(k, 1, first_step=first)
                first += k
            got.append((c.download(), c.energy()))
    assert np.array_equal(got[0][0], got[1][0]) and got[0][1] == got[1][1]
