"""1D problems: runs of steps in one launch against steps launched one by one, at
every axis length (one lane per line up to eight waves).  FP64 differs by rounding
only: 9 steps of some 100 roundings (1.1e-16) a point stay below 1e-12; FP32
(6e-8 a rounding) below 1e-5, the bar of its psi elsewhere."""
import numpy as np
import pytest

import gpue_amd as G
from tests.conftest import rel_l2, seeded_psi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [64, 32])
@pytest.mark.parametrize("n", [16, 32, 48, 64, 96, 128, 192, 256, 384, 512, 1024, 2048, 4096])
@pytest.mark.parametrize("plan", [0, 1])
def test_line_runs_equal_single_steps(n, plan, prec):
    runs, single = [], []
    for out, graph_steps in ((runs, 8), (single, 0)):
        with G.Context(dimnum=1, xDim=n, xMax=8.0, g=30.0, gpe=1, corotating=1, gdt=1e-3, dt=1e-3, precision=prec) as c:
            c.set_graph_steps(graph_steps)
            c.set_variants((plan, 0, 0))
            psi = seeded_psi(c.shape, [c.grid(0)], seed=8, phase=True)
            c.upload(psi)
            c.parsum()
            r, e = c.evolve(9, 0, energy_every=4)   # energies after steps 0, 4 and 8
            out.append((c.download(), e))
            c.evolve(7, 1)
            c.set_field(G.FIELD_AX, 0.2 * np.cos(c.grid(0)))
            c.evolve(1, 0, first_step=9)
            c.evolve(6, 1, first_step=10)
            out.append((c.download(), np.array(c.energy())))
    tol = 1e-12 if prec == 64 else 1e-5
    for (a, ea), (b, eb) in zip(runs, single):
        assert rel_l2(a, b) <= tol
        assert len(ea) == len(eb) and np.all(np.abs(ea - eb) <= tol * np.abs(eb))
