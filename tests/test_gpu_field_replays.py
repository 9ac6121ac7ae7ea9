"""Captured blocks of time-dependent steps, replayed at several first steps: one graph of
eight steps many times over, and calls longer than two default blocks, against steps
launched one by one.  Up to 110 steps of some 40 roundings (1.1e-16) a point on two sides
stay below 1e-12 even if they all add up."""
import numpy as np
import pytest

import gpue_amd as G
from tests.conftest import rel_l2, seeded_psi

pytestmark = pytest.mark.gpu
TOL = 1e-12

FIELDS = {
    "V": {G.FIELD_V: "0.5*(x*x+y*y)*(1+0.5*sin(300*t))"},
    "VK": {G.FIELD_V: "0.5*(x*x+y*y)+x*sin(200*t)", G.FIELD_K: "0.5*(x*x+y*y)*(1+0.3*cos(100*t))"},
    "A": {G.FIELD_AX: "0-y*0.3*cos(200*t)", G.FIELD_AY: "x*0.3*cos(200*t)"},
}


@pytest.mark.parametrize("gauge", [0, 1])
@pytest.mark.parametrize("fields", sorted(FIELDS))
@pytest.mark.parametrize("block", [8, None])
def test_replays_follow_the_time(block, fields, gauge):
    got = []
    for steps in (block, 0):
        with G.Context(dimnum=2, xDim=48, yDim=64, xMax=6.0, yMax=6.0, g=10.0, gpe=1, corotating=gauge, omega=0.3,
                       gdt=1e-3, dt=1e-3) as c:
            c.upload(seeded_psi(c.shape, [c.grid(0), c.grid(1)], seed=5, phase=True))
            c.parsum()
            if steps is not None:
                c.set_graph_steps(steps)
            for which, e in FIELDS[fields].items():
                c.set_field_eqn(which, e)
            out = []
            for gstate, first, n in ((1, 0, 40), (1, 40, 70), (1, 13, 25), (0, 110, 33), (0, 7, 17)):
                c.evolve(n, gstate, first_step=first)
                out.append((c.download(), c.energy()))
            got.append(out)
    for (a, ea), (b, eb) in zip(*got):
        assert rel_l2(a, b) <= TOL
        assert np.all(np.abs(np.array(ea) - np.array(eb)) <= TOL * np.abs(np.array(eb)))
