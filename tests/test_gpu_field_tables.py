"""Time-dependent equation fields: the per-point program evaluator (k_fields_at)
against the evaluator of static equations, and captured blocks of steps (two V
tables, fused real-time boundaries) against steps launched one by one.

The two sides do the same arithmetic on the same values, in another order at
most: up to 48 steps of some 40 roundings (1.1e-16) a point stay below 1e-12
even if they all add up.
"""
import numpy as np
import pytest

import gpue_amd as G
from tests.conftest import rel_l2, seeded_psi

pytestmark = pytest.mark.gpu
TOL = 1e-12


def make(n, gauge=0, **kw):
    c = G.Context(dimnum=2, xDim=n[0], yDim=n[1], xMax=6.0, yMax=6.0, g=10.0, gpe=1, corotating=gauge, omega=0.3,
                  gdt=1e-3, dt=1e-3, **kw)
    c.upload(seeded_psi(c.shape, [c.grid(0), c.grid(1)], seed=5, phase=True))
    c.parsum()
    return c


# every operator, both stack depths (programs of up to 4 slots and of 5 to 8), one
# point per lane and four (grids above 2^19 points); "0*t" makes them time dependent
@pytest.mark.parametrize("n", [(48, 32), (96, 16), (1024, 1024)])
@pytest.mark.parametrize("expr", [
    "0.5*(x*x+y*y)+0.3*cos(x)*sin(y)",
    "0.1*exp(0-(x*x+y*y)/4)+sqrt(1+x*x)+0.01*tan(0.1*y)+pow(x,2)/9",
    "jn(1,x)+0.2*(x-y)^2",
    "0.1*(x+(y+(x*(y+(x*(0.5*y))))))",
    "2+sin(1.5)*cos(0.25)",
])
def test_evaluator_matches_static_fields(n, expr):
    a, b = make(n), make(n)
    a.set_field_eqn(G.FIELD_V, expr)
    b.set_field_eqn(G.FIELD_V, "(" + expr + ")+0*t")
    for c in (a, b):
        c.evolve(4, 1)
    assert rel_l2(b.download(), a.download()) <= TOL
    a.close()
    b.close()


CASES = {
    "V": {G.FIELD_V: "0.5*(x*x+y*y)*(1+0.5*sin(300*t))"},
    "VK": {G.FIELD_V: "0.5*(x*x+y*y)+x*sin(200*t)", G.FIELD_K: "0.5*(x*x+y*y)*(1+0.3*cos(100*t))"},
    "A": {G.FIELD_AX: "0-y*0.3*cos(200*t)", G.FIELD_AY: "x*0.3*cos(200*t)"},
    "VA": {G.FIELD_V: "0.5*(x*x+y*y)*(1+0.5*sin(300*t))", G.FIELD_AX: "0-y*0.3*(1+50*t)"},
}


# blocks of 8 and 2 steps and single ones, from even and odd first steps; a static V
# afterwards drops the second table
@pytest.mark.parametrize("gauge", [0, 1])
@pytest.mark.parametrize("case", sorted(CASES))
def test_blocks_equal_single_steps(case, gauge):
    blocks, single = make((48, 64), gauge), make((48, 64), gauge)
    single.set_graph_steps(0)
    for c in (blocks, single):
        for which, e in CASES[case].items():
            c.set_field_eqn(which, e)
    for gstate, first, steps in ((0, 0, 13), (1, 13, 21), (1, 40, 8), (0, 7, 6)):
        for c in (blocks, single):
            c.evolve(steps, gstate, first_step=first)
        assert rel_l2(blocks.download(), single.download()) <= TOL, (gstate, first, steps)
        (ea, ma), (eb, mb) = blocks.energy(), single.energy()
        assert abs(ea - eb) <= TOL * abs(eb) and abs(ma - mb) <= TOL * abs(mb)
    for c in (blocks, single):
        c.set_field_eqn(G.FIELD_V, "0.5*(x*x+y*y)")
        c.evolve(10, 1)
    assert rel_l2(blocks.download(), single.download()) <= TOL
    blocks.close()
    single.close()
