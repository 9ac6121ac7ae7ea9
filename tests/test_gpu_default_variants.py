"""The variants a context starts with, on either side of the sizes where the rule changes,
against wide lines on whole-width tiles for every sweep."""
import numpy as np
import pytest

import gpue_amd as G
from tests.conftest import rel_l2, seeded_psi

pytestmark = pytest.mark.gpu

SHAPES = [(512, 512), (1024, 512), (512, 1024), (1024, 1024), (2048, 1024), (1024, 2048), (2048, 2048), (4096, 1024),
          (128, 64, 128), (128, 128, 96), (192, 192, 48), (192, 96, 192), (64, 64, 512), (256, 64, 256), (48, 256, 384)]


# Three imaginary and three real steps.  A step is about 60 roundings a point (1.1e-16, all
# aligned: 6.6e-15; FP32 6e-8, a random walk: 5e-7), six of them on two sides.
@pytest.mark.parametrize("prec,bound", [(64, 1e-13), (32, 6e-6)])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("tables", [False, True], ids=["rotating", "tables"])
def test_defaults_agree_with_wide_lines(shape, prec, bound, tables):
    dim = len(shape)
    kw = dict(dimnum=dim, xDim=shape[0], yDim=shape[1], zDim=shape[2] if dim == 3 else 1, xMax=6.0, yMax=6.0, zMax=6.0,
              g=20.0, gpe=1, gdt=1e-4, dt=1e-4, precision=prec)
    if not tables:
        kw.update(corotating=1, omega=0.5)
    got = []
    for variants in (None, (0, 0, 0)):
        with G.Context(**kw) as c:
            axes = [c.grid(a) for a in range(dim)]
            if tables:
                k2 = [c.grid(3 + a) ** 2 for a in range(dim)]
                add = lambda u: sum(v.reshape([-1 if dim - 1 - j == a else 1 for j in range(dim)]) for a, v in enumerate(u))
                c.set_field(G.FIELD_V, 0.4 * add([x * x for x in axes]))
                c.set_field(G.FIELD_K, 0.45 * add(k2))
            if variants:
                c.set_variants(variants)
            c.upload(seeded_psi(c.shape, axes, seed=9, phase=True))
            c.evolve(3, 0)
            c.evolve(3, 1)
            got.append(c.download())
    assert rel_l2(got[0], got[1]) <= bound
