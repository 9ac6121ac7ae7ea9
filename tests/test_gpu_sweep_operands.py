"""Operands and reductions of the sweeps at the sizes where they can go wrong:
norm partials reduced inside the next step's first sweep (one to four chunks of
1024 partials, workgroups of one line up to many), and phases beyond the range of
the reduced sincos (the library path, one point at a time)."""
import numpy as np
import pytest

import gpue_amd as G
from tests.conftest import rel_l2, seeded_psi

pytestmark = pytest.mark.gpu


# steps of one call leave the norm to the next step's first sweep; steps of separate
# calls are closed by the finalize kernel: the same additions, bit for bit
@pytest.mark.parametrize("prec", [64, 32])
@pytest.mark.parametrize("n", [(16, 16), (48, 16), (16, 4096), (2048, 64), (384, 1024), (512, 2048)])
@pytest.mark.parametrize("gauge", [0, 1])
def test_deferred_norm_equals_finalize(n, gauge, prec):
    out = []
    for steps in (1, 6):
        with G.Context(dimnum=2, xDim=n[0], yDim=n[1], xMax=6.0, yMax=6.0, g=50.0, gpe=1, corotating=gauge, omega=0.4,
                       gdt=1e-3, precision=prec) as c:
            c.upload(seeded_psi(c.shape, [c.grid(0), c.grid(1)], seed=4, phase=True))
            c.parsum()
            for s in range(0, 6, steps):
                c.evolve(steps, 0, first_step=s)
            out.append(c.download())
    assert np.array_equal(out[0], out[1])


# V*dt/2 = 2m exactly (dt = 2^-10, V a multiple of 2^12), m up to 2^22: some points of a
# lane take short polynomials, some the reduction, some the library; one step with
# periodic reference phases of 2m from numpy.  FP64 error bound: about 60 roundings of
# 1.1e-16 a point, 1e-13 with room for the worst alignment.
@pytest.mark.parametrize("n", [(64, 48), (16, 512), (1024, 32)])
@pytest.mark.parametrize("variants", [None, (0, 0, 0), (1, 1, 1)])
def test_large_phases(n, variants):
    rng = np.random.default_rng(7)
    nx, ny = n
    m = np.where(rng.uniform(size=(ny, nx)) < 0.7, 0, rng.integers(-2 ** 22, 2 ** 22, (ny, nx)))
    m[:, 0] = 2 ** 22 - 1
    dt = 2.0 ** -10
    with G.Context(dimnum=2, xDim=nx, yDim=ny, xMax=6.0, yMax=6.0, gdt=dt, dt=dt) as c:
        if variants:
            c.set_variants(variants)
        c.set_field(G.FIELD_V, m * 2.0 ** 12)
        psi = seeded_psi(c.shape, [c.grid(0), c.grid(1)], seed=6, phase=True)
        c.upload(psi)
        c.evolve(1, 1)
        got = c.download()
        kx, ky = c.grid(3), c.grid(4)
    half = np.exp(-2j * m.astype(float))
    K = 0.5 * (kx[None, :] ** 2 + ky[:, None] ** 2)
    ref = half * np.fft.ifft2(np.exp(-1j * K * dt) * np.fft.fft2(half * psi))
    assert rel_l2(got, ref) <= 1e-13
