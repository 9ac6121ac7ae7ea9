"""FP32 real-time phases beyond the range of the reduced sincos: V*dt/2 = 2m exactly (dt =
2^-10, V a multiple of 2^12), m up to 2^20, so that some points of a lane take the short
forms and some the library.  One step against numpy in 64 bits; a step is some 60 roundings
of 6e-8 a point, a random walk of 5e-7, so 5e-6 is ten times that."""
import numpy as np
import pytest

import gpue_amd as G
from tests.conftest import rel_l2, seeded_psi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(64, 48), (16, 512), (1024, 32), (32, 4096)])
@pytest.mark.parametrize("variants", [None, (0, 0, 0), (1, 1, 1)])
def test_large_phases(n, variants):
    rng = np.random.default_rng(7)
    nx, ny = n
    m = np.where(rng.uniform(size=(ny, nx)) < 0.7, 0, rng.integers(-2 ** 20, 2 ** 20, (ny, nx)))
    m[:, 0] = 2 ** 20 - 1
    dt = 2.0 ** -10
    with G.Context(dimnum=2, xDim=nx, yDim=ny, xMax=6.0, yMax=6.0, gdt=dt, dt=dt, precision=32) as c:
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
    assert rel_l2(got, ref) <= 5e-6
