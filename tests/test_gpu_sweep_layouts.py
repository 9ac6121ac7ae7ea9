"""LDS exchange layouts of every plan and tile width: each supported length along the row
and the strided axis, next to an axis that fills no tile, in all kernel variants."""
import numpy as np
import pytest

import gpue_amd as G
from tests.conftest import rel_l2, seeded_psi

pytestmark = pytest.mark.gpu

LENGTHS = [16, 32, 48, 64, 96, 128, 192, 256, 384, 512, 1024, 2048, 4096]


# One real-time step against numpy.  FP64 as in the operand tests: about 60 roundings of
# 1.1e-16 a point.  FP32: psi in and out, two V/2, two transforms an axis of up to 12
# butterfly levels, about 60 roundings of 6e-8 that add up like a random walk: 5e-7; 2e-6
# leaves a factor of four.
@pytest.mark.parametrize("prec,bound", [(64, 1e-13), (32, 2e-6)])
@pytest.mark.parametrize("n", LENGTHS)
@pytest.mark.parametrize("axis", [0, 1])
def test_every_variant_of_a_length(axis, n, prec, bound):
    nx, ny = (n, 48) if axis == 0 else (48, n)
    dt = 2.0 ** -6 * min(1.0, 64.0 / n) ** 2   # K dt of 2 rad at most on the long axis
    with G.Context(dimnum=2, xDim=nx, yDim=ny, xMax=6.0, yMax=6.0, gdt=dt, dt=dt, precision=prec) as c:
        x, y, kx, ky = c.grid(0), c.grid(1), c.grid(3), c.grid(4)
        psi = seeded_psi(c.shape, [x, y], seed=8, phase=True)
        half = np.exp(-0.25j * dt * (x[None, :] ** 2 + y[:, None] ** 2))
        K = 0.5 * (kx[None, :] ** 2 + ky[:, None] ** 2)
        ref = half * np.fft.ifft2(np.exp(-1j * K * dt) * np.fft.fft2(half * psi))
        for v in range(6):
            c.set_variants((v % 4, v, 0))
            c.upload(psi)
            c.evolve(1, 1)
            assert rel_l2(c.download(), ref) <= bound, f"variant {v}"
