"""psi transfers on either side of the sizes where the way they take changes: 2 MiB (one
chunk), 8 MiB (chunk size, uploads) and 16 MiB (threads) on the device."""
import numpy as np
import pytest

import gpue_amd as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [64, 32])
@pytest.mark.parametrize("shape", [(32, 32), (32, 48), (32, 64), (48, 64), (128, 192), (128, 256), (256, 384), (256, 512),
                                   (384, 512), (1024, 512), (1024, 1024)])
def test_roundtrip(shape, prec):
    rng = np.random.default_rng(3)
    with G.Context(dimnum=2, xDim=shape[0], yDim=shape[1], xMax=5.0, yMax=5.0, precision=prec) as c:
        for _ in range(2):
            psi = rng.standard_normal(c.shape) + 1j * rng.standard_normal(c.shape)
            c.upload(psi)
            want = psi if prec == 64 else psi.astype(np.complex64).astype(np.complex128)
            assert np.array_equal(c.download(), want)


# an upload takes back a pending norm, whatever the order of its parts
def test_upload_drops_pending_norm():
    rng = np.random.default_rng(4)
    with G.Context(dimnum=2, xDim=64, yDim=48, xMax=5.0, yMax=5.0, gdt=1e-3) as c:
        psi = rng.standard_normal(c.shape) + 1j * rng.standard_normal(c.shape)
        c.upload(psi)
        c.evolve(3, 0)
        c.upload(psi)
        assert np.array_equal(c.download(), psi)
        c.evolve(1, 1)
        a = c.download()
    with G.Context(dimnum=2, xDim=64, yDim=48, xMax=5.0, yMax=5.0, gdt=1e-3) as c:
        c.upload(psi)
        c.evolve(1, 1)
        assert np.array_equal(c.download(), a)
