"""psi through the pinned chunks, both ways: one chunk and a part of one, the edges of
the chunk sizes, transfers that use threads, and several at once.  Doubles come back
as they were, FP32 psi rounded to nearest."""
import threading

import numpy as np
import pytest

import gpue_amd as G

pytestmark = pytest.mark.gpu

# psi of 256 B, 1 MiB, 2 MiB, 2.25, 8, 9, 12, 13.5, 16, 32 and 54 MiB in FP64 (half in FP32)
SHAPES = [(16,), (256, 256), (256, 512), (384, 384), (512, 1024), (192, 64, 48), (192, 4096), (96, 96, 96),
          (1024, 1024), (2048, 1024), (192, 192, 96)]


def make(shape, prec):
    dims = dict(zip(("xDim", "yDim", "zDim"), shape))
    return G.Context(dimnum=len(shape), xMax=5.0, yMax=5.0, zMax=5.0, precision=prec, **dims)


def roundtrip(shape, prec, seed):
    rng = np.random.default_rng(seed)
    with make(shape, prec) as c:
        for _ in range(2):
            psi = rng.standard_normal(c.shape) + 1j * rng.standard_normal(c.shape)
            c.upload(psi)
            want = psi if prec == 64 else psi.astype(np.complex64).astype(np.complex128)
            if not np.array_equal(c.download(), want):
                return False
    return True


@pytest.mark.parametrize("prec", [64, 32])
@pytest.mark.parametrize("shape", SHAPES)
def test_roundtrip(shape, prec):
    assert roundtrip(shape, prec, 1)


def test_several_at_once():
    ok = []
    shapes = [(1024, 1024), (192, 192, 96), (256, 256), (384, 1024), (96, 96, 96)]
    ts = [threading.Thread(target=lambda s=s, p=p, k=k: ok.append(roundtrip(s, p, k)))
          for k, (s, p) in enumerate((s, p) for s in shapes for p in (64, 32))]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert ok == [True] * len(ts)
