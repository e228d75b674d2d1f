"""Resampling around the least array that goes through the pinned slots, 8 MiB, up or
down or both: the same sums of products as numpy's, bit for bit.
"""
import numpy as np
import pytest

pytest.importorskip("torch")

from radlite_amd import engine

pytestmark = pytest.mark.gpu

ROWS = (8 << 20) // 8 // 32                        # rows of 32 channels in 8 MiB


@pytest.mark.parametrize("nrays,npix", [(ROWS - 1, ROWS - 1), (ROWS, ROWS), (ROWS + 1, 100),
                                        (100, ROWS + 1)])
def test_resample(nrays, npix):
    rng = np.random.default_rng(nrays)
    img = rng.normal(size=(nrays, 32))
    vtx = rng.integers(-1, nrays, size=(npix, 2)).astype(np.int32)
    w = rng.normal(size=(npix, 2))
    ref = np.zeros((npix, 32))
    for k in range(2):
        v = vtx[:, k]
        ref = np.where((v >= 0)[:, None], ref + w[:, k:k + 1] * img[np.maximum(v, 0)], ref)
    rt = engine.Raytracer(0, "fp64")
    for _ in range(2):
        assert np.array_equal(rt.resample_image(img, vtx, w), ref.T)
    rt.close()
