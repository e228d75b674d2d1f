"""Large host arrays through the pinned slots: arrays around the least size taken
that way (16 MiB) and of several pieces with a remainder, up and down.  The
resampled image is a sum of products in a fixed order, the same in numpy: equal
bit for bit.
"""
import numpy as np
import pytest

pytest.importorskip("torch")

from radlite_amd import engine

pytestmark = pytest.mark.gpu

MIB16 = (16 << 20) // 8


@pytest.mark.parametrize("nrays,npix,nfr", [
    (MIB16 // 64 - 1, MIB16 // 64 - 1, 64),       # one row short of it
    (MIB16 // 64, MIB16 // 64, 64),               # exactly
    (40009, 50021, 61),                           # 19.5 and 24.4 MB, odd
])
def test_resample_through_slots(nrays, npix, nfr):
    rng = np.random.default_rng(nrays)
    img = rng.normal(size=(nrays, nfr))
    vtx = rng.integers(-1, nrays, size=(npix, 3)).astype(np.int32)
    w = rng.normal(size=(npix, 3))
    ref = np.zeros((npix, nfr))
    for k in range(3):
        v = vtx[:, k]
        ref = np.where((v >= 0)[:, None], ref + w[:, k:k + 1] * img[np.maximum(v, 0)], ref)
    rt = engine.Raytracer(0, "fp64")
    for _ in range(2):                            # a first call, and one on kept buffers
        out = rt.resample_image(img, vtx, w)
        assert np.array_equal(out, ref.T)
    rt.close()
