"""The packed (block, channel) pairs of the formal solution, at the sizes where
their bookkeeping can go wrong, against the CPU oracle: channel counts around a
chunk (256) and a second one, rays around the 64 block records held at a time
(512 nodes), channels finer than the line (a block's pairs are the whole
chunk), channels coarser than it (few pairs per block, many blocks per batch),
and channel tilings that cut a block's pairs.

Tolerances: 1e-10 of every channel of the spectrum in FP64, 1e-5 of the largest
in FP32; the images of all tilings are the same bits.
"""
import sys

import numpy as np
import pytest

import pyorc
from radlite_amd import engine, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nr,nth,nphi,nfr,vmax", [
    (30, 20, 4, 255, 25.0), (30, 20, 4, 256, 25.0), (30, 20, 4, 257, 25.0),
    (12, 9, 4, 513, 2.0), (40, 24, 4, 300, 1.0), (150, 60, 2, 9, 60.0),
    (240, 110, 2, 40, 30.0), (270, 130, 2, 33, 30.0)])
def test_pairs_against_oracle(nr, nth, nphi, nfr, vmax):
    disk = synth.make_disk(nr, nth, seed=nr, sigma_t=0.1)
    lines = synth.single_line()
    v, dv = synth.passband(vmax, nfr)
    ri = synth.run_inputs(disk, lines, synth.lte_pops(disk, lines), nphi=nphi, dbdr=1,
                          b_extra=-2, vmax=v, dv=dv, incl_deg=50.0)
    n, vm = engine.passband(ri.vmax, ri.dv)
    assert n == nfr
    ref = pyorc.Oracle(pyorc.Prepared(ri)).line_spectrum(0, want_image=False, skip_mode=1)
    for precision in ("fp64", "fp32"):
        print(f"[gpu] pairs {nr}x{nth} {nfr} ch {precision}", file=sys.stderr, flush=True)
        rt = engine.Raytracer(0, precision)
        rt.load_run(ri)
        rt.setup_rays([ri.incl_deg * 0.0174532925199], ri.nphi, ri.b_extra, ri.dbdr)
        items = [(0, 0, nfr, vm, engine.SKIP_NONE)]
        fl, im, _ = rt.trace(items, want_image=True)
        if precision == "fp64":
            assert (np.abs(fl[0] - ref["flux"]) <= 1e-10 * np.abs(ref["flux"])).all()
        else:
            assert np.abs(fl[0] - ref["flux"]).max() <= 1e-5 * np.abs(ref["flux"]).max()
        for cw in (16, 64):                          # whatever the chunk, the same bits
            rt.set_option(engine.OPT_TILE, cw)
            _, ic, _ = rt.trace(items, want_image=True)
            assert np.array_equal(ic[0], im[0])
        rt.close()
