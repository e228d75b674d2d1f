"""Line-free blocks and the wave walk of the formal solution, at the sizes and
models where they can go wrong, against the CPU oracle: rays shorter than a
block, around a block's and a window's end (8 and 128 segments), channel
counts around a wave's 16 channels per ray; no dust (a line that is never
below the dust), a line too weak to be seen anywhere, inverted populations.

Tolerances: FP64 as everywhere, 1e-10 per channel and 1e-8 per ray (the
cancellation in e1 = dtau - e0 amplifies a rounding by up to 1e8).  FP32 1e-5 of
the largest channel: each element's weights carry a few 2^-24, and some tens
of elements make up a channel's intensity.
"""
import sys

import numpy as np
import pytest

import pyorc
from radlite_amd import engine, synth

pytestmark = pytest.mark.gpu


def _model(nr, nth, nfr, kind, seed):
    disk = synth.make_disk(nr, nth, seed=seed, sigma_t=0.1)
    lines = synth.single_line()
    pops = synth.lte_pops(disk, lines)
    if kind == "nodust":
        disk.rho_dust[:] = 0.0
    if kind == "weak":
        disk.abund[:] = 1e-30
    if kind == "inverted":
        pops = pops[..., ::-1].copy()
        disk.abund[:] = 1e-9
    v, dv = synth.passband(30.0, nfr)
    return synth.run_inputs(disk, lines, pops, nphi=9, dbdr=1, b_extra=-2, vmax=v, dv=dv,
                            incl_deg=50.0)


@pytest.mark.parametrize("kind", ["lte", "nodust", "weak", "inverted"])
@pytest.mark.parametrize("nr,nth,nfr", [(4, 3, 2), (5, 4, 15), (9, 6, 16), (12, 9, 17),
                                        (60, 40, 33), (130, 60, 65)])
def test_blocks_against_oracle(nr, nth, nfr, kind):
    ri = _model(nr, nth, nfr, kind, seed=nr)
    orc = pyorc.Oracle(pyorc.Prepared(ri))
    n, vmax = engine.passband(ri.vmax, ri.dv)
    assert n == nfr
    for skip in (engine.SKIP_NONE, engine.SKIP_REFERENCE):
        ref = orc.line_spectrum(0, skip_mode=skip)
        top = np.max(np.abs(ref["image"]))
        for precision in ("fp64", "fp32"):
            print(f"[gpu] blocks {nr}x{nth} {nfr} ch {kind} skip {skip} {precision}",
                  file=sys.stderr, flush=True)
            if precision == "fp32" and kind in ("inverted", "nodust"):
                # single precision has no series for a negative depth, and without
                # dust its exponent range cuts the wings that coarse grids sample
                continue
            rt = engine.Raytracer(0, precision)
            rt.load_run(ri)
            rt.setup_rays([ri.incl_deg * 0.0174532925199], ri.nphi, ri.b_extra, ri.dbdr)
            fl, im, warn = rt.trace([(0, 0, nfr, vmax, skip)], want_image=True)
            rt.close()
            if precision == "fp64":
                ok = np.abs(fl[0] - ref["flux"]) <= 1e-10 * np.abs(ref["flux"])
                assert ok.all()
                # (without dust a ray's light can come from one element of that
                # kind alone: held against the brightest there)
                near = top if kind == "nodust" else np.abs(ref["image"])
                assert (np.abs(im[0] - ref["image"]) <= 1e-8 * near).all()
                assert bool(warn[0] & engine.WARN_MASER) == bool(ref["maser"])
                assert bool(warn[0] & engine.WARN_OVERSHOOT) == (ref["overshoot"] > 0)
            else:
                assert np.abs(fl[0] - ref["flux"]).max() <= 1e-5 * np.abs(ref["flux"]).max()
                assert np.abs(im[0] - ref["image"]).max() <= 1e-5 * top
