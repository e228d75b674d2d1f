"""The formal solution of few channels (up to 64), whose sparse windows take their
pairs from any number of blocks: against the CPU oracle at channel counts around a
group of 64, one to two channels a block and whole blocks of pairs, rays around one
and several windows of 64 blocks; and in calls that mix them with items of many
channels, in any order, bit for bit as each item alone.

Tolerances: 1e-10 of every channel of the spectrum in FP64, 1e-5 of the largest in
FP32, as for many channels; chunks of 16 channels give the same bits.
"""
import sys

import numpy as np
import pytest

import pyorc
from radlite_amd import engine, synth

pytestmark = pytest.mark.gpu


def _load(nr, nth, nphi, nfr, vmax, nlines=1):
    disk = synth.make_disk(nr, nth, seed=nr, sigma_t=0.1)
    lines = synth.single_line() if nlines == 1 else synth.random_lines(nlines, seed=2)
    v, dv = synth.passband(vmax, nfr)
    return synth.run_inputs(disk, lines, synth.lte_pops(disk, lines), nphi=nphi, dbdr=1,
                            b_extra=-2, vmax=v, dv=dv, incl_deg=50.0)


def _raytracer(ri, precision):
    rt = engine.Raytracer(0, precision)
    rt.load_run(ri)
    rt.setup_rays([ri.incl_deg * 0.0174532925199], ri.nphi, ri.b_extra, ri.dbdr)
    return rt


@pytest.mark.parametrize("nr,nth,nphi,nfr,vmax", [
    (6, 4, 4, 2, 20.0), (30, 20, 4, 3, 25.0), (240, 110, 2, 9, 45.0), (270, 130, 2, 13, 30.0),
    (60, 40, 4, 40, 30.0), (60, 40, 4, 63, 45.0), (60, 40, 4, 64, 45.0), (60, 40, 4, 65, 45.0),
    (240, 110, 2, 64, 1.0)])
def test_against_oracle(nr, nth, nphi, nfr, vmax):
    ri = _load(nr, nth, nphi, nfr, vmax)
    n, vm = engine.passband(ri.vmax, ri.dv)
    assert n == nfr
    for skip in (engine.SKIP_NONE, engine.SKIP_REFERENCE):
        ref = pyorc.Oracle(pyorc.Prepared(ri)).line_spectrum(0, want_image=False, skip_mode=skip)
        for precision in ("fp64", "fp32"):
            print(f"[gpu] few channels {nr}x{nth} {nfr} ch skip {skip} {precision}",
                  file=sys.stderr, flush=True)
            rt = _raytracer(ri, precision)
            items = [(0, 0, nfr, vm, skip)]
            fl, im, _ = rt.trace(items, want_image=True)
            if precision == "fp64":
                assert (np.abs(fl[0] - ref["flux"]) <= 1e-10 * np.abs(ref["flux"])).all()
            else:
                assert np.abs(fl[0] - ref["flux"]).max() <= 1e-5 * np.abs(ref["flux"]).max()
            rt.set_option(engine.OPT_TILE, 16)       # and the persistent grid
            _, ic, _ = rt.trace(items, want_image=True)
            assert np.array_equal(ic[0], im[0])
            rt.close()


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("nfrs", [(9, 100, 12, 300, 64, 65), (100, 9), (64, 64), (65, 65),
                                  (65, 2, 2, 2, 257)])
def test_mixed_calls_equal_single_ones(nfrs, precision):
    ri = _load(30, 20, 6, 9, 30.0, nlines=len(nfrs))
    print(f"[gpu] mixed channel counts {nfrs} {precision}", file=sys.stderr, flush=True)
    rt = _raytracer(ri, precision)
    items = [(il, 0, n, 30.0, il % 2) for il, n in enumerate(nfrs)]
    together = rt.trace(items, want_image=True)
    rt.set_option(engine.OPT_TILE, 32)
    persistent = rt.trace(items, want_image=True)
    for k, it in enumerate(items):
        alone = rt.trace([it], want_image=True)
        for got in (together, persistent):
            assert np.array_equal(got[0][k], alone[0][0]), it
            assert np.array_equal(got[1][k], alone[1][0]), it
            assert got[2][k] == alone[2][0], it
    rt.close()
