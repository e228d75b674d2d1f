"""Lines of negative rest frequency (a level file whose upper level lies below
the lower one in energy): the channel velocities dnu/nu0 descend.  Spectrum and
image against the CPU oracle, populations as a normal line's and inverted (as
the reversed levels' own Boltzmann factors are), around one and several groups
of 64 channels and a second chunk; and the device-physics gradient by (block,
channel) pairs against the sweep that steps every channel through every
segment.

Tolerances as for lines of positive frequency, each relative to the largest
value (the negative frequency makes the line's emission negative, so that single
channels can pass through 0): FP64 1e-10 in the spectrum and 1e-8 in the image,
FP32 1e-5; gradients 1e-13 (FP64) and 4e-6 (FP32) of the table's largest.
"""
import sys

import numpy as np
import pytest

torch = pytest.importorskip("torch")

import pyorc
from radlite_amd import diff, engine, synth

pytestmark = pytest.mark.gpu


def _model(nr, nth, nfr, vmax, abund, inverted):
    disk = synth.make_disk(nr, nth, seed=nr, sigma_t=0.1)
    disk.abund[:] = abund
    lines = synth.single_line()
    pops = synth.lte_pops(disk, lines)
    if inverted:
        pops = pops[..., ::-1].copy()
    v, dv = synth.passband(vmax, nfr)
    ri = synth.run_inputs(disk, lines, pops, nphi=6, dbdr=1, b_extra=-2, vmax=v, dv=dv,
                          incl_deg=50.0)
    ri.E_cm = np.asarray(ri.E_cm)[::-1].copy()
    return ri


@pytest.mark.parametrize("inverted", [False, True])
@pytest.mark.parametrize("nr,nth,nfr,vmax", [
    (10, 8, 3, 30.0), (20, 12, 33, 30.0), (60, 40, 50, 30.0), (30, 20, 65, 12.0),
    (30, 20, 257, 25.0)])
def test_spectrum_against_oracle(nr, nth, nfr, vmax, inverted):
    ri = _model(nr, nth, nfr, vmax, 1e-9 if inverted else 1e-4, inverted)
    prep = pyorc.Prepared(ri)
    assert (prep.nu0 < 0.0).all()
    n, vm = engine.passband(ri.vmax, ri.dv)
    assert n == nfr
    for skip in (engine.SKIP_NONE, engine.SKIP_REFERENCE):
        ref = pyorc.Oracle(prep).line_spectrum(0, skip_mode=skip)
        # the line is seen: it is not the dust's spectrum
        assert np.ptp(ref["flux"]) > 1e-6 * np.abs(ref["flux"]).max()
        for precision in ("fp64", "fp32"):
            if precision == "fp32" and inverted:
                continue          # single precision has no series for a negative depth
            print(f"[gpu] descending {nr}x{nth} {nfr} ch skip {skip} {precision}",
                  file=sys.stderr, flush=True)
            rt = engine.Raytracer(0, precision)
            rt.load_run(ri)
            rt.setup_rays([ri.incl_deg * 0.0174532925199], ri.nphi, ri.b_extra, ri.dbdr)
            fl, im, warn = rt.trace([(0, 0, nfr, vm, skip)], want_image=True)
            rt.close()
            tol = (1e-10, 1e-8) if precision == "fp64" else (1e-5, 1e-5)
            assert np.abs(fl[0] - ref["flux"]).max() <= tol[0] * np.abs(ref["flux"]).max()
            assert np.abs(im[0] - ref["image"]).max() <= tol[1] * np.abs(ref["image"]).max()
            if precision == "fp64":
                assert bool(warn[0] & engine.WARN_MASER) == bool(ref["maser"])


def _gradient(nfr, precision, keep):
    ri = _model(24, 16, nfr, 30.0, 1e-9, True)
    m = diff.SpectrumModel(ri, precision=precision, incl_rad=[0.87])
    assert m.tables.nu0[0] < 0.0
    m.rt.set_option(engine.OPT_CKPT, keep)
    rng = np.random.default_rng(nfr)
    shape = ri.rho_gas.shape
    x = [torch.from_numpy(a).requires_grad_(True)
         for a in (ri.t_dust[0].copy(), np.log(1e-9) + 0.1 * rng.normal(size=shape),
                   0.1 + 0.05 * rng.random(shape))]
    f = m.flux_from_physics_device(*x)
    (f * torch.from_numpy(rng.normal(size=nfr)) * 1e20).sum().backward()
    m.close()
    return f.detach().numpy(), [a.grad.numpy() for a in x]


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("nfr", [9, 65])
def test_gradient_pairs_against_segments(nfr, precision):
    fa, ga = _gradient(nfr, precision, 1)
    fb, gb = _gradient(nfr, precision, 2)
    assert np.isfinite(fb).all() and all(np.isfinite(g).all() for g in gb)
    assert np.abs(fa - fb).max() <= (1e-14 if precision == "fp64" else 1e-6) * np.abs(fb).max()
    for a, b in zip(ga, gb):
        assert np.abs(b).max() > 0.0
        assert np.abs(a - b).max() <= (1e-13 if precision == "fp64" else 4e-6) * np.abs(b).max()
