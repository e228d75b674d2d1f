"""The reverse sweep by (block, channel) pairs (taken when I is kept through
the ray) against the sweep from checkpoints every two segments, which steps
every channel through every segment.

Tolerance: a gradient is a sum over rays and channels of lambda times an
element's derivative.  lambda is a product of up to a few hundred factors,
rounded in another order: sqrt(300) 2^-24 = 1e-6 of it (FP32), 2e-15 (FP64),
and a channel that does not see the line drops 2^-30 (2^-60) of the line's
gradient.  Taken four times that in FP32 and, for sums that cancel, 1e-13 in
FP64, relative to the largest gradient of the table.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from radlite_amd import engine, synth

pytestmark = pytest.mark.gpu


def _run(nr, nth, nfr, precision, kind, keep):
    disk = synth.make_disk(nr, nth, seed=3, sigma_t=0.1)
    lines = synth.single_line()
    pops = synth.lte_pops(disk, lines)
    if kind == "nodust":
        disk.rho_dust[:] = 0.0
    if kind == "weak":
        disk.abund *= 1e-9
    if kind == "inverted":
        pops = pops[..., ::-1].copy()
        disk.abund[:] = 1e-9
    v, dv = synth.passband(30.0, nfr)
    ri = synth.run_inputs(disk, lines, pops, nphi=6, dbdr=1, b_extra=-2, vmax=v, dv=dv,
                          incl_deg=50.0)
    rt = engine.Raytracer(0, precision)
    rt.load_run(ri)
    rt.setup_rays([0.87], ri.nphi, ri.b_extra, ri.dbdr)
    items = [(0, 0, nfr, 0.5 * (nfr - 1) * dv, engine.SKIP_NONE)]
    g = [np.random.default_rng(nfr).normal(size=nfr) * 1e20]
    rt.set_option(engine.OPT_CKPT, keep)
    f, gr = rt.adjoint(items, g)
    rt.close()
    return f, gr


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
# channels around the batch of 64 pairs and the group of 64 channels; rays of
# less than a window of 16 blocks and of several
@pytest.mark.parametrize("nr,nth,nfr,kind", [
    (6, 4, 2, "lte"), (10, 8, 9, "lte"), (10, 8, 63, "lte"), (12, 7, 64, "lte"),
    (12, 7, 65, "lte"), (90, 40, 24, "lte"), (40, 24, 257, "lte"), (24, 16, 33, "weak"),
    (24, 16, 33, "nodust"), (24, 16, 33, "inverted")])
def test_pairs_against_segments(nr, nth, nfr, kind, precision):
    if precision == "fp32" and kind in ("inverted", "nodust"):
        # single precision has no series for a negative depth, and without dust
        # its exponent range cuts the wings that coarse grids sample
        pytest.skip("not a single-precision model")
    fa, ga = _run(nr, nth, nfr, precision, kind, 1)
    fb, gb = _run(nr, nth, nfr, precision, kind, 2)
    assert np.array_equal(fa[0], fb[0])
    tol = 1e-13 if precision == "fp64" else 4e-6
    for k in ga:
        s = np.abs(gb[k]).max()
        print(k, np.abs(ga[k] - gb[k]).max() / s if s else 0.0, flush=True)
        assert np.abs(ga[k] - gb[k]).max() <= tol * s, k
