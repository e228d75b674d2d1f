"""Single precision on models that FP64 cannot vouch for (no dust, where its exponent
range cuts the wings that coarse grids sample; inverted populations): the formal
solution by blocks and packed pairs against the single-precision forward of the
adjoint's tape at a checkpoint interval of 2, which steps every channel through
every segment, and the maser flag against FP64's.

Tolerance 1e-5 of the largest channel, as for single precision elsewhere: each
element's weights carry a few 2^-24, in another order in the two.
"""
import sys

import numpy as np
import pytest

from radlite_amd import engine, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["nodust", "inverted"])
@pytest.mark.parametrize("nr,nth,nfr", [(4, 3, 2), (9, 6, 16), (60, 40, 33), (130, 60, 65),
                                        (60, 40, 257)])
def test_blocks_against_segments(nr, nth, nfr, kind):
    disk = synth.make_disk(nr, nth, seed=nr, sigma_t=0.1)
    lines = synth.single_line()
    pops = synth.lte_pops(disk, lines)
    if kind == "nodust":
        disk.rho_dust[:] = 0.0
    else:
        pops = pops[..., ::-1].copy()
        disk.abund[:] = 1e-9
    v, dv = synth.passband(30.0, nfr)
    ri = synth.run_inputs(disk, lines, pops, nphi=9, dbdr=1, b_extra=-2, vmax=v, dv=dv,
                          incl_deg=50.0)
    n, vmax = engine.passband(ri.vmax, ri.dv)
    assert n == nfr
    items = [(0, 0, nfr, vmax, engine.SKIP_NONE)]
    print(f"[gpu] single precision {nr}x{nth} {nfr} ch {kind}", file=sys.stderr, flush=True)
    warn = {}
    for precision in ("fp64", "fp32"):
        rt = engine.Raytracer(0, precision)
        rt.load_run(ri)
        rt.setup_rays([ri.incl_deg * 0.0174532925199], ri.nphi, ri.b_extra, ri.dbdr)
        fl, _, w = rt.trace(items)
        warn[precision] = int(w[0]) & engine.WARN_MASER
        if precision == "fp32":
            rt.set_option(engine.OPT_CKPT, 2)
            ref = rt.trace_tape(items)[0]
            assert np.isfinite(ref).all()
            assert np.abs(fl[0] - ref).max() <= 1e-5 * np.abs(ref).max()
        rt.close()
    assert warn["fp32"] == warn["fp64"]
