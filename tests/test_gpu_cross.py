"""The crossing pass by one wave per ray (few rays in a launch) against the one
by a thread per ray (many): the same rays, taken alone and in a launch of eight
inclinations that exceeds the bound, give the same bits in every intensity,
from the face-on to the edge-on disk, on grids whose rays have from a handful to
several hundred crossings; the exactly face-on disk, whose outermost rays the
reference stops at, is refused by both.
"""
import sys

import numpy as np
import pytest

from radlite_amd import engine, synth

pytestmark = pytest.mark.gpu

INCS = [x * 0.0174532925199 for x in (2.0, 4.0, 30.0, 45.0, 61.0, 80.0, 89.0, 90.0)]


@pytest.mark.parametrize("nr,nth,nphi,dbdr,b_extra", [
    (4, 3, 320, 9, -2), (17, 31, 250, 2, -5), (33, 32, 160, 2, -1), (64, 65, 150, 1, -7),
    (130, 40, 96, 1, -2)])
def test_wave_equals_thread(nr, nth, nphi, dbdr, b_extra):
    disk = synth.make_disk(nr, nth, seed=nr, sigma_t=0.1)
    lines = synth.single_line()
    v, dv = synth.passband(30.0, 3)
    ri = synth.run_inputs(disk, lines, synth.lte_pops(disk, lines), nphi=nphi, dbdr=dbdr,
                          b_extra=b_extra, vmax=v, dv=dv, incl_deg=30.0)
    nfr, vmax = engine.passband(ri.vmax, ri.dv)
    print(f"[gpu] crossings {nr}x{nth} {nphi} angles", file=sys.stderr, flush=True)
    rt = engine.Raytracer(0, "fp64")
    rt.load_run(ri)
    rays = rt.setup_rays(INCS, nphi, b_extra, dbdr)
    assert sum(rays) > 80000 >= max(rays)
    items = [(0, i, nfr, vmax, engine.SKIP_NONE) for i in range(len(INCS))]
    _, together, _ = rt.trace(items, want_image=True)
    nodes = rt.stats()["nodes"]
    alone = 0
    for i, inc in enumerate(INCS):
        rt.setup_rays([inc], nphi, b_extra, dbdr)
        _, im, _ = rt.trace([(0, 0, nfr, vmax, engine.SKIP_NONE)], want_image=True)
        alone += rt.stats()["nodes"]
        assert np.array_equal(im[0], together[i]), inc
    assert alone == nodes
    for incs in ([0.0], [0.0] + INCS[1:]):
        rt.setup_rays(incs, nphi, b_extra, dbdr)
        with pytest.raises(engine.RadliteError) as e:
            rt.trace([(0, i, nfr, vmax, engine.SKIP_NONE) for i in range(len(incs))])
        assert e.value.code == 13
    rt.close()
