"""Device memory of resampling: it decides nothing for the traces (their budget is
taken at the first of them), and what it keeps for the next call is bounded and
given back when a trace's budget is small.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from radlite_amd import engine, synth

pytestmark = pytest.mark.gpu

MB = 1 << 20


def _resample(rt, mb):
    """A resampling whose image and output are mb MiB each."""
    n = mb * MB // 8 // 64
    rt.resample_image(np.ones((n, 64)), np.zeros((n, 1), np.int32), np.ones((n, 1)))


def _free():
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


def test_budget_is_taken_at_the_first_trace():
    first = engine.Raytracer(0, "fp64")
    _resample(first, 64)
    held = torch.empty(4 << 30, dtype=torch.uint8, device="cuda")
    other = engine.Raytracer(0, "fp64")
    a, b = first.memory_info()["budget"], other.memory_info()["budget"]
    # what the first context keeps (138 MiB) counts for it in full and is not free
    # for the other: 60% of the 4 GiB, had the budget been taken before, is 2.6e9
    assert abs(a - b) < 0.3e9
    first.close()
    other.close()
    del held
    torch.cuda.empty_cache()


def test_kept_buffers_are_given_back():
    disk = synth.make_disk(12, 8, seed=1)
    lines = synth.single_line()
    v, dv = synth.passband(30.0, 9)
    ri = synth.run_inputs(disk, lines, synth.lte_pops(disk, lines), nphi=6, dbdr=1, b_extra=-2,
                          vmax=v, dv=dv, incl_deg=50.0)
    nfr, vmax = engine.passband(ri.vmax, ri.dv)
    rt = engine.Raytracer(0, "fp64")
    rt.load_run(ri)
    items = [(0, 0, nfr, vmax, engine.SKIP_NONE)]

    def trace():
        rt.setup_rays([0.87], ri.nphi, ri.b_extra, ri.dbdr)
        return rt.trace(items)[0][0]

    _resample(rt, 8)                       # the pinned slots and the context's own
    ref = trace()
    start = _free()
    _resample(rt, 256)
    kept = start - _free()
    assert kept >= 500 * MB                # for the next call
    rt.set_memory_budget(kept + 4 * MB)
    assert np.array_equal(trace(), ref)
    assert start - _free() <= 64 * MB      # given back
    rt.set_memory_budget(0)
    _resample(rt, 600)                     # above the bound: not kept
    assert start - _free() <= 64 * MB
    rt.close()
