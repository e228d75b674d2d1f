"""The single-precision spectrum of the adjoint's forward by blocks (maps of the
intensity, composed in double and rounded once a block) is no further from the
double-precision one than the forward that steps the intensity through every
segment (a checkpoint interval of 2): the rounding of ten segments' steps is
replaced by one, so that over several models the mean error has to be smaller.
"""
import sys

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from radlite_amd import diff, engine, synth

pytestmark = pytest.mark.gpu

SIZES = [(40, 24, 24, 30.0), (90, 40, 64, 30.0), (24, 16, 33, 5.0), (60, 40, 9, 45.0),
         (120, 60, 100, 30.0)]


def _flux(nr, nth, nfr, vmax, seed, precision, factor, keep):
    disk = synth.make_disk(nr, nth, seed=seed, sigma_t=0.1)
    disk.abund *= factor
    lines = synth.single_line()
    v, dv = synth.passband(vmax, nfr)
    ri = synth.run_inputs(disk, lines, synth.lte_pops(disk, lines), nphi=8, dbdr=1, b_extra=-2,
                          vmax=v, dv=dv, incl_deg=50.0)
    m = diff.SpectrumModel(ri, precision=precision, incl_rad=[0.87])
    m.rt.set_option(engine.OPT_CKPT, keep)
    rng = np.random.default_rng(seed)
    x = [torch.from_numpy(a).requires_grad_(True)
         for a in (ri.t_dust[0].copy(), np.log(disk.abund) + 0.1 * rng.normal(size=disk.abund.shape),
                   0.1 + 0.05 * rng.random(disk.abund.shape))]
    f = m.flux_from_physics_device(*x).detach().numpy()
    m.close()
    return f


@pytest.mark.parametrize("factor", [1.0, 1e-9, 1e3])
def test_maps_are_no_further_off(factor):
    err = {1: [], 2: []}
    for size in SIZES:
        for seed in (0, 1, 2):
            ref = _flux(*size, seed, "fp64", factor, 2)
            for keep in err:
                f = _flux(*size, seed, "fp32", factor, keep)
                err[keep].append(np.sqrt(np.mean((f - ref) ** 2)) / np.abs(ref).max())
    print(f"[gpu] abundance x {factor:g}: by maps {np.mean(err[1]):.2e}, by segments "
          f"{np.mean(err[2]):.2e}", file=sys.stderr, flush=True)
    assert np.mean(err[1]) <= np.mean(err[2])
