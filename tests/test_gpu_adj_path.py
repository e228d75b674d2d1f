"""Which reverse sweep runs.  The gradients on the tables are by segments also
where the device formed the tables (rl_set_physics): the same bits as with the
same tables set by the caller, from a tape and without one.  The gradients on
the physical fields alone are by (block, channel) pairs as long as the tables
are rl_set_physics's, whatever else has been set since; they differ from those by
segments by rounding (bounds of test_gpu_adj_blocks.py).
"""
import numpy as np
import pytest

from radlite_amd import engine, synth
from radlite_amd.diff import kappa_at_lines

pytestmark = pytest.mark.gpu


def _make(precision, nlines=1):
    disk = synth.make_disk(24, 16, seed=4, sigma_t=0.1)
    lines = synth.single_line() if nlines == 1 else synth.random_lines(nlines, seed=1)
    v, dv = synth.passband(30.0, 33)
    ri = synth.run_inputs(disk, lines, synth.lte_pops(disk, lines), nphi=6, dbdr=1, b_extra=-2,
                          vmax=v, dv=dv, incl_deg=50.0)
    rt = engine.Raytracer(0, precision)
    tb = rt.load_run(ri)
    _rays(rt, ri)
    ka, ks = (np.array([kappa_at_lines(ri.cont_nu, k[0], tb.nu0)])
              for k in (ri.kappa_abs, ri.kappa_scat))
    rt.set_level_data(np.asarray(ri.E_cm, float) * synth.K_PER_CM, np.asarray(ri.g, float))
    rt.set_dust_species(ri.rho_dust, ka, ks)
    nfr, vmax = engine.passband(ri.vmax, ri.dv)
    items = [(il, 0, nfr, vmax, engine.SKIP_NONE) for il in range(len(ri.A))]
    g = [1e20 * np.random.default_rng(il).normal(size=nfr) for il in range(len(ri.A))]
    return ri, rt, items, g


def _rays(rt, ri):
    rt.setup_rays([ri.incl_deg * 0.0174532925199], ri.nphi, ri.b_extra, ri.dbdr)


def _physics(rt, ri):
    rt.set_physics(ri.t_dust[0], np.full(ri.rho_gas.shape, 0.1), log_abund=np.log(ri.abund))


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("nlines", [1, 3])
def test_table_gradients_do_not_depend_on_who_formed_the_tables(nlines, precision):
    ri, rt, items, g = _make(precision, nlines)
    _physics(rt, ri)
    _, alone = rt.adjoint(items, g)                    # its own forward
    rt.trace_tape(items)
    _, taped = rt.adjoint(items, g)                    # from a tape
    _, again = rt.adjoint(items, g)
    t = rt.get_tables()
    rt.set_medium(ri.rho_gas, t["abund"], ri.vel, t["lw"], ri.umass_av, float(t["lw"].max()))
    rt.set_levels(t["pops"])
    rt.set_dust_line(t["jd"], t["ad"])
    _, ref = rt.adjoint(items, g)
    rt.close()
    for k in ref:
        assert np.abs(ref[k]).max() > 0.0
        for got in (alone, taped, again):
            assert np.array_equal(got[k], ref[k]), k


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_pairs_as_long_as_the_tables_are_the_physics(precision):
    ri, rt, items, g = _make(precision)
    info = lambda: (rt.adjoint_pairs() > 0, rt.adjoint_info()[1])
    _physics(rt, ri)
    rt.trace_tape(items)
    rt.adjoint(items, g, outputs=())
    assert info() == (True, 1)
    ref = rt.physics_adjoint()
    # another view set since (and the star): the same tables, the same sweep
    for tape in (True, False):
        _rays(rt, ri)
        rt.set_outer_bc(ri.outer_bc)
        if tape:
            rt.trace_tape(items)
        rt.adjoint(items, g, outputs=())
        assert info() == (True, int(tape))
        got = rt.physics_adjoint()
        assert all(np.array_equal(got[k], ref[k]) for k in ref)
    # a table asked for: by segments, from a tape taken by blocks too, which is
    # then one by segments
    rt.trace_tape(items)
    rt.adjoint(items, g, outputs=("g_rho",))
    assert info() == (False, 0)
    got = rt.physics_adjoint()
    tol = 1e-13 if precision == "fp64" else 4e-6
    for k in ref:
        assert np.abs(got[k] - ref[k]).max() <= tol * np.abs(ref[k]).max(), k
    rt.adjoint(items, g, outputs=("g_ad",))
    assert info() == (False, 1)
    # a table set by the caller: by segments
    rt.set_levels(rt.get_tables()["pops"])
    rt.adjoint(items, g, outputs=())
    assert info() == (False, 0)
    _physics(rt, ri)
    rt.adjoint(items, g, outputs=())
    assert info() == (True, 0)
    rt.set_option(engine.OPT_CKPT, 2)
    rt.adjoint(items, g, outputs=())
    assert info() == (False, 0)
    rt.close()
