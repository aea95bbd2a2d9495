"""River discharges on the GPU against the oracle, bit for bit: one-level meshes (stepped and
graph-replayed), multi-level meshes and spherical grids (discharge area from spharea), FP64 and
FP32, and the discharge cells found again after a remesh."""
import numpy as np
import pytest

import bg_flood_amd as bgf
from bg_flood_amd import scenarios
from oracle import pyoracle as po
from tests._util import domain_for, oracle_for, orc_param_with

pytestmark = pytest.mark.gpu


def rivers_for(L):
    """Two rivers in a domain of side L: a small one and a wide one straddling block edges."""
    return [(0.2 * L, 0.23 * L, 0.5 * L, 0.52 * L, [0.0, 6.0, 200.0], [0.0, 25.0, 5.0]),
            (0.6 * L, 0.75 * L, 0.24 * L, 0.26 * L, [0.0, 1e6], [12.0, 12.0])]


def compare(d, o):
    m = bgf.interior_mask(d.nblkmem, d.active)
    st = d.get_state()
    for k in ("h", "u", "v"):
        a, b = st[k][m], o.get(k)[m]
        assert np.array_equal(a, b), "%s: max diff %g" % (k, np.abs(a - b).max())


def run_pair(sc, prec, nsteps, graph, L, rivers=None):
    print("case rivers %s nblk=%d graph=%s" % (prec, sc["param"]["nblk"], graph), flush=True)
    d = domain_for(sc, precision=prec)
    o = oracle_for(sc, precision=prec)
    rv = rivers if rivers is not None else rivers_for(L)
    d.set_rivers(rv)
    o.set_rivers(rv)
    lg = bgf.Loop(nextoutputtime=1e9, dt=0, dtmax=0, totaltime=0)
    lo = po.OrcLoop(nextoutputtime=1e9, dt=0, dtmax=0, totaltime=0)
    d.init_dt(lg)
    o.init_loop(lo)
    if graph:
        d.run(lg, nsteps)
        for _ in range(nsteps):
            o.step(lo)
            lo.totaltime += lo.dt
        assert lg.totaltime == lo.totaltime
    else:
        for k in range(nsteps):
            d.step(lg)
            o.step(lo)
            assert lg.dt == lo.dt, "step %d" % k
            lg.totaltime += lg.dt
            lo.totaltime += lo.dt
    compare(d, o)
    return d, o


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_one_level_rivers_exact(prec):
    sc = scenarios.gaussian_hump(n=64, dx=4.0, depth=1.0, amp=0.0, precision=prec, aoibnd=0)
    run_pair(sc, prec, 40, False, 256.0)
    run_pair(sc, prec, 40, True, 256.0)


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_multi_level_rivers_exact(prec):
    sc = scenarios.amr_basin(precision=prec, island=True, amp=0.3)
    L = sc["nbx"] * 16 * sc["param"]["dx"]
    run_pair(sc, prec, 30, False, L)
    run_pair(sc, prec, 30, True, L)


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_spherical_rivers_exact(prec):
    sc = scenarios.spherical_basin(lat0=40.0, lat_c=40.3, dx=0.01, amp=0.2, precision=prec)
    p = sc["param"]
    rivers = [(p["xo"] + 0.2, p["xo"] + 0.23, p["yo"] + 0.3, p["yo"] + 0.32, [0.0, 8.0, 1e4], [0.0, 40.0, 10.0]),
              (p["xo"] + 0.47, p["xo"] + 0.52, p["yo"] + 0.1, p["yo"] + 0.105, [0.0, 1e6], [15.0, 15.0])]
    run_pair(sc, prec, 30, False, 0.0, rivers)
    run_pair(sc, prec, 30, True, 0.0, rivers)


def test_rivers_after_remesh():
    from tests.test_gpu_remesh import scenario, NBX, NBY, DX
    sc = scenario("fp64")
    L = NBX * 16 * DX
    d, o = run_pair(sc, "fp64", 8, False, L)
    lg = bgf.Loop(nextoutputtime=1e9, dt=0, dtmax=0, totaltime=0)
    lo = po.OrcLoop(nextoutputtime=1e9, dt=0, dtmax=0, totaltime=0)
    d.init_dt(lg)
    o.init_loop(lo)
    for cycle in range(3):
        ref = d.refine_flags("zs", 2, 1e-3)
        co = np.zeros(d.nblkmem, np.uint8)
        co[d.active] = 1 - ref[d.active]
        blocks, nb, nm, remap = bgf.adapt_mesh(d.param, d.blocks, ref, co, NBX, NBY)
        d.remesh(blocks, nb, nm, remap)
        o.remesh(orc_param_with(o.p, nblk=nb, nblkmem=nm), blocks, remap)
        compare(d, o)
        for _ in range(8):
            d.step(lg)
            o.step(lo)
            assert lg.dt == lo.dt
            lg.totaltime += lg.dt
            lo.totaltime += lo.dt
        compare(d, o)


@pytest.mark.parametrize("mesh", ["one level", "three levels"])
@pytest.mark.parametrize("n", [2, 3, 4, 5, 2000])
def test_long_series_late_in_the_run(n, mesh):
    """A rain and a river series of few and many entries, from times before, on and between the entries and
    past the last: both stages and every workgroup look the entries up."""
    sc = scenarios.gaussian_hump(n=48, dx=4.0, depth=1.0, amp=0.1, precision="fp64") if mesh == "one level" else \
        scenarios.amr_basin(nbx=3, nby=3, precision="fp64", island=True, amp=0.1)
    L = sc["nbx"] * 16 * sc["param"]["dx"]
    rng = np.random.default_rng(n)
    t = np.cumsum(rng.uniform(0.5, 2.0, n))
    rivers = [(0.2 * L, 0.4 * L, 0.5 * L, 0.6 * L, list(t), list(rng.uniform(1.0, 30.0, n)))]
    rain = rng.uniform(5.0, 100.0, n)
    d, o = domain_for(sc, precision="fp64"), oracle_for(sc, precision="fp64")
    for x in (d, o):
        x.set_rivers(rivers)
        x.set_rain_series(t, rain)
    start = sorted({t[0], t[1] - 0.01, t[n // 2], t[n // 2] - 0.02, t[-2], t[-1], t[-1] + 3.0})
    lg = bgf.Loop(nextoutputtime=1e9, dt=0, dtmax=0, totaltime=0)
    lo = po.OrcLoop(nextoutputtime=1e9, dt=0, dtmax=0, totaltime=0)
    d.init_dt(lg)
    o.init_loop(lo)
    for at in start:
        print("case series of %d, %s, at %g" % (n, mesh, at), flush=True)
        lg.totaltime = lo.totaltime = float(at)
        d.run(lg, 3)
        o.run(lo, 3)
        assert (lg.dt, lg.totaltime) == (lo.dt, lo.totaltime)
        compare(d, o)
    d.close()
