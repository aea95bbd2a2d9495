"""Boundary types 2 (Dirichlet) and 3 (absorbing) on the GPU against the oracle, bit for bit, with
time-varying water levels, on one-level meshes (stepped and graph-replayed) and multi-level meshes,
FP64 and FP32; with Param.zsoffset, a boundary taper and a type-4 side; with segments of their own
polygons (a corner block follows the later segment); with level maps (frames interpolated in time,
sampled at each face) and Param.zsinit; with a device level map read in place; and with the
segments' blocks found again after remeshing."""
import numpy as np
import pytest

import bg_flood_amd as bgf
from bg_flood_amd import scenarios
from oracle import pyoracle as po
from tests._util import domain_for, oracle_for

pytestmark = pytest.mark.gpu

LEVELS = {0: (2, [0.0, 4.0, 30.0], [0.0, 0.4, -0.2]),    # left: Dirichlet, rising then falling
          1: (3, [0.0, 100.0], [0.0, 0.0]),               # right: absorbing
          2: (3, [0.0, 10.0, 40.0], [0.1, -0.1, 0.2]),    # bottom: absorbing with a moving level
          3: (0, [], [])}                                  # top: wall


OPTIONS = None  # (zsoffset, bndtaper, inittime) set by the options test, (changed levels, type 4 top)


def configure(x):
    levels = dict(LEVELS)
    if OPTIONS:
        levels[3] = (4, [], [])
    for side, (btype, t, z) in levels.items():
        x.set_boundary(side, btype, t, z)
    if OPTIONS:
        x.set_boundary_options(*OPTIONS)


def compare(d, o):
    m = bgf.interior_mask(d.nblkmem, d.active)
    st = d.get_state()
    for k in ("h", "u", "v"):
        a, b = st[k][m], o.get(k)[m]
        assert np.array_equal(a, b), "%s: max diff %g" % (k, np.abs(a - b).max())


def run_pair(sc, prec, nsteps, graph):
    print("case boundary %s nblk=%d graph=%s" % (prec, sc["param"]["nblk"], graph), flush=True)
    d = domain_for(sc, precision=prec)
    o = oracle_for(sc, precision=prec)
    configure(d)
    configure(o)
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
    return lo.totaltime


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_one_level_boundaries_exact(prec):
    sc = scenarios.gaussian_hump(n=64, dx=4.0, depth=2.0, amp=0.3, radius=20.0, precision=prec, aoibnd=1)
    t = run_pair(sc, prec, 60, graph=False)
    assert t > 10.0
    run_pair(sc, prec, 60, graph=True)


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_multi_level_boundaries_exact(prec):
    sc = scenarios.amr_basin(precision=prec, island=True, amp=0.5, aoibnd=1)
    run_pair(sc, prec, 40, graph=False)
    run_pair(sc, prec, 40, graph=True)


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_offset_taper_and_type_4_exact(prec):
    """zsoffset 0.05 m, a 20 s taper from t = -3 s, and the top side of type 4, on both kernel
    families."""
    global OPTIONS
    OPTIONS = (0.05, 20.0, -3.0)
    try:
        sc = scenarios.gaussian_hump(n=64, dx=4.0, depth=2.0, amp=0.3, radius=20.0, precision=prec, aoibnd=1)
        run_pair(sc, prec, 60, graph=False)
        run_pair(sc, prec, 60, graph=True)
        sc = scenarios.amr_basin(precision=prec, island=True, amp=0.5, aoibnd=1)
        run_pair(sc, prec, 40, graph=True)
    finally:
        OPTIONS = None


def test_fast_kernels_take_the_boundaries():
    sc = scenarios.gaussian_hump(n=64, dx=4.0, depth=2.0, amp=0.3, radius=20.0, precision="fp32", aoibnd=1)
    d = domain_for(sc, precision="fp32_fast")
    e = domain_for(sc, precision="fp32")
    configure(d)
    configure(e)
    for x in (d, e):
        L = bgf.Loop(nextoutputtime=1e9, dt=0, dtmax=0, totaltime=0)
        x.init_dt(L)
        x.run(L, 80)
    m = bgf.interior_mask(d.nblkmem, d.active)
    a, b = d.get_state()["h"][m], e.get_state()["h"][m]
    assert np.max(np.abs(a - b)) < 1e-3


def poly_segments(sc):
    """A moving absorbing level on the left side, a wall on top, a Dirichlet polygon over the left
    part of the bottom side (the bottom-left corner block goes to the polygon, the later segment;
    the top-left one to the wall)."""
    p = sc["param"]
    L = sc["nbx"] * 16 * p["dx"]
    xo, yo = p["xo"], p["yo"]
    # the polygon reaches 0.05 L into the domain: a block's box starts at its first cell centre
    top = yo + 0.05 * L
    return [dict(type=3, side=0, t=[0.0, 20.0, 60.0], z=[0.0, 0.3, 0.1]),
            dict(type=0, side=3),
            dict(type=2, poly=[(xo - 5, yo - 5), (xo + 0.45 * L, yo - 5), (xo + 0.45 * L, top), (xo - 5, top)],
                 t=[0.0, 1e6], z=[0.2, 0.2])]


def map_segments(sc):
    """The right side absorbing with a two-frame level map, the bottom Dirichlet with a one-frame
    map, the left absorbing without forcing (at Param.zsinit)."""
    p = sc["param"]
    L = sc["nbx"] * 16 * p["dx"]
    xo, yo = p["xo"], p["yo"]
    xs = xo - 30.0 + np.arange(0, L + 60.0, 0.13 * L)
    ys = yo - 30.0 + np.arange(0, L + 60.0, 0.11 * L)
    X, Y = np.meshgrid((xs - xo) / L, (ys - yo) / L)
    f0 = (0.25 * X - 0.1 * Y).astype(np.float32)
    f1 = (0.3 - 0.2 * X + 0.15 * np.sin(4 * Y)).astype(np.float32)
    segs = [dict(type=3, side=1), dict(type=2, side=2), dict(type=3, side=0)]
    maps = {0: (np.stack([f0, f1]), xs[0], ys[0], xs[1] - xs[0], ys[1] - ys[0], 2.0, 30.0),
            1: (np.full((3, 4), 0.15, np.float32), xo - L, yo - L, 1.5 * L, L, 0.0, 1.0)}
    return segs, maps


def run_segments(sc, prec, nsteps, graph, segs, maps=None, options=None):
    print("case boundary segments %s nblk=%d graph=%s maps=%s" % (prec, sc["param"]["nblk"], graph, bool(maps)),
          flush=True)
    d = domain_for(sc, precision=prec)
    o = oracle_for(sc, precision=prec)
    for x in (d, o):
        x.set_boundary_segments(segs)
        for k, m in (maps or {}).items():
            x.set_boundary_map(k, *m)
        if options:
            x.set_boundary_options(**options)
    bd = d.boundary_blocks()
    bo = o.boundary_blocks()[:len(bd)]
    assert np.array_equal(bd, bo)
    for k in range(len(segs)):
        assert (bd == k).any(), "segment %d claims no block" % k
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
def test_polygon_segments_exact(prec):
    sc = scenarios.gaussian_hump(n=64, dx=4.0, depth=2.0, amp=0.3, radius=20.0, precision=prec, aoibnd=1)
    run_segments(sc, prec, 60, False, poly_segments(sc))
    run_segments(sc, prec, 60, True, poly_segments(sc), options=dict(zsoffset=0.02, bndtaper=15.0))
    sc = scenarios.amr_basin(precision=prec, island=True, amp=0.5, aoibnd=1)
    run_segments(sc, prec, 40, True, poly_segments(sc))


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_level_maps_exact(prec):
    sc = scenarios.gaussian_hump(n=64, dx=4.0, depth=2.0, amp=0.3, radius=20.0, precision=prec, aoibnd=0)
    segs, maps = map_segments(sc)
    run_segments(sc, prec, 60, False, segs, maps, options=dict(zsinit=0.05))
    run_segments(sc, prec, 60, True, segs, maps, options=dict(zsinit=0.05, bndtaper=10.0))
    sc = scenarios.amr_basin(precision=prec, island=True, amp=0.5, aoibnd=0)
    segs, maps = map_segments(sc)
    run_segments(sc, prec, 40, True, segs, maps, options=dict(zsinit=0.05))


def test_device_level_map_exact():
    """A level map the caller keeps on the device (WLmap.now_g), read in place: the run of the same
    values given as a one-frame map, bit for bit."""
    from tests._util import DeviceArray
    sc = scenarios.gaussian_hump(n=64, dx=4.0, depth=2.0, amp=0.3, radius=20.0, precision="fp32", aoibnd=1)
    segs, maps = map_segments(sc)
    frames, xo, yo, dx, dy, _, _ = maps[0]
    d = domain_for(sc, precision="fp32")
    o = oracle_for(sc, precision="fp32")
    d.set_boundary_segments(segs[:1])
    o.set_boundary_segments(segs[:1])
    now = DeviceArray(np.ascontiguousarray(frames[1], np.float32))
    d.set_boundary_map_device(0, now, xo, yo, dx, dy)
    o.set_boundary_map(0, frames[1], xo, yo, dx, dy)
    lg = bgf.Loop(nextoutputtime=1e9, dt=0, dtmax=0, totaltime=0)
    lo = po.OrcLoop(nextoutputtime=1e9, dt=0, dtmax=0, totaltime=0)
    d.init_dt(lg)
    o.init_loop(lo)
    d.run(lg, 40)
    for _ in range(40):
        o.step(lo)
        lo.totaltime += lo.dt
    compare(d, o)
    d.close()
    now.free()


def test_segments_follow_the_remesh():
    """Segments on an adaptive mesh: after each adapt-and-remesh cycle the boundary blocks are
    assigned again, as the oracle assigns them, and the runs stay bit-identical."""
    from tests.test_gpu_remesh import scenario, NBX, NBY, DX
    from tests._util import orc_param_with
    sc = scenario("fp64")
    L = NBX * 16 * DX
    segs = [dict(type=3, side=1, t=[0.0, 1e6], z=[0.1, 0.1]),
            dict(type=2, poly=[(-5, L * 0.3), (30, L * 0.3), (30, L * 0.7), (-5, L * 0.7)], t=[0.0, 1e6], z=[0.3, 0.3])]
    d, o = run_segments(sc, "fp64", 8, False, segs)
    lg = bgf.Loop(nextoutputtime=1e9, dt=0, dtmax=0, totaltime=0)
    lo = po.OrcLoop(nextoutputtime=1e9, dt=0, dtmax=0, totaltime=0)
    d.init_dt(lg)
    o.init_loop(lo)
    for cycle in range(3):
        print("case segments after remesh, cycle %d" % cycle, flush=True)
        ref = d.refine_flags("zs", 2, 1e-3)
        co = np.zeros(d.nblkmem, np.uint8)
        co[d.active] = 1 - ref[d.active]
        blocks, nb, nm, remap = bgf.adapt_mesh(d.param, d.blocks, ref, co, NBX, NBY)
        d.remesh(blocks, nb, nm, remap)
        o.remesh(orc_param_with(o.p, nblk=nb, nblkmem=nm), blocks, remap)
        bd = d.boundary_blocks()
        assert np.array_equal(bd, o.boundary_blocks()[:len(bd)])
        for k in range(6):
            d.step(lg)
            o.step(lo)
            assert lg.dt == lo.dt, (cycle, k)
            lg.totaltime += lg.dt
            lo.totaltime += lo.dt
        compare(d, o)


@pytest.mark.parametrize("mesh", ["one level", "three levels"])
@pytest.mark.parametrize("n", [2, 3, 4, 2000])
def test_long_level_series(n, mesh):
    """Level series of few and many entries on two sides, from times before, on and between the entries and
    past the last."""
    sc = scenarios.gaussian_hump(n=48, dx=4.0, depth=1.0, amp=0.1, precision="fp64") if mesh == "one level" else \
        scenarios.amr_basin(nbx=3, nby=3, precision="fp64", island=True, amp=0.1)
    rng = np.random.default_rng(n)
    t = np.cumsum(rng.uniform(0.5, 2.0, n))
    d, o = domain_for(sc, precision="fp64"), oracle_for(sc, precision="fp64")
    for x in (d, o):
        x.set_boundary(0, 2, t, 0.3 * np.sin(t))
        x.set_boundary(3, 3, t, 0.2 * np.cos(t))
    lg = bgf.Loop(nextoutputtime=1e9, dt=0, dtmax=0, totaltime=0)
    lo = po.OrcLoop(nextoutputtime=1e9, dt=0, dtmax=0, totaltime=0)
    d.init_dt(lg)
    o.init_loop(lo)
    for at in sorted({t[0] - 0.1, t[0], t[1] - 0.01, t[n // 2], t[n // 2] - 0.02, t[-2], t[-1], t[-1] + 3.0}):
        print("case level series of %d, %s, at %g" % (n, mesh, at), flush=True)
        lg.totaltime = lo.totaltime = float(at)
        d.run(lg, 3)
        o.run(lo, 3)
        assert (lg.dt, lg.totaltime) == (lo.dt, lo.totaltime)
        compare(d, o)
    d.close()
