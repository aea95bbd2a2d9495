"""Continuous batching on the GPU: requests that arrive while others run are admitted as slots free
up, run overlapped, and each result (maximum depth, gauge series) is bit-identical to the same
request served alone."""
import ctypes

import numpy as np
import pytest

import bg_flood_amd as bgf
from bg_flood_amd import scenarios, serving
from tests._util import hip

pytestmark = pytest.mark.gpu


def rain_request(k, n, horizon):
    sc = scenarios.rain_terrain(n=n, dx=5.0, amp=8.0 + k, rain=40.0 + 10 * k, manning=0.03, seed=100 + k,
                                precision="fp32")
    cells = [(i + 1) + (j + 1) * 18 + b * 324 for i, j, b in ((3, 4, 0), (8, 8, 1), (15, 0, 2), (7, 9, 3))]
    return serving.Request(k, sc, horizon, gauges=cells, gauge_every=3)


def amr_request(k, horizon):
    sc = scenarios.amr_basin(precision="fp32", island=True, amp=1.0 + 0.2 * k)
    cells = [(i + 1) + (j + 1) * 18 + b * 324 for i, j, b in ((5, 5, 0), (9, 2, 7))]
    return serving.Request(k, sc, horizon, gauges=cells)


def make_requests():
    return [rain_request(0, 64, 120.0), rain_request(1, 96, 60.0), rain_request(2, 48, 200.0),
            amr_request(3, 8.0), rain_request(4, 80, 90.0), rain_request(5, 64, 150.0)]


def common_param(reqs):
    return dict(reqs[0].sc["param"], precision="fp32_comp")


def test_mixed_stream_matches_requests_served_alone():
    reqs = make_requests()
    arrivals = np.array([0.0, 0.0, 0.05, 0.05, 0.1, 0.12])
    # room for about two members at a time: later arrivals wait for slots
    cap = 2 * max(r.sc["param"]["nblkmem"] for r in reqs if not r.multilevel) + 8
    srv, wall = serving.serve(reqs, arrivals, common_param(reqs), max_blocks=cap, max_members=4, chunk=16,
                              time_limit=120.0)
    print("served %d requests in %.2f s" % (len(srv.done), wall), flush=True)
    assert len(srv.done) == len(reqs)
    for r in reqs:
        assert r.latency is not None and r.latency >= 0
        assert r.result["totaltime"] == pytest.approx(r.horizon, rel=1e-6)
    for r0 in reqs:
        alone = [make_requests()[r0.rid]]
        s1, _ = serving.serve(alone, np.array([0.0]), common_param(reqs), max_blocks=cap, max_members=4, chunk=16)
        a, b = r0.result, alone[0].result
        assert np.array_equal(a["maxdepth"], b["maxdepth"]), r0.rid
        assert np.array_equal(a["gauges"], b["gauges"]), r0.rid
        assert np.array_equal(a["times"], b["times"]), r0.rid
        s1.close()
    srv.close()


# ---- the serving configuration's mix against the oracle ---------------------------------------
def tsunami_request(k, horizon):
    """An AMR tsunami request on the benchmark's geometry (3 levels, 20 x 10 km, shelf, island)."""
    sc = quadratic_friction(scenarios.tsunami(amp=1.5, seed=21, precision="fp32"))
    act = sc["blocks"]["active"]
    cells = [(i + 1) + (j + 1) * 18 + act[b] * 324 for i, j, b in ((3, 4, 0), (8, 8, 40), (15, 0, 200),
                                                                      (7, 9, len(act) // 2))]
    return serving.Request(k, sc, horizon, gauges=cells, gauge_every=5)


def oracle_result(req):
    """The request run by the FP32 oracle to its horizon: running maximum depth (from the initial
    state for multi-level requests, whose statistics include it; from 0 for batch members, whose
    running maximum starts at 0) and the gauges sampled after every gauge_every-th step."""
    from oracle import pyoracle as po
    from tests._util import oracle_for
    import bg_flood_amd as bgf
    sc = req.sc
    o = oracle_for(sc, precision="fp32")
    lo = po.OrcLoop(nextoutputtime=req.horizon, dt=0, dtmax=0, totaltime=0)
    o.init_loop(lo)
    hmax = np.asarray(sc["h"], np.float32).copy() if req.multilevel else np.zeros(len(sc["h"]), np.float32)
    vals, times = [], []
    n = 0
    while lo.totaltime < req.horizon:
        o.step(lo)
        lo.totaltime += lo.dt
        n += 1
        h = o.get("h")
        hmax = np.maximum(hmax, h)
        if req.gauges and n % req.gauge_every == 0:
            vals.append(h[req.gauges])
            times.append(lo.totaltime)
    p = sc["param"]
    mask = bgf.interior_mask(p["nblkmem"], sc["blocks"]["active"][:p["nblk"]])
    return np.where(mask, hmax, 0), np.array(vals, np.float32).T, np.array(times), lo.totaltime, n


def quadratic_friction(sc, cf=0.002):
    """The scenario with quadratic bottom friction instead of Manning's: the Manning law takes a cube
    root, which neither the host's libm nor the GPU's math library rounds correctly, so only runs
    without it can be compared with the oracle bit for bit (Manning runs are compared within
    tolerances in test_gpu_parity.py and test_gpu_configs.py)."""
    sc["param"] = dict(sc["param"], frictionmodel=0)
    sc["cf"] = np.full(len(sc["cf"]), np.float32(cf), np.float32)
    return sc


def wet_rain_request(k, n, horizon):
    """A rain request that starts with 0.3 m of water over its terrain (so it takes tens of steps)."""
    r = rain_request(k, n, horizon)
    quadratic_friction(r.sc)
    p = r.sc["param"]
    import bg_flood_amd as bgf
    m = bgf.interior_mask(p["nblkmem"], r.sc["blocks"]["active"][:p["nblk"]])
    r.sc["h"] = np.where(m, np.float32(0.3), np.float32(0)).astype(np.float32)
    return r


def test_mix_with_a_tsunami_request_matches_the_oracle():
    """The serving mix (rain requests in the shared batch, an AMR tsunami request on its own handle,
    arriving while others run) served in FP32 reference arithmetic: every request's maximum-depth grid
    and gauge series equal the oracle's run of that request alone, bit for bit (quadratic friction,
    see quadratic_friction)."""
    reqs = [wet_rain_request(0, 64, 90.0), wet_rain_request(1, 96, 60.0), tsunami_request(2, 6.0),
            wet_rain_request(3, 80, 120.0)]
    arrivals = np.array([0.0, 0.02, 0.04, 0.06])
    cap = sum(r.sc["param"]["nblkmem"] for r in reqs if not r.multilevel)
    common = dict(reqs[0].sc["param"], precision="fp32")
    srv, wall = serving.serve(reqs, arrivals, common, max_blocks=cap, max_members=4, chunk=16, time_limit=300.0)
    print("served %d requests in %.2f s" % (len(srv.done), wall), flush=True)
    assert len(srv.done) == len(reqs)
    for r in reqs:
        print("case serving vs oracle: request %d (%s, %d cells)" % (r.rid, "amr" if r.multilevel else "rain",
                                                                    r.cells), flush=True)
        hmax, gv, gt, t_end, nsteps = oracle_result(r)
        res = r.result
        assert res["totaltime"] == t_end
        assert np.array_equal(res["maxdepth"], hmax), "max diff %g" % np.abs(res["maxdepth"] - hmax).max()
        assert np.array_equal(res["times"], gt)
        assert np.array_equal(np.asarray(res["gauges"])[:, :gt.size], gv)
        assert gt.size == nsteps // r.gauge_every and nsteps >= 20
    srv.close()


def test_admission_is_first_fit():
    """A request too large for the room left waits without holding back a smaller one behind it."""
    big, small, first = rain_request(0, 128, 30.0), rain_request(1, 48, 30.0), rain_request(2, 96, 1e6)
    nb = lambda r: r.sc["param"]["nblkmem"]
    cap = nb(big) + nb(small)  # the big one only fits once `first` has left
    assert nb(big) > cap - nb(first) >= nb(small)
    common = dict(first.sc["param"], precision="fp32")
    srv = serving.Server(common, max_blocks=cap, max_members=4, chunk=8)
    srv.submit(first)
    srv.poll()
    srv.submit(big)
    srv.submit(small)
    srv._admit()
    assert [r.rid for r in srv.waiting] == [0]
    assert any(r is small for r in srv.members.values())
    srv.close()


def _device_bytes_free():
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert hip().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


@pytest.mark.parametrize("kind", ["domain", "batch"])
def test_admission_counts_the_memory_of_a_multi_level_slot(kind):
    """A multi-level domain's and batch's device memory for many block slots against what admission
    counts for them: no more than counted (allocations are rounded up: 2 %), and most of it used."""
    slots = 100000
    sc = scenarios.amr_basin(precision="fp32")
    print("case memory of %d slots, %s" % (slots, kind), flush=True)
    small = dict(sc["param"])
    bgf.Domain(small, sc["blocks"]).close()  # the runtime's own first allocations
    before = _device_bytes_free()
    if kind == "domain":
        x = bgf.Domain(dict(small, nblkmem=slots), sc["blocks"])
    else:
        x = bgf.Batch(small, slots, 8)
    used = before - _device_bytes_free()
    x.close()
    counted = serving.AMR_BYTES_PER_BLOCK * slots
    assert 0.9 * counted < used < 1.02 * counted, (used, counted)
