"""Where the launches change form: cell sizes far from one (the division by the cell size in multiply-adds),
read-backs whose blocks just fill, miss and pass a piece of the pinned memory, run lengths about the captured
graph's, runs that stop early after an odd step, and multi-level meshes below and above the size from which
the dt reduction has a launch of its own.  The exact kernels keep the oracle's operations and get_state
copies, so every comparison is bit for bit."""
import numpy as np
import pytest

import bg_flood_amd as bgf
from bg_flood_amd import scenarios
from oracle import pyoracle as po
from tests._util import domain_for, oracle_for

pytestmark = pytest.mark.gpu


def loop(cls=bgf.Loop):
    return cls(nextoutputtime=1e9, dt=0, dtmax=0, totaltime=0)


def against_oracle(sc, prec, steps):
    d, o = domain_for(sc, precision=prec), oracle_for(sc, precision=prec)
    lg, lo = loop(), loop(po.OrcLoop)
    d.init_dt(lg)
    o.init_loop(lo)
    for _ in range(steps):  # step by step: a run would stop where dt falls below dtmin
        d.step(lg)
        o.step(lo)
        assert lg.dt == lo.dt and lg.dt > 0
        lg.totaltime += lg.dt
        lo.totaltime += lo.dt
    m = bgf.interior_mask(d.nblkmem, d.active)
    st = d.get_state()
    for k in ("h", "u", "v"):
        assert np.array_equal(st[k][m], o.get(k)[m]), k
    assert np.abs(st["u"][m]).max() > 0
    d.close()


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("dx", [1.0 / 3.0, 1e-4, 3e6])
def test_cell_sizes(dx, prec):
    print("case cell size %g %s" % (dx, prec), flush=True)
    sc = scenarios.gaussian_hump(n=48, dx=dx, depth=2.0, amp=0.5, radius=5 * dx, precision=prec, aoibnd=1)
    against_oracle(sc, prec, 8)


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("nbx,nby", [(1, 1), (127, 1), (16, 16), (257, 1)])
def test_read_back_leaves_the_other_cells(nbx, nby, prec):
    print("case read-back %d blocks %s" % (nbx * nby, prec), flush=True)
    p, blocks, _, _ = scenarios.uniform(16 * nbx, 16 * nby, 1.0, prec)
    rng = np.random.default_rng(nbx)
    T = np.float64 if prec == "fp64" else np.float32
    n = p["nblkmem"] * 324
    zb, h, u, v, cf = (rng.random(n).astype(T) for _ in range(5))
    d = bgf.Domain(p, blocks)
    d.set_state(zb, h, u, v, cf)
    m = bgf.interior_mask(d.nblkmem, d.active)
    want = dict(zs=zb + h, h=h, u=u, v=v)
    for fields in (("zs", "h", "u", "v"), ("zs",), ("h", "v")):
        out = {k: np.full(n, -7, T) for k in fields}
        rc = bgf.lib().bgf_get_state(d.h, *[out[k].ctypes.data if k in out else None for k in ("zs", "h", "u", "v")])
        assert rc == 0
        for k in fields:
            assert np.array_equal(out[k][m], want[k][m]) and (out[k][~m] == -7).all(), k
    d.close()


MESHES = {"one level": lambda: scenarios.gaussian_hump(n=64, dx=4.0, depth=2.0, amp=0.3, radius=20.0, precision="fp32"),
          "two levels": lambda: scenarios.amr_basin(nbx=4, nby=3, maxlevel=1, precision="fp32")}


@pytest.mark.parametrize("mesh", list(MESHES))
@pytest.mark.parametrize("steps", [1, 15, 16, 17, 24])
def test_run_lengths(steps, mesh):
    print("case run of %d, %s" % (steps, mesh), flush=True)
    sc = MESHES[mesh]()
    a, b = domain_for(sc), domain_for(sc)
    la, lb = loop(), loop()
    a.init_dt(la)
    b.init_dt(lb)
    for _ in range(2):  # the second run finds the graph captured
        a.run(la, steps)
        for _ in range(steps):
            b.step(lb)
            lb.totaltime += lb.dt
    assert (la.dt, la.totaltime) == (lb.dt, lb.totaltime)
    sa, sb = a.get_state(), b.get_state()
    assert all(np.array_equal(sa[k], sb[k]) for k in sa)
    a.close()
    b.close()


@pytest.mark.parametrize("mesh", list(MESHES))
@pytest.mark.parametrize("steps", [8, 9, 32])
def test_run_stops_after_an_odd_step(steps, mesh):
    print("case run of %d stopped, %s" % (steps, mesh), flush=True)
    sc = MESHES[mesh]()
    a, b = domain_for(sc), domain_for(sc)
    la, lb = loop(), loop()
    a.init_dt(la)
    b.init_dt(lb)
    for _ in range(5):
        b.step(lb)
        lb.totaltime += lb.dt
    a.run(la, steps, endtime=lb.totaltime)
    assert (la.dt, la.totaltime) == (lb.dt, lb.totaltime)
    sa, sb = a.get_state(), b.get_state()
    assert all(np.array_equal(sa[k], sb[k]) for k in sa)
    a.close()
    b.close()


@pytest.mark.parametrize("part,above", [(0.3, False), (0.45, True)])
def test_multi_level_reduction(part, above):
    def refine(l, x, y):
        return np.random.default_rng([7, l, x, y]).random() < part

    sc = scenarios.amr_basin(nbx=48, nby=40, maxlevel=1, depth=1.5, amp=0.8, precision="fp32", refine=refine)
    n = sc["param"]["nblk"]
    print("case multi-level reduction, %d blocks" % n, flush=True)
    assert (n > 4096) == above
    against_oracle(sc, "fp32", 3)


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_read_back_grows_with_the_members(prec):
    """Members of one batch read in turn, from one block to more than a piece of the pinned memory holds and
    back, all fields and some: the pieces grow from read to read."""
    T = np.float64 if prec == "fp64" else np.float32
    sides = [(1, 1), (3, 1), (17, 2), (40, 9), (2, 1)]
    parts = [scenarios.uniform(16 * nx, 16 * ny, 1.0, prec)[:2] for nx, ny in sides]
    rng = np.random.default_rng(2)
    b = bgf.Batch(parts[0][0], sum(p["nblkmem"] for p, _ in parts), len(parts))
    held = []
    for p, blocks in parts:
        n = p["nblkmem"] * 324
        a = [(1.0 + rng.random(n)).astype(T) for _ in range(5)]
        held.append((b.add(p, blocks, *a, endtime=1e9), p, blocks, a))
    for order in (range(len(held)), reversed(range(len(held)))):
        for k in order:
            mid, p, blocks, (zb, h, u, v, _) = held[k]
            print("case read-back of member %d, %d blocks, %s" % (k, p["nblk"], prec), flush=True)
            m = bgf.interior_mask(p["nblkmem"], blocks["active"][:p["nblk"]])
            n = p["nblkmem"] * 324
            want = dict(zs=zb + h, h=h, u=u, v=v)
            for fields in (("u",), ("zs", "h", "u", "v")):
                out = {f: np.full(n, -7, T) for f in fields}
                rc = bgf.lib().bgf_batch_get_state(b.h, mid, *[out[f].ctypes.data if f in out else None
                                                               for f in ("zs", "h", "u", "v")])
                assert rc == 0
                for f in fields:
                    assert np.array_equal(out[f][m], want[f][m]) and (out[f][~m] == -7).all(), f
    b.close()
