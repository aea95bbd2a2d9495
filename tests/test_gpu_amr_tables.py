"""Neighbour tables that are no quadtree's, which the library accepts as long as indexes and levels are in
range: a side whose second half alone is finer (its halo is filled by the launch that meshes of four levels
use) and a finer block that does not name its coarser neighbour (every block then stores its faces and waits),
alone and beside a regular member in one batch, against the oracle bit for bit."""
import numpy as np
import pytest

import bg_flood_amd as bgf
from bg_flood_amd import scenarios
from oracle import pyoracle as po
from tests._util import domain_for, oracle_for

pytestmark = pytest.mark.gpu

SIDES = (("LeftBot", "LeftTop", "RightBot", "RightTop"), ("RightBot", "RightTop", "LeftBot", "LeftTop"),
         ("BotLeft", "BotRight", "TopLeft", "TopRight"), ("TopLeft", "TopRight", "BotLeft", "BotRight"))


def mesh(prec, levels):
    return scenarios.amr_basin(nbx=4, nby=4, dx=10.0, maxlevel=levels, depth=1.5, amp=0.8, precision=prec, island=True,
                               frictionmodel=0, cf=0.002)


def edit(sc, kind, side):
    """The tables with one side changed; side: index of SIDES, the side of the coarser block."""
    b = {k: np.array(v) for k, v in sc["blocks"].items()}
    lev, act = b["level"], b["active"][:sc["param"]["nblk"]]
    first, second, back1, back2 = SIDES[side]
    ib = next(i for i in act if lev[b[first][i]] > lev[i] and lev[b[second][i]] > lev[i])
    if kind == "odd":
        b[first][ib] = next(i for i in act if i != ib and lev[i] == lev[ib])
    elif kind == "all":
        n = b[second][ib]
        b[back1][n] = b[back2][n] = next(i for i in act if i != n and lev[i] == lev[n])
    return dict(sc, blocks=b)


def loop(cls):
    return cls(nextoutputtime=1e9, dt=0, dtmax=0, totaltime=0)


def against(sc, prec, steps, dt, totaltime, state):
    o, lo = oracle_for(sc, precision=prec), loop(po.OrcLoop)
    o.init_loop(lo)
    o.run(lo, steps)
    assert (dt, totaltime) == (lo.dt, lo.totaltime)
    m = bgf.interior_mask(sc["param"]["nblkmem"], sc["blocks"]["active"][:sc["param"]["nblk"]])
    for k in ("h", "u", "v"):
        assert np.array_equal(state[k][m], o.get(k)[m]), k
    assert (state["h"][m] <= sc["param"]["eps"]).any() and np.abs(state["u"][m]).max() > 0


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("levels", [1, 2])
@pytest.mark.parametrize("side", range(4))
@pytest.mark.parametrize("kind", ["odd", "all"])
def test_tables_that_are_no_quadtree(kind, side, levels, prec):
    print("case table %s, side %d, %d levels, %s" % (kind, side, levels + 1, prec), flush=True)
    sc = edit(mesh(prec, levels), kind, side)
    d = domain_for(sc, precision=prec)
    lg = loop(bgf.Loop)
    d.init_dt(lg)
    d.run(lg, 20)
    against(sc, prec, 20, lg.dt, lg.totaltime, d.get_state())
    d.close()


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("kind", ["odd", "all"])
def test_beside_a_regular_member(kind, prec):
    print("case table %s in a batch, %s" % (kind, prec), flush=True)
    mem = [mesh(prec, 2), edit(mesh(prec, 2), kind, 1), mesh(prec, 1)]
    T = np.float64 if prec == "fp64" else np.float32
    b = bgf.Batch(dict(mem[0]["param"], precision=prec, minlevel=0, maxlevel=2), sum(m["param"]["nblkmem"] for m in mem), 3)
    ids = [b.add(dict(m["param"], precision=prec), m["blocks"], *[np.asarray(m[k]).astype(T) for k in
                                                                  ("zb", "h", "u", "v", "cf")], endtime=1e9) for m in mem]
    b.run(20)
    for mid, m in zip(ids, mem):
        lb, _ = b.loop(mid)
        against(m, prec, 20, lb.dt, lb.totaltime, b.get_state(mid))
    b.close()
