"""The multi-level stage on scattered quadtrees against the oracle, bit for bit: meshes refined at
random blocks (every kind of side next to every other, coarse blocks that end beside a coarser one, as
the halo cells at the end of a half side need) with an island through the refinement boundaries, on two
and three levels (the halo formed in the stage) and four (the halo filled level by level)."""
import numpy as np
import pytest

import bg_flood_amd as bgf
from bg_flood_amd import scenarios
from oracle import pyoracle as po
from tests._util import domain_for, oracle_for

pytestmark = pytest.mark.gpu

FACING = {"LeftBot": "RightBot", "RightBot": "LeftBot", "BotLeft": "TopLeft", "TopLeft": "BotLeft"}
ADJOINING = {"LeftBot": (("BotLeft", "BotRight"), ("TopLeft", "TopRight")),
             "RightBot": (("BotLeft", "BotRight"), ("TopLeft", "TopRight")),
             "BotLeft": (("LeftBot", "LeftTop"), ("RightBot", "RightTop")),
             "TopLeft": (("LeftBot", "LeftTop"), ("RightBot", "RightTop"))}


def scattered(levels, seed, prec, aoibnd=0):
    nbx, nby, part = (8, 7, 0.2) if levels == 3 else (5, 4, 0.45)

    def refine(l, x, y):
        return np.random.default_rng([seed, l, x, y]).random() < part

    sc = scenarios.amr_basin(nbx=nbx, nby=nby, maxlevel=levels, depth=1.5, amp=0.8, precision=prec, island=True,
                             aoibnd=aoibnd, frictionmodel=0, cf=0.002, refine=refine)
    assert sc["param"]["maxlevel"] - sc["param"]["minlevel"] == levels
    return sc


def chains(sc):
    """Coarse neighbours that end, on the block's half, beside a still coarser block."""
    b, n = sc["blocks"], 0
    lev = b["level"]
    for ib in range(sc["param"]["nblk"]):
        for side, back in FACING.items():
            C = b[side][ib]
            if lev[C] >= lev[ib]:
                continue
            first = b[back][C] == ib
            n += lev[b[ADJOINING[side][0 if first else 1][0]][C]] < lev[C]
    return n


def compare(sc, prec, steps):
    d, o = domain_for(sc, precision=prec), oracle_for(sc, precision=prec)
    lg = bgf.Loop(nextoutputtime=1e9, dt=0, dtmax=0, totaltime=0)
    lo = po.OrcLoop(nextoutputtime=1e9, dt=0, dtmax=0, totaltime=0)
    d.init_dt(lg)
    o.init_loop(lo)
    d.run(lg, steps)
    o.run(lo, steps)
    assert lg.dt == lo.dt and lg.totaltime == lo.totaltime
    m = bgf.interior_mask(d.nblkmem, d.active)
    st = d.get_state()
    for k in ("h", "u", "v"):
        assert np.array_equal(st[k][m], o.get(k)[m]), k
    assert (st["h"][m] <= sc["param"]["eps"]).any() and (st["h"][m] > 1.0).any()
    d.close()


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("levels,seed,aoibnd", [(1, 3, 0), (2, 4, 0), (2, 5, 1), (3, 6, 0)])
def test_scattered_quadtrees(levels, seed, aoibnd, prec):
    sc = scattered(levels, seed, prec, aoibnd)
    print("case scattered levels=%d seed=%d %s nblk=%d chains=%d" % (levels, seed, prec, sc["param"]["nblk"],
                                                                     chains(sc)), flush=True)
    if levels > 1:
        assert chains(sc) > 0
    compare(sc, prec, 25)
