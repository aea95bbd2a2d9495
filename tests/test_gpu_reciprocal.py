"""The exact faces where the spread of the wave speeds has a significand of ones: the one divisor at which
the correction that follows the hardware reciprocal stops short of the rounded quotient, because its last
sum is a tie.  Still water of a depth with such a speed stands beside water of another depth; the exact
kernels keep the oracle's operations, so the comparison is bit for bit."""
import numpy as np
import pytest

import bg_flood_amd as bgf
from bg_flood_amd import scenarios
from oracle import pyoracle as po
from tests._util import domain_for, oracle_for

pytestmark = pytest.mark.gpu

GRAV = 8.0  # a power of two: g h is exact


def deep(T):
    """A depth whose still faces divide by a number of a significand of ones: twice the wave speed."""
    ulp = np.finfo(T).eps
    for k in range(1, 9):
        h = T(4.0 - k * ulp) / T(GRAV)
        b = T(2.0) * np.sqrt(T(GRAV) * h)
        if np.frexp(b)[0] == T(1.0) - ulp / T(2.0):
            return h
    raise AssertionError("no such depth")


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("mesh", ["one level", "three levels"])
def test_spread_of_ones(mesh, prec):
    print("case spread of ones, %s %s" % (mesh, prec), flush=True)
    T = np.float64 if prec == "fp64" else np.float32
    if mesh == "one level":
        sc = scenarios.gaussian_hump(n=64, dx=4.0, depth=2.0, amp=0.1, radius=20.0, precision=prec)
        width = 64 * 4.0
    else:
        sc = scenarios.amr_basin(nbx=4, nby=4, dx=10.0, maxlevel=2, precision=prec)
        width = 4 * 16 * 10.0
    sc["param"]["g"] = GRAV
    X, Y = scenarios.cell_coords_levels(sc["blocks"], sc["param"]["nblkmem"], 0.0, 0.0, sc["param"]["dx"], np.float64)
    m = bgf.interior_mask(sc["param"]["nblkmem"], sc["blocks"]["active"][:sc["param"]["nblk"]])
    sc["zb"] = np.zeros_like(sc["zb"])
    # the deeper water in the middle half along x and along y: its edges cross blocks and levels
    inside = (abs(X / width - 0.5) < 0.27) & (abs(Y / width - 0.5) < 0.23)
    sc["h"] = np.where(m, np.where(inside, deep(T), T(0.375)), T(0)).astype(T)
    d, o = domain_for(sc, precision=prec), oracle_for(sc, precision=prec)
    lg = bgf.Loop(nextoutputtime=1e9, dt=0, dtmax=0, totaltime=0)
    lo = po.OrcLoop(nextoutputtime=1e9, dt=0, dtmax=0, totaltime=0)
    d.init_dt(lg)
    o.init_loop(lo)
    for _ in range(3):
        d.step(lg)
        o.step(lo)
        assert lg.dt == lo.dt and lg.dt > 0
    st = d.get_state()
    for k in ("h", "u", "v"):
        assert np.array_equal(st[k][m], o.get(k)[m]), k
    assert np.abs(st["u"][m]).max() > 0
    d.close()
