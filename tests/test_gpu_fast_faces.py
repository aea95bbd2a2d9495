"""The predictor's tendencies of the FAST kernels by themselves, cell by cell against the FP64 oracle: states
with dry cells and films between wet ones, rough and smooth beds, walls and Neumann sides, where each cell's
source depends on which of its neighbours are wet.

One step of 1e-7 s (its end is an output time) leaves the stage state where it was, so the oracle's tendencies
after it are those of the same state to 1e-7 s of change.  A face is some 50 operations on quantities of up to
h (|u| + c) for the mass and h (|u| + c)^2 for the momentum, each rounded to 2^-23 at the worst (hardware
reciprocals and square roots among them), and a cell takes four faces and two sources over the cell size: 64
roundings of that size for each bound the error."""
import numpy as np
import pytest

import bg_flood_amd as bgf
from bg_flood_amd import scenarios
from oracle import pyoracle as po
from tests._util import domain_for, hip, oracle_for

pytestmark = pytest.mark.gpu

N, DX, EPS, GRAV = 64, 4.0, 1e-4, 9.81


def state(kind, aoibnd, seed):
    rng = np.random.default_rng(seed)
    p, blocks, nbx, nby = scenarios.uniform(N, N, DX, "fp32", aoibnd=aoibnd, frictionmodel=0, cf=0.0)
    n = p["nblkmem"] * 324
    X, Y = scenarios.cell_coords(blocks, p["nblkmem"], 0.0, 0.0, DX, np.float64)
    if kind == "rough":
        zb = rng.uniform(-2.0, 2.0, n)
        wet, film = rng.random(n) < 0.6, rng.random(n) < 0.1
    else:
        zb = 1.2 * np.sin(X / 30.0) * np.cos(Y / 25.0) + rng.uniform(-0.02, 0.02, n)
        wet = zb < 0.5 + 0.1 * rng.random(n)
        film = rng.random(n) < 0.03
    h = np.where(film, 0.5 * EPS, np.where(wet, np.where(kind == "rough", rng.uniform(0.01, 2.0, n),
                                                         np.maximum(0.8 - zb, 0.01)), 0.0))
    moving = h > EPS
    u = np.where(moving, rng.uniform(-1.0, 1.0, n) if kind == "rough" else np.cos(X / 20.0 + seed), 0.0)
    v = np.where(moving, rng.uniform(-1.0, 1.0, n) if kind == "rough" else np.sin(Y / 15.0), 0.0)
    m = bgf.interior_mask(p["nblkmem"], blocks["active"][:p["nblk"]])
    sc = dict(param=p, blocks=blocks, nbx=nbx, nby=nby)
    for k, a in (("zb", zb), ("h", h), ("u", u), ("v", v), ("cf", 0.0 * h)):
        sc[k] = np.where(m, a, 0.0).astype(np.float32)
    return sc


def tendencies(d, name, nblk):
    out = np.empty((nblk, 16, 16), np.float32)
    assert hip().hipMemcpy(out.ctypes.data, d.device_array(name), out.nbytes, 2) == 0
    return out


@pytest.mark.parametrize("prec", ["fp32_fast", "fp32_comp"])
@pytest.mark.parametrize("aoibnd", [0, 1])
@pytest.mark.parametrize("kind", ["rough", "smooth"])
def test_tendencies_of_wet_and_dry_cells(kind, aoibnd, prec):
    worst = {}
    for seed in range(4):
        print("case FAST faces %s, sides %d, seed %d, %s" % (kind, aoibnd, seed, prec), flush=True)
        sc = state(kind, aoibnd, seed)
        nblk = sc["param"]["nblk"]
        wide = dict(sc, param=dict(sc["param"], precision="fp64"))
        for k in ("zb", "h", "u", "v", "cf"):
            wide[k] = sc[k].astype(np.float64)
        d, o = domain_for(sc, precision=prec), oracle_for(wide, precision="fp64")
        lg = bgf.Loop(nextoutputtime=1e-7, dt=0, dtmax=0, totaltime=0)
        lo = po.OrcLoop(nextoutputtime=1e-7, dt=0, dtmax=0, totaltime=0)
        d.init_dt(lg)
        o.init_loop(lo)
        d.step(lg)
        o.step(lo)
        assert abs(lg.dt - 1e-7) < 1e-13 and abs(lo.dt - 1e-7) < 1e-13
        h = sc["h"].astype(np.float64)
        speed = (np.hypot(sc["u"], sc["v"]) + np.sqrt(GRAV * h)).max()
        size = dict(dh=h.max() * speed, dhu=h.max() * speed ** 2, dhv=h.max() * speed ** 2)
        act = sc["blocks"]["active"][:nblk]
        dry = h.reshape(-1, 18, 18)[act, 1:-1, 1:-1] <= EPS
        for k in ("dh", "dhu", "dhv"):
            want = o.get(k).reshape(-1, 18, 18)[act, 1:-1, 1:-1]
            err = np.abs(tendencies(d, k, sc["param"]["nblkmem"])[act] - want)
            bound = 6 * 64 * 2.0 ** -23 * size[k] / DX
            worst[k] = max(worst.get(k, 0.0), err.max() / bound)
            assert err.max() <= bound, (k, err.max(), bound, dry.reshape(-1)[err.argmax()])
            # dry cells beside wet ones have tendencies far above the bound: their sources are seen
            assert (np.abs(want[dry]) > 100 * bound).sum() > 20
        d.close()
    print("worst errors over their bounds", worst)
