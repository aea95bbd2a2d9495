"""bgf_step_noalloc, the one-level step that allocates nothing, called through the C ABI on device
arrays, against bgf_step (the handle's step) on the same inputs: dt, dtmax and the new h, u, v of
every interior cell bit-identical, in FP64, FP32 and FP32_FAST, over two calls in a row of which the
second has fewer blocks (the scratch array keeps the first call's contents), and over two chained
steps.  Sizes beyond the scratch array and the compensated form are refused before any launch."""
import ctypes

import numpy as np
import pytest

import bg_flood_amd as bgf
from bg_flood_amd import scenarios
from tests._util import DeviceArray, domain_for, hip, interior

pytestmark = pytest.mark.gpu

BLOCK_DEV_KEYS = ("active", "LeftBot", "RightBot", "BotLeft", "TopLeft")


def _lib():
    L = bgf.lib()
    vp = ctypes.c_void_p
    L.bgf_step_noalloc.argtypes = [ctypes.POINTER(bgf.BgfParam), ctypes.POINTER(bgf.BgfBlocks)] + [vp] * 8 + [
        ctypes.POINTER(bgf.Loop), vp]
    L.bgf_step_noalloc.restype = ctypes.c_int
    return L


def _dev(a):
    return DeviceArray(np.ascontiguousarray(a))


class DeviceDomain:
    """A scenario's arrays in device memory the caller allocated itself (hipMalloc)."""

    def __init__(self, sc, prec):
        self.sc = sc
        self.param = dict(sc["param"], precision=prec)
        T = np.float64 if prec == "fp64" else np.float32
        self.T = T
        nbm = self.param["nblkmem"]
        keep = {}
        host = bgf._blocks_struct(sc["blocks"], nbm, keep)
        del host
        self.blk = {k: _dev(keep[k]) for k in BLOCK_DEV_KEYS}
        self.B = bgf.BgfBlocks()
        for k in BLOCK_DEV_KEYS:
            setattr(self.B, k, ctypes.cast(ctypes.c_void_p(self.blk[k].ptr), ctypes.POINTER(ctypes.c_int)))
        self.a = {k: _dev(np.asarray(sc[k], T)) for k in ("zb", "cf", "h", "u", "v")}
        for k in ("h", "u", "v"):
            self.a[k + "o"] = self.a[k].copy()
        self.P = bgf._param_struct(self.param)

    def step(self, L, loop):
        a = self.a
        assert hip().hipDeviceSynchronize() == 0
        rc = L.bgf_step_noalloc(ctypes.byref(self.P), ctypes.byref(self.B), a["zb"].ptr, a["cf"].ptr, a["h"].ptr,
                                a["u"].ptr, a["v"].ptr, a["ho"].ptr, a["uo"].ptr, a["vo"].ptr, ctypes.byref(loop), None)
        assert rc == 0, L.bgf_last_error().decode()
        # the result becomes the next step's input
        for k in ("h", "u", "v"):
            a[k], a[k + "o"] = a[k + "o"], a[k]

    def state(self):
        return {k: self.a[k].numpy() for k in ("h", "u", "v")}


def _scenario(n, prec):
    return scenarios.rain_terrain(n=n, dx=5.0, amp=10.0, rain=200.0, manning=0.03, seed=3,
                                  precision="fp64" if prec == "fp64" else "fp32")


def _check_against_handle(L, n, prec, nsteps):
    sc = _scenario(n, prec)
    print("case no-alloc step: %s, %d x %d cells, %d steps" % (prec, n, n, nsteps), flush=True)
    d = domain_for(sc, precision=prec)
    lg = bgf.Loop(nextoutputtime=1e9, dt=0, dtmax=0, totaltime=0)
    d.init_dt(lg)
    dd = DeviceDomain(sc, prec)
    ln = bgf.Loop(nextoutputtime=1e9, dt=lg.dt, dtmax=lg.dtmax, totaltime=0)
    for k in range(nsteps):
        d.step(lg)
        dd.step(L, ln)
        assert ln.dt == lg.dt and ln.dtmax == lg.dtmax, (k, ln, lg)
        lg.totaltime += lg.dt
        ln.totaltime += ln.dt
    m = interior(sc)
    ref = d.get_state()
    got = dd.state()
    for k in ("h", "u", "v"):
        assert np.array_equal(got[k][m], ref[k][m]), (prec, n, k)
    assert got["h"][m].max() > 0  # the rain has wetted the domain: the steps were not trivial
    d.close()


@pytest.mark.parametrize("prec", ["fp64", "fp32", "fp32_fast"])
def test_noalloc_matches_the_handle_step_then_a_smaller_call(prec):
    L = _lib()
    _check_against_handle(L, 256, prec, 3)  # 256 blocks
    _check_against_handle(L, 128, prec, 2)  # then 64 blocks: the scratch keeps the first call's contents


def test_noalloc_refuses_what_it_cannot_hold():
    L = _lib()
    sc = _scenario(128, "fp32")
    dd = DeviceDomain(sc, "fp32_comp")
    loop = bgf.Loop(nextoutputtime=1e9, dt=1.0, dtmax=1.0, totaltime=0)
    a = dd.a
    args = (a["zb"].ptr, a["cf"].ptr, a["h"].ptr, a["u"].ptr, a["v"].ptr, a["ho"].ptr, a["uo"].ptr, a["vo"].ptr)
    rc = L.bgf_step_noalloc(ctypes.byref(dd.P), ctypes.byref(dd.B), *args, ctypes.byref(loop), None)
    assert rc == 5 and b"COMP" in L.bgf_last_error()
    big = bgf._param_struct(dict(dd.param, precision="fp32", nblk=21619, nblkmem=21619))
    rc = L.bgf_step_noalloc(ctypes.byref(big), ctypes.byref(dd.B), *args, ctypes.byref(loop), None)
    assert rc == 1 and b"21618" in L.bgf_last_error()
    big64 = bgf._param_struct(dict(dd.param, precision="fp64", nblk=10866, nblkmem=10866))
    rc = L.bgf_step_noalloc(ctypes.byref(big64), ctypes.byref(dd.B), *args, ctypes.byref(loop), None)
    assert rc == 1 and b"10865" in L.bgf_last_error()


def _spread(sc, slots, seed):
    """The scenario with its blocks in random slots of `slots` ones, in another order of the list."""
    p, b = sc["param"], sc["blocks"]
    n = p["nblk"]
    rng = np.random.default_rng(seed)
    at = np.full(p["nblkmem"], -1)
    at[b["active"][:n]] = np.append(rng.permutation(slots - 1)[:n - 1], slots - 1)
    out = dict(sc, param=dict(p, nblkmem=slots))
    blocks = {}
    for k, v in b.items():
        v = np.asarray(v)
        if k == "active":
            w = rng.permutation(at[v[:n]]).astype(v.dtype)
        else:
            w = np.zeros(slots, v.dtype)
            w[at[b["active"][:n]]] = at[v[b["active"][:n]]] if k not in ("level", "xo", "yo") else v[b["active"][:n]]
        blocks[k] = w
    out["blocks"] = blocks
    for k in ("zb", "h", "u", "v", "cf"):
        a = np.zeros((slots, 324), np.asarray(sc[k]).dtype)
        a[at[b["active"][:n]]] = np.asarray(sc[k]).reshape(-1, 324)[b["active"][:n]]
        out[k] = a.reshape(-1)
    return out, at


# slots as many as the blocks, a few unused, and more than the scratch holds at the top of the arrays with all
# used ones below (the declared count alone does not decide)
@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("slots,declared", [(64, 64), (97, 97), (1500, 1500), (97, 30000)])
def test_noalloc_with_unused_slots(slots, declared, prec):
    L = _lib()
    print("case no-alloc step: %s, 64 blocks in %d of %d slots" % (prec, slots, declared), flush=True)
    sc = _scenario(128, prec)
    sp, at = _spread(sc, slots, slots)
    d = domain_for(sc, precision=prec)
    lg = bgf.Loop(nextoutputtime=1e9, dt=0, dtmax=0, totaltime=0)
    d.init_dt(lg)
    dd = DeviceDomain(sp, prec)
    dd.P.nblkmem = declared
    ln = bgf.Loop(nextoutputtime=1e9, dt=lg.dt, dtmax=lg.dtmax, totaltime=0)
    for _ in range(2):
        d.step(lg)
        dd.step(L, ln)
        assert ln.dt == lg.dt and ln.dtmax == lg.dtmax
    ref, got = d.get_state(), dd.state()
    n = sc["param"]["nblk"]
    act = sc["blocks"]["active"][:n]
    for k in ("h", "u", "v"):
        a, b = ref[k].reshape(-1, 18, 18)[act, 1:-1, 1:-1], got[k].reshape(-1, 18, 18)[at[act], 1:-1, 1:-1]
        assert np.array_equal(a, b), k
    d.close()


def test_noalloc_refuses_slots_it_cannot_hold():
    L = _lib()
    sc = _scenario(128, "fp32")
    sp, _ = _spread(sc, 22000, 1)
    dd = DeviceDomain(sp, "fp32")
    loop = bgf.Loop(nextoutputtime=1e9, dt=1.0, dtmax=1.0, totaltime=0)
    a = dd.a
    rc = L.bgf_step_noalloc(ctypes.byref(dd.P), ctypes.byref(dd.B), a["zb"].ptr, a["cf"].ptr, a["h"].ptr, a["u"].ptr,
                            a["v"].ptr, a["ho"].ptr, a["uo"].ptr, a["vo"].ptr, ctypes.byref(loop), None)
    assert rc == 1 and b"21999" in L.bgf_last_error()
