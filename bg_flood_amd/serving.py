"""Continuous batching of flood-solve requests on one GPU.

A request is one scenario to run to its own simulated horizon; the result is its maximum-depth
grid and the time series of up to 16 gauges.  One-level (Cartesian) requests join a shared
bg_flood_amd.Batch as members: they are admitted while block slots, member slots and the HBM
budget allow, advance together (each with its own dt) in chunks of steps, and leave the batch as
soon as they reach their horizon, which frees room for the requests still waiting.  Multi-level
(AMR) requests join a second batch, of multi-level domains, made for the parameters of the first
one that arrives (grid spacing, levels, physics): its members advance together through one set
of multi-level launches, each with its own dt, on their own stream, so those launches overlap the
one-level batch's on the device.  A multi-level request whose parameters differ from that batch's
runs on its own Domain handle and stream.  Maximum depth and gauges are recorded on the GPU for
every request.  Admission is first fit in arrival order, so a large request waiting for room does
not hold back the smaller ones behind it (up to an age limit that keeps it from starving).  A
member's arithmetic does not depend on the other members (same kernels, its own dt, its own gauge
sampling counted in its own steps), so a result is the same whether the request ran alone or in
the mix.

There is no counterpart in the reference, which runs one scenario per process
(src/Mainloop.cu:17-91); the outputs follow its max-depth and gauge outputs
(src/Meanmax.cu, src/Mainloop.cu:359-500).
"""
import collections
import time

import numpy as np

from . import BS, Batch, BgfError, Domain, Loop, interior_mask

# HBM bytes of one block slot in the batch (h, u, v twice, zb, cf, dh, dhu, dhv, max depth,
# compensation) and of one block slot of a multi-level domain or batch: the cells' arrays (those
# without the compensation, the eight face-flux arrays, the pre-prolongation copy of h, and in a
# domain the remesh staging of the bed and the roughness instead of the max depth), the gather
# recipes (132 entries of 24 bytes), the neighbour record (64) and the block lists and tables.
BATCH_BYTES_PER_BLOCK = 13 * BS * 4
AMR_BYTES_PER_BLOCK = 22 * BS * 4 + 132 * 24 + 64 + 160


class Request:
    """A solve request: scenario dict (param, blocks, nbx, nby, zb, h, u, v, cf), horizon in
    simulated seconds and up to 16 gauge cells (memloc indices)."""

    def __init__(self, rid, scenario, horizon, gauges=(), gauge_every=10):
        self.rid = rid
        self.sc = scenario
        self.horizon = float(horizon)
        self.gauges = list(gauges)[:16]
        self.gauge_every = int(gauge_every)
        self.multilevel = scenario["param"]["maxlevel"] > scenario["param"]["minlevel"]
        self.submitted = None
        self.finished = None
        self.result = None
        self.cells = scenario["param"]["nblk"] * 256
        self.cell_updates = 0

    @property
    def latency(self):
        return None if self.finished is None else self.finished - self.submitted


# Parameters a multi-level request must share with the multi-level batch to join it.
AMR_SHARED = ("g", "eps", "CFL", "theta", "dx", "delta", "frictionmodel", "aoibnd", "ForceMassConserve", "lat",
              "mask", "rain_on", "wetdryfix", "spherical")


class Server:
    def __init__(self, common, max_blocks, max_members=128, hbm_budget=250e9, chunk=40, max_bypass_s=30.0,
                 amr_max_blocks=24000, amr_max_members=32):
        self.batch = Batch(common, max_blocks, max_members)
        self.batch.track_maxdepth(True)
        self.precision = common["precision"]
        self.max_blocks = max_blocks
        self.budget = float(hbm_budget)
        self.used = BATCH_BYTES_PER_BLOCK * max_blocks  # the batch is allocated up front
        self.chunk = int(chunk)
        self.max_bypass_s = float(max_bypass_s)
        self.waiting = collections.deque()
        self.members = {}  # member id -> request
        self.domains = []  # [request, Domain, Loop, bytes]
        self.done = []
        self.cell_updates_amr = 0
        # the multi-level batch, made at the first multi-level request
        self.amr_batch = None
        self.amr_common = None
        self.amr_max_blocks = int(amr_max_blocks)
        self.amr_max_members = int(amr_max_members)
        self.amr_members = {}  # member id -> request

    # ------------------------------------------------------------ requests
    def submit(self, req, now=None):
        req.submitted = time.perf_counter() if now is None else now
        self.waiting.append(req)

    def _fits_ever(self, r):
        """Whether the request could be admitted into an empty server at all."""
        p = r.sc["param"]
        if r.multilevel:
            return BATCH_BYTES_PER_BLOCK * self.max_blocks + AMR_BYTES_PER_BLOCK * p["nblkmem"] <= self.budget
        return p["nblkmem"] <= self.max_blocks

    def _amr_joins(self, p):
        """Whether a multi-level request can join the multi-level batch (making it if there is none
        and the memory allows)."""
        if self.amr_batch is None:
            need = AMR_BYTES_PER_BLOCK * self.amr_max_blocks
            if p["nblkmem"] > self.amr_max_blocks or self.used + need > self.budget:
                return False
            self.amr_common = dict(p, precision=self.precision if self.precision in ("fp64", "fp32") else "fp32")
            self.amr_batch = Batch(self.amr_common, self.amr_max_blocks, self.amr_max_members)
            self.amr_batch.track_maxdepth(True)
            self.used += need
        c = self.amr_common
        return (all(p[k] == c[k] for k in AMR_SHARED if k in c and k in p) and p["minlevel"] >= c["minlevel"]
                and p["maxlevel"] <= c["maxlevel"])

    def _try_admit(self, r):
        """Admits one request if its memory (and, for batch members, a block and member slot) is free
        now; returns whether it was admitted."""
        p = r.sc["param"]
        if r.multilevel and self._amr_joins(p):
            try:
                mid = self.amr_batch.add(p, r.sc["blocks"], r.sc["zb"], r.sc["h"], r.sc["u"], r.sc["v"],
                                         r.sc["cf"], endtime=r.horizon)
            except BgfError:
                return False  # no block or member slot free until a member leaves
            if r.gauges:
                self.amr_batch.set_gauges(mid, r.gauges, every=r.gauge_every)
            self.amr_members[mid] = r
            return True
        if r.multilevel:
            need = AMR_BYTES_PER_BLOCK * p["nblkmem"]
            if self.used + need > self.budget:
                return False
            d = Domain(dict(p, precision=self.precision), r.sc["blocks"])
            d.set_state(r.sc["zb"], r.sc["h"], r.sc["u"], r.sc["v"], r.sc["cf"])
            L = Loop(nextoutputtime=r.horizon, dt=0, dtmax=0, totaltime=0)
            d.init_dt(L)
            d.set_stats(max=True)  # the running maximum of h, every step, on the GPU
            if r.gauges:
                d.set_gauges(r.gauges, every=r.gauge_every)  # sampled on the GPU, counted in its own steps
            self.domains.append([r, d, L, need])
            self.used += need
            return True
        try:
            mid = self.batch.add(p, r.sc["blocks"], r.sc["zb"], r.sc["h"], r.sc["u"], r.sc["v"], r.sc["cf"],
                                 endtime=r.horizon)
        except BgfError:
            return False  # no block or member slot free until a member leaves
        if r.gauges:
            self.batch.set_gauges(mid, r.gauges, every=r.gauge_every)
        self.members[mid] = r
        return True

    def _admit(self, now=None):
        """First fit in arrival order: a request that does not fit yet does not hold back smaller ones
        behind it, unless it has waited longer than `max_bypass_s` (then nothing overtakes it, so
        large requests are not starved).  Requests that cannot fit even an empty server fail."""
        now = time.perf_counter() if now is None else now
        kept = collections.deque()
        blocked = False
        while self.waiting:
            r = self.waiting.popleft()
            if not self._fits_ever(r):
                r.result = dict(error="request larger than the server's capacity")
                r.finished = now
                self.done.append(r)
                continue
            if blocked or not self._try_admit(r):
                kept.append(r)
                if now - r.submitted > self.max_bypass_s:
                    blocked = True
        self.waiting = kept

    # ------------------------------------------------------------ serving
    def poll(self):
        """One scheduling round: admit, advance everything by one chunk, harvest finished requests."""
        self._admit()
        if self.members:
            self.batch.run_async(self.chunk)
        if self.amr_members:
            self.amr_batch.run_async(self.chunk)
        for rec in self.domains:
            rec[1].run_async(rec[2], self.chunk, endtime=rec[0].horizon)
        for rec in self.domains:
            self._sync_domain(rec)
        if self.amr_members:
            before = self.amr_batch.stats()["cell_updates"]
            self.amr_batch.sync()
            self.cell_updates_amr += self.amr_batch.stats()["cell_updates"] - before
            now = time.perf_counter()
            for mid in list(self.amr_members):
                L, done = self.amr_batch.loop(mid)
                if done:
                    r = self.amr_members.pop(mid)
                    info = self.amr_batch.members[mid]
                    mask = interior_mask(info["nblkmem"], info["active"])
                    h0 = np.asarray(r.sc["h"], np.float32)
                    hmax = np.maximum(self.amr_batch.maxdepth(mid), h0)  # the initial state counts too
                    gv, gt = self.amr_batch.gauges(mid)
                    r.result = dict(maxdepth=np.where(mask, hmax, 0), gauges=gv[:len(r.gauges)] if r.gauges else None,
                                    times=gt, totaltime=L.totaltime)
                    r.finished = now
                    self.amr_batch.remove(mid)
                    self.done.append(r)
        if self.members:
            self.batch.sync()
            now = time.perf_counter()
            for mid in list(self.members):
                L, done = self.batch.loop(mid)
                if done:
                    r = self.members.pop(mid)
                    mask = interior_mask(self.batch.members[mid]["nblkmem"], self.batch.members[mid]["active"])
                    hmax = np.where(mask, self.batch.maxdepth(mid), 0)
                    gv, gt = self.batch.gauges(mid)
                    r.result = dict(maxdepth=hmax, gauges=gv[:len(r.gauges)], times=gt, totaltime=L.totaltime)
                    r.finished = now
                    self.batch.remove(mid)
                    self.done.append(r)
        now = time.perf_counter()
        for rec in list(self.domains):
            r, d, L = rec[0], rec[1], rec[2]
            if L.totaltime >= r.horizon:
                p = r.sc["param"]
                mask = interior_mask(p["nblkmem"], r.sc["blocks"]["active"][:p["nblk"]])
                h0 = np.asarray(r.sc["h"], np.float32)
                hmax = np.maximum(d.stat("hmax").astype(np.float32), h0)  # the initial state counts too
                gv, gt = d.gauges() if r.gauges else (None, np.zeros(0))
                r.result = dict(maxdepth=np.where(mask, hmax, 0), gauges=gv, times=gt, totaltime=L.totaltime)
                r.finished = now
                d.close()
                self.used -= rec[3]
                self.domains.remove(rec)
                self.done.append(r)

    def _sync_domain(self, rec):
        r, d, L = rec[0], rec[1], rec[2]
        d.sync(L)
        n = d.last_run_steps()
        r.cell_updates += n * r.cells
        self.cell_updates_amr += n * r.cells

    def busy(self):
        return bool(self.waiting or self.members or self.domains or self.amr_members)

    def stats(self):
        return self.batch.stats()

    def close(self):
        for rec in self.domains:
            rec[1].close()
        self.domains = []
        self.batch.close()
        if self.amr_batch is not None:
            self.amr_batch.close()
            self.amr_batch = None


def serve(requests, arrivals, common, max_blocks, max_members=128, hbm_budget=250e9, chunk=40, time_limit=600.0):
    """Feeds requests to a Server at their arrival times (seconds from the start, real time) and
    serves until all are done or time_limit passes.  Returns (server, wall seconds)."""
    srv = Server(common, max_blocks, max_members, hbm_budget, chunk)
    order = np.argsort(arrivals)
    t0 = time.perf_counter()
    k = 0
    while True:
        now = time.perf_counter() - t0
        while k < len(order) and arrivals[order[k]] <= now:
            srv.submit(requests[order[k]], now=t0 + arrivals[order[k]])
            k += 1
        if not srv.busy():
            if k >= len(order):
                break
            time.sleep(min(0.002, max(0.0, arrivals[order[k]] - now)))
            continue
        srv.poll()
        if time.perf_counter() - t0 > time_limit:
            break
    return srv, time.perf_counter() - t0
