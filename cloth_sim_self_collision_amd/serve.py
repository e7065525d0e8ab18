"""Serving many cloth simulations on one GPU with continuous batching.

Requests (a cloth and a number of steps) arrive over time.  The server keeps
every admitted simulation resident on the device (mesh, matrix, factor, BVH,
state) until it finishes.  Admitted requests join one of a few *lanes* by
size (vertex count); each lane is a host thread that steps its resident
cloths together, one ``cs_batch_step(1)`` per tick, and picks up newly
admitted requests at the next tick.  Optionally, large requests
(``solo_from`` vertices and up) run alone instead, each on a thread and
stream of its own with the plain step.  Lanes (and solo requests) run
concurrently, so small cloths tick at their own pace instead of waiting for
the largest resident cloth, and the work of all of them overlaps on the
device.  Cloths are
created (host setup and upload) by a small pool of threads, so a large
cloth's setup does not hold back the admission of the ones after it.

Admission is by resident device footprint: a request is admitted once it has
arrived and its estimated footprint (BYTES_PER_VERTEX_ESTIMATE per vertex, or
the measured ``cs_cloth_memory`` once created and after each step) fits the HBM budget beside the
resident ones.  A request that can never fit, whose cloth cannot be created,
whose step fails or whose solve turns non-finite gets an error result while
the others continue.  Requests can be cancelled (``Server.cancel``) or evicted
(``Server.evict``: its state and simulated time are saved, its device memory
is released and it is admitted again later, continuing exactly where it
stopped).  A creation that runs out of device memory while others are
resident is retried after they retire.

Each cloth's trajectory is bit-identical to stepping it alone (the batched
kernels run each cloth's arithmetic unchanged), so "the same alone and in the
mix" holds exactly, not only within a tolerance.

Reported per request: the final state, the latency of each of its steps (the
wall time of its lane's tick that advanced it) and its queueing delay; per
run: aggregate vertex-steps/s and p50/p99 step latency.

Wire format (JSON lines, `python -m cloth_sim_self_collision_amd.serve`):

  request  {"id": any JSON value, "scene": a scene configuration
            (scene.from_config; one cloth), "steps": int >= 1,
            "arrival": seconds after the start (optional, default 0),
            "precision": "f64" (default, bit-identical to the reference)
                         or "mixed" (FP32 preconditioner coefficients; served
                         only while every step's ILU(0)-PCG converges),
            "return": subset of ["x", "v"] (optional, default ["x"])}
  result   {"id", "status": "ok", "vertices", "triangles", "steps",
            "arrival", "queued_s", "admitted_s", "finished_s",
            "step_ms": [...], "pcg_iters": [...], "impulse_applied": [...],
            "n_prox": [...], "n_ccd": [[...] per step],
            "x": {"dtype": "<f8", "shape": [np, 3], "data": base64}, "v": ...}
           or {"id", "status": "error", "error": message} for a request
           that cannot be served (bad record, unknown scene, precision, too
           large for the budget, a failed or non-finite step, a mixed-precision
           step whose solve did not converge, cancelled).

Results are written as requests finish, one line each, in completion order.
"""
from __future__ import annotations

import base64
import concurrent.futures as cf
import dataclasses
import json
import sys
import threading
import time
from typing import Callable, Iterable, List, Optional, TextIO

import numpy as np

from . import _lib
from . import scene
from .scene import Cloth, SplitMix64
from .sim import DeviceBatch, DeviceCloth

# admission estimate before a cloth exists on the device: bytes per vertex of
# the resident footprint (cs_cloth_memory of grids at creation: 9956 at 65k
# vertices, 9940 at 100k, 9920 at 1M, rounded up).  The real footprint counts
# from the creation on, and again after each step (contact buffers grow: 10151,
# 10414 and 10990 after a step of the same cloths).
BYTES_PER_VERTEX_ESTIMATE = 10240
# a request is refused only where this much does not fit the budget; between
# the two it is admitted when nothing else is resident
LEAST_BYTES_PER_VERTEX = 8192

# lane boundaries by vertex count: six lanes, [0, 2500), [2500, 8000), ...,
# [60000, inf).  A lane's tick lasts as long as its slowest member's step, so
# members of similar size waste little; measured on a 64-request stream of the
# serving workload (1e3..2e5 triangles): 141 000 vertex-steps/s with these
# six lanes against 129 000 with five (2500, 8000, 21846, 50000), 122 000
# with eight and 84 000 with every cloth of 21846 vertices or more alone.
DEFAULT_LANES = (2500, 8000, 16000, 30000, 60000)
# PCG variant per default lane (CS_OPT_PCG): the two smallest lanes run each
# cloth's whole solve in one workgroup (one launch per step instead of about
# seven per PCG iteration), the others one launch per PCG operation
DEFAULT_LANE_PCG = (2, 2, 0, 0, 0, 0)
_OPT_PCG = 2
# requests of at least this many vertices are stepped alone, each by its own
# thread on its own stream, instead of joining a lane (None: never)
DEFAULT_SOLO_FROM: Optional[int] = None
# Per lane: how many instances of the lane may step at once, and how long an
# idle instance gathers members before its first tick (seconds).  A request
# that arrives while every instance of its lane is in a tick starts another
# instance (up to the limit) instead of waiting for the next tick, and an
# instance that starts from idle waits this window for the requests arriving
# just after (a tick cannot take members once it runs).  Default: off
# (one instance, no window) in every lane.
DEFAULT_LANE_INSTANCES = (1, 1, 1, 1, 1, 1)
DEFAULT_LANE_WINDOW = (0.0, 0.0, 0.0, 0.0, 0.0, 0.0)
# cloths created at once on admission (host setup and upload)
CREATORS = 4
_NONFINITE = "the solve produced an infinite or NaN displacement (the ILU(0)-PCG iterate overflowed)"
_OPT_PRECISION = 3


def _step_error(req: "Request", st: dict) -> Optional[str]:
    """Why a step's result cannot be served, or None."""
    if st["status"] != 0:
        return _NONFINITE
    if (req.precision == "mixed" and st["pcg_iters"] >= req.cloth.pcg_maxit and
            not st["pcg_conv"] < req.cloth.pcg_tol):
        return ("mixed precision is served only where ILU(0)-PCG converges: this step stopped "
                f"at the cap of {req.cloth.pcg_maxit} iterations (residual ratio "
                f"{st['pcg_conv']:.3g}); request precision f64")
    return None


@dataclasses.dataclass
class Request:
    rid: object  # any JSON value on the wire
    cloth: Cloth
    steps: int
    arrival: float = 0.0  # seconds after the start of the run
    returns: tuple = ("x",)  # arrays of the final state in the wire result
    precision: str = "f64"  # or "mixed"


@dataclasses.dataclass
class Result:
    rid: int
    xyz: np.ndarray
    uvw: np.ndarray
    step_ms: List[float]
    queued_s: float
    admitted_s: float
    finished_s: float
    vertices: int
    pcg_iters: List[int]
    impulse_applied: List[bool] = dataclasses.field(default_factory=list)
    n_prox: List[int] = dataclasses.field(default_factory=list)
    n_ccd: List[list] = dataclasses.field(default_factory=list)


@dataclasses.dataclass
class Failure:
    rid: object
    error: str


@dataclasses.dataclass
class _Active:
    req: Request
    dev: Optional[DeviceCloth] = None
    done: int = 0
    step_ms: List[float] = dataclasses.field(default_factory=list)
    pcg_iters: List[int] = dataclasses.field(default_factory=list)
    impulse_applied: List[bool] = dataclasses.field(default_factory=list)
    n_prox: List[int] = dataclasses.field(default_factory=list)
    n_ccd: List[list] = dataclasses.field(default_factory=list)
    admitted_s: float = -1.0
    memory: int = 0
    saved: Optional[tuple] = None  # (x, v, t) of an evicted request
    cancel: bool = False
    evict: bool = False


class _Lane:
    """One host thread stepping a set of resident cloths together, or (solo)
    one cloth alone with the plain step until it leaves."""

    def __init__(self, server: "Server", index: int, solo: Optional[_Active] = None,
                 tune: bool = False):
        self.server = server
        self.index = index
        self.inbox: List[_Active] = []
        self.active: List[_Active] = []
        self.batch: Optional[DeviceBatch] = None
        self.members: tuple = ()
        self.ticks = 0
        self.solo = solo
        self.tuner = _VariantTuner() if tune and solo is None else None
        self.window = 0.0     # seconds an idle instance gathers members before a tick
        self.in_tick = False  # stepping now (set under the server's lock)
        target = self._run if solo is None else self._run_solo
        self.thread = threading.Thread(target=target, name=f"lane{index}", daemon=True)

    def _close_batch(self):
        if self.batch is not None:
            self.batch.close()
        self.batch = None
        self.members = ()

    def _run(self):
        srv = self.server
        try:
            while True:
                with srv.cv:
                    while not self.inbox and not self.active and not srv.stopping:
                        srv.cv.wait(0.05)
                    if srv.stopping and not self.inbox and not self.active:
                        return
                    if not self.active and self.window > 0.0:
                        # from idle: gather the requests arriving within the
                        # window into this first tick
                        until = srv.clock() + self.window
                        while not srv.stopping and srv.clock() < until:
                            srv.cv.wait(min(0.02, max(0.0, until - srv.clock())))
                    self.active.extend(self.inbox)
                    self.inbox.clear()
                    going = [a for a in self.active if a.cancel or a.evict]
                if going:
                    self._close_batch()  # before any member cloth is destroyed
                    for a in going:
                        self.active.remove(a)
                        self._leave(a, "cancelled" if a.cancel else None)
                if not self.active:
                    self._close_batch()
                    continue
                key = tuple(id(a.dev) for a in self.active)
                if key != self.members:
                    self._close_batch()
                    self.batch = DeviceBatch([a.dev for a in self.active])
                    self.members = key
                    if srv.profile:
                        self.batch.profile(True)
                variant = self._choose_variant()
                with srv.cv:
                    self.in_tick = True
                ts = srv.clock()
                try:
                    stats = self.batch.step(1)
                except _lib.ClothSimError as e:
                    # the whole tick failed: every member gets the error
                    self._close_batch()
                    srv.log(f"lane {self.index}: step failed: {e}")
                    for a in list(self.active):
                        self.active.remove(a)
                        self._leave(a, f"step failed: {e}")
                    continue
                finally:
                    with srv.cv:
                        self.in_tick = False
                dt_ms = (srv.clock() - ts) * 1e3
                self.ticks += 1
                if variant is not None:
                    self.tuner.record(variant, dt_ms / sum(a.dev.np_ for a in self.active))
                if srv.profile:
                    # per-class device time of this tick's shared launches, and
                    # what each member did in it
                    prof = self.batch.profile_read()
                    self.batch.profile(True)
                    rec = {"lane": self.index, "t0_s": ts - srv.t0, "ms": dt_ms, "prof": prof,
                           "members": [(a.dev.np_, a.dev.nnz, st["pcg_iters"], st["status"])
                                       for a, st in zip(self.active, stats)]}
                    with srv.cv:
                        srv.tick_log.append(rec)
                leaving = []
                for a, st in zip(list(self.active), stats):
                    err = _step_error(a.req, st)
                    if err is not None:
                        leaving.append((a, err, False))
                        continue
                    self._record(a, st, dt_ms)
                    if a.done >= a.req.steps:
                        leaving.append((a, None, True))
                if leaving:
                    self._close_batch()  # before any member cloth is destroyed
                    for a, err, fin in leaving:
                        self.active.remove(a)
                        self._leave(a, err, finished=fin)
        except BaseException as e:  # noqa: BLE001 - reported, the server stops
            with srv.cv:
                srv.fatal = e
                srv.cv.notify_all()
        finally:
            self._close_batch()

    def _choose_variant(self) -> Optional[int]:
        """With autotuning, the PCG variant of this tick for every member
        (None: not tuned, the members keep the lane's variant).  Only lanes
        whose members all allow the one-workgroup solve are tuned."""
        if self.tuner is None:
            return None
        v = self.tuner.pick()
        try:
            for a in self.active:
                a.dev.set_option(_OPT_PCG, v)
        except _lib.ClothSimError:
            for a in self.active:  # a member too large for one workgroup
                a.dev.set_option(_OPT_PCG, 0)
            return None
        return v

    def _record(self, a: _Active, st: dict, dt_ms: float) -> None:
        a.done += 1
        a.step_ms.append(dt_ms)
        a.pcg_iters.append(st["pcg_iters"])
        a.impulse_applied.append(bool(st["impulse_applied"]))
        a.n_prox.append(int(st["n_prox"]))
        a.n_ccd.append([int(c) for c in st["n_ccd"][:st["n_ccd_pass"]]])
        # contact buffers grow with the contacts met: admission counts them
        mem = a.dev.memory()
        if mem > a.memory:
            with self.server.cv:
                self.server.resident += mem - a.memory
                a.memory = mem

    def _run_solo(self):
        """Step one cloth alone (its own stream) until it finishes, fails, is
        cancelled or evicted."""
        srv = self.server
        a = self.solo
        try:
            if srv.profile:
                a.dev.profile(True)
            while True:
                if a.cancel or a.evict:
                    self._leave(a, "cancelled" if a.cancel else None)
                    return
                ts = srv.clock()
                try:
                    st = a.dev.step(1)
                except _lib.ClothSimError as e:
                    self._leave(a, f"step failed: {e}")
                    return
                dt_ms = (srv.clock() - ts) * 1e3
                self.ticks += 1
                if srv.profile:
                    rec = {"lane": self.index, "t0_s": ts - srv.t0, "ms": dt_ms,
                           "prof": a.dev.profile_read(),
                           "members": [(a.dev.np_, a.dev.nnz, st["pcg_iters"], st["status"])]}
                    a.dev.profile(True)
                    with srv.cv:
                        srv.tick_log.append(rec)
                err = _step_error(a.req, st)
                if err is not None:
                    self._leave(a, err)
                    return
                self._record(a, st, dt_ms)
                if a.done >= a.req.steps:
                    self._leave(a, None, finished=True)
                    return
        except BaseException as e:  # noqa: BLE001 - reported, the server stops
            with srv.cv:
                srv.fatal = e
                srv.cv.notify_all()

    def _leave(self, a: _Active, error: Optional[str], finished: bool = False):
        """Retire a request from this lane: result, error, or eviction."""
        srv = self.server
        res = None
        if finished:
            x, v = a.dev.get_state()
            res = Result(rid=a.req.rid, xyz=x, uvw=v, step_ms=a.step_ms,
                         queued_s=max(0.0, a.admitted_s - a.req.arrival) if srv.realtime else 0.0,
                         admitted_s=a.admitted_s, finished_s=srv.clock() - srv.t0,
                         vertices=a.req.cloth.np_, pcg_iters=a.pcg_iters,
                         impulse_applied=a.impulse_applied, n_prox=a.n_prox, n_ccd=a.n_ccd)
        elif error is None:  # eviction: keep the state, release the device memory
            x, v = a.dev.get_state()
            a.saved = (x, v, a.dev.time)
        a.dev.close()
        a.dev = None
        with srv.cv:
            srv.resident -= a.memory
            a.memory = 0
            if res is not None:
                srv._finish(a, res)
            elif error is not None:
                srv._fail(a.req.rid, error)
                srv.live.discard(id(a))
            else:
                a.evict = False
                srv.pending.append(a)
                srv.pending.sort(key=lambda q: (q.req.arrival, str(q.req.rid)))
            srv.cv.notify_all()


class _VariantTuner:
    """Picks a lane's PCG variant from measured ticks: the one-workgroup solve
    (2) or one launch per PCG operation (0), by the lower recent tick time per
    member vertex.  Each variant is tried on the first ticks, and the one not
    in use again every `explore` ticks, so the choice follows the lane's
    membership.  Results are the same with either variant."""

    def __init__(self, explore: int = 8, keep: int = 4):
        self.samples = {0: [], 2: []}
        self.explore = explore
        self.keep = keep
        self.n = 0

    def pick(self) -> int:
        self.n += 1
        for v in (2, 0):
            if not self.samples[v]:
                return v
        best = min(self.samples, key=lambda v: sum(self.samples[v]) / len(self.samples[v]))
        return (2 if best == 0 else 0) if self.n % self.explore == 0 else best

    def record(self, v: int, ms_per_vertex: float) -> None:
        self.samples[v] = (self.samples[v] + [ms_per_vertex])[-self.keep:]


class Server:
    """Continuous batching over resident simulations in concurrent lanes.

    hbm_budget_bytes: device memory the resident cloths may hold;
    lanes: vertex-count boundaries of the lanes (one lane per interval; () is
    a single lane that steps every resident cloth together);
    lane_pcg: the PCG variant (CS_OPT_PCG) of each lane's cloths, one value
    per lane (0 automatic, 2 the whole solve in one workgroup per cloth, for
    cloths that allow it); None: DEFAULT_LANE_PCG when lanes is
    DEFAULT_LANES, else automatic everywhere;
    profile: time each tick's shared launches by kernel class (HIP events on
    the lane's stream) and keep a record per tick in tick_log;
    autotune: each lane picks its PCG variant from its measured ticks
    (_VariantTuner) instead of lane_pcg;
    solo_from: requests of at least this many vertices are stepped alone by a
    thread of their own (plain steps on the cloth's stream) instead of
    joining a lane, so a large cloth never paces smaller ones (None: never);
    lane_instances / lane_window: per lane, how many instances may step at
    once (a request arriving while every instance is in a tick starts
    another) and how long an idle instance gathers members before its first
    tick (seconds); None: DEFAULT_LANE_INSTANCES / DEFAULT_LANE_WINDOW.
    Set GPU_MAX_HW_QUEUES (HIP's hardware queues per process, 4 by default)
    to at least the number of lanes plus solo requests before HIP starts, or
    streams share queues and their kernels run one after another."""

    def __init__(self, hbm_budget_bytes: int, clock: Callable[[], float] = time.perf_counter,
                 on_result: Optional[Callable[["Result"], None]] = None,
                 on_error: Optional[Callable[["Failure"], None]] = None,
                 lanes: tuple = DEFAULT_LANES, lane_pcg: Optional[tuple] = None,
                 profile: bool = False, solo_from: Optional[int] = DEFAULT_SOLO_FROM,
                 autotune: bool = False, lane_instances: Optional[tuple] = None,
                 lane_window: Optional[tuple] = None):
        if lane_pcg is None:
            lane_pcg = DEFAULT_LANE_PCG if tuple(lanes) == DEFAULT_LANES else (0,) * (len(lanes) + 1)
        if lane_instances is None:
            lane_instances = DEFAULT_LANE_INSTANCES if tuple(lanes) == DEFAULT_LANES \
                else (1,) * (len(lanes) + 1)
        if lane_window is None:
            lane_window = DEFAULT_LANE_WINDOW if tuple(lanes) == DEFAULT_LANES \
                else (0.0,) * (len(lanes) + 1)
        if len(lane_pcg) != len(lanes) + 1:
            raise ValueError("lane_pcg needs one value per lane")
        if len(lane_instances) != len(lanes) + 1 or min(lane_instances) < 1:
            raise ValueError("lane_instances needs one value of at least 1 per lane")
        if len(lane_window) != len(lanes) + 1 or min(lane_window) < 0.0:
            raise ValueError("lane_window needs one value of at least 0 per lane")
        self.lane_pcg = tuple(int(v) for v in lane_pcg)
        self.lane_instances = tuple(int(v) for v in lane_instances)
        self.lane_window = tuple(float(v) for v in lane_window)
        self.profile = bool(profile)
        self.autotune = bool(autotune)
        self.solo_from = solo_from
        self.solo_lanes: List[_Lane] = []
        self.lanes: dict = {}
        self.tick_log: List[dict] = []
        self.budget = int(hbm_budget_bytes)
        self.clock = clock
        self.on_result = on_result
        self.on_error = on_error
        self.bounds = tuple(lanes)
        self.cv = threading.Condition()
        self.pending: List[_Active] = []
        self.results: List[Result] = []
        self.failures: List[Failure] = []
        self.live: set = set()
        self.resident = 0
        self.stopping = False
        self.fatal: Optional[BaseException] = None
        self.realtime = True
        self.t0 = 0.0
        self._by_rid: dict = {}

    def log(self, msg: str) -> None:
        print(f"[serve] {msg}", file=sys.stderr, flush=True)

    def _lane_of(self, np_: int) -> int:
        k = 0
        while k < len(self.bounds) and np_ >= self.bounds[k]:
            k += 1
        return k

    def _finish(self, a: _Active, res: Result):  # with cv held
        self.results.append(res)
        self.live.discard(id(a))
        if self.on_result is not None:
            self.on_result(res)

    def _fail(self, rid, msg: str):  # with cv held
        f = Failure(rid, msg)
        self.failures.append(f)
        if self.on_error is not None:
            self.on_error(f)

    def cancel(self, rid) -> None:
        """Drop request rid: pending ones at once, resident ones at their
        lane's next tick; it gets an error result "cancelled"."""
        with self.cv:
            for a in list(self.pending):
                if a.req.rid == rid:
                    self.pending.remove(a)
                    self.live.discard(id(a))
                    self._fail(rid, "cancelled")
            a = self._by_rid.get(rid)
            if a is not None and a.dev is not None:
                a.cancel = True
            self.cv.notify_all()

    def evict(self, rid) -> None:
        """Move resident request rid off the device at its lane's next tick
        (state and time saved, memory released); it is admitted again like a
        pending request and continues from the saved state."""
        with self.cv:
            a = self._by_rid.get(rid)
            if a is not None and a.dev is not None:
                a.evict = True
            self.cv.notify_all()

    def run(self, requests: List[Request], *, realtime: bool = True,
            control: Optional[Callable[["Server", float], None]] = None) -> dict:
        """Serve `requests` (arrival times in seconds from now).  realtime: a
        request is admitted only once its arrival time has passed; if not,
        every request counts as arrived at once (throughput runs).  control,
        if given, is called from the admission loop with the elapsed time
        (for cancel/evict)."""
        self.realtime = realtime
        self.solo_lanes = []
        self.pending = [_Active(req=r) for r in sorted(requests, key=lambda r: (r.arrival, str(r.rid)))]
        self._by_rid = {a.req.rid: a for a in self.pending}
        self.live = {id(a) for a in self.pending}
        # lanes are created as requests need them, one per (size interval,
        # precision, PCG tolerance and cap): a batch's cloths share all of these
        self.lanes = {}
        pool = cf.ThreadPoolExecutor(max_workers=CREATORS, thread_name_prefix="create")
        creating: list = []
        self.t0 = self.clock()
        try:
            with self.cv:
                for a in list(self.pending):
                    need = a.req.cloth.np_ * LEAST_BYTES_PER_VERTEX
                    if need > self.budget:
                        self.pending.remove(a)
                        self.live.discard(id(a))
                        self._fail(a.req.rid, f"needs about {need} bytes of device memory, more "
                                              f"than the budget of {self.budget}")
            while True:
                for f in [f for f in creating if f.done()]:
                    f.result()  # an unexpected error in a creation stops the server
                    creating.remove(f)
                now = self.clock() - self.t0
                if control is not None:
                    control(self, now)
                with self.cv:
                    if self.fatal is not None:
                        raise self.fatal
                    if not self.live:
                        break
                    cand = None
                    for a in self.pending:
                        if realtime and a.req.arrival > now:
                            break
                        need = max(a.memory, a.req.cloth.np_ * BYTES_PER_VERTEX_ESTIMATE)
                        if self.resident + need <= self.budget or self.resident == 0:
                            cand = a
                        break  # admission in arrival order
                    if cand is not None:
                        self.pending.remove(cand)
                        cand.memory = cand.req.cloth.np_ * BYTES_PER_VERTEX_ESTIMATE
                        self.resident += cand.memory
                if cand is None:
                    with self.cv:
                        nxt = [a.req.arrival - now for a in self.pending[:1] if realtime]
                        self.cv.wait(max(0.0, min([0.02] + nxt)))
                    continue
                creating.append(pool.submit(self._admit, cand))
        finally:
            pool.shutdown(wait=True)
            with self.cv:
                self.stopping = True
                lanes = [ln for group in self.lanes.values() for ln in group]
                for ln in lanes:
                    for a in ln.active + ln.inbox:
                        a.cancel = True
                for ln in self.solo_lanes:
                    ln.solo.cancel = True
                self.cv.notify_all()
            for ln in lanes + self.solo_lanes:
                ln.thread.join()
        wall = self.clock() - self.t0
        lat = np.array([m for r in self.results for m in r.step_ms])
        vsteps = sum(r.vertices * len(r.step_ms) for r in self.results)
        return {"results": sorted(self.results, key=lambda r: str(r.rid)),
                "failures": list(self.failures), "wall_s": wall,
                "ticks": sum(ln.ticks for ln in lanes + self.solo_lanes),
                "lanes": [ln.ticks for ln in lanes], "solo": [ln.ticks for ln in self.solo_lanes],
                "vertex_steps_per_s": vsteps / wall if wall > 0 else 0.0,
                "p50_step_ms": float(np.percentile(lat, 50)) if len(lat) else 0.0,
                "p99_step_ms": float(np.percentile(lat, 99)) if len(lat) else 0.0}

    def _admit(self, a: _Active) -> None:
        """Create the cloth of an admitted request (outside the lock) and hand
        it to its lane; creation failures become errors or a later retry."""
        try:
            dev = DeviceCloth(a.req.cloth)
            if a.saved is not None:
                x, v, t = a.saved
                dev.set_state(x, v)
                dev.time = t
                a.saved = None
        except _lib.ClothSimError as e:
            with self.cv:
                self.resident -= a.memory
                a.memory = 0
                if e.status in (2, 3) and self.resident > 0:
                    # device memory exhausted while others are resident: retry later
                    self.pending.insert(0, a)
                else:
                    self.live.discard(id(a))
                    self._fail(a.req.rid, f"cannot create the cloth: {e}")
                self.cv.notify_all()
            return
        lane = self._lane_of(a.req.cloth.np_)
        if a.req.precision == "mixed":
            try:
                dev.set_option(_OPT_PRECISION, 1)
            except _lib.ClothSimError as e:
                dev.close()
                with self.cv:
                    self.resident -= a.memory
                    a.memory = 0
                    self.live.discard(id(a))
                    self._fail(a.req.rid, f"mixed precision is not available for this cloth: {e}")
                    self.cv.notify_all()
                return
        elif self.lane_pcg[lane] != 0:
            try:
                dev.set_option(_OPT_PCG, self.lane_pcg[lane])
            except _lib.ClothSimError:
                pass  # a cloth the variant does not apply to keeps the automatic one
        with self.cv:
            mem = dev.memory()
            self.resident += max(mem, a.memory) - a.memory
            a.memory = max(mem, a.memory)
            a.dev = dev
            if a.admitted_s < 0:
                a.admitted_s = self.clock() - self.t0
            if self.solo_from is not None and a.req.cloth.np_ >= self.solo_from:
                ln = _Lane(self, sum(len(g) for g in self.lanes.values()) +
                           len(self.solo_lanes), solo=a)
                self.solo_lanes.append(ln)
                ln.thread.start()
            else:
                cl = a.req.cloth
                key = (lane, a.req.precision, cl.pcg_tol, cl.pcg_maxit)
                group = self.lanes.setdefault(key, [])
                # an instance not in a tick takes the request into its next
                # tick; if every one is stepping, another instance starts
                # (up to the lane's limit), else the first one takes it
                ln = next((x for x in group if not x.in_tick), None)
                if ln is None and len(group) < self.lane_instances[lane]:
                    # the one-workgroup solve that the tuner tries is FP64 only
                    ln = _Lane(self, sum(len(g) for g in self.lanes.values()) +
                               len(self.solo_lanes),
                               tune=self.autotune and a.req.precision == "f64")
                    ln.window = self.lane_window[lane]
                    group.append(ln)
                    ln.thread.start()
                elif ln is None:
                    ln = group[0]
                ln.inbox.append(a)
            self.cv.notify_all()


def run_plain(requests: List[Request], first_states: bool = False) -> dict:
    """The same requests one after another, each cloth stepped alone (the
    plain GPU step), for comparison.  A request whose step fails is recorded
    in "failures" and contributes no steps.  first_states: also return each
    request's positions after its first step ("first": rid -> x), read
    outside the timed steps."""
    t0 = time.perf_counter()
    results, lat, failures = [], [], []
    first = {}
    t_read = 0.0
    vsteps = 0
    for r in sorted(requests, key=lambda r: (r.arrival, str(r.rid))):
        try:
            with DeviceCloth(r.cloth) as d:
                ms = []
                for k in range(r.steps):
                    t1 = time.perf_counter()
                    d.step(1)
                    ms.append((time.perf_counter() - t1) * 1e3)
                    if first_states and k == 0:
                        t2 = time.perf_counter()
                        first[r.rid] = d.get_state()[0]
                        t_read += time.perf_counter() - t2
                x, v = d.get_state()
        except _lib.ClothSimError as e:
            failures.append(Failure(r.rid, str(e)))
            continue
        lat += ms
        vsteps += r.cloth.np_ * r.steps
        results.append((r.rid, x, v))
    wall = time.perf_counter() - t0 - t_read
    lat = np.array(lat)
    return {"results": results, "failures": failures, "wall_s": wall, "first": first,
            "vertex_steps_per_s": vsteps / wall if wall > 0 else 0.0,
            "p50_step_ms": float(np.percentile(lat, 50)) if len(lat) else 0.0,
            "p99_step_ms": float(np.percentile(lat, 99)) if len(lat) else 0.0}


def poisson_requests(count: int, rate_per_s: float, *, seed: int = 0, tri_range=(1.0e3, 2.0e5),
                     aspect_range=(1.0, 4.0), step_range=(50, 300), pcg_maxit: int = 1000) -> list:
    """The serving workload as wire requests: Poisson arrivals at `rate_per_s`;
    rectangular grids whose triangle count is log-uniform in `tri_range` and
    aspect ratio uniform in `aspect_range`, the longer side 1 m; steps uniform
    in `step_range`; each dropped from a height in [0.3, 0.8] m onto its own
    sphere or box, with the batch workload's physics (dt 0.01).

    The longer side runs along the fast vertex index (vertex (ix, iy) is
    ix * ny + iy, ny >= nx).  With the longer side along the slow index the
    reference's natural-order ILU(0) overflows on the larger of these meshes
    (489 x 151 vertices: a NaN solve; 151 x 489: finite), so this orientation
    keeps every mesh of the range servable."""
    rng = SplitMix64(seed)
    t = 0.0
    out = []
    for k in range(count):
        t += -np.log(1.0 - rng.uniform()) / rate_per_s
        tri = float(np.exp(np.log(tri_range[0]) +
                           (np.log(tri_range[1]) - np.log(tri_range[0])) * rng.uniform()))
        asp = aspect_range[0] + (aspect_range[1] - aspect_range[0]) * rng.uniform()
        # 2 (n_short - 1)(n_long - 1) triangles with n_long - 1 = aspect (n_short - 1)
        ns = max(3, int(round(np.sqrt(tri / (2.0 * asp)))) + 1)
        nl = max(3, int(round(asp * (ns - 1))) + 1)
        steps = step_range[0] + int(rng.uniform() * (step_range[1] - step_range[0] + 1))
        h = 0.3 + 0.5 * rng.uniform()
        ob = ({"kind": "sphere", "center": [0.0, 0.0, 0.0], "radius": 0.3} if rng.uniform() < 0.5
              else {"kind": "box", "center": [0.0, 0.0, 0.0], "half": [0.25, 0.25, 0.25]})
        js = int(rng.next_u64() & 0x7FFFFFFF)
        out.append({"id": k, "steps": steps, "arrival": t,
                    "scene": {"scene": "drop", "n": ns, "ny": nl, "side": 1.0, "height": h,
                              "obstacle": ob, "seed": js, "pcg_maxit": pcg_maxit,
                              "name": f"req{k}_{ns}x{nl}"}})
    return out


def poisson_stream(count: int, rate_per_s: float, **kw) -> List[Request]:
    """poisson_requests parsed into Requests."""
    return [parse_request(r, k) for k, r in enumerate(poisson_requests(count, rate_per_s, **kw))]


# ---------------------------------------------------------------------------
# wire format

PRECISIONS = ("f64", "mixed")


def encode_array(a: np.ndarray) -> dict:
    """A float64 array as {"dtype": "<f8", "shape", "data": base64 of its bytes}."""
    a = np.ascontiguousarray(a, dtype="<f8")
    return {"dtype": "<f8", "shape": list(a.shape), "data": base64.b64encode(a.tobytes()).decode()}


def decode_array(obj: dict) -> np.ndarray:
    if obj.get("dtype") != "<f8":
        raise ValueError("only <f8 arrays")
    a = np.frombuffer(base64.b64decode(obj["data"]), dtype="<f8")
    return a.reshape(obj["shape"]).copy()


def parse_request(obj: dict, index: int = 0) -> Request:
    """A wire request (see the module docstring) as a Request; ValueError
    with the reason if it cannot be served."""
    if not isinstance(obj, dict):
        raise ValueError("a request is a JSON object")
    rid = obj.get("id", index)
    if "scene" not in obj:
        raise ValueError("missing 'scene'")
    steps = obj.get("steps")
    if not isinstance(steps, int) or isinstance(steps, bool) or steps < 1:
        raise ValueError("'steps' must be an integer >= 1")
    prec = obj.get("precision", "f64")
    if prec not in PRECISIONS:
        raise ValueError(f"precision {prec!r} is not served (served: {', '.join(PRECISIONS)})")
    arrival = float(obj.get("arrival", 0.0))
    if not arrival >= 0.0:
        raise ValueError("'arrival' must be >= 0")
    returns = tuple(obj.get("return", ["x"]))
    if not set(returns) <= {"x", "v"}:
        raise ValueError("'return' takes 'x' and/or 'v'")
    cloth = scene.from_config(obj["scene"])
    if isinstance(cloth, list):
        raise ValueError("a request carries one cloth (use one request per cloth)")
    return Request(rid=rid, cloth=cloth, steps=steps, arrival=arrival, returns=returns,
                   precision=prec)


def result_record(r: Result, req: Optional[Request] = None) -> dict:
    out = {"id": r.rid, "status": "ok", "precision": req.precision if req is not None else None,
           "vertices": r.vertices,
           "triangles": req.cloth.nt if req is not None else None, "steps": len(r.step_ms),
           "arrival": req.arrival if req is not None else None,
           "queued_s": r.queued_s, "admitted_s": r.admitted_s, "finished_s": r.finished_s,
           "step_ms": r.step_ms, "pcg_iters": r.pcg_iters,
           "impulse_applied": r.impulse_applied, "n_prox": r.n_prox, "n_ccd": r.n_ccd}
    returns = req.returns if req is not None else ("x",)
    if "x" in returns:
        out["x"] = encode_array(r.xyz.reshape(-1, 3))
    if "v" in returns:
        out["v"] = encode_array(r.uvw.reshape(-1, 3))
    return out


def error_record(rid, message: str) -> dict:
    return {"id": rid, "status": "error", "error": message}


def serve_jsonl(lines: Iterable[str], out: TextIO, *, hbm_budget_bytes: int,
                realtime: bool = True) -> dict:
    """Serve the JSON-lines requests in `lines`, writing one result line per
    request to `out` as each finishes (error lines first, for requests that
    cannot be served).  Returns the run summary of Server.run."""
    reqs, by_rid = [], {}
    for k, line in enumerate(lines):
        line = line.strip()
        if not line:
            continue
        rid = k
        try:
            obj = json.loads(line)
            rid = obj.get("id", k) if isinstance(obj, dict) else k
            req = parse_request(obj, k)
        except (ValueError, KeyError, TypeError) as e:
            out.write(json.dumps(error_record(rid, str(e))) + "\n")
            out.flush()
            continue
        key = len(reqs)  # internal id: wire ids need not be unique or hashable
        by_rid[key] = req
        reqs.append(dataclasses.replace(req, rid=key))

    def emit(r: Result):  # called with the server's lock held: lines never interleave
        req = by_rid[r.rid]
        rec = result_record(dataclasses.replace(r, rid=req.rid), req)
        out.write(json.dumps(rec) + "\n")
        out.flush()

    def emit_error(f: Failure):
        out.write(json.dumps(error_record(by_rid[f.rid].rid, f.error)) + "\n")
        out.flush()

    if not reqs:
        return {"results": [], "failures": [], "wall_s": 0.0, "ticks": 0,
                "vertex_steps_per_s": 0.0, "p50_step_ms": 0.0, "p99_step_ms": 0.0}
    return Server(hbm_budget_bytes, on_result=emit, on_error=emit_error).run(reqs,
                                                                           realtime=realtime)


def main(argv=None) -> int:
    import argparse
    ap = argparse.ArgumentParser(description="Serve cloth simulations on one GPU (JSON lines).")
    ap.add_argument("--requests", default="-", help="request lines (default: stdin)")
    ap.add_argument("--results", default="-", help="result lines (default: stdout)")
    ap.add_argument("--budget-gb", type=float, default=64.0, help="HBM budget for resident cloths")
    ap.add_argument("--no-realtime", action="store_true",
                    help="admit every request at once (ignore arrival times)")
    ap.add_argument("--setup-cache", default=None, help="directory of cached per-mesh setups")
    ap.add_argument("--make-poisson", type=int, default=0, metavar="COUNT",
                    help="write COUNT requests of the Poisson serving workload and exit")
    ap.add_argument("--rate", type=float, default=4.0, help="--make-poisson arrival rate, 1/s")
    ap.add_argument("--seed", type=int, default=0, help="--make-poisson seed")
    args = ap.parse_args(argv)
    if args.make_poisson > 0:
        fout = sys.stdout if args.results == "-" else open(args.results, "w")
        for r in poisson_requests(args.make_poisson, args.rate, seed=args.seed):
            fout.write(json.dumps(r) + "\n")
        if fout is not sys.stdout:
            fout.close()
        return 0
    if args.setup_cache:
        from . import _lib
        _lib.set_setup_cache(args.setup_cache)
    fin = sys.stdin if args.requests == "-" else open(args.requests)
    fout = sys.stdout if args.results == "-" else open(args.results, "w")
    try:
        summary = serve_jsonl(fin, fout, hbm_budget_bytes=int(args.budget_gb * 2**30),
                              realtime=not args.no_realtime)
    finally:
        if fin is not sys.stdin:
            fin.close()
        if fout is not sys.stdout:
            fout.close()
    print(json.dumps({k: v for k, v in summary.items() if k not in ("results", "failures")}),
          file=sys.stderr)
    return 0


if __name__ == "__main__":
    sys.exit(main())
