"""Continuous-batching server for design sweeps of many independent solves.

Requests (grid size, SDF geometry, source, probes, step count) arrive over
time. The server keeps each admitted solve's fields and tables resident in HBM
(one ``FDTDSolver`` per request, built through the public API), admits waiting
requests whenever an active-slot and the HBM budget allow, and advances all
active solves together with the batched step kernel (one launch per step over
every solve's strips, captured in a hipGraph per chunk). While a chunk runs on
the GPU the host builds the next arrivals' scenes, so set-up overlaps device
work. A finished solve's probe traces are copied out and its memory released.

The batched kernel executes, for each solve, exactly the per-wave arithmetic of
the single-solve kernel, so every result is bit-identical alone and in the mix
(tests/test_gpu_serving.py checks that).

Reported: solves/s and latency (arrival -> result) p50/p99, next to running
the same requests one at a time through plain ``FDTDSolver(backend="mi355x")``.
"""

from __future__ import annotations

import time
from dataclasses import dataclass, field

import numpy as np

from . import _native
from .boundaries import PML
from .geometry import Box, Cylinder, Difference, SDFPrimitive, Union
from .grid import UniformGrid
from .solver import FDTDSolver
from .sources import GaussianPulse
from .tuning import pick_tiling

BYTES_PER_CELL_RESIDENT = 2 * 16 + 3   # ping-pong fields + flags + mask + material ids


@dataclass
class SolveRequest:
    rid: int
    shape: tuple[int, int, int]
    resolution: float
    pml_depth: int
    geometry: SDFPrimitive | np.ndarray | None
    source: GaussianPulse
    probes: list
    steps: int
    arrival: float = 0.0          # seconds after the stream starts

    @property
    def cells(self) -> int:
        return int(np.prod(self.shape))

    @property
    def footprint(self) -> int:
        return self.cells * BYTES_PER_CELL_RESIDENT + self.steps * (len(self.probes) * 4 + 8)


@dataclass
class SolveResult:
    rid: int
    traces: dict
    arrival: float
    admitted: float
    finished: float

    @property
    def latency(self) -> float:
        return self.finished - self.arrival


def build_solver(req: SolveRequest, device: int = 0, tiling=None) -> FDTDSolver:
    """The request as a plain single-solve FDTDSolver (also the one-at-a-time path)."""
    s = FDTDSolver(grid=UniformGrid(req.shape, req.resolution), c=343.0, rho=1.204, backend="mi355x",
                   device=device, tiling=tiling)
    if req.geometry is not None:
        s.set_geometry(req.geometry)
    if req.pml_depth:
        s.add_boundary(PML(depth=req.pml_depth))
    s.add_source(GaussianPulse(position=tuple(req.source.position), frequency=req.source.frequency,
                               bandwidth=req.source.bandwidth, amplitude=req.source.amplitude))
    for q, p in enumerate(req.probes):
        s.add_probe(f"probe{q}", tuple(int(v) for v in p))
    return s


def tune_shapes(requests, rows: int = 2, planes=(1, 2, 4, 8), steps: int = 20, device: int = 0) -> dict:
    """Autotune the launch shape of every distinct grid shape in `requests`
    before serving them: for each shape, an air box of that shape with PML
    is timed with each candidate (rows, planes) strip (``autotune.autotune``,
    device time over `steps` steps) and the fastest is stored in the tiling
    cache, where ``pick_tiling`` (used by the server and by single solves)
    finds it. They are shapes of single steps, which batches in passes take for the
    steps that passes leave. `rows` is the batched sweep's row count, so only the
    strip length along i is chosen per shape. Returns {shape: (tiling, ms per step)}.

    Measured on the 64-request sweep (62 shapes, tuned in 0.2 s), one step per
    launch: the tuned
    single-solve strips (planes 2 for 30 shapes, 4 for 26, 8 for 5, 1 for 1)
    served the batch at 11.6 solves/s against 13.2 with the heuristic's
    shorter strips, which keep more waves in flight when many solves share
    the GPU; the server therefore keeps the heuristic unless a cache entry
    exists."""
    from .autotune import autotune
    out = {}
    for shape in sorted({tuple(r.shape) for r in requests}):
        s = FDTDSolver(grid=UniformGrid(shape, 1e-3), c=343.0, rho=1.204, backend="mi355x", device=device)
        s.add_boundary(PML(depth=8))
        s.add_probe("probe", tuple(n // 2 for n in shape))
        cands = [(rows, p, 1) for p in planes if p <= shape[0]]
        best, table = autotune(s, candidates=cands, steps=steps, store=True)
        out[shape] = (best, min(t[3] for t in table))
        del s
    return out


def sweep_requests(n: int = 64, rate: float = 40.0, seed: int = 1234, steps=(2000, 8000),
                   dims=tuple(range(64, 193, 16))) -> list[SolveRequest]:
    """Seeded Poisson stream of enclosure solves (the design-sweep workload).

    Each axis is drawn from 64..192 in steps of 16, 1 mm cells, PML 8-12; a box
    enclosure with 6-12-cell walls and one cylindrical port (radius 4-10, length
    10-40) through its -x wall; a Gaussian pulse of 200 Hz-4 kHz at a seeded
    interior point; 1-4 probes inside; step count uniform in [2000, 8000].
    Inter-arrival times are exponential with mean 1/rate seconds.
    """
    rng = np.random.default_rng(seed)
    t = 0.0
    out = []
    dx = 1e-3
    for rid in range(n):
        t += float(rng.exponential(1.0 / rate))
        shape = tuple(int(rng.choice(dims)) for _ in range(3))
        pml = int(rng.integers(8, 13))
        wall = int(rng.integers(6, 13))
        lo = np.array([pml + 4] * 3)
        hi = np.array(shape) - pml - 4
        wall = min(wall, int((hi - lo).min()) // 2 - 3)   # keep a cavity on small test grids
        outer = Box(min_corner=tuple(lo * dx), max_corner=tuple(hi * dx))
        inner = Box(min_corner=tuple((lo + wall) * dx), max_corner=tuple((hi - wall) * dx))
        r = int(rng.integers(4, 11))
        plen = int(rng.integers(10, 41))
        cy, cz = (lo[1] + hi[1]) / 2 * dx, (lo[2] + hi[2]) / 2 * dx
        x0 = lo[0] * dx
        port = Cylinder(p1=(x0 - 0.5 * plen * dx, cy, cz), p2=(x0 + 0.5 * plen * dx + wall * dx, cy, cz),
                        radius=r * dx)
        domain = Box(min_corner=(-1.0, -1.0, -1.0), max_corner=(2.0, 2.0, 2.0))
        geom = Union(Difference(domain, Difference(outer, inner)), port)
        cav_lo, cav_hi = lo + wall + 2, hi - wall - 2
        src = tuple(int(v) for v in rng.integers(cav_lo, cav_hi))
        f = float(rng.uniform(200.0, 4000.0))
        probes = [tuple(int(v) for v in rng.integers(cav_lo, cav_hi)) for _ in range(int(rng.integers(1, 5)))]
        steps_n = int(rng.integers(steps[0], steps[1] + 1))
        out.append(SolveRequest(rid, shape, dx, pml, geom, GaussianPulse(position=src, frequency=f), probes,
                                steps_n, t))
    return out


@dataclass
class _Slot:
    req: SolveRequest
    solver: FDTDSolver | None
    admitted: float
    done: int = 0
    host_trace: object = None


@dataclass
class ServeStats:
    results: list = field(default_factory=list)
    wall: float = 0.0
    chunks: int = 0
    max_active: int = 0

    @property
    def solves_per_s(self) -> float:
        return len(self.results) / self.wall if self.wall > 0 else 0.0

    def latency_pct(self, q: float) -> float:
        return float(np.percentile([r.latency for r in self.results], q))

    def summary(self) -> dict:
        return {"solves": len(self.results), "wall_s": round(self.wall, 3),
                "solves_per_s": round(self.solves_per_s, 3),
                "p50_s": round(self.latency_pct(50), 3), "p99_s": round(self.latency_pct(99), 3),
                "chunks": self.chunks, "max_active": self.max_active}


class SweepServer:
    """Continuous batching of uniform-grid solves on one GPU.

    Admission: a waiting request is admitted while an active slot, the HBM
    budget and the active-cell cap allow. The default cap (``max_cells``, 6M
    cells: about 200 MB of fields) keeps the active solves inside the 256 MB
    Infinity Cache, where the batched sweep runs faster than from HBM, and
    still fills the GPU; admitting more only stretches every solve's latency
    (the device is shared). None admits without a cell cap. ``policy`` orders
    the waiting requests: "sjf" (least work, cells x steps, first: lowest mean
    latency, but the largest requests wait for every smaller one),
    "aged" (least work first with an age credit: by arrival time plus the
    request's work at the nominal batched rate, so a request that has waited
    as long as a smaller one needs outranks it) or "fifo" (arrival order).
    ``rows``: rows per wave strip of the
    batched sweep; 2 (many short strips) measured 9% faster than 4 on the
    64-request sweep, whose solves all fit the cache. ``use_graph`` (the
    default): each chunk (its step launches and the launch that moves the
    solves' counters) is replayed as one captured hipGraph; the graph is
    captured once per chunk length and wave capacity and stays valid while
    the table of active solves changes between chunks. Enqueueing the kernels
    one by one instead (False) measured the same on the 64-request sweep
    (13.95-14.00 against 13.88-13.99 solves/s, one step per launch)."""

    CACHE_RESIDENT_CELLS = 6 << 20
    # batched rate (cell-updates per second) that converts a request's work
    # into seconds for the "aged" order: about that of a cache-resident batch
    # stepped one by one (in passes the 64-request sweep runs at 265e9; the
    # smaller rate gives small requests the more credit)
    NOMINAL_RATE = 120e9

    def __init__(self, device: int = 0, rows: int = 2, chunk: int = 100, max_active: int = 64,
                 hbm_budget: int | None = None, use_graph: bool = True,
                 max_cells: int | None = CACHE_RESIDENT_CELLS, policy: str = "aged"):
        import torch
        if policy not in ("fifo", "sjf", "aged"):
            raise ValueError(f"policy must be 'fifo', 'sjf' or 'aged', not {policy!r}")
        self.device = device
        self.rows = rows
        self.chunk = chunk
        self.max_active = max_active
        self.max_cells = max_cells
        self.policy = policy
        self.use_graph = use_graph
        if hbm_budget is None:
            free, _total = torch.cuda.mem_get_info(device)
            hbm_budget = int(free * 0.6)
        self.hbm_budget = hbm_budget
        self._stream = torch.cuda.current_stream(torch.device(f"cuda:{device}"))
        h = _native._vp()
        _native.call("fdtd_batch_create", device, self._stream.cuda_stream, rows, _native.C.byref(h))
        self._batch = h.value

    def close(self) -> None:
        if self._batch:
            _native.load().fdtd_batch_destroy(self._batch)
            self._batch = None

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass

    def _set_batch(self, slots: list[_Slot]) -> None:
        ctxs = (_native._vp * max(len(slots), 1))(*[s.solver._ctx for s in slots])
        limits = np.array([s.req.steps for s in slots] or [0], dtype=np.int64)
        _native.call("fdtd_batch_set", self._batch, ctxs, limits.ctypes.data, len(slots))

    def serve(self, requests: list[SolveRequest], realtime: bool = True) -> ServeStats:
        """Serve a stream; arrival times are honoured against the wall clock
        when ``realtime`` (otherwise every request is available at t=0).

        The loop never waits for the chunk it has just launched: up to two
        chunks are queued on the stream; table updates, trace copies of
        finished solves (into pinned memory) and the next chunk are enqueued
        behind the running one, and new scenes are built on a second stream
        meanwhile. A solve that finishes is dropped from the table for the next
        chunk and freed once its trace copy has completed."""
        import collections

        import torch
        pending = sorted(requests, key=lambda r: r.arrival)
        stats = ServeStats()
        active: list[_Slot] = []
        retiring: collections.deque = collections.deque()   # (event, [slots])
        inflight: collections.deque = collections.deque()   # chunk events
        used = 0
        t0 = time.perf_counter()
        now = lambda: time.perf_counter() - t0  # noqa: E731
        dev = torch.device(f"cuda:{self.device}")
        build_stream = torch.cuda.Stream(dev)
        built: dict[int, tuple] = {}

        def build(r: SolveRequest):
            with torch.cuda.stream(build_stream):
                s = build_solver(r, self.device, tiling=(self.rows, pick_tiling(r.shape)[1], 1))
                s._prepare(r.steps)
            ev = torch.cuda.Event()
            ev.record(build_stream)
            return s, ev

        def waiting(limit_time: float) -> list[SolveRequest]:
            """Requests arrived by limit_time, in admission order."""
            arrived = [r for r in pending if not realtime or r.arrival <= limit_time]
            if self.policy == "sjf":
                arrived.sort(key=lambda r: (r.cells * r.steps, r.arrival))
            elif self.policy == "aged":
                arrived.sort(key=lambda r: (r.arrival + r.cells * r.steps / self.NOMINAL_RATE, r.rid))
            return arrived

        def prebuild(limit_time: float) -> None:
            for r in waiting(limit_time):
                if len(built) >= 4:
                    break
                if r.rid not in built:
                    built[r.rid] = build(r)

        def harvest(block: bool) -> None:
            while retiring and (block or retiring[0][0].query()):
                ev, slots = retiring.popleft()
                ev.synchronize()
                t = now()
                for sl in slots:
                    sv = sl.solver
                    sv._advance_host(sl.req.steps)
                    host = sl.host_trace
                    traces = {name: np.ascontiguousarray(host[:, q].numpy(), dtype=np.float32)
                              for q, name in enumerate(sv._probe_order)}
                    stats.results.append(SolveResult(sl.req.rid, traces, sl.req.arrival, sl.admitted, t))
                    sl.solver = None
                    sl.host_trace = None
                block = False

        active_cells = 0
        while pending or active or retiring:
            tnow = now()
            changed = False
            for r in waiting(tnow):
                if len(active) >= self.max_active or (active and used + r.footprint > self.hbm_budget):
                    break
                if active and self.max_cells is not None and active_cells + r.cells > self.max_cells:
                    break
                pending.remove(r)
                s, ev = built.pop(r.rid, None) or build(r)
                self._stream.wait_event(ev)
                active.append(_Slot(r, s, now()))
                used += r.footprint
                active_cells += r.cells
                changed = True
            if changed:
                self._set_batch(active)
            if active:
                stats.max_active = max(stats.max_active, len(active))
                _native.call("fdtd_batch_step_n", self._batch, self.chunk, 1 if self.use_graph else 0)
                stats.chunks += 1
                finished = []
                for sl in active:
                    sl.done += min(self.chunk, sl.req.steps - sl.done)
                    if sl.done >= sl.req.steps:
                        finished.append(sl)
                if finished:
                    for sl in finished:
                        tr = sl.solver._trace[:sl.req.steps]
                        sl.host_trace = torch.empty(tr.shape, dtype=tr.dtype, pin_memory=True)
                        sl.host_trace.copy_(tr, non_blocking=True)
                        active.remove(sl)
                        used -= sl.req.footprint
                        active_cells -= sl.req.cells
                    ev = torch.cuda.Event()
                    ev.record(self._stream)
                    retiring.append((ev, finished))
                    self._set_batch(active)
                cev = torch.cuda.Event()
                cev.record(self._stream)
                inflight.append(cev)
                prebuild(now() + 0.05)
                while len(inflight) > 2:
                    inflight.popleft().synchronize()
                harvest(False)
            else:
                harvest(bool(retiring) and not pending)
                if pending and realtime and not retiring:
                    prebuild(pending[0].arrival)
                    wait = pending[0].arrival - now()
                    if wait > 0:
                        time.sleep(min(wait, 0.01))
        torch.cuda.synchronize(self.device)
        stats.wall = now()
        built.clear()
        return stats


def serve_one_at_a_time(requests: list[SolveRequest], device: int = 0, realtime: bool = True,
                        graph_chunk: int = 0) -> ServeStats:
    """Baseline: each request runs alone through plain FDTDSolver, in arrival order."""
    import torch
    stats = ServeStats()
    t0 = time.perf_counter()
    now = lambda: time.perf_counter() - t0  # noqa: E731
    for r in sorted(requests, key=lambda x: x.arrival):
        if realtime and r.arrival > now():
            time.sleep(r.arrival - now())
        start = now()
        s = build_solver(r, device)
        s.step_n(r.steps, graph_chunk=graph_chunk)
        traces = s.get_probe_data()
        torch.cuda.synchronize(device)
        stats.results.append(SolveResult(r.rid, traces, r.arrival, start, now()))
        stats.max_active = 1
        del s
    stats.wall = now()
    return stats
