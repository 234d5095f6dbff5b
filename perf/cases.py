"""Performance cases of the contact-tracing path: what a program does with
this package, through its public entry points, over the sizes it is used at.

kind     one pass
stage    one tick of the stage calls from positions in host memory
         (Workbench.tick), its meetings back on the host, sorted; with
         `record`, its contact pairs too (Workbench.contacts)
run      `ticks` ticks of a device-resident trace (Workbench.run_ticks), plain
         launches or replayed graphs; the last tick's meetings and the
         running totals
batch    the same for many cities at once (Batch.run_ticks)
serve    one served tick of location updates, then tracing queries answered
         on it (Server.tick / submit / drain / result)
kv       `ticks` ticks with the sorted key-value output on, then a flush with
         all of its parts copied out (Workbench.kv_flush)
project  lon/lat points of a trace to planar metres (project_device)

A trace goes forward for `ticks` ticks and back again, so that a context can
run on for any number of passes with every object moving one step per tick.
Every context has run one such loop before its first pass: runs of contact
are under way and meetings end at every tick.
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

from glint_pipeline_amd import autotune, gen, runtime

GAP = 50.0   # street grid of the walkers, metres


# ------------------------------------------------------------------- cases
def listed() -> list[dict]:
    return [
        # the smallest calls: a few thousand objects ticked from host memory, contact pairs
        # read back every tick (an interactive check of a scene)
        {"name": "stage_3k_contacts", "kind": "stage", "n": 3000, "density": 0.012, "hot": False, "cap": 16,
         "precision": "fp64", "record": True},
        # a quarter of a million objects in hotspots, fed from host memory one tick per call, as
        # a program that receives every tick's positions runs it
        {"name": "stage_250k_hotspots", "kind": "stage", "n": 250_007, "density": 0.0111, "hot": True, "cap": 200,
         "precision": "fp32guard", "record": False},
        # the plain CPU workload: 100k walkers in a 10 km box, FP64, plain launches
        {"name": "run_100k_uniform", "kind": "run", "n": 100_000, "density": 0.001, "hot": False, "cap": 200,
         "precision": "fp64", "graph": False, "ticks": 8, "schema": "dynamic", "geo": False, "reach": 2.0, "min": 5},
        # the plain GPU workload: 1M walkers in a 30 km box, FP64, plain launches
        {"name": "run_1m_uniform", "kind": "run", "n": 1_000_000, "density": 1.0 / 900, "hot": False, "cap": 200,
         "precision": "fp64", "graph": False, "ticks": 8, "schema": "dynamic", "geo": False, "reach": 2.0, "min": 5},
        # the headline workload: 10M objects, 80% of them in 64 hotspots of a 30 km box, FP32
        # guard band, replayed graphs of 8 ticks
        {"name": "run_10m_hotspots", "kind": "run", "n": 10_000_000, "density": 1.0 / 90, "hot": True, "cap": 320,
         "precision": "fp32guard", "graph": True, "ticks": 8, "schema": "dynamic", "geo": False, "reach": 2.0,
         "min": 5},
        # a lon/lat trace on the reference's geography predicates
        {"name": "run_300k_lonlat", "kind": "run", "n": 300_001, "density": 1.0 / 900, "hot": False, "cap": 200,
         "precision": "fp64", "graph": False, "ticks": 8, "schema": "dynamic", "geo": True, "reach": 2.0, "min": 5},
        # the tree rebuilt every tick (the dynamic schema off), 2M objects in hotspots
        {"name": "run_2m_grid_rebuild", "kind": "run", "n": 2_000_000, "density": 1.0 / 90, "hot": True, "cap": 200,
         "precision": "fp32guard", "graph": True, "ticks": 8, "schema": "grid", "geo": False, "reach": 2.0, "min": 5},
        # 32 cities of 50k to 2M objects in one batch, replayed graphs of 8 ticks
        {"name": "batch_32_cities", "kind": "batch", "count": 32, "smallest": 50_000, "largest": 2_000_000,
         "graph": True, "ticks": 8},
        # 20M resident objects of which a tenth moves per tick, 50 queries a tick
        {"name": "serve_20m", "kind": "serve", "n": 20_000_000, "move": 0.1, "queries": 50},
        # meetings organised as sorted key-value files every 8 ticks
        {"name": "kv_400k_hotspots", "kind": "kv", "n": 400_000, "density": 1.0 / 90, "cap": 200, "ticks": 8,
         "graph": False},
        # 10 ticks of a million lon/lat points brought to metres
        {"name": "project_10m_points", "kind": "project", "n": 10_000_000},
    ]


def _log(rng, lo: float, hi: float) -> int:
    return int(math.floor(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng) -> dict:
    kind = rng.choice(["stage", "stage", "run", "run", "run", "batch", "serve", "kv", "project"])
    if kind == "stage":
        record = rng.random() < 0.4
        return {"kind": kind, "n": _log(rng, 1000, 30_000 if record else 500_000), "density": 10 ** rng.uniform(-3, -1.9),
                "hot": rng.random() < 0.5, "cap": rng.choice([16, 32, 50, 128, 200]),
                "precision": rng.choice(["fp64", "fp32guard"]), "record": record}
    if kind == "run":
        form = rng.choice(["dynamic", "dynamic", "dynamic", "grid", "geo"])
        hot = rng.random() < 0.5
        top = {"dynamic": 5_000_000 if hot else 10_000_000, "grid": 3_000_000, "geo": 1_000_000}[form]
        return {"kind": kind, "n": _log(rng, 20_000, top), "density": 10 ** rng.uniform(-3.05, -1.95 if hot else -2.5),
                "hot": hot and form != "geo", "cap": rng.choice([200, 320, 512] if form == "grid" else [50, 128, 200, 320, 512]),
                "precision": "fp64" if form == "geo" else rng.choice(["fp64", "fp32guard"]),
                "graph": rng.random() < 0.5, "ticks": rng.choice([4, 7, 8, 12]),
                "schema": "grid" if form == "grid" else "dynamic", "geo": form == "geo",
                "reach": rng.choice([1.5, 2.0] if form == "grid" else [1.5, 2.0, 3.0]), "min": rng.choice([2, 3, 5])}
    if kind == "batch":
        return {"kind": kind, "count": rng.randrange(3, 33), "smallest": _log(rng, 5_000, 50_000),
                "largest": _log(rng, 60_000, 1_500_000), "graph": rng.random() < 0.7, "ticks": rng.choice([4, 8])}
    if kind == "serve":
        return {"kind": kind, "n": _log(rng, 100_000, 20_000_000), "move": rng.choice([0.02, 0.1, 0.3, 1.0]),
                "queries": rng.randrange(1, 51)}
    if kind == "kv":
        return {"kind": kind, "n": _log(rng, 10_000, 800_000), "density": 10 ** rng.uniform(-3, -1.95),
                "cap": rng.choice([50, 200, 320]), "ticks": rng.choice([4, 8, 12]), "graph": rng.random() < 0.5}
    return {"kind": kind, "n": _log(rng, 1000, 60_000_000)}


# ------------------------------------------------------------------ inputs
def _workload(case: dict, seed: int) -> gen.Workload:
    """Walkers at `density` objects per square metre in a box of whole blocks;
    in hotspots, 80% of them in Gaussians (sigma 200 m, Zipf 1.1), one to
    every 156250 objects as in the 10M workload."""
    n = case["n"]
    side = max(2 * GAP, math.ceil(math.sqrt(n / case["density"]) / GAP) * GAP)
    w = gen.uniform_city(n, 1, side, seed=seed, grid_capacity=case["cap"], reach_distance=case.get("reach", 2.0),
                         min_meet_time=case.get("min", 5))
    if case["hot"]:
        w.num_hotspots = max(1, round(n / 156_250))
        w.hotspot_fraction = 0.8
        w.hotspot_sigma = min(200.0, side / 8)
    return w


def _pairs(case: dict) -> float:
    """Contact pairs per tick a program would size its buffers for: 70 per
    object in hotspots (what the headline workload reaches), a share of an
    object's neighbourhood elsewhere."""
    n, r = case["n"], case.get("reach", 2.0)
    if case.get("hot"):
        return 70.0 * n * (r / 2.0) ** 2
    return max(0.2, 60.0 * case["density"] * r * r) * n


class _Trace:
    """2*ticks snapshots in device memory: forward ticks 0..T-1, then ticks
    T..1 in reverse; block 0 and block 1 follow each other in turn."""

    def __init__(self, w: gen.Workload, ticks: int, degrees=None):
        self.size, self.ticks = 16 * w.num_objects, ticks
        self.buf = runtime.DeviceBuffer(self.size * 2 * ticks)
        g = gen.Generator(w)
        if degrees is None:
            self.buf.upload(g.positions(), 0)
            runtime.DeviceWalkers(g).walk(ticks, self.buf, self.size)
        else:
            for t in range(ticks + 1):
                xy = (g.positions() if t == 0 else g.step()).reshape(-1, 2)
                self.buf.upload(degrees(xy), self.size * t)
        for k in range(1, ticks):
            runtime._check(runtime.lib().glint_device_copy(
                self.buf.address(self.size * (ticks + k)), self.buf.address(self.size * (ticks - k)), self.size),
                "glint_device_copy")

    def block(self, half: int) -> int:
        return self.buf.address(self.size * self.ticks * half)


class _LonLat:
    """Degrees of a walk in metres near (lon0, lat0), and its box with a metre of margin."""

    def __init__(self, lon0: float = -87.63, lat0: float = 41.88):
        p = runtime.projection_for_box(lon0, lat0)
        self.lon0, self.lat0, self.fx, self.fy = lon0, lat0, p.deg_per_m_lon, p.deg_per_m_lat

    def degrees(self, xy: np.ndarray) -> np.ndarray:
        return np.stack([self.lon0 + xy[:, 0] * self.fx, self.lat0 + xy[:, 1] * self.fy], axis=1)

    def box(self, side: float) -> tuple:
        return (self.lon0 - self.fx, self.lat0 - self.fy, self.lon0 + (side + 1) * self.fx,
                self.lat0 + (side + 1) * self.fy)


class _State:
    """What a program holds between passes; device buffers go with it."""

    def __init__(self, case: dict):
        self.case, self.kind, self.tick, self.half = case, case["kind"], 0, 0


# ----------------------------------------------------------------- outputs
TOTALS = ("ticks", "contacts", "contacts_border", "distinct_pairs", "meetings", "units", "border_objects",
          "max_contacts_tick", "max_meetings_tick", "max_leaf_count", "tests")


def _totals(wb: runtime.Workbench) -> list[int]:
    t = wb.totals()
    return [int(t[k]) for k in TOTALS]


class _Rows:
    """Rows of results in a buffer of a fixed number of rows, as a program
    that hands them on keeps them; the rows past the last are zero."""

    def __init__(self, rows: int, columns: int, dtype, device: bool = False):
        self.buf = torch.zeros((rows, columns), dtype=dtype, device="cuda") if device else \
            np.zeros((rows, columns), dtype=dtype)
        self.used = 0

    def cut(self, k: int):
        """The first k rows, about to be written."""
        if k > len(self.buf):
            raise ValueError(f"{k} rows, room for {len(self.buf)}")
        if k < self.used:
            self.buf[k:self.used] = 0
        self.used = k
        return self.buf[:k]

    def put(self, rows):
        self.cut(len(rows))[:] = rows
        return self.buf


def _last_meetings(s: _State, contexts: list) -> torch.Tensor:
    """The last tick's meetings of every context, ordered by context and pair,
    on the device: (context, pid_a, pid_b, start, end) rows."""
    parts = []
    for i, wb in enumerate(contexts):
        ptr, cnt = ctypes.c_void_p(), ctypes.c_uint64()
        runtime._check(runtime.lib().glint_device_meetings(wb.h, ctypes.byref(ptr), ctypes.byref(cnt)),
                       "glint_device_meetings", wb.h)
        m = torch.empty((cnt.value, 4), dtype=torch.int32, device="cuda")
        if cnt.value:
            runtime._check(runtime.lib().glint_device_copy(m.data_ptr(), ptr, 16 * cnt.value), "glint_device_copy")
        parts.append(torch.nn.functional.pad(m, (1, 0), value=i))
    rows = torch.cat(parts)
    bits = 31 if len(contexts) == 1 else 21   # objects per context
    key = (rows[:, 0].long() << (2 * bits)) | (rows[:, 1].long() << bits) | rows[:, 2].long()
    return s.meetings.put(rows[torch.argsort(key)])


# ----------------------------------------------------------------- prepare
def _run_state(case: dict, seed: int, **extra) -> _State:
    s = _State(case)
    w = _workload(case, seed)
    pairs = _pairs(case)
    params = {"precision": case.get("precision", "fp32guard"), "grid_capacity": case["cap"], "join_tile": 256,
              "table_threads": 512, "load_factor": 3.0 if case["hot"] else 0.75, "schema": case.get("schema", "dynamic")}
    cfg = autotune.config_for(w, params, pairs, graph_ticks=case["ticks"] if case["graph"] else 0, **extra)
    degrees = None
    if case.get("geo"):
        ll = _LonLat()
        degrees = ll.degrees
        cfg.low_x, cfg.low_y, cfg.high_x, cfg.high_y = ll.box(w.side)
        cfg.geography = 1
    s.trace = _Trace(w, case["ticks"], degrees)
    s.wb = runtime.Workbench(cfg)
    s.meetings = _Rows(3 * w.num_objects + 1024, 5, torch.int32, device=True)
    for _ in range(2):
        _advance(s)
    return s


def _advance(s: _State) -> None:
    s.wb.run_ticks(s.trace.block(s.half), s.tick, s.case["ticks"], latencies=False)
    s.tick += s.case["ticks"]
    s.half ^= 1


def _stage_state(case: dict, seed: int) -> _State:
    s = _State(case)
    w = _workload(case, seed)
    w.min_meet_time = 3
    g = gen.Generator(w)
    forward = [g.positions().copy()] + [g.step().copy() for _ in range(6)]
    s.points = forward + forward[-2:0:-1]
    pairs = _pairs(case)
    prec = runtime.PRECISION_FP64 if case["precision"] == "fp64" else runtime.PRECISION_FP32_GUARD
    s.wb = runtime.Workbench(runtime.make_config(
        w.num_objects, w.box(), grid_capacity=case["cap"], min_meet_time=w.min_meet_time, precision=prec,
        record_contacts=case["record"], unit_capacity=8 * w.num_objects + 4096,
        contact_capacity=int(1.5 * pairs) + (1 << 20)))
    s.meetings = _Rows(2 * w.num_objects + 1024, 4, np.int32)
    if case["record"]:
        s.contacts = _Rows(int(pairs) + 1024, 1, np.int64)
    for _ in range(len(s.points)):
        _stage_tick(s)
    return s


def _stage_tick(s: _State) -> np.ndarray:
    m = s.wb.tick(s.points[s.tick % len(s.points)], s.tick)
    s.tick += 1
    return m


def _batch_state(case: dict, seed: int) -> _State:
    s = _State(case)
    ws = gen.batched_cities(case["count"], seed=4, n_min=case["smallest"], n_max=case["largest"])
    cfgs, s.traces = [], []
    for i, w in enumerate(ws):
        w.seed = 1000 * seed + i
        params = autotune.params_for(autotune.size_class(w.num_objects))
        cfgs.append(autotune.config_for(w, params, autotune.pairs_estimate("batched", w.num_objects),
                                        graph_ticks=case["ticks"]))
        s.traces.append(_Trace(w, case["ticks"]))
    s.batch = runtime.Batch(cfgs, graph_ticks=case["ticks"] if case["graph"] else 0)
    s.meetings = _Rows(sum(w.num_objects for w in ws) // 2 + 4096, 5, torch.int32, device=True)
    for _ in range(2):
        _batch_advance(s)
    return s


def _batch_advance(s: _State) -> None:
    s.batch.run_ticks([t.block(s.half) for t in s.traces], s.tick, s.case["ticks"], latencies=False)
    s.tick += s.case["ticks"]
    s.half ^= 1


STEPS = 4            # update lists held by a serving state, each used forward and back
SERVE_WARM = 72      # ticks of history: one block of the meeting index and a tail


def _serve_state(case: dict, seed: int) -> _State:
    s = _State(case)
    n = case["n"]
    w = gen.uniform_city(n, 1, gen.city_side(n), seed=seed, grid_capacity=200)
    w.move_fraction = case["move"]
    w.min_meet_time = 2
    params = dict(autotune.params_for(autotune.size_class(n)), precision="fp32guard")
    cfg = autotune.config_for(w, params, autotune.pairs_estimate("batched", n), graph_ticks=0,
                              meeting_log_capacity=1 << max(20, math.ceil(math.log2(n)) + 1))
    g = gen.Generator(w)
    full = torch.from_numpy(g.positions().copy()).cuda()
    points = full.clone().view(-1, 2)
    walkers = runtime.DeviceWalkers(g)
    pids, xy, count = runtime.DeviceBuffer(4 * n + 16), runtime.DeviceBuffer(16 * n), runtime.DeviceBuffer(4)
    forward, back = [], []
    for _ in range(STEPS):
        k = walkers.step_updates(pids, xy, count)
        p = torch.empty((k + 3) // 4 * 4, dtype=torch.int32, device="cuda")
        to = torch.empty((k, 2), dtype=torch.float64, device="cuda")
        runtime._check(runtime.lib().glint_device_copy(p.data_ptr(), pids.address(), 4 * p.numel()), "glint_device_copy")
        runtime._check(runtime.lib().glint_device_copy(to.data_ptr(), xy.address(), 16 * k), "glint_device_copy")
        p = p[:k].clone()
        was = points[p.long()]
        points[p.long()] = to
        forward.append((p, to))
        back.insert(0, (p, was))
    s.updates = forward + back
    rng = np.random.default_rng(seed)
    s.queries = []
    for _ in range(2 * case["queries"]):
        seeds = rng.choice(n, size=int(rng.integers(1, min(10_001, n))), replace=False).astype(np.uint32)
        s.queries.append((seeds, int(rng.integers(8, SERVE_WARM)), 2 if rng.random() < 0.2 else 1))
    s.hop1, s.hop2 = (_Rows(2 * min(10_001, n) * case["queries"] + 4096, 4, np.int32) for _ in range(2))
    torch.cuda.synchronize()
    s.wb = runtime.Workbench(cfg)
    s.server = runtime.Server(s.wb, arena_bytes=2 << 30, max_running=16)
    s.server.tick(0, d_full_xy=full.data_ptr())
    s.wb.synchronize()
    s.tick = 1
    for _ in range(SERVE_WARM):
        _serve_tick(s)
        s.server.poll()
    s.wb.synchronize()
    return s


def _serve_tick(s: _State) -> None:
    p, xy = s.updates[(s.tick - 1) % len(s.updates)]
    s.server.tick(s.tick, d_pids=p.data_ptr(), d_xy=xy.data_ptr(), k=p.numel())
    s.tick += 1


# a flush's parts: keys and boxes of the files and of the oversize buffer and
# the packed keys vary in length, the others are as many as objects or files
KV_VARIABLE = (runtime.KV_KEYS, runtime.KV_BOXES, runtime.KV_OVERSIZE_KEYS, runtime.KV_OVERSIZE_BOXES,
               runtime.KV_PACKED)


def _kv_parts(case: dict) -> dict:
    files = 100
    return {runtime.KV_KEYS: (0, 2, np.int64), runtime.KV_BOXES: (0, 4, np.float32),
            runtime.KV_OVERSIZE_KEYS: (0, 2, np.int64), runtime.KV_OVERSIZE_BOXES: (0, 4, np.float32),
            runtime.KV_SIDS: (case["n"], 1, np.int16), runtime.KV_CTFS: (files, runtime.CTF_DTYPE.itemsize, np.uint8),
            runtime.KV_BITMAPS: (files, 8192, np.uint8), runtime.KV_OVERSIZE_BITMAP: (1, 8192, np.uint8),
            runtime.KV_PACKED: (0, 16, np.uint8)}


def _kv_flush(s: _State) -> dict:
    """A flush, every part copied to the program's own buffers."""
    summary = s.wb.kv_flush(copy=False)["summary"]
    lib, out = runtime.lib(), {"summary": [summary[k] for k in sorted(summary)]}
    for part, rows in s.parts.items():
        size = ctypes.c_uint64()
        runtime._check(lib.glint_kv_part_size(s.wb.h, part, ctypes.byref(size)), "glint_kv_part_size", s.wb.h)
        row = rows.buf.itemsize * rows.buf.shape[1]
        to = rows.cut(-(-size.value // row))
        runtime._check(lib.glint_kv_copy(s.wb.h, part, to.ctypes.data if size.value else None, size.value),
                       "glint_kv_copy", s.wb.h)
        if size.value % row:
            to[-1, size.value % row:] = 0
        out[f"part{part}"] = rows.buf
    return out


def prepare(case: dict, seed: int):
    kind = case["kind"]
    if kind == "stage":
        return _stage_state(case, seed)
    if kind == "run":
        return _run_state(case, seed)
    if kind == "batch":
        return _batch_state(case, seed)
    if kind == "serve":
        return _serve_state(case, seed)
    if kind == "kv":
        full = dict(case, hot=True, precision="fp32guard", schema="dynamic")
        capacity = 2 * case["ticks"] * max(1 << 16, case["n"])
        s = _run_state(full, seed, kv_capacity=capacity, kv_split_num=10)
        s.parts = {part: _Rows(capacity if part in KV_VARIABLE else n, columns, dtype)
                   for part, (n, columns, dtype) in _kv_parts(case).items()}
        _kv_flush(s)
        return s
    s = _State(case)
    g = torch.Generator(device="cuda").manual_seed(seed)
    p = torch.rand((case["n"], 2), dtype=torch.float64, device="cuda", generator=g)
    s.points = torch.stack([-87.94 + 0.42 * p[:, 0], 41.64 + 0.39 * p[:, 1]], dim=1)   # a city's box, degrees
    s.projection = runtime.projection_for_box(-87.94, 41.64)
    s.out = torch.empty_like(s.points)
    torch.cuda.synchronize()
    return s


# --------------------------------------------------------------------- run
def run(s):
    if s.kind == "stage":
        out = {"meetings": s.meetings.put(_stage_tick(s).view(np.int32))}
        if s.case["record"]:
            out["contacts"] = s.contacts.put(s.wb.contacts().view(np.int64)[:, None])
        return out
    if s.kind == "run":
        _advance(s)
        return {"meetings": _last_meetings(s, [s.wb]), "totals": _totals(s.wb)}
    if s.kind == "batch":
        _batch_advance(s)
        return {"meetings": _last_meetings(s, s.batch.contexts),
                "totals": np.array([_totals(wb) for wb in s.batch.contexts], dtype=np.int64)}
    if s.kind == "serve":
        _serve_tick(s)
        last, q = s.tick - 1, s.case["queries"]
        at = (last % 2) * q
        ids = [s.server.submit(seeds, max(0, last - window), last, hops)
               for seeds, window, hops in s.queries[at:at + q]]
        s.server.drain()
        answers = [s.server.result(i) for i in ids]
        return {"hop1": s.hop1.put(np.concatenate([a for a, _ in answers]).view(np.int32)),
                "hop2": s.hop2.put(np.concatenate([b for _, b in answers]).view(np.int32)),
                "counts": np.array([[len(a), len(b)] for a, b in answers], dtype=np.int64)}
    if s.kind == "kv":
        _advance(s)
        return _kv_flush(s)
    runtime.project_device(s.projection, s.points.data_ptr(), s.out.data_ptr(), s.case["n"])
    return s.out


# ----------------------------------------------------- work and exact values
def work(case: dict) -> dict:
    """Positions in; per tick the run of every continuing pair read and
    written (12 B: pair and start), of which an eighth of the contacts are; a
    distance for every pair of a half-full leaf."""
    kind = case["kind"]
    if kind == "project":
        return {"bytes": 32.0 * case["n"], "flops": 4.0 * case["n"]}

    def ticks(n, pairs, cap, count):
        return {"bytes": count * (16.0 * n + 24.0 * pairs / 8), "flops": count * 6.0 * n * cap / 4}

    if kind == "batch":
        ws = gen.batched_cities(case["count"], seed=4, n_min=case["smallest"], n_max=case["largest"])
        n = sum(w.num_objects for w in ws)
        return ticks(n, 0.1 * n, 200, case["ticks"])
    if kind == "serve":
        one = ticks(case["n"], 0.1 * case["n"], 200, 1)
        return {"bytes": one["bytes"] + 20.0 * case["move"] * case["n"], "flops": one["flops"]}
    pairs = _pairs(dict(case, hot=case.get("hot", True)))
    return ticks(case["n"], pairs, case["cap"], case.get("ticks", 1))


def exact(case: dict, seed: int):
    """Planar metres of the projected points; every other kind returns whole
    numbers and copies of its inputs."""
    if case["kind"] != "project":
        return None
    s = prepare(case, seed)
    p = s.points.cpu().numpy()
    q = s.projection
    return np.stack([(p[:, 0] - q.lon0) / q.deg_per_m_lon, (p[:, 1] - q.lat0) / q.deg_per_m_lat], axis=1)
