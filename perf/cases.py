"""Performance cases of the spatial join engine: what a program that binds the engine has it do, over the range it is used on.

Every case goes through the library's public entry points: the requests through the C ABI with row callbacks, as the
daemon and any foreign-language client call it, the rest through the Python binding (``gsj.Context``, ``gsj.Scheduler``,
``gsj.copy_parse``, ``gsj.subdivide``, ``gsj.dedup``). Layers are resident before the call, as in the engine's use; what counts is one request:
candidate search, exact refinement, compaction and the rows in host memory. Inputs are the library's own deterministic
synthetic layers: star polygons in grid cells under region tiles with shared jittered borders, the jittered parcel
mesh with shared, overlapping and separated sides and lognormal vertex counts, and uniform plus clustered points.
"""
import ctypes as C
import math
import os
import sys

import numpy as np

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_ROOT, "postgis-cuda_amd"))

import gsj  # noqa: E402

X0, Y0, CELL = -95.5, 38.5, 1.0 / 1549   # the parcel mesh: 1549 cells to the degree
GRID_CELL = 0.001                        # the parcel grid's cell
EXACT_PARCELS = 20_000                   # plain numpy clips this many parcels in a few seconds

_ctx = None


def _context():
    """the program's one context (one GPU), kept for all requests as a server keeps it"""
    global _ctx
    if _ctx is None:
        _ctx = gsj.Context(0)
    return _ctx


def listed():
    return [
        # a map click's worth of parcels under four regions: launches and host waits are all of it
        {"name": "join_area_tile", "kind": "join", "nx": 13, "ny": 11, "k": 2, "segs": 40, "what": "area"},
        # the ordinary overlay request: 10k parcels of 4-12 vertices under 16 regions of 2000 vertices, with areas
        {"name": "join_area_10k", "kind": "join", "nx": 100, "ny": 100, "k": 4, "segs": 500, "what": "area"},
        # a county's parcels against large regions with the DE-9IM matrix of every row
        {"name": "join_relate_250k", "kind": "join", "nx": 517, "ny": 489, "k": 4, "segs": 500, "what": "relate"},
        # topology check of one town: subdivided parcels with themselves, DE-9IM
        {"name": "self_relate_50k", "kind": "self", "nx": 229, "ny": 223, "subdiv": 256, "what": "relate"},
        # the benchmark's request at the size of a large county
        {"name": "self_relate_1M", "kind": "self", "nx": 1103, "ny": 997, "subdiv": 256, "what": "relate"},
        # geocoded addresses into parcels
        {"name": "points_in_parcels_3M", "kind": "pip", "points": 3_000_017, "nx": 701, "ny": 687, "subdiv": 256},
        # neighbours within 5 m with the distance of every row
        {"name": "dwithin_self_300k", "kind": "dwithin", "nx": 557, "ny": 541, "d": 5.0, "report": True},
        # addresses within 25 m of a parcel with the distance
        {"name": "points_dwithin_200k", "kind": "pdist", "points": 200_003, "nx": 401, "ny": 383, "d": 25.0, "report": True},
        # overlaps that survive a setback on both sides
        {"name": "erode_self_250k", "kind": "erode", "nx": 503, "ny": 499, "ra": 0.5, "rb": 0.75},
        # connected blocks of parcels
        {"name": "cluster_400k", "kind": "cluster", "nx": 641, "ny": 619, "subdiv": 256},
        # the served stream: small windowed requests of every kind over one resident layer, four lanes
        {"name": "served_windows_64", "kind": "served", "nx": 811, "ny": 797, "requests": 64},
        # a layer's load: the binary COPY stream parsed, deduplicated, subdivided and made resident with its tree
        {"name": "load_60k", "kind": "load", "nx": 251, "ny": 239, "subdiv": 64},
    ]


def draw(rng):
    def side(lo, hi):   # cells, with a ragged aspect
        n, a = math.exp(rng.uniform(math.log(lo), math.log(hi))), math.exp(rng.uniform(-0.2, 0.2))
        return max(3, int(math.sqrt(n) * a) | rng.randint(0, 1)), max(3, int(math.sqrt(n) / a))

    def span(lo, hi):
        return int(math.exp(rng.uniform(math.log(lo), math.log(hi)))) | rng.randint(0, 1)

    kind = rng.choice(["join", "join", "self", "self", "pip", "dwithin", "pdist", "erode", "cluster", "served", "load"])
    if kind == "join":
        nx, ny = side(100, 250_000)
        return {"kind": kind, "nx": nx, "ny": ny, "k": rng.choice([2, 4, 8]), "segs": span(20, 600), "what": rng.choice(["area", "relate"])}
    if kind == "self":
        nx, ny = side(1_000, 900_000)
        return {"kind": kind, "nx": nx, "ny": ny, "subdiv": rng.choice([0, 64, 256]), "what": rng.choice(["area", "relate"])}
    if kind == "pip":
        nx, ny = side(1_000, 450_000)
        return {"kind": kind, "points": span(1_000, 3_000_000), "nx": nx, "ny": ny, "subdiv": rng.choice([0, 256])}
    if kind == "dwithin":
        nx, ny = side(1_000, 280_000)
        return {"kind": kind, "nx": nx, "ny": ny, "d": round(rng.uniform(1.0, 8.0), 3), "report": rng.random() < 0.5}
    if kind == "pdist":
        nx, ny = side(1_000, 140_000)
        return {"kind": kind, "points": span(1_000, 180_000), "nx": nx, "ny": ny, "d": round(rng.uniform(1.0, 25.0), 3), "report": rng.random() < 0.5}
    if kind == "erode":
        nx, ny = side(1_000, 230_000)
        return {"kind": kind, "nx": nx, "ny": ny, "ra": round(rng.uniform(0.5, 3.0), 3), "rb": round(rng.uniform(0.5, 3.0), 3)}
    if kind == "cluster":
        nx, ny = side(1_000, 380_000)
        return {"kind": kind, "nx": nx, "ny": ny, "subdiv": rng.choice([0, 256])}
    if kind == "served":
        nx, ny = side(20_000, 600_000)
        return {"kind": kind, "nx": nx, "ny": ny, "requests": rng.randint(8, 60)}
    nx, ny = side(1_000, 55_000)
    return {"kind": "load", "nx": nx, "ny": ny, "subdiv": rng.choice([32, 64, 256])}


# ------------------------------------------------------------------------------------------- inputs
def _mesh(case, seed):
    return gsj.generate("parcels_mesh", nx=case["nx"], ny=case["ny"], x0=X0, y0=Y0, w=CELL, h=CELL, seed=seed)


def _grid(case, seed):
    P = gsj.generate("parcels_grid", nx=case["nx"], ny=case["ny"], seed=seed)
    sx, sy = np.random.default_rng(seed).uniform(0.0, GRID_CELL, 2)   # the regions' borders fall anywhere in a parcel's cell
    R = gsj.generate("regions_grid", nx=case["nx"], ny=case["ny"], x0=-118.5 + sx, y0=34.0 + sy, kx=case["k"], ky=case["k"], edge_segs=case["segs"],
                     seed=seed)
    return P, R


def _points(case, seed):
    return gsj.generate_points(n=case["points"], x0=X0, y0=Y0, w=case["nx"] * CELL, h=case["ny"] * CELL,
                               clusters=max(1, case["points"] // 5000), sigma_m=50.0, seed=seed)


def _window_parcels(case, win):
    """no window meets more parcels than this: its cells, one more to each side for jitter and bulges"""
    return (min(case["nx"], math.ceil((win[2] - win[0]) / CELL) + 4)) * (min(case["ny"], math.ceil((win[3] - win[1]) / CELL) + 4))


def _window_requests(case, seed):
    """(kind, rows' second column, options, fields) of the stream's requests: 35% intersects + area, 20% relate, 20%
    dwithin, 20% eroded intersects, 5% cluster, at random places. The windows' sizes and kinds are the case's own (lognormal
    in area around a few hundred parcels), so that the streams of two seeds cost the same."""
    shape, rng = np.random.default_rng([case["nx"], case["ny"], case["requests"]]), np.random.default_rng(seed)
    n, W, H = case["requests"], case["nx"] * CELL, case["ny"] * CELL
    out = []
    for i in range(n):
        s = min(CELL * math.sqrt(math.exp(shape.normal(math.log(400.0), 1.3))), W, H)
        u, d, ra, rb = shape.uniform(), shape.uniform(1.0, 50.0), shape.uniform(0.5, 3.0), shape.uniform(0.5, 3.0)
        cx, cy = X0 + s / 2 + rng.uniform() * (W - s), Y0 + s / 2 + rng.uniform() * (H - s)
        win = (cx - s / 2, cy - s / 2, cx + s / 2, cy + s / 2)
        if u < 0.35:
            out.append((gsj.REQ_JOIN, "area", _opts(want_area=True, upper=True, window=win), {}))
        elif u < 0.55:
            out.append((gsj.REQ_JOIN, "code", _opts(want_relate=True, upper=True, window=win), {}))
        elif u < 0.75:
            out.append((gsj.REQ_DWITHIN, None, _opts(upper=True, window=win), {"d": d, "same": 1}))
        elif u < 0.95:
            out.append((gsj.REQ_INTERSECTS_BUFFERED, None, _opts(upper=True, window=win), {"ra": ra, "rb": rb, "same": 1}))
        else:
            out.append((gsj.REQ_CLUSTER_ROWS, None, _opts(window=win), {}))
    return out


class _Sink:
    """Row arrays a program keeps: a callback's buffers are valid until it returns, so it moves the rows out of them. The
    arrays are as long as a request of this case can need; the rows past ``n`` stay zero."""

    def __init__(self, cap, second=None, dtype=None):
        self.cap, self.n = cap, 0
        self.pairs = np.zeros((cap, 2), np.uint32)
        self.second, self.value = second, (np.zeros(cap, dtype) if second else None)

    def take(self, pairs, value, n):
        if self.n + n > self.cap:
            return 1
        C.memmove(self.pairs.ctypes.data + 8 * self.n, pairs, 8 * n)
        if value:
            w = self.value.itemsize
            C.memmove(self.value.ctypes.data + w * self.n, value, w * n)
        self.n += n
        return 0

    def out(self):
        o = {"rows": self.n, "pairs": self.pairs}
        if self.second:
            o[self.second] = self.value
        return o

    def rows_cb(self):
        return gsj.ROWS_CB(lambda user, pairs, area, code, n: self.take(pairs, area or code, n))

    def points_cb(self):
        return gsj.POINTS_CB(lambda user, pairs, where, n: self.take(pairs, where, n))

    def dist_cb(self):
        return gsj.DIST_CB(lambda user, pairs, dist, n: self.take(pairs, dist, n))


def _opts(want_area=False, want_relate=False, upper=False, window=None):
    o = gsj.JoinOpts()
    o.want_area, o.want_relate, o.upper = int(want_area), int(want_relate), int(upper)
    if window is not None:
        o.has_window = 1
        o.window[:] = window
    return o


def _join_sink(what, cap):
    return _Sink(cap, "area", np.float64) if what == "area" else _Sink(cap, "code", np.uint32)


def prepare(case, seed):
    ctx, kind, n = _context(), case["kind"], case["nx"] * case["ny"]
    st = {"case": case, "ctx": ctx}
    if kind == "join":
        P, R = _grid(case, seed)
        st["P"], st["R"] = ctx.polys(P, build_bvh=False), ctx.polys(R)
        sink = _join_sink(case["what"], 9 * n + 100)
        st.update(sink=sink, cb=sink.rows_cb(), opts=_opts(want_area=case["what"] == "area", want_relate=case["what"] == "relate"))
        return st
    hs = _mesh(case, seed)
    if kind == "load":
        st["stream"] = gsj.copy_write(hs, srid=4326)
        cap, capv = 2 * n + 1000, 24 * n + 20_000   # a parcel holds 13 vertices on average
        st["cap"] = (cap, capv)
        st["out"] = {"gro": np.zeros(cap, np.uint64), "rvo": np.zeros(2 * cap, np.uint64), "parent": np.zeros(cap, np.uint32),
                     "members": np.zeros(cap, np.uint32), "origin": np.zeros((cap, 2)), "ext": np.zeros((cap, 2)),
                     "box": np.zeros((cap, 4), np.float32), "xy": np.zeros((capv, 2)), "length": np.zeros(cap)}
        return st
    if case.get("subdiv"):
        hs = gsj.subdivide(hs, case["subdiv"])
    st["R"] = ctx.polys(hs)
    if kind in ("pip", "pdist"):
        st["P"] = ctx.points(_points(case, seed))
    if kind == "self":
        sink = _join_sink(case["what"], 5 * n + 100)
        st.update(sink=sink, cb=sink.rows_cb(), opts=_opts(want_area=case["what"] == "area", want_relate=case["what"] == "relate", upper=True))
    elif kind == "pip":
        sink = _Sink(2 * case["points"] + 100, "where", np.uint8)
        st.update(sink=sink, cb=sink.points_cb(), opts=_opts())
    elif kind in ("dwithin", "pdist"):
        sink = _Sink(8 * case["points"] if kind == "pdist" else 7 * n, *(("dist", np.float64) if case["report"] else ()))
        st.update(sink=sink, cb=sink.dist_cb(), opts=_opts(upper=kind == "dwithin"))
    elif kind == "erode":
        sink = _Sink(4 * n + 100)
        st.update(sink=sink, cb=sink.dist_cb(), opts=_opts(upper=True))
    elif kind == "served":
        st["sched"] = gsj.Scheduler(ctx, lanes=4)
        st["requests"], st["sinks"], st["cbs"] = [], [], []
        for k, what, o, kw in _window_requests(case, seed):
            req = gsj.Request()
            req.kind, req.P, req.R, req.opts = k, st["R"].h, st["R"].h, o
            for f, v in kw.items():
                setattr(req, f, v)
            sink = _join_sink(what, 0) if what else _Sink(0)
            st["requests"].append(req)
            st["sinks"].append(sink)
        # all requests' rows in one set of arrays: request i's part is as long as its window's parcels can need
        caps = [12 * _window_parcels(case, req.opts.window) for req in st["requests"]]
        st["pairs"] = np.zeros((sum(caps), 2), np.uint32)
        at = 0
        for req, sink, cap in zip(st["requests"], st["sinks"], caps):
            sink.cap, sink.pairs = cap, st["pairs"][at:at + cap]
            if sink.second:
                sink.value = np.zeros(cap, sink.value.dtype)
            if req.kind in (gsj.REQ_JOIN, gsj.REQ_CLUSTER_ROWS):
                req.rows_cb = sink.rows_cb()
            else:
                req.dist_cb = sink.dist_cb()
            at += cap
        st["area"] = np.zeros(sum(s.cap for s in st["sinks"] if s.second == "area"))
        st["code"] = np.zeros(sum(s.cap for s in st["sinks"] if s.second == "code"), np.uint32)
        for name in ("area", "code"):
            at = 0
            for s in st["sinks"]:
                if s.second == name:
                    s.value = st[name][at:at + s.cap]
                    at += s.cap
    return st


# ------------------------------------------------------------------------------------------- one pass
def _check(rc):
    if rc != gsj.GSJ_OK:
        raise gsj.GsjError(rc, gsj.load().gsj_last_error().decode())


def run(state):
    case, ctx, lib = state["case"], state["ctx"], gsj.load()
    kind = case["kind"]
    if kind == "cluster":
        return ctx.cluster(state["R"])[0]
    if kind == "load":
        return _load(state)
    if kind == "served":
        return _served(state)
    sink, R = state["sink"], state["R"].h
    sink.n = 0
    args = (C.byref(state["opts"]), state["cb"], None, C.byref(gsj.JoinStats()))
    if kind == "join":
        _check(lib.gsj_join(ctx.h, state["P"].h, R, *args))
    elif kind == "self":
        _check(lib.gsj_join(ctx.h, R, R, *args))
    elif kind == "pip":
        _check(lib.gsj_points_in_polygons(ctx.h, state["P"].h, R, *args))
    elif kind == "dwithin":
        _check(lib.gsj_dwithin(ctx.h, R, R, case["d"], 1, int(case["report"]), *args))
    elif kind == "pdist":
        _check(lib.gsj_points_dwithin(ctx.h, state["P"].h, R, case["d"], int(case["report"]), *args))
    else:
        _check(lib.gsj_intersects_buffered(ctx.h, R, R, case["ra"], case["rb"], 1, None, *args))
    return sink.out()


def _served(state):
    lib, s = gsj.load(), state["sched"].h
    tickets, ticket = [], C.c_uint64()
    for req, sink in zip(state["requests"], state["sinks"]):
        sink.n = 0
        _check(lib.gsj_submit(s, C.byref(req), C.byref(ticket)))
        tickets.append(ticket.value)
    for t in tickets:
        _check(lib.gsj_wait(s, t, None, None))
    return {"rows": np.array([sink.n for sink in state["sinks"]]), "pairs": state["pairs"], "area": state["area"], "code": state["code"]}


def _load(state):
    ctx, out = state["ctx"], state["out"]
    layer = gsj.copy_parse(ctx, state["stream"], want_ids=False)
    distinct, moff, midx = gsj.dedup(layer.polys, ctx)
    pieces = gsj.subdivide(distinct, state["case"]["subdiv"], ctx)
    L = ctx.polys(pieces)
    state["layer"] = L   # resident from here on; the one before it is released, as a reload does
    if pieces.n + 1 > state["cap"][0] or pieces.nr + 1 > 2 * state["cap"][0] or pieces.nv > state["cap"][1]:
        raise ValueError("more pieces than this case expects")
    for name, a in (("gro", pieces.gro), ("rvo", pieces.rvo), ("parent", pieces.parent), ("members", midx)):
        out[name][:len(a)] = a

    def p(name, t):
        return out[name].ctypes.data_as(C.POINTER(t))

    # the prepared arrays as the device holds them
    _check(gsj.load().gsj_layer_export(L.h, p("origin", C.c_double), p("ext", C.c_double), p("box", C.c_float), p("xy", C.c_double),
                                       p("length", C.c_double)))
    return {"sizes": np.array([pieces.n, pieces.nr, pieces.nv, len(moff) - 1]), **out}


# ------------------------------------------------------------------------------------------- what a pass cannot do without
_GEOM = 60   # bytes of one geometry's records (origin, extent, offsets, box); vertices are 16 bytes each
_MESH_V, _GRID_V = 13.0, 9.0   # stored vertices of a mesh and of a grid parcel


def work(case):
    kind, n = case["kind"], case["nx"] * case["ny"]
    if kind == "join":
        nr = case["k"] ** 2
        rows = n * 1.02
        b = n * (_GEOM + 16 * _GRID_V) + nr * (_GEOM + 64 * case["segs"]) + rows * (16 if case["what"] == "area" else 12)
        return {"bytes": b, "flops": rows * 600.0}
    mesh = n * (_GEOM + 16 * _MESH_V)
    if kind == "self":
        return {"bytes": mesh + 3.3 * n * (16 if case["what"] == "area" else 12), "flops": 3.3 * n * 1400.0}
    if kind == "pip":
        return {"bytes": mesh + case["points"] * (16 + 9), "flops": case["points"] * 1.5 * 60.0}
    if kind == "dwithin":
        return {"bytes": mesh + 5.0 * n * (16 if case["report"] else 8), "flops": 5.0 * n * 1000.0}
    if kind == "pdist":
        return {"bytes": mesh + case["points"] * (16 + 3 * (16 if case["report"] else 8)), "flops": case["points"] * 4 * 1000.0}
    if kind == "erode":
        return {"bytes": mesh + 8.0 * n, "flops": 3.0 * n * 2000.0}
    if kind == "cluster":
        return {"bytes": mesh + 4.0 * n, "flops": 3.3 * n * 300.0}
    if kind == "served":
        m = case["requests"] * min(900.0, n)
        return {"bytes": m * (_GEOM + 16 * _MESH_V + 40), "flops": m * 3.3 * 1000.0}
    # load: the stream in, the pieces and the prepared arrays out
    return {"bytes": n * (16 * _MESH_V + 30) + n * (16 * _MESH_V + 2 * _GEOM), "flops": n * _MESH_V * 30.0}


# ------------------------------------------------------------------------------------------- areas in plain numpy
def _inside(px, py, ax, ay, bx, by):
    """even-odd membership of points (k) in the ring with edges a -> b (m)"""
    py, px = py[:, None], px[:, None]
    span = (ay[None] > py) != (by[None] > py)
    with np.errstate(divide="ignore", invalid="ignore"):
        x = ax[None] + (py - ay[None]) / (by - ay)[None] * (bx - ax)[None]
    return (np.count_nonzero(span & (x > px), axis=1) & 1) == 1


def _part(A, B, near):
    """twice the area contributed by A's edges inside B (rings of (k, 4) edges x0 y0 x1 y1; near: B's edges by A's box)"""
    x0, y0, x1, y1 = A.T
    dx, dy = x1 - x0, y1 - y0
    t = np.full((len(A), len(near) + 2), 1.0)
    t[:, 0] = 0.0
    if len(near):
        ux, uy, vx, vy = near.T
        fx, fy = vx - ux, vy - uy
        with np.errstate(divide="ignore", invalid="ignore"):
            den = dx[:, None] * fy[None] - dy[:, None] * fx[None]
            wx, wy = ux[None] - x0[:, None], uy[None] - y0[:, None]
            s, u = (wx * fy[None] - wy * fx[None]) / den, (wx * dy[:, None] - wy * dx[:, None]) / den
        ok = (den != 0) & (s > 0) & (s < 1) & (u >= 0) & (u <= 1)
        t[:, 2:] = np.where(ok, s, 1.0)
        t.sort(axis=1)
    lo, hi = t[:, :-1], t[:, 1:]
    e, k = np.nonzero(hi > lo)
    a, b = lo[e, k], hi[e, k]
    m = 0.5 * (a + b)
    mx, my = x0[e] + dx[e] * m, y0[e] + dy[e] * m
    w = _inside(mx, my, B[:, 0], B[:, 1], B[:, 2], B[:, 3])
    p0x, p0y, p1x, p1y = x0[e] + dx[e] * a, y0[e] + dy[e] * a, x0[e] + dx[e] * b, y0[e] + dy[e] * b
    return float(np.sum(np.where(w, p0x * p1y - p0y * p1x, 0.0)))


def _edges(xy):
    return np.concatenate([xy[:-1], xy[1:]], axis=1)


def _by(E, box):
    """E's edges whose boxes meet the box"""
    return E[(np.maximum(E[:, 0], E[:, 2]) >= box[0]) & (np.minimum(E[:, 0], E[:, 2]) <= box[2]) &
             (np.maximum(E[:, 1], E[:, 3]) >= box[1]) & (np.minimum(E[:, 1], E[:, 3]) <= box[3])]


def _morton_order(boxes):
    """indices of boxes in the order of the interleaved 32-bit positions of their centres, x first (the tree's leaf order)"""
    c = 0.5 * (boxes[:, :2] + boxes[:, 2:])
    lo, hi = c.min(axis=0), c.max(axis=0)
    q = np.floor((c - lo) * np.where(hi > lo, 4294967295.0 / np.where(hi > lo, hi - lo, 1.0), 0.0)).astype(np.uint64)

    def key(x, y):
        return sum(((int(x) >> b & 1) << (2 * b + 1)) | ((int(y) >> b & 1) << (2 * b)) for b in range(32))

    return sorted(range(len(boxes)), key=lambda i: (key(*q[i]), i))


def exact(case, seed):
    """Intersection areas by splitting every edge at its crossings and summing the parts inside the other polygon. The
    rows, DE-9IM codes and labels are whole numbers; geography distances have no plain closed form."""
    if case["kind"] != "join" or case["what"] != "area" or case["nx"] * case["ny"] > EXACT_PARCELS:
        return None
    P, R = _grid(case, seed)
    regions = [np.asarray(R.xy[int(R.rvo[g]):int(R.rvo[g + 1])]) for g in range(R.n)]
    boxes = np.array([[*r.min(axis=0), *r.max(axis=0)] for r in regions])
    order = _morton_order(boxes)
    area = []
    for a in range(P.n):
        A = np.asarray(P.xy[int(P.rvo[a]):int(P.rvo[a + 1])])
        lo, hi = A.min(axis=0), A.max(axis=0)
        EA = _edges(A - lo)
        for g in order:
            if boxes[g, 0] > hi[0] or boxes[g, 2] < lo[0] or boxes[g, 1] > hi[1] or boxes[g, 3] < lo[1]:
                continue
            EB = _edges(regions[g] - lo)
            row = _by(EB, (-1e9, 0.0, 1e9, hi[1] - lo[1]))        # the edges a horizontal ray from the parcel can meet
            near = _by(row, (0.0, 0.0, hi[0] - lo[0], hi[1] - lo[1]))
            s = _part(EA, row, near)
            if len(near):
                s += _part(near, EA, EA)
            if s > 0:
                area.append(0.5 * s)
    full = np.zeros(9 * P.n + 100)
    full[:len(area)] = area
    return {"rows": None, "pairs": None, "area": full}
