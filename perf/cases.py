"""The work that a user of the library has it do, as timed cases.

Every case goes through hsync's public entry points: reductions and scans of one
array, batches of many ragged scans or sums, graph searches (one source, 64
sources), shortest paths, PageRank, and the device-wide barrier and semaphore
under contention.  Sizes are those of bench.py and the tests (2^24 sums, 2^28
scans, 512 ragged segments, R-MAT graphs up to scale 22 with edge factor 16, 1024
workgroups), smaller and ragged ones, and meshes with gaps, which stand for the
road networks that the graph programs are run on (high diameter, degree <= 4).

listed() names the cases, draw() makes more of the same ranges, prepare() builds
what a program holds before the call (inputs, the arena, the resident graph and
the work space), run() is one call, exact() the same results from plain torch.
"""
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.getcwd(), "tpds22-artifact_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

DEV = "cuda"
INF = 2**31 - 1
ALPHA, TOL = 0.85, 1e-6


def listed():
    return [
        # the smallest call: a sum of a few thousand values, taken as a number
        {"name": "reduce_small", "kind": "reduce", "n": 4099, "hi": 255, "take": True},
        # the headline sum: 2^24 values, enqueued among other work
        {"name": "reduce_2p24", "kind": "reduce", "n": 1 << 24, "hi": 255, "take": False},
        # the headline scan: 2^28 values, inclusive
        {"name": "scan_2p28", "kind": "scan", "n": 1 << 28, "hi": 15, "inclusive": True},
        # a batch of ragged scans in one launch, lengths log-uniform in 2^10..2^22
        {"name": "scan_batch_512", "kind": "batch", "op": "scan", "nseg": 512, "lo": 10.0, "top": 22.0, "inclusive": True},
        # many short rows (the row sums of a ragged table): 1..2^11 values each
        {"name": "rows_30011", "kind": "batch", "op": "reduce", "nseg": 30011, "lo": 0.0, "top": 11.0, "inclusive": True},
        # one search over a large power-law graph
        {"name": "bfs_rmat22", "kind": "bfs", "graph": "rmat", "n": 1 << 22, "ef": 16},
        # 64 searches at once, the headline of the batched search
        {"name": "msbfs_rmat22", "kind": "msbfs", "graph": "rmat", "n": 1 << 22, "ef": 16, "nsrc": 64},
        # one shortest-path run over a road-like mesh: thousands of small rounds
        {"name": "sssp_mesh", "kind": "sssp", "graph": "mesh", "h": 1000, "w": 1100, "delta": 10000},
        # 64 shortest-path runs at once over a power-law graph
        {"name": "mssp_rmat21", "kind": "mssp", "graph": "rmat", "n": 1 << 21, "ef": 16, "nsrc": 64},
        # ranks of a large power-law graph to an L1 change below 1e-6
        {"name": "pagerank_rmat22", "kind": "pagerank", "graph": "rmat", "n": 1 << 22, "ef": 16},
        # device-wide barrier episodes of a full data-exchanging grid
        {"name": "barrier_1024", "kind": "barrier", "wgs": 1024, "ldst": 16, "episodes": 200},
        # a semaphore of 16 units, 9 readers to 1 writer, 1024 workgroups
        {"name": "semaphore_1024", "kind": "semaphore", "sem": 4, "wgs": 1024, "capacity": 16, "ldst": 16, "iters": 2},
    ]


def draw(rng):
    def logint(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["reduce", "scan", "batch", "batch", "bfs", "msbfs", "sssp", "mssp", "pagerank", "barrier", "semaphore"])
    if kind == "reduce":
        return {"kind": kind, "n": logint(100, 1 << 28), "hi": rng.choice([15, 255, 2**32 - 1]), "take": rng.random() < 0.5}
    if kind == "scan":
        return {"kind": kind, "n": logint(100, 1 << 28), "hi": rng.choice([15, 255, 2**32 - 1]), "inclusive": rng.random() < 0.5}
    if kind == "batch":
        nseg = logint(1, 65536)
        top = rng.uniform(4.0, min(24.0, 27.0 - math.log2(nseg) + 2.0))
        return {"kind": kind, "op": rng.choice(["scan", "reduce"]), "nseg": nseg, "lo": rng.uniform(0.0, top), "top": top,
                "inclusive": rng.random() < 0.5}
    if kind == "barrier":
        return {"kind": kind, "wgs": rng.choice([256, 512, 1024, 2048, rng.randrange(8, 2048)]), "ldst": rng.randrange(1, 17),
                "episodes": rng.randrange(20, 400)}
    if kind == "semaphore":
        return {"kind": kind, "sem": 4, "wgs": rng.choice([256, 512, 1024, 2048]), "capacity": rng.choice([1, 16, 256]),
                "ldst": rng.randrange(1, 17), "iters": 1}
    if kind in ("bfs", "sssp") and rng.random() < 0.4:
        c = {"kind": kind, "graph": "mesh", "h": rng.randrange(50, 1000), "w": rng.randrange(50, 1000)}
    else:
        top = 1 << (21 if kind == "mssp" else 22)
        c = {"kind": kind, "graph": "rmat", "n": logint(1 << 12, top), "ef": rng.randrange(4, 17)}
    if kind in ("msbfs", "mssp"):
        c["nsrc"] = rng.choice([64, rng.randrange(1, 65)])
    if kind == "sssp":
        c["delta"] = rng.choice([10000, rng.randrange(100, 20000)])
    return c


# ---------------------------------------------------------------------------
# inputs


def _gen(seed, device=DEV):
    g = torch.Generator(device=device)
    g.manual_seed(seed)
    return g


def _values(n, hi, seed):
    if hi >= 2**31:
        return torch.randint(-2**31, 2**31, (n,), generator=_gen(seed), device=DEV, dtype=torch.int32)
    return torch.randint(0, hi + 1, (n,), generator=_gen(seed), device=DEV, dtype=torch.int32)


def _total(case):
    """Values of a batch: the segments times the mean of the log-uniform lengths."""
    lo, top = case["lo"], max(case["top"], case["lo"] + 1e-6)
    return max(1, int(case["nseg"] * (2.0**top - 2.0**lo) / ((top - lo) * math.log(2.0))))


def _offsets(case, seed):
    """Log-uniform lengths, scaled to the batch's total (short ones may become empty)."""
    rng = np.random.default_rng(seed)
    ends = np.cumsum(np.exp2(rng.uniform(case["lo"], case["top"], case["nseg"])))
    return np.concatenate([[0], np.rint(ends * (_total(case) / ends[-1]))]).astype(np.uint64)


def _edges(case, seed):
    """n, and the directed edges as one sorted tensor of u * n + v without repeats or self loops."""
    g = _gen(seed)
    if case["graph"] == "mesh":  # 4-neighbour mesh, both directions, one street in eight missing
        h, w = case["h"], case["w"]
        at = torch.arange(h * w, device=DEV).view(h, w)
        a = torch.cat([at[:, :-1].reshape(-1), at[:-1, :].reshape(-1)])
        b = torch.cat([at[:, 1:].reshape(-1), at[1:, :].reshape(-1)])
        keep = torch.rand(a.numel(), generator=g, device=DEV) >= 0.125
        a, b = a[keep], b[keep]
        n = h * w
        return n, torch.sort(torch.cat([a * n + b, b * n + a]))[0]
    # R-MAT, (a, b, c) = (0.57, 0.19, 0.19); ids at or above n are left out, so n is any number
    n, m = case["n"], case["n"] * case["ef"]
    u = torch.zeros(m, dtype=torch.int64, device=DEV)
    v = torch.zeros(m, dtype=torch.int64, device=DEV)
    for _ in range(max(1, (n - 1).bit_length())):
        r = torch.rand(m, generator=g, device=DEV)
        ub = r >= 0.76
        vb = ((r >= 0.57) & ~ub) | (r >= 0.95)
        u = u * 2 + ub
        v = v * 2 + vb
    keep = (u != v) & (u < n) & (v < n)
    return n, torch.unique(u[keep] * n + v[keep])


def _graph_parts(case, seed):
    """n, row, u, v, w on the device (64-bit), w the weights of a shortest-path case."""
    n, key = _edges(case, seed)
    u, v = torch.div(key, n, rounding_mode="floor"), key % n
    row = torch.zeros(n + 1, dtype=torch.int64, device=DEV)
    row[1:] = torch.cumsum(torch.bincount(u, minlength=n), 0)
    w = torch.randint(1, 256, (key.numel(),), generator=_gen(seed + 7), device=DEV) if case["kind"] in ("sssp", "mssp") else None
    return n, row, u, v, w


def _sources(case, row, seed):
    deg = (row[1:] - row[:-1]).cpu()
    have = torch.nonzero(deg).view(-1)
    at = torch.randint(0, have.numel(), (case.get("nsrc", 1),), generator=_gen(seed + 13, "cpu"))
    return [int(s) for s in have[at]]


# ---------------------------------------------------------------------------


def prepare(case, seed):
    import hsync as hs
    kind = case["kind"]
    st = {"case": case, "hs": hs, "arena": hs.Arena()}
    if kind in ("reduce", "scan"):
        x = st["x"] = _values(case["n"], case["hi"], seed)
        if kind == "reduce":
            st["out"] = torch.empty(1, dtype=torch.int32, device=DEV)
            st["partials"] = torch.empty(2048, dtype=torch.int32, device=DEV)
        else:
            st["out"] = torch.empty_like(x)
    elif kind == "batch":
        st["off"] = _offsets(case, seed)
        st["x"] = _values(int(st["off"][-1]), 15, seed)
        if case["op"] == "scan":
            st["out"] = torch.empty_like(st["x"])
    elif kind == "barrier":
        st["storage"] = torch.rand(case["wgs"] * 256 * (case["ldst"] + 1), generator=_gen(seed), device=DEV)
    elif kind == "semaphore":
        st["storage"] = torch.rand(256 * (case["ldst"] + 1), generator=_gen(seed), device=DEV)
        st["handle"] = st["arena"].sem_create(case["sem"], case["sem"], case["capacity"])
    else:
        import hsync.graph as G
        n, row, u, v, w = _graph_parts(case, seed)
        host = [None if t is None else t.to(torch.int32).cpu().numpy().view(np.uint32) for t in (row, v, w)]
        st["srcs"] = _sources(case, row, seed)
        del u, v, w, row
        st["G"], st["g"] = G, G.Graph(*host, transposed=kind in ("bfs", "msbfs", "pagerank"))
        lib = hs.load()
        import ctypes
        nb = ctypes.c_uint64(0)
        g, nsrc = st["g"], len(st["srcs"])
        size = {"bfs": lambda: lib.hs_bfs_work_size(g.n, g.m, ctypes.byref(nb)),
                "sssp": lambda: lib.hs_sssp_work_size(g.n, g.m, ctypes.byref(nb)),
                "pagerank": lambda: lib.hs_pagerank_work_size(g.n, g.m, ctypes.byref(nb)),
                "msbfs": lambda: lib.hs_msbfs_work_size(g.n, g.m, nsrc, ctypes.byref(nb)),
                "mssp": lambda: lib.hs_mssp_work_size(g.n, g.m, nsrc, ctypes.byref(nb))}[kind]
        if size() != 0:
            raise RuntimeError("work size")
        st["work"] = torch.empty(nb.value, dtype=torch.uint8, device=DEV)
        if kind == "pagerank":
            st["out"] = torch.empty(n, dtype=torch.float32, device=DEV)
        elif kind in ("bfs", "sssp"):
            st["out"] = torch.empty(n, dtype=torch.int32, device=DEV)
        else:
            st["out"] = torch.empty((nsrc, n), dtype=torch.int32, device=DEV)
            st["srcs"] = G.device_sources(st["srcs"])
    torch.cuda.synchronize()
    return st


def run(st):
    case, hs, arena = st["case"], st["hs"], st["arena"]
    kind = case["kind"]
    if kind == "reduce":
        if case["take"]:  # the plain call: the sum as a Python number
            return hs.reduce_i32(arena, st["x"])
        return hs.reduce_i32(arena, st["x"], out=st["out"], partials=st["partials"], sync=False)
    if kind == "scan":
        return hs.scan_u32(arena, st["x"], inclusive=case["inclusive"], out=st["out"], sync=False)
    if kind == "batch":
        if case["op"] == "scan":
            return hs.scan_batch_u32(st["x"], st["off"], inclusive=case["inclusive"], out=st["out"], sync=False)
        return hs.reduce_batch_i32(st["x"], st["off"], sync=False)
    if kind == "barrier":
        hs.barrier_bench(arena, "xcd", st["storage"], case["wgs"], 256, case["ldst"], case["episodes"], check=False, sync=False)
        return st["storage"]
    if kind == "semaphore":
        hs.sem_bench(arena, case["sem"], st["handle"], st["storage"], case["wgs"], 256, case["ldst"], case["iters"], 10, sync=False)
        return st["storage"]
    G, g = st["G"], st["g"]
    if kind == "bfs":
        return G.bfs(arena, g, st["srcs"][0], level=st["out"], work=st["work"], sync=False)[0]
    if kind == "sssp":
        return G.sssp(arena, g, st["srcs"][0], delta=case["delta"], dist=st["out"], work=st["work"], sync=False)[0]
    if kind == "msbfs":
        return G.msbfs(arena, g, st["srcs"], levels=st["out"], work=st["work"], sync=False)
    if kind == "mssp":
        return G.mssp(arena, g, st["srcs"], dist=st["out"], work=st["work"], sync=False)[0]
    return G.pagerank(arena, g, alpha=ALPHA, tol=TOL, rank=st["out"], work=st["work"], sync=False)[0]


def work(case):
    kind = case["kind"]
    if kind == "reduce":
        return {"bytes": 4 * case["n"], "flops": case["n"]}
    if kind == "scan":
        return {"bytes": 8 * case["n"], "flops": case["n"]}
    if kind == "batch":
        n = _total(case)
        return {"bytes": (8 if case["op"] == "scan" else 4) * n + 12 * case["nseg"], "flops": n}
    if kind == "barrier":
        # every thread reads and writes its lines once an episode
        return {"bytes": 8 * case["wgs"] * 256 * case["ldst"] * case["episodes"], "flops": 0}
    if kind == "semaphore":
        return {"bytes": 4 * 256 * case["ldst"] * case["wgs"] * case["iters"], "flops": 0}
    if case["graph"] == "mesh":
        n, m = case["h"] * case["w"], int(3.5 * case["h"] * case["w"])
    else:
        n, m = case["n"], case["n"] * case["ef"]
    nsrc = case.get("nsrc", 1)
    if kind in ("bfs", "msbfs"):
        return {"bytes": 4 * n + 4 * m + 4 * n * nsrc, "flops": 0}
    if kind in ("sssp", "mssp"):
        return {"bytes": 4 * n + 8 * m + 4 * n * nsrc, "flops": m * nsrc}
    # about 18 iterations to the tolerance, each over the in-edges and the vertex state
    return {"bytes": 18 * (4 * m + 16 * n), "flops": 18 * 2 * m}


# ---------------------------------------------------------------------------
# the same results from plain torch


def _as_i32(t):
    """The low 32 bits of 64-bit integers."""
    return (((t + 2**31) & 0xFFFFFFFF) - 2**31).to(torch.int32)


def _sum_batch(x, off):
    ends = torch.cat([torch.zeros(1, dtype=torch.int64, device=DEV), torch.cumsum(x, 0, dtype=torch.int64)])
    at = torch.from_numpy(off.astype(np.int64)).to(DEV)
    return ends, at


def _paths(n, u, v, w, srcs):
    """Distances by rounds of relaxation over all edges until nothing changes."""
    out = torch.empty((len(srcs), n), dtype=torch.int32, device=DEV)
    w32 = w.to(torch.int32)
    for k, s in enumerate(srcs):
        d = torch.full((n,), INF, dtype=torch.int32, device=DEV)
        d[s] = 0
        while True:
            du = d[u]
            cand = torch.where(du == INF, du, du + w32)
            new = d.scatter_reduce(0, v, cand, "amin")
            if torch.equal(new, d):
                break
            d = new
        out[k] = d
    return out


def _levels(n, u, v, srcs):
    """Levels of up to 64 searches, a level at a time for all of them."""
    out = torch.full((len(srcs), n), INF, dtype=torch.int32, device=DEV)
    for k, s in enumerate(srcs):
        out[k, s] = 0
        front = torch.zeros(n, dtype=torch.bool, device=DEV)
        front[s] = True
        level = 0
        while True:
            level += 1
            to = v[front[u]]
            front = torch.zeros(n, dtype=torch.bool, device=DEV)
            front[to] = True
            front &= out[k] == INF
            if not bool(front.any()):
                break
            out[k][front] = level
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "reduce":
        s = int(_values(case["n"], case["hi"], seed).sum(dtype=torch.int64))
        s = (s + 2**31) % 2**32 - 2**31
        return s if case["take"] else torch.tensor([s], dtype=torch.int32, device=DEV)
    if kind == "scan":
        x = _values(case["n"], case["hi"], seed)
        s = torch.cumsum(x, 0, dtype=torch.int64)
        return _as_i32(s if case["inclusive"] else s - x)
    if kind == "batch":
        off = _offsets(case, seed)
        x = _values(int(off[-1]), 15, seed)
        ends, at = _sum_batch(x, off)
        if case["op"] == "reduce":
            return _as_i32(ends[at[1:]] - ends[at[:-1]])
        s = ends[1:] if case["inclusive"] else ends[:-1]
        return _as_i32(s - torch.repeat_interleave(ends[at[:-1]], at[1:] - at[:-1]))
    if kind == "barrier":
        # each episode shifts every segment by one line: its first `episodes` lines end as line 0
        L, e = case["ldst"], case["episodes"]
        s = torch.rand(case["wgs"] * 256 * (L + 1), generator=_gen(seed), device=DEV).view(-1, L + 1, 16)
        at = (torch.arange(L + 1, device=DEV) - e).clamp(min=0)
        return s[:, at].reshape(-1)
    if kind == "semaphore":
        L, e = case["ldst"], -(-case["wgs"] // 10) * case["iters"]
        s = torch.rand(256 * (L + 1), generator=_gen(seed), device=DEV).view(-1, L + 1, 16)
        at = (torch.arange(L + 1, device=DEV) - e).clamp(min=0)
        return s[:, at].reshape(-1)
    n, row, u, v, w = _graph_parts(case, seed)
    if kind == "pagerank":
        a = float(np.float32(ALPHA))
        deg = (row[1:] - row[:-1]).double()
        x = torch.full((n,), 1.0 / n, dtype=torch.float64, device=DEV)
        while True:
            c = torch.where(deg > 0, x / deg.clamp(min=1), torch.zeros_like(x))
            base = (1.0 - a) / n + a * float(x[deg == 0].sum()) / n
            y = torch.zeros(n, dtype=torch.float64, device=DEV).index_add_(0, v, c[u]) * a + base
            change = float((y - x).abs().sum())
            x = y
            if change < float(np.float32(TOL)):
                return x
    srcs = _sources(case, row, seed)
    if kind in ("bfs", "msbfs"):
        out = _levels(n, u, v, srcs)
    elif kind == "mssp" and len(srcs) * u.numel() > 4e8:
        return None  # minutes of relaxation rounds
    else:
        out = _paths(n, u, v, w, srcs)
    return out[0] if kind in ("bfs", "sssp") else out
