"""Performance cases: the work that users of the engine have it do, through the
Python entry points (``kites_amd.DeviceGraph``), from a graph resident in HBM
to the vertex values in the caller's arrays.

Graphs are drawn on the GPU from the seed alone: R-MAT (a = .57, b = c = .19),
the 4-neighbour grid and disjoint unions of uneven R-MAT graphs, which are the
families that the benchmark, the tests and the scheduler's training use.

``listed()`` gives the named cases, ``draw(rng)`` one more of the same ranges,
``prepare(case, seed)`` the resident graph and the sources, ``run(state)`` one
pass, ``work(case)`` what a pass cannot do without and ``exact(case, seed)``
the 64-bit values of the one path that computes in floating point.
"""
import math

import numpy as np
import torch

import kites_amd as K
from kites_amd import scheduler

TOL = 1e-4
DAMPING = 0.85


def listed():
    return [
        # the smallest call: one query on a graph of Wiki-Vote's size (latency)
        {"name": "sssp-7k", "kind": "sssp", "n": 7115, "ef": 15, "wmax": 64, "sched": "auto"},
        # ordinary single-source queries with the default options
        {"name": "bfs-1m", "kind": "bfs", "n": 1 << 20, "ef": 16, "wmax": 1, "sched": "auto"},
        # a max-min reduction (not the native-min path), ragged vertex count
        {"name": "widest-200k", "kind": "widest", "n": 200003, "ef": 16, "wmax": 255,
         "sched": "auto"},
        # the headline workload: R-MAT scale 22, learned schedule
        {"name": "sssp-4m-learned", "kind": "sssp", "n": 1 << 22, "ef": 16, "wmax": 255,
         "sched": "learned"},
        # connected components of an undirected graph, ragged vertex count
        {"name": "cc-777k", "kind": "cc", "n": 777777, "ef": 8, "wmax": 1, "sched": "learned"},
        # high-diameter graphs: thousands of iterations with small frontiers
        {"name": "bfs-grid-2048", "kind": "grid_bfs", "rows": 2048, "cols": 2048, "wmax": 100},
        {"name": "sssp-grid-1500x1111", "kind": "grid_sssp", "rows": 1500, "cols": 1111,
         "wmax": 100, "delta": 800},
        # many sources of one graph in one run, every column returned
        {"name": "batch64-1m", "kind": "batch", "n": 1 << 20, "ef": 16, "wmax": 255, "k": 64},
        {"name": "bfs256-256k", "kind": "bfs256", "n": 1 << 18, "ef": 16, "wmax": 1, "k": 256},
        # 200 independent graphs of uneven sizes in one run
        {"name": "graphs-200", "kind": "graphs", "count": 200, "lo": 10, "hi": 16, "wmax": 255},
        # float PageRank, ordered sums
        {"name": "pagerank-1m", "kind": "pagerank", "n": 1 << 20, "ef": 16, "wmax": 1},
        # an edge list in host memory to BFS levels: graph build and one query
        {"name": "build-bfs-1m", "kind": "build", "n": 1000003, "ef": 16, "wmax": 255},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["sssp", "bfs", "widest", "cc", "grid_bfs", "grid_sssp", "batch", "bfs256",
                       "graphs", "pagerank", "build"])
    c = {"kind": kind, "wmax": rng.choice([1, 64, 100, 255])}
    if kind in ("grid_bfs", "grid_sssp"):
        c["rows"], c["cols"] = _log_int(rng, 60, 2000), _log_int(rng, 60, 2000)
        if kind == "grid_sssp":
            c["rows"], c["cols"] = _log_int(rng, 60, 1400), _log_int(rng, 60, 1100)
            c["wmax"] = rng.choice([64, 100, 255])
            c["delta"] = 8 * c["wmax"]
    elif kind == "graphs":
        c["count"], c["lo"] = rng.randint(3, 150), 10
        c["hi"] = rng.randint(11, 16)
    else:
        most = {"sssp": 4000000, "bfs": 4000000, "widest": 1000000, "cc": 1000000,
                "batch": 1000000, "bfs256": 250000, "pagerank": 1000000, "build": 1000000}[kind]
        c["n"] = _log_int(rng, 1000, most)
        c["ef"] = rng.randint(4, 8 if kind == "cc" else 16)
        if kind in ("sssp", "bfs", "cc"):
            c["sched"] = rng.choice(["auto", "learned"])
        elif kind == "widest":
            c["sched"] = "auto"
        elif kind == "batch":
            c["k"] = rng.randint(1, 64)
        elif kind == "bfs256":
            c["k"] = rng.randint(1, 256)
    return c


# ---- inputs ------------------------------------------------------------------

def _rmat(gen, n, draws):
    """`draws` R-MAT endpoints below n, as drawn (self-loops and repeats
    included)."""
    scale = max(1, (n - 1).bit_length())
    dev = gen.device
    got, have = [], 0
    while have < draws:
        k = draws if not have else max(1024, 2 * (draws - have))
        s = torch.zeros(k, dtype=torch.int32, device=dev)
        d = torch.zeros(k, dtype=torch.int32, device=dev)
        for _ in range(scale):
            r = torch.rand(k, generator=gen, device=dev)
            down = r >= 0.76                          # quadrants c, d
            right = (r >= 0.95) | ((r >= 0.57) & ~down)   # quadrants b, d
            s = 2 * s + down
            d = 2 * d + right
        keep = (s < n) & (d < n)
        got.append((s[keep], d[keep]))
        have += got[-1][0].numel()
    s, d = (torch.cat([g[i] for g in got])[:draws].to(torch.int32) for i in (0, 1))
    return s, d


def _weights(gen, m, wmax):
    return torch.randint(1, wmax + 1, (m,), generator=gen, device=gen.device, dtype=torch.int32)


def _grid(gen, rows, cols, wmax):
    idx = torch.arange(rows * cols, dtype=torch.int32, device=gen.device).view(rows, cols)
    a, b, u, v = (x.reshape(-1) for x in (idx[:, :-1], idx[:, 1:], idx[:-1], idx[1:]))
    s, d = torch.cat([a, b, u, v]), torch.cat([b, a, v, u])
    return s, d, _weights(gen, s.numel(), wmax)


def _edges(case, seed):
    """(n, src, dst, w, sources) of a case, tensors on the GPU."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    kind = case["kind"]
    if kind in ("grid_bfs", "grid_sssp"):
        rows, cols = case["rows"], case["cols"]
        s, d, w = _grid(gen, rows, cols, case["wmax"])
        r, c = np.random.default_rng(seed).integers(0, [1 + rows // 32, 1 + cols // 32])
        return rows * cols, s, d, w, [int(r) * cols + int(c)]   # near a corner
    if kind == "graphs":
        pick = np.random.default_rng(case["count"])   # the sizes are the case's
        off, ss, dd, sources = 0, [], [], []
        for _ in range(case["count"]):
            n = 1 << int(pick.integers(case["lo"], case["hi"] + 1))
            s, d = _rmat(gen, n, int(pick.integers(8, 33)) * n)
            sources.append(off + torch.bincount(s, minlength=n).argmax())
            ss.append(s + off)
            dd.append(d + off)
            off += n
        s, d = torch.cat(ss), torch.cat(dd)
        return off, s, d, _weights(gen, s.numel(), case["wmax"]), torch.stack(sources).tolist()
    n = case["n"]
    s, d = _rmat(gen, n, case["ef"] * n)
    if kind == "cc":
        s, d = torch.cat([s, d]), torch.cat([d, s])
    deg = torch.bincount(s, minlength=n)
    if kind in ("batch", "bfs256"):
        # uniform among the vertices with out-edges
        cand = torch.nonzero(deg).flatten()
        at = torch.randperm(cand.numel(), generator=gen, device=gen.device)
        sources = cand[at.repeat(-(-case["k"] // at.numel()))[:case["k"]]].tolist()
    else:
        sources = [int(deg.argmax())]
    return n, s, d, _weights(gen, s.numel(), case["wmax"]), sources


def prepare(case, seed):
    n, s, d, w, sources = _edges(case, seed)
    s, d, w = (x.cpu().numpy().view(np.uint32) for x in (s, d, w))
    st = {"kind": case["kind"], "sources": np.array(sources, np.uint32), "case": case}
    if case["kind"] == "build":
        st.update(n=n, edges=(s, d, w))
        return st
    st["g"], _ = K.DeviceGraph.from_edges(n, s, d, w, dedup=True)
    if case.get("sched") == "learned" or case["kind"] == "graphs":
        st["g"].set_model(scheduler.load_model())
    return st


# ---- one pass ----------------------------------------------------------------

def run(st):
    kind, src = st["kind"], st["sources"]
    if kind == "build":
        g, _ = K.DeviceGraph.from_edges(st["n"], *st["edges"], dedup=True)
        out, _ = g.solve("bfs", int(src[0]))
        g.close()
    elif kind in ("sssp", "bfs", "widest", "cc"):
        out, _ = st["g"].solve(kind, int(src[0]), sched=st["case"]["sched"])
    elif kind == "grid_bfs":
        out, _ = st["g"].solve("bfs", int(src[0]))
    elif kind == "grid_sssp":
        out, _ = st["g"].solve("sssp", int(src[0]), delta=st["case"]["delta"])
    elif kind == "batch":
        out, _ = st["g"].batch("sssp", src)
    elif kind == "bfs256":
        out, _ = st["g"].bfs256(src)
    elif kind == "graphs":
        st["g"].init_sources("sssp", src)
        st["g"].run("sssp", sched="learned")
        out = st["g"].values()
    else:
        out, _ = st["g"].pagerank(damping=DAMPING, tol=TOL)
        return out
    return out.view(np.int32)


def work(case):
    """Each input array read once, each output written once: the offsets, the
    column indices (and the weights where the path uses them) and the values;
    one operation per edge and column."""
    kind = case["kind"]
    if kind in ("grid_bfs", "grid_sssp"):
        n = case["rows"] * case["cols"]
        m = 4 * n - 2 * (case["rows"] + case["cols"])
    elif kind == "graphs":
        sizes = [1 << s for s in range(case["lo"], case["hi"] + 1)]
        n = case["count"] * sum(sizes) // len(sizes)
        m = 20 * n
    else:
        n, m = case["n"], case["n"] * case["ef"] * (2 if kind == "cc" else 1)
    cols = case.get("k", 1)
    weighted = kind in ("sssp", "widest", "grid_sssp", "batch", "graphs", "build")
    edge = 12 if kind == "build" else 8 if weighted else 4
    return {"bytes": edge * m + 4 * (n + 1) + 4 * n * cols, "flops": m * cols}


def exact(case, seed):
    """PageRank in 64 bits: Jacobi sweeps over the active vertices, a vertex
    moving while its value changes by more than the tolerance.  The other
    paths compute whole numbers."""
    if case["kind"] != "pagerank":
        return None
    n, s, d, _, _ = _edges(case, seed)
    key = torch.unique(d.long() * n + s.long())
    d, s = key // n, key % n
    keep = s != d
    s, d = s[keep], d[keep]
    npad = -(-n // 128) * 128
    share = DAMPING / torch.bincount(s, minlength=npad).double()[s]
    end = torch.bincount(d, minlength=npad).cumsum(0)   # the edges are in order of d
    zero = torch.zeros(1, dtype=torch.float64, device=s.device)
    value = torch.ones(npad, dtype=torch.float64, device=s.device)
    active = torch.ones(npad, dtype=torch.bool, device=s.device)
    while True:
        upto = torch.cat([zero, (value[s] * share).cumsum(0)])[end]
        new = 1.0 - DAMPING + torch.diff(upto, prepend=zero)
        moved = active & ((new - value).abs() > TOL)
        if not bool(moved.any()):
            return value.cpu().numpy()
        value = torch.where(moved, new, value)
        active = torch.zeros_like(active)
        active[d[moved[s]]] = True
