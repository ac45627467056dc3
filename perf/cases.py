"""The framework's work as a set of measurable cases.

Each case is one solve through the C ABI that the library's hosts call
(include/gdb_amd.h, here over the ctypes binding), with the launch shape left
to the tuning table (wgs = 0) and the tuned variant, as bench.py, the
command-line tools and the integration notes run it.  Graphs, priorities and
outputs are device arrays, as the C ABI takes them; a solve returns when it is
done, so a pass needs no further synchronisation.

Graph families and sizes are those of the repository's own benchmark,
autotuner and full-size tests: R-MAT (0.57, 0.19, 0.19) with edge factor 16,
4-neighbour grids with 5% of the edges removed, and G(n, p) of average degree
8, all as sorted int32 CSR without self-loops or duplicate edges.  They are
generated on the device from the seed.

  listed case        what it stands for in use
  color_rmat10       the smallest solve: one launch, discovery, ~70 rounds of
                     barriers on 1024 vertices (latency)
  color_rmat14       Pannotia colouring of a skewed graph, a few hundred
                     rounds with little work each (barrier-bound)
  mis_rmat22         Pannotia MIS on the largest graph in use (128 M edges):
                     few rounds, random gathers
  bc_rmat22_s16      Pannotia betweenness of the same graph, 16 sources, the
                     undirected case (the CSR is its own transpose)
  bc_directed_s8     betweenness of a directed graph with its transpose, the
                     forward and backward sweep walking different arrays
  bfs_rmat20         Lonestar worklist BFS, the shallow skewed graph: a
                     handful of wide iterations
  sssp_rmat18        Lonestar worklist SSSP on the same family
  sssp_grid1024      Lonestar worklist SSSP on a road-like graph: thousands
                     of short iterations
  sssp_pull_rmat16   Pannotia pull Bellman-Ford over the in-edge CSR of a
                     directed graph
  mst_rmat18         Lonestar minimum spanning forest
  batch_grid2048     the headline: BFS and SSSP of one large grid side by
                     side in one persistent launch, owner-partitioned ranges
  batch_1024graphs   the batched engine as a server of many small graphs:
                     1024 graphs x (BFS, SSSP, colouring) in one launch

draw() spreads over the same families: the sizes between the smallest and the
largest listed ones, odd sizes, rectangular grids, index-ordered and permuted
priorities, narrow and wide weights, directed and undirected graphs.
"""
import ctypes as C
import math

import numpy as np
import torch

import gpu_discovery_barrier_amd as gdb

EDGE_FACTOR = 16


def listed():
    return [
        {"name": "color_rmat10", "kind": "color", "graph": "rmat", "scale": 10, "order": "index"},
        {"name": "color_rmat14", "kind": "color", "graph": "rmat", "scale": 14, "order": "perm"},
        {"name": "mis_rmat22", "kind": "mis", "graph": "rmat", "scale": 22, "order": "perm"},
        {"name": "bc_rmat22_s16", "kind": "bc", "graph": "rmat", "scale": 22, "sources": 16, "directed": False},
        {"name": "bc_directed_s8", "kind": "bc", "graph": "rmat", "scale": 15, "sources": 8, "directed": True},
        {"name": "bfs_rmat20", "kind": "bfs", "graph": "rmat", "scale": 20},
        {"name": "sssp_rmat18", "kind": "sssp", "graph": "rmat", "scale": 18, "whi": 100},
        {"name": "sssp_grid1024", "kind": "sssp", "graph": "grid", "rows": 1024, "cols": 1024, "whi": 255},
        {"name": "sssp_pull_rmat16", "kind": "pull", "graph": "rmat", "scale": 16, "directed": True, "whi": 100},
        {"name": "mst_rmat18", "kind": "mst", "graph": "rmat", "scale": 18, "whi": 100},
        {"name": "batch_grid2048", "kind": "pair", "graph": "grid", "rows": 2048, "cols": 2048, "whi": 255,
         "delta": 12288},
        {"name": "batch_1024graphs", "kind": "many", "graphs": 1024, "whi": 100, "delta": 200},
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    def rmat(lo, hi):
        # A vertex count between the powers of two is as common in use as one of them.
        return {"graph": "rmat", "n": log_int(1 << lo, 1 << hi)}

    def grid(lo, hi):
        r = log_int(lo, hi)
        return {"graph": "grid", "rows": r, "cols": max(2, min(hi, int(r * rng.uniform(0.5, 2.0))))}

    def gnp(lo, hi):
        return {"graph": "gnp", "n": log_int(lo, hi)}

    kind = rng.choice(["color", "mis", "bc", "bfs", "sssp", "pull", "mst", "pair", "many"])
    if kind == "color":
        g = rng.choice([rmat(9, 15), grid(24, 400), gnp(500, 60000)])
        return {"kind": kind, **g, "order": rng.choice(["index", "perm"])}
    if kind == "mis":
        return {"kind": kind, **rng.choice([rmat(11, 21), grid(64, 1500), gnp(1000, 500000)]), "order": "perm"}
    if kind == "bc":
        directed = rng.random() < 0.5
        return {"kind": kind, **(rmat(10, 15) if directed else rmat(10, 19)), "sources": rng.randint(3, 16),
                "directed": directed}
    if kind == "bfs":
        return {"kind": kind, **rng.choice([rmat(11, 20), grid(64, 1000), gnp(1000, 500000)])}
    if kind == "sssp":
        return {"kind": kind, **rng.choice([rmat(11, 18), grid(64, 900), gnp(1000, 200000)]),
                "whi": rng.choice([10, 100, 255])}
    if kind == "pull":
        return {"kind": kind, **rng.choice([{**rmat(10, 17), "directed": True}, grid(32, 160), gnp(1000, 100000)]),
                "whi": rng.choice([10, 100, 255])}
    if kind == "mst":
        return {"kind": kind, **rng.choice([rmat(10, 17), grid(64, 1000), gnp(1000, 300000)]),
                "whi": rng.choice([10, 100, 255])}
    if kind == "pair":
        return {"kind": kind, **grid(200, 1800), "whi": rng.choice([100, 255]), "delta": rng.choice([6144, 12288])}
    return {"kind": "many", "graphs": log_int(48, 900), "whi": rng.choice([10, 100]), "delta": rng.choice([100, 200])}


# ---- graphs -----------------------------------------------------------------
def _rng(seed):
    return torch.Generator("cuda").manual_seed(seed)


def _rmat_pairs(n, count, gen):
    """`count` directed R-MAT draws over n vertices (the recursion runs over
    the next power of two; draws outside [0, n) are folded back)."""
    scale = max(1, (n - 1).bit_length())
    src = torch.zeros(count, dtype=torch.int64, device="cuda")
    dst = torch.zeros(count, dtype=torch.int64, device="cuda")
    for _ in range(scale):
        u = torch.rand(count, generator=gen, device="cuda")
        down = u >= 0.76
        right = ((u >= 0.57) & (u < 0.76)) | (u >= 0.95)
        src = src * 2 + down
        dst = dst * 2 + right
    return src % n, dst % n


def _grid_pairs(rows, cols, gen):
    ids = torch.arange(rows * cols, device="cuda").view(rows, cols)
    a = torch.cat([ids[:, :-1].reshape(-1), ids[:-1, :].reshape(-1)])
    b = torch.cat([ids[:, 1:].reshape(-1), ids[1:, :].reshape(-1)])
    keep = torch.rand(a.numel(), generator=gen, device="cuda") >= 0.05
    return a[keep], b[keep]


def _vertices(case):
    if case["graph"] == "grid":
        return case["rows"] * case["cols"]
    return case["n"] if "n" in case else 1 << case["scale"]


def _keys(case, gen):
    """Sorted, unique keys src * n + dst of the graph's directed edges."""
    n = _vertices(case)
    if case["graph"] == "rmat":
        a, b = _rmat_pairs(n, EDGE_FACTOR * n, gen)
    elif case["graph"] == "grid":
        a, b = _grid_pairs(case["rows"], case["cols"], gen)
    else:
        a = torch.randint(0, n, (4 * n,), generator=gen, device="cuda")
        b = torch.randint(0, n, (4 * n,), generator=gen, device="cuda")
    keep = a != b
    a, b = a[keep], b[keep]
    k = a * n + b
    if not case.get("directed"):
        k = torch.cat([k, b * n + a])
    return torch.unique_consecutive(torch.sort(k)[0])


def _offsets(src, n):
    row = torch.zeros(n + 1, dtype=torch.int64, device="cuda")
    row[1:] = torch.cumsum(torch.bincount(src, minlength=n), 0)
    return row.to(torch.int32)


def _weights(a, b, n, seed, whi):
    """A weight in [1, whi] per undirected edge, from a hash of its ends."""
    h = (torch.minimum(a, b) * n + torch.maximum(a, b) + (seed << 24)) * 0x9E3779B97F4A7C1
    h = (h ^ (h >> 29)) * 0xBF58476D1CE4E5B
    h = (h ^ (h >> 32)) & 0x7FFFFFFF
    return (1 + h % whi).to(torch.int32)


def _graph(case, seed, transpose=False):
    """(row, col, w) of the case's graph; with `transpose`, of its in-edges."""
    gen = _rng(seed)
    n = _vertices(case)
    k = _keys(case, gen)
    a, b = k // n, k % n
    if transpose:
        k = torch.sort(b * n + a)[0]
        a, b = k // n, k % n
    w = _weights(a, b, n, seed, case["whi"]) if "whi" in case else None
    return _offsets(a, n), b.to(torch.int32), w


def _priorities(n, order, seed):
    p = torch.arange(n, device="cuda") if order == "index" else torch.randperm(n, generator=_rng(seed + 1), device="cuda")
    return (p.double() / (n + 1)).float()


def _sources(row, count, seed):
    has = torch.nonzero(row[1:] > row[:-1]).view(-1)
    pick = torch.randperm(has.numel(), generator=_rng(seed + 2), device="cuda")[:count]
    return torch.sort(has[pick])[0].to(torch.int32)


def _many_sizes(count):
    """The batch's graph sizes: half G(n, p) with n log-uniform in [256,
    65536], half square grids with a side in [16, 256]; fixed by the count, so
    that another seed gives other edges and weights of the same sizes."""
    r = np.random.default_rng(count)
    gnp = [("gnp", int(math.exp(r.uniform(math.log(256), math.log(65536))))) for _ in range(count - count // 2)]
    return gnp + [("grid", int(r.integers(16, 257))) for _ in range(count // 2)]


# ---- prepare / run ----------------------------------------------------------
class _State:
    """Inputs, outputs and the context of one program."""

    def __init__(self, case):
        self.case = case
        self.lib = gdb.lib()
        self.ctx = gdb.Context()
        self.opts = gdb.Opts.make(wgs=0, variant=gdb.VARIANT_TUNED)
        self.stats = gdb.Stats()


def _task(algo, n, m, row, col, w, out, source=0, values=None, delta=0, owned=0):
    t = gdb.Task()
    t.algo, t.n, t.m, t.source, t.delta, t.owned = algo, n, m, source, delta, owned
    t.row, t.col, t.out = row.data_ptr(), col.data_ptr(), out.data_ptr()
    t.w = w.data_ptr() if w is not None else None
    t.node_value = values.data_ptr() if values is not None else None
    return t


def _prepare_many(s, case, seed):
    gen = _rng(seed)
    sizes = _many_sizes(case["graphs"])
    ns = [n if f == "gnp" else n * n for f, n in sizes]
    # The G(n, p) graphs are drawn together: a disjoint union, split by rows.
    gn = [n for f, n in sizes if f == "gnp"]
    off = torch.tensor(np.concatenate([[0], np.cumsum(gn)]), device="cuda")
    count = torch.tensor([4 * n for n in gn], device="cuda")
    which = torch.repeat_interleave(torch.arange(len(gn), device="cuda"), count)
    span = torch.tensor(gn, device="cuda")[which]
    total = int(off[-1])
    a = (torch.rand(which.numel(), generator=gen, device="cuda", dtype=torch.float64) * span).long() + off[which]
    b = (torch.rand(which.numel(), generator=gen, device="cuda", dtype=torch.float64) * span).long() + off[which]
    keep = a != b
    a, b = a[keep], b[keep]
    k = torch.unique_consecutive(torch.sort(torch.cat([a * total + b, b * total + a]))[0])
    src, dst = k // total, k % total
    rows = _offsets(src, total)
    w = _weights(src, dst, total, seed, case["whi"])
    bounds = rows[off].tolist()
    offs = off.tolist()
    dst = dst.to(torch.int32)
    graphs = []
    for i in range(len(gn)):
        lo, hi = bounds[i], bounds[i + 1]
        graphs.append(((rows[offs[i]:offs[i + 1] + 1] - lo).contiguous(), dst[lo:hi] - offs[i], w[lo:hi].clone()))
    side_of = {}
    for f, side in sizes:
        if f != "grid":
            continue
        if side not in side_of:  # a full grid of a given side has one shape
            n = side * side
            ids = torch.arange(n, device="cuda").view(side, side)
            e = torch.cat([torch.stack([ids[:, :-1].reshape(-1), ids[:, 1:].reshape(-1)], 1),
                           torch.stack([ids[:-1, :].reshape(-1), ids[1:, :].reshape(-1)], 1)])
            k = torch.sort(torch.cat([e[:, 0] * n + e[:, 1], e[:, 1] * n + e[:, 0]]))[0]
            side_of[side] = (k // n, k % n, _offsets(k // n, n), n)
        a, b, row, n = side_of[side]
        graphs.append((row.clone(), b.to(torch.int32), _weights(a, b, n, seed + len(graphs), case["whi"])))
    # One output array; every task writes its own slice (64-entry aligned).
    starts = np.concatenate([[0], np.cumsum([(n + 63) // 64 * 64 for n in ns for _ in range(3)])])
    s.out = torch.zeros(int(starts[-1]), dtype=torch.int32, device="cuda")
    tasks = []
    s.keep = graphs
    s.values = []
    for i, ((row, col, w), n) in enumerate(zip(graphs, ns)):
        nv = _priorities(n, "index", 0)
        s.values.append(nv)
        o = [s.out[int(starts[3 * i + j]):] for j in range(3)]
        m = col.numel()
        tasks.append(_task(gdb.TASK_BFS, n, m, row, col, w, o[0]))
        tasks.append(_task(gdb.TASK_SSSP, n, m, row, col, w, o[1], delta=case["delta"]))
        tasks.append(_task(gdb.TASK_COLOR, n, m, row, col, w, o[2], values=nv))
    s.tasks = (gdb.Task * len(tasks))(*tasks)


def prepare(case, seed):
    s = _State(case)
    kind = case["kind"]
    if kind == "many":
        _prepare_many(s, case, seed)
        torch.cuda.synchronize()
        return s
    n = s.n = _vertices(case)
    if kind == "pull":
        s.row, s.col, s.w = _graph(case, seed, transpose=True)
    else:
        s.row, s.col, s.w = _graph(case, seed)
    s.m = s.col.numel()
    if kind in ("color", "mis"):
        s.values = _priorities(n, case["order"], seed)
        s.out = torch.empty(n, dtype=torch.int32, device="cuda")
    elif kind == "bc":
        s.row_t, s.col_t = (s.row, s.col) if not case["directed"] else _graph(case, seed, transpose=True)[:2]
        s.sources = _sources(s.row, case["sources"], seed)
        s.out = torch.empty(n, dtype=torch.float32, device="cuda")
    elif kind == "mst":
        s.answer = (C.c_ulonglong(0), C.c_int(0), C.c_int(0))
    else:
        # The first vertex that has an edge.
        s.source = int(torch.nonzero(s.row[1:] > s.row[:-1])[0])
        s.out = torch.empty(n, dtype=torch.int32, device="cuda")
    if kind == "pair":
        s.out_s = torch.empty(n, dtype=torch.int32, device="cuda")
        t = [_task(gdb.TASK_BFS, n, s.m, s.row, s.col, s.w, s.out, s.source, owned=1),
             _task(gdb.TASK_SSSP, n, s.m, s.row, s.col, s.w, s.out_s, s.source, delta=case["delta"], owned=1)]
        s.tasks = (gdb.Task * 2)(*t)
    torch.cuda.synchronize()
    return s


def run(s):
    lib, h, o, st, kind = s.lib, s.ctx.h, C.byref(s.opts), C.byref(s.stats), s.case["kind"]
    if kind in ("pair", "many"):
        gdb.check(lib.gdb_batch_solve(h, s.tasks, len(s.tasks), 0, o, st), "gdb_batch_solve")
        return [s.out, s.out_s] if kind == "pair" else s.out
    n, m, row, col = s.n, s.m, s.row.data_ptr(), s.col.data_ptr()
    if kind == "mst":
        wt, ed, cp = s.answer
        gdb.check(lib.gdb_mst(h, n, m, row, col, s.w.data_ptr(), C.byref(wt), C.byref(ed), C.byref(cp), o, st), "gdb_mst")
        return {"weight": wt.value, "edges": ed.value, "components": cp.value}
    out = s.out.data_ptr()
    if kind == "color":
        gdb.check(lib.gdb_color(h, n, m, row, col, s.values.data_ptr(), out, o, st), "gdb_color")
    elif kind == "mis":
        gdb.check(lib.gdb_mis(h, n, m, row, col, s.values.data_ptr(), out, o, st), "gdb_mis")
    elif kind == "bc":
        gdb.check(lib.gdb_bc(h, n, m, row, col, s.row_t.data_ptr(), s.col_t.data_ptr(), s.sources.data_ptr(),
                             s.sources.numel(), out, o, st), "gdb_bc")
    elif kind == "bfs":
        gdb.check(lib.gdb_bfs_worklist(h, n, m, row, col, s.source, out, o, st), "gdb_bfs_worklist")
    elif kind == "sssp":
        gdb.check(lib.gdb_sssp_worklist(h, n, m, row, col, s.w.data_ptr(), s.source, out, o, st), "gdb_sssp_worklist")
    else:
        gdb.check(lib.gdb_sssp_pull(h, n, m, row, col, s.w.data_ptr(), s.source, out, o, st), "gdb_sssp_pull")
    return s.out


# ---- work / exact -----------------------------------------------------------
def _edges(case):
    """Expected directed edges (R-MAT loses more to duplicates when small)."""
    n = _vertices(case)
    if case["graph"] == "grid":
        return int(1.9 * (2 * n - case["rows"] - case["cols"]))
    if case["graph"] == "gnp":
        return 8 * n
    kept = min(0.97, 0.81 + 0.018 * (math.log2(n) - 14))
    return int((1 if case.get("directed") else 2) * EDGE_FACTOR * n * kept)


def work(case):
    """Row offsets, columns (and weights) read once, outputs written once; one
    add and one compare per edge that a solve has to look at."""
    kind = case["kind"]
    if kind == "many":
        b = f = 0
        for fam, n in _many_sizes(case["graphs"]):
            m = 8 * n if fam == "gnp" else 4 * n * (n - 1)
            n = n if fam == "gnp" else n * n
            b += 3 * (4 * n + 4 * m + 4 * n) + 4 * m + 4 * n
            f += 2 * 3 * m
        return {"bytes": b, "flops": f}
    n, m = _vertices(case), _edges(case)
    graph, passes = 4 * (n + 1) + 4 * m, 1
    if kind in ("color", "mis"):
        b = graph + 4 * n + 4 * n
    elif kind == "bc":
        b = graph * (2 if case["directed"] else 1) + 4 * n
        passes = 2 * case["sources"]
    elif kind == "bfs":
        b = graph + 4 * n
    elif kind == "pair":
        b = 2 * graph + 4 * m + 8 * n
        passes = 2
    elif kind == "mst":
        b = graph + 4 * m
    else:
        b = graph + 4 * m + 4 * n
    return {"bytes": b, "flops": 2 * m * passes}


def exact(case, seed):
    """Betweenness in 64 bits: Brandes, one sum over each row's edges per
    level; every other case returns whole numbers."""
    if case["kind"] != "bc":
        return None
    n = _vertices(case)

    def row_sums(row, col):
        row, col = row.long(), col.long()
        return lambda x: torch.segment_reduce(x[col], "sum", offsets=row, initial=0.0)

    row, col, _ = _graph(case, seed)
    over_out = row_sums(row, col)
    over_in = row_sums(*_graph(case, seed, transpose=True)[:2]) if case["directed"] else over_out
    bc = torch.zeros(n, dtype=torch.float64, device="cuda")
    for s in _sources(row, case["sources"], seed).tolist():
        level = torch.full((n,), -1, dtype=torch.int32, device="cuda")
        sigma = torch.zeros(n, dtype=torch.float64, device="cuda")
        level[s], sigma[s], depth = 0, 1.0, 0
        while True:
            paths = over_in(torch.where(level == depth, sigma, 0.0))
            new = (level == -1) & (paths > 0)
            if not bool(new.any()):
                break
            depth += 1
            level[new] = depth
            sigma = torch.where(new, paths, sigma)
        delta = torch.zeros(n, dtype=torch.float64, device="cuda")
        for d in range(depth - 1, -1, -1):
            share = torch.where(level == d + 1, (1.0 + delta) / sigma.clamp(min=1.0), 0.0)
            delta = torch.where(level == d, sigma * over_out(share), delta)
        delta[s] = 0.0
        bc += delta
    return bc
