"""Parity of MIS, pull SSSP, BC and the worklist BFS / SSSP with the oracle,
for every schedule, through the C ABI.

Bars: MIS sets, SSSP distances and BFS levels bit-exact; BC (FP32) within
1e-4 relative of the FP64 Brandes oracle entry by entry, |got - want| <=
1e-4 * |want|, with an absolute floor of 1e-6 that only matters for entries
that are (near) zero."""
import ctypes as C

import numpy as np
import pytest

import gpu_discovery_barrier_amd as gdb
import oracle
from conftest import csr_from_edges, grid_csr, load_fixtures, values_of

pytestmark = pytest.mark.gpu
FX = load_fixtures()

SCHEDS = [
    dict(schedule=gdb.SCHED_PERSISTENT, variant=gdb.VARIANT_PLAIN),
    dict(schedule=gdb.SCHED_PERSISTENT, variant=gdb.VARIANT_TUNED),
    dict(schedule=gdb.SCHED_RELAUNCH, variant=gdb.VARIANT_PLAIN),
    dict(schedule=gdb.SCHED_RELAUNCH, variant=gdb.VARIANT_PLAIN, relaunch_check=5),
]
SID = lambda s: "-".join(map(str, s.values()))
BC_RTOL = 1e-4
BC_ATOL = 1e-6


@pytest.fixture(scope="module")
def ctx():
    c = gdb.Context()
    yield c
    c.close()


def dev(row, col, w=None):
    w = np.ones_like(col) if w is None else w
    return gdb.DeviceCSR(gdb.CSR(row.size - 1, row, col, w))


def bc_close(got, want):
    """Per-entry relative bar: |got - want| <= 1e-4 |want|, floor 1e-6."""
    want = np.asarray(want, np.float64)
    err = np.abs(got.astype(np.float64) - want)
    ok = err <= np.maximum(BC_RTOL * np.abs(want), BC_ATOL)
    assert ok.all(), (np.flatnonzero(~ok)[:10], got[~ok][:10], want[~ok][:10])
    nz = want != 0
    return float((err[nz] / np.abs(want[nz])).max()) if nz.any() else 0.0


# ---------------------------------------------------------------- MIS
@pytest.mark.parametrize("sched", SCHEDS, ids=SID)
@pytest.mark.parametrize("fx", FX["mis"], ids=lambda f: f["name"])
def test_mis_fixtures(ctx, fx, sched):
    row, col, _ = csr_from_edges(fx["n"], fx["edges"])
    got, _ = gdb.mis(ctx, dev(row, col), gdb.DeviceBuffer.from_numpy(values_of(fx)),
                     gdb.Opts.make(wgs=64, **sched))
    assert got.tolist() == fx["s"]


@pytest.mark.parametrize("sched", SCHEDS, ids=SID)
@pytest.mark.parametrize("vals", ["id", "perm"])
def test_mis_rmat(ctx, sched, vals):
    g = gdb.gen_rmat(15, 16, seed=3)
    nv = gdb.pannotia_values(g.n) if vals == "id" else \
        gdb.permutation(g.n, 3).astype(np.float32) / np.float32(g.n + 1)
    want, rounds = oracle.mis_ref(g.row, g.col, nv)
    got, st = gdb.mis(ctx, dev(g.row, g.col), gdb.DeviceBuffer.from_numpy(nv), gdb.Opts.make(**sched))
    print(vals, SID(sched), st.as_dict())
    assert (got == want).all()
    assert st.rounds == rounds


@pytest.mark.parametrize("extra", [0, 1, 31])
@pytest.mark.parametrize("deg", [1, 15, 16, 17, 79, 80, 81, 300])
def test_mis_one_deciding_edge(ctx, deg, extra):
    """Hubs of one degree, each with its only smaller neighbour at another place
    of its row; the leaves of neighbouring hubs are joined, for further rounds."""
    spots = sorted({0, 3, 4, deg // 2, 14, 15, 16, 17, deg - 1} & set(range(deg)))
    hubs = len(spots)
    n = hubs * (deg + 1) + extra
    nv = np.empty(n, np.float32)
    nv[:hubs] = 2.0 + np.arange(hubs)
    nv[hubs:] = 100.0 + gdb.permutation(n - hubs, deg + 1).astype(np.float32)
    edges = []
    for h, p in enumerate(spots):
        leaves = hubs + h * deg + np.arange(deg)
        nv[leaves[p]] = 1.0 + h / 100
        edges += [(h, int(u)) for u in leaves]
        edges += [(int(u), hubs + (int(u) - hubs + deg) % (hubs * deg)) for u in leaves if hubs > 1]
    row, col, _ = csr_from_edges(n, edges)
    want, rounds = oracle.mis_ref(row, col, nv)
    got, st = gdb.mis(ctx, dev(row, col), gdb.DeviceBuffer.from_numpy(nv), gdb.Opts.make())
    assert (got == want).all() and st.rounds == rounds


@pytest.mark.parametrize("n", [1, 255, 256, 257, 1025])
@pytest.mark.parametrize("wgs,groups", [(64, 1), (256, 3), (0, 0)])
def test_bfs_sweep(ctx, n, wgs, groups):
    """Iterations of more than 100000 edges, by one row and by many, among small
    ones; sizes around what one trip of the sweep covers."""
    rng = np.random.default_rng(n)
    chain = np.arange(n - 1)
    mid = n // 2
    src = np.concatenate([np.zeros(120000, np.int64), chain, rng.integers(0, max(1, mid), 130000)])
    dst = np.concatenate([rng.integers(0, max(1, mid), 120000), chain + 1, rng.integers(0, n - n // 4, 130000)])
    order = np.argsort(src, kind="stable")
    row = np.zeros(n + 1, np.int32)
    row[1:] = np.cumsum(np.bincount(src, minlength=n))
    col = dst[order].astype(np.int32)
    for source in {0, n - 1}:
        want, rounds = oracle.bfs_worklist_ref(row, col, source)
        got, st = gdb.bfs_worklist(ctx, dev(row, col), source, gdb.Opts.make(wgs=wgs, groups=groups))
        assert (got == want).all() and st.rounds == rounds


# ---------------------------------------------------------------- pull SSSP
@pytest.mark.parametrize("sched", SCHEDS, ids=SID)
@pytest.mark.parametrize("fx", FX["sssp_pull"], ids=lambda f: f["name"])
def test_sssp_pull_fixtures(ctx, fx, sched):
    row, col, w = csr_from_edges(fx["n"], fx["edges"], fx["w"])
    got, _ = gdb.sssp_pull(ctx, dev(row, col, w), 0, gdb.Opts.make(wgs=64, **sched))
    assert got.tolist() == fx["dist"]


@pytest.mark.parametrize("sched", SCHEDS, ids=SID)
def test_sssp_pull_rmat(ctx, sched):
    g = gdb.gen_rmat(14, 16, seed=5, wlo=1, whi=100)
    gt = g.transpose()
    want, rounds = oracle.sssp_pull_ref(gt.row, gt.col, gt.w, 0)
    got, st = gdb.sssp_pull(ctx, dev(gt.row, gt.col, gt.w), 0, gdb.Opts.make(**sched))
    print(SID(sched), st.as_dict())
    assert (got == want).all()
    assert st.rounds == rounds


@pytest.mark.parametrize("sched", SCHEDS[:2], ids=SID)
def test_sssp_pull_round_cap_grid(ctx, sched):
    # 30x3 grid: hop diameter 31 > n-1?  No: n = 90; use a path so the cap binds.
    n = 40
    row, col, w = csr_from_edges(n, [(i, i + 1) for i in range(n - 1)], [3] * (n - 1))
    want, rounds = oracle.sssp_pull_ref(row, col, w, 0)
    got, st = gdb.sssp_pull(ctx, dev(row, col, w), 0, gdb.Opts.make(wgs=64, **sched))
    assert (got == want).all() and want[-1] == oracle.PANNOTIA_INF and st.rounds == rounds


# ---------------------------------------------------------------- BC
@pytest.mark.parametrize("sched", SCHEDS[:3], ids=SID)
@pytest.mark.parametrize("fx", FX["bc"], ids=lambda f: f["name"])
def test_bc_fixtures(ctx, fx, sched):
    row, col, _ = csr_from_edges(fx["n"], fx["edges"])
    g = dev(row, col)
    got, _ = gdb.bc(ctx, g, g, np.array(fx["sources"], np.int32), gdb.Opts.make(wgs=64, **sched))
    bc_close(got, fx["bc"])


@pytest.mark.parametrize("sched", SCHEDS[:3], ids=SID)
def test_bc_rmat(ctx, sched):
    g = gdb.gen_rmat(13, 16, seed=3)
    src = gdb.permutation(g.n, 3)[:16]
    want = oracle.bc_brandes_tb(g.row, g.col, src)
    d = dev(g.row, g.col)
    got, st = gdb.bc(ctx, d, d, src, gdb.Opts.make(**sched))
    print(SID(sched), st.as_dict())
    bc_close(got, want)


@pytest.mark.parametrize("sched", SCHEDS, ids=SID)
def test_bc_rmat15_64_sources(ctx, sched):
    # R-MAT 15 with 64 sources: eight full eight-source sweeps on the tuned
    # schedule, 64 single-source passes on the others.
    g = gdb.gen_rmat(15, 16, seed=3)
    deg = np.diff(g.row)
    src = gdb.permutation(g.n, 15)
    src = src[deg[src] > 0][:64].astype(np.int32)
    want = oracle.bc_brandes_tb(g.row, g.col, src)
    d = dev(g.row, g.col)
    got, st = gdb.bc(ctx, d, d, src, gdb.Opts.make(**sched))
    rel = bc_close(got, want)
    print(SID(sched), st.as_dict(), "max rel", rel)
    assert (want > 0).sum() > g.n // 4  # most vertices carry a nonzero centrality


def test_bc_close_rejects_small_entries_off():
    # The bar must catch a wrong small entry: zeroing the smallest nonzero
    # oracle value fails it, as does a 2e-4 relative error on one entry.
    g = gdb.gen_rmat(10, 16, seed=3)
    src = gdb.permutation(g.n, 3)[:8]
    want = oracle.bc_brandes_tb(g.row, g.col, src)
    k = int(np.argmin(np.where(want > 0, want, np.inf)))
    bad = want.astype(np.float32).copy()
    bad[k] = 0
    with pytest.raises(AssertionError):
        bc_close(bad, want)
    j = int(np.argmax(want))
    bad = want.astype(np.float32).copy()
    bad[j] *= 1 + 2e-4
    with pytest.raises(AssertionError):
        bc_close(bad, want)


def test_bc_sweeps_partial_batch_and_repeated_sources(ctx):
    # Eight sources per sweep: 13 sources leave a partial last sweep, and a
    # source listed twice (within one sweep and across two) is counted twice,
    # as the single-source kernels and the oracle count it.
    g = gdb.gen_rmat(12, 16, seed=21)
    p = gdb.permutation(g.n, 21)
    src = np.concatenate([p[:5], p[:1], p[5:11], p[1:2]]).astype(np.int32)  # repeats in and across sweeps
    d = dev(g.row, g.col)
    want = oracle.bc_brandes_tb(g.row, g.col, src)
    for sched in SCHEDS[:3]:
        got, _ = gdb.bc(ctx, d, d, src, gdb.Opts.make(**sched))
        bc_close(got, want)


@pytest.mark.parametrize("n", [1023, 1024, 1030])
@pytest.mark.parametrize("directed", [False, True])
@pytest.mark.parametrize("wgs,groups", [(64, 4), (256, 3), (0, 0)])
def test_bc_step_with_many_edges(ctx, n, directed, wgs, groups):
    """A random core of 130 edges per vertex and a path of seven: steps that sweep
    between steps that claim, two batches of sources, around a trip's vertices."""
    rng = np.random.default_rng(n)
    core = n - 7
    a = np.concatenate([rng.integers(0, core, 130 * core), np.arange(core - 1, n - 1)])
    b = np.concatenate([rng.integers(0, core, 130 * core), np.arange(core, n)])
    key = a * n + b
    key = np.unique(key if directed else np.concatenate([key, b * n + a]))
    key = key[key // n != key % n]

    def csr(k):
        row = np.zeros(n + 1, np.int32)
        row[1:] = np.cumsum(np.bincount(k // n, minlength=n))
        return row, (k % n).astype(np.int32)

    row, col = csr(key)
    assert len(col) > 120000
    src = np.concatenate([[n - 1], rng.permutation(n)[:10]]).astype(np.int32)
    want = oracle.bc_brandes_tb(row, col, src)
    g = dev(row, col)
    gt = dev(*csr(np.sort(key % n * n + key // n))) if directed else g
    got, _ = gdb.bc(ctx, g, gt, src, gdb.Opts.make(wgs=wgs, groups=groups))
    bc_close(got, want)


def test_bc_tuned_is_deterministic(ctx):
    g = gdb.gen_rmat(12, 16, seed=8)
    src = gdb.permutation(g.n, 8)[:8]
    d = dev(g.row, g.col)
    a, _ = gdb.bc(ctx, d, d, src, gdb.Opts.make(variant=gdb.VARIANT_TUNED))
    b, _ = gdb.bc(ctx, d, d, src, gdb.Opts.make(variant=gdb.VARIANT_TUNED, wgs=1024, groups=7))
    assert (a == b).all()


# ---------------------------------------------------------------- worklist BFS / SSSP
@pytest.mark.parametrize("sched", SCHEDS, ids=SID)
@pytest.mark.parametrize("fx", FX["bfs"], ids=lambda f: f["name"])
def test_bfs_fixtures(ctx, fx, sched):
    if "rows" in fx:
        row, col, _ = grid_csr(fx["rows"], fx["cols"])
    else:
        row, col, _ = csr_from_edges(fx["n"], fx["edges"])
    got, _ = gdb.bfs_worklist(ctx, dev(row, col), 0, gdb.Opts.make(wgs=64, **sched))
    assert got.tolist() == fx["dist"]


@pytest.mark.parametrize("sched", SCHEDS, ids=SID)
@pytest.mark.parametrize("fx", FX["sssp_worklist"], ids=lambda f: f["name"])
def test_sssp_worklist_fixtures(ctx, fx, sched):
    row, col, w = csr_from_edges(fx["n"], fx["edges"], fx["w"])
    got, _ = gdb.sssp_worklist(ctx, dev(row, col, w), 0, gdb.Opts.make(wgs=64, **sched))
    assert got.tolist() == fx["dist"]


@pytest.mark.parametrize("sched", SCHEDS, ids=SID)
def test_bfs_sssp_grid(ctx, sched):
    g = gdb.gen_grid(256, 256, 0.05, seed=2, wlo=1, whi=255)
    d = dev(g.row, g.col, g.w)
    want_b, iters = oracle.bfs_worklist_ref(g.row, g.col, 0)
    got_b, st = gdb.bfs_worklist(ctx, d, 0, gdb.Opts.make(**sched))
    print("bfs", SID(sched), st.as_dict())
    assert (got_b == want_b).all()
    assert st.rounds == iters
    want_s, _ = oracle.sssp_worklist_ref(g.row, g.col, g.w, 0)
    got_s, st = gdb.sssp_worklist(ctx, d, 0, gdb.Opts.make(**sched))
    print("sssp", SID(sched), st.as_dict())
    assert (got_s == want_s).all()


@pytest.mark.parametrize("sched", SCHEDS[:2], ids=SID)
def test_bfs_sssp_rmat(ctx, sched):
    g = gdb.gen_rmat(15, 16, seed=6, wlo=1, whi=255)
    d = dev(g.row, g.col, g.w)
    got_b, _ = gdb.bfs_worklist(ctx, d, 0, gdb.Opts.make(**sched))
    assert (got_b == oracle.bfs_tb(g.row, g.col, 0)).all()
    got_s, _ = gdb.sssp_worklist(ctx, d, 0, gdb.Opts.make(**sched))
    assert (got_s.astype(np.int64) == oracle.dijkstra_tb(g.row, g.col, g.w, 0)).all()


def test_verify_distances_kernel(ctx):
    g = gdb.gen_grid(64, 64, 0.05, seed=2, wlo=1, whi=255)
    d = dev(g.row, g.col, g.w)
    want, _ = oracle.sssp_worklist_ref(g.row, g.col, g.w, 0)
    good = gdb.DeviceBuffer.from_numpy(want)
    assert gdb.verify_distances(ctx, d, good, weighted=True) == 0
    bad = want.copy()
    bad[100] += 1000
    n_bad = oracle.verify_distances_ref(g.row, g.col, g.w, bad)
    assert n_bad > 0
    assert gdb.verify_distances(ctx, d, gdb.DeviceBuffer.from_numpy(bad), weighted=True) == n_bad


def test_bc_directed_graph_uses_transpose(ctx):
    # Arcs u -> v with u < v only: the in-edge CSR differs from the CSR, so
    # the tuned kernel takes its two-walk path (pull in-edges, push out-edges).
    g = gdb.gen_rmat(11, 16, seed=12)
    src = np.repeat(np.arange(g.n, dtype=np.int32), np.diff(g.row))
    keep = src < g.col
    row = np.zeros(g.n + 1, np.int32)
    np.add.at(row, src[keep] + 1, 1)
    dg_h = gdb.CSR(g.n, np.cumsum(row).astype(np.int32), g.col[keep].astype(np.int32),
                   g.w[keep].astype(np.int32))
    gt_h = dg_h.transpose()
    sources = np.array([0, 1, 2, 5, 9, 17], np.int32)
    want = oracle.bc_brandes_tb(dg_h.row, dg_h.col, sources)
    d, dt = dev(dg_h.row, dg_h.col), dev(gt_h.row, gt_h.col)
    for sched in SCHEDS[:3]:
        got, _ = gdb.bc(ctx, d, dt, sources, gdb.Opts.make(**sched))
        bc_close(got, want)


def test_bc_symmetric_walk_matches_two_walks(ctx):
    # The same symmetric graph passed once (one walk per frontier vertex) and
    # as a separate transpose copy (two walks) gives the same centralities.
    g = gdb.gen_rmat(12, 16, seed=13)
    src = gdb.permutation(g.n, 13)[:8]
    d1, d2 = dev(g.row, g.col), dev(g.row, g.col)
    o = gdb.Opts.make(variant=gdb.VARIANT_TUNED)
    a, _ = gdb.bc(ctx, d1, d1, src, o)
    b, _ = gdb.bc(ctx, d1, d2, src, o)
    bc_close(a, oracle.bc_brandes_tb(g.row, g.col, src))
    bc_close(b, oracle.bc_brandes_tb(g.row, g.col, src))


def symmetric_multigraph(scale, seed):
    # An R-MAT graph with every fifth undirected edge doubled (both arcs) and
    # a self-loop on every seventh vertex; still symmetric.
    g = gdb.gen_rmat(scale, 16, seed=seed)
    src = np.repeat(np.arange(g.n, dtype=np.int32), np.diff(g.row))
    dst = np.asarray(g.col, np.int32)
    fwd = np.flatnonzero(src < dst)[::5]
    loops = np.arange(0, g.n, 7, dtype=np.int32)
    s = np.concatenate([src, src[fwd], dst[fwd], loops])
    d = np.concatenate([dst, dst[fwd], src[fwd], loops])
    order = np.lexsort((d, s))
    s, d = s[order], d[order]
    row = np.zeros(g.n + 1, np.int32)
    np.add.at(row, s + 1, 1)
    return np.cumsum(row).astype(np.int32), d.astype(np.int32)


def test_bc_multigraph_duplicate_edges_and_self_loops(ctx):
    # Parallel edges count once per edge in sigma and delta (as in the
    # oracle); a self-loop never joins a level.  Eleven sources: a full
    # eight-source sweep and a partial one, one source with a self-loop.
    row, col = symmetric_multigraph(11, 4)
    n = row.size - 1
    src = np.concatenate([[0, 7], gdb.permutation(n, 4)[:9]]).astype(np.int32)
    want = oracle.bc_brandes_tb(row, col, src)
    d = dev(row, col)
    for sched in SCHEDS[:3]:
        got, _ = gdb.bc(ctx, d, d, src, gdb.Opts.make(**sched))
        bc_close(got, want)


@pytest.mark.parametrize("sched", SCHEDS[:3], ids=SID)
def test_worklist_multigraph_parallel_edges_with_different_weights(ctx, sched):
    # Parallel edges carry different weights, so two slots of one lane can
    # relax the same vertex with different candidates in one step.
    row, col = symmetric_multigraph(11, 6)
    w = (np.arange(col.size, dtype=np.int64) * 7919 % 97 + 1).astype(np.int32)
    d = dev(row, col, w)
    for source in (0, 5, 1000):
        got_b, _ = gdb.bfs_worklist(ctx, d, source, gdb.Opts.make(**sched))
        assert (got_b == oracle.bfs_tb(row, col, source)).all()
        got_s, _ = gdb.sssp_worklist(ctx, d, source, gdb.Opts.make(**sched))
        assert (got_s.astype(np.int64) == oracle.dijkstra_tb(row, col, w, source)).all()


@pytest.mark.parametrize("hops", [0, 8])
def test_batch_multigraph_parallel_edges_with_different_weights(ctx, hops):
    row, col = symmetric_multigraph(11, 6)
    w = (np.arange(col.size, dtype=np.int64) * 7919 % 97 + 1).astype(np.int32)
    d = dev(row, col, w)
    ob = gdb.DeviceBuffer.empty(row.size - 1, np.uint32)
    os_ = gdb.DeviceBuffer.empty(row.size - 1, np.uint32)
    tasks = [gdb.make_task(gdb.TASK_BFS, d, ob, 3, hops=hops),
             gdb.make_task(gdb.TASK_SSSP, d, os_, 3, delta=40, hops=hops)]
    gdb.batch_solve(ctx, tasks, 2, gdb.Opts.make(wgs=128, groups=4))
    assert (ob.to_numpy() == oracle.bfs_tb(row, col, 3)).all()
    assert (os_.to_numpy().astype(np.int64) == oracle.dijkstra_tb(row, col, w, 3)).all()


@pytest.mark.parametrize("wgs,groups", [(64, 1), (64, 9), (256, 64), (1024, 4)])
@pytest.mark.parametrize("leaves", [1023, 1024, 1025, 2049, 40000])
def test_worklist_long_rows_and_stages(ctx, wgs, groups, leaves):
    # Two hubs of `leaves` edges one level apart (rows at the edges of the
    # per-wave and per-piece walks), whose leaves overflow a small group's
    # push stage, then a second ring of vertices behind the leaves.
    n = 2 + 2 * leaves
    edges = [(0, 1)] + [(h, 2 + i) for h in range(2) for i in range(leaves)]
    edges += [(2 + i, 2 + leaves + i) for i in range(leaves)]
    src = np.array([a for a, _ in edges] + [b for _, b in edges], np.int64)
    dst = np.array([b for _, b in edges] + [a for a, _ in edges], np.int64)
    wt = np.random.default_rng(leaves).integers(1, 50, len(edges))
    wt = np.concatenate([wt, wt])
    order = np.lexsort((dst, src))
    row = np.concatenate([[0], np.cumsum(np.bincount(src, minlength=n))]).astype(np.int32)
    d = dev(row, dst[order].astype(np.int32), wt[order].astype(np.int32))
    o = gdb.Opts.make(wgs=wgs, groups=groups, variant=gdb.VARIANT_TUNED)
    source = n - 1
    got_b, st = gdb.bfs_worklist(ctx, d, source, o)
    want_b, iters = oracle.bfs_worklist_ref(row, dst[order].astype(np.int32), source)
    assert (got_b == want_b).all() and st.rounds == iters
    got_s, _ = gdb.sssp_worklist(ctx, d, source, o)
    assert (got_s.astype(np.int64) == oracle.dijkstra_tb(row, dst[order].astype(np.int32),
                                                          wt[order].astype(np.int32), source)).all()


def local_graph(name):
    rng = np.random.default_rng(7)
    if name == "path":
        n = 5000
        src = np.arange(n - 1)
        return csr_directed(n, np.concatenate([src, src + 1]), np.concatenate([src + 1, src]), rng, 100)
    if name == "chain_one_way":  # reached from the low end only
        return csr_directed(3000, np.arange(2999), np.arange(1, 3000), rng, 9)
    if name == "band6":  # six edges a vertex, up to 40 apart, parallel edges and self-loops kept
        src = np.repeat(np.arange(20000), 6)
        return csr_directed(20000, src, np.clip(src + rng.integers(-40, 41, src.size), 0, 19999), rng, 50)
    if name == "grid_shuffled":  # the same grid without locality: iteration queues
        g = gdb.gen_grid(150, 150, 0.05, seed=3, wlo=1, whi=255)
        g = g.relabel(gdb.permutation(g.n, 5))
        return g.row, g.col, g.w
    rows, cols, hole, whi = {"grid": (160, 97, 0.05, 255), "holes": (120, 130, 0.35, 10), "tall": (2000, 7, 0.0, 3),
                             "wide": (3, 9001, 0.0, 255), "two_ranges": (128, 110, 0.0, 100),
                             "tiny": (2, 3, 0.0, 5)}[name]
    g = gdb.gen_grid(rows, cols, hole, seed=4, wlo=1, whi=whi)
    return g.row, g.col, g.w


def csr_directed(n, src, dst, rng, whi):
    order = np.lexsort((dst, src))
    row = np.concatenate([[0], np.cumsum(np.bincount(src, minlength=n))]).astype(np.int32)
    return row, dst[order].astype(np.int32), rng.integers(0, whi, src.size).astype(np.int32)


@pytest.mark.parametrize("name", ["path", "chain_one_way", "band6", "grid_shuffled", "grid", "holes", "tall", "wide",
                                  "two_ranges", "tiny"])
def test_worklist_open_shape_on_local_graphs(ctx, name):
    # The shape left open takes the owner-partitioned solve on local graphs:
    # equal to the iteration queues (a given shape) and to the oracle, for the
    # first, a middle and the last vertex as the source.
    row, col, w = local_graph(name)
    n = row.size - 1
    if name == "band6":
        w[::1000] = 2000000000  # at or above the unreachable distance: never relaxed
    d = dev(row, col, w)
    for source in (0, n // 2, n - 1):
        want_b, iters = oracle.bfs_worklist_ref(row, col, source)
        want_s, _ = oracle.sssp_worklist_ref(row, col, w, source)
        for wgs, groups in ((0, 0), (256, 64)):
            o = gdb.Opts.make(wgs=wgs, groups=groups, variant=gdb.VARIANT_TUNED)
            got_b, st = gdb.bfs_worklist(ctx, d, source, o)
            assert (got_b == want_b).all() and st.rounds == iters, (name, source, wgs)
            got_s, _ = gdb.sssp_worklist(ctx, d, source, o)
            assert (got_s == want_s).all(), (name, source, wgs)


@pytest.mark.parametrize("wgs,groups", [(0, 0), (64, 2), (256, 64)])
@pytest.mark.parametrize("leaves", [16, 17, 1024, 1025, 2500])
def test_sssp_pull_row_lengths(ctx, wgs, groups, leaves):
    # A hub that gathers from `leaves` vertices, which it reaches through a
    # second hub: in-edge rows at the edges of the per-lane, per-wave and
    # per-piece walks, with the change in the last edge of the long row.
    n = leaves + 3
    rng = np.random.default_rng(leaves)
    src = np.concatenate([np.arange(1, leaves + 1), np.zeros(leaves, np.int64), [leaves + 1, 0]])
    dst = np.concatenate([np.full(leaves, leaves + 1), np.arange(1, leaves + 1), [leaves + 2, leaves + 2]])
    wt = np.concatenate([rng.integers(5, 90, leaves), rng.integers(5, 90, leaves), [1, 500]])
    wt[leaves - 1] = wt[2 * leaves - 1] = 1  # the shortest way runs over the last leaf
    order = np.lexsort((dst, src))
    row = np.concatenate([[0], np.cumsum(np.bincount(src, minlength=n))]).astype(np.int32)
    gt = gdb.CSR(n, row, dst[order].astype(np.int32), wt[order].astype(np.int32)).transpose()
    want, rounds = oracle.sssp_pull_ref(gt.row, gt.col, gt.w, 0)
    got, st = gdb.sssp_pull(ctx, dev(gt.row, gt.col, gt.w), 0, gdb.Opts.make(wgs=wgs, groups=groups,
                                                                            variant=gdb.VARIANT_TUNED))
    assert (got == want).all() and st.rounds == rounds


@pytest.mark.parametrize("leaves", [4095, 4096, 4097, 6145, 30000])
def test_bc_rows_walked_by_a_group(ctx, leaves):
    # Two hubs sharing `leaves` neighbours, with a second ring behind them:
    # rows at the edges of the per-wave and per-group walks; the sums do not
    # depend on the launch shape.
    n = 2 + leaves + leaves // 3
    edges = [(h, 2 + i) for h in range(2) for i in range(leaves)]
    edges += [(2 + 3 * i, 2 + leaves + i) for i in range(leaves // 3)]
    a = np.array(edges, np.int64)
    src, dst = np.concatenate([a[:, 0], a[:, 1]]), np.concatenate([a[:, 1], a[:, 0]])
    order = np.lexsort((dst, src))
    row = np.concatenate([[0], np.cumsum(np.bincount(src, minlength=n))]).astype(np.int32)
    col = dst[order].astype(np.int32)
    d = dev(row, col)
    sources = np.array([0, 2, n - 1, 1, 5, 7, 11, 2 + leaves, 3, n // 2], np.int32)
    want = oracle.bc_brandes_mt(row, col, sources)
    first = None
    for wgs, groups in ((512, 0), (64, 5), (256, 16), (0, 0)):
        got, _ = gdb.bc(ctx, d, d, sources, gdb.Opts.make(wgs=wgs, groups=groups, variant=gdb.VARIANT_TUNED))
        bc_close(got, want)
        first = got if first is None else first
        assert (got == first).all(), (wgs, groups)


@pytest.mark.parametrize("wgs,groups", [(0, 0), (64, 3), (512, 16)])
@pytest.mark.parametrize("nsrc", [1, 2, 8, 11])
@pytest.mark.parametrize("shape", ["random", "layers", "levels253", "levels256", "hub"])
def test_bc_directed_sweeps(ctx, shape, nsrc, wgs, groups):
    # Sources of a directed graph share sweeps with a byte of level each:
    # skipping levels, back edges, the deepest search a byte holds and one
    # beyond it (solved source by source), and a row walked by waves.
    rng = np.random.default_rng(nsrc)
    if shape == "random":
        n = 3000
        src, dst = rng.integers(0, n, 15000), rng.integers(0, n, 15000)
    elif shape == "layers":  # forward edges of any length, a few back
        n = 900
        src = rng.integers(0, n, 4000)
        dst = np.minimum(n - 1, src + rng.integers(1, 60, 4000))
        dst[::50] = rng.integers(0, n, dst[::50].size)
    elif shape == "hub":
        n = 5000
        src = np.concatenate([np.arange(1, 2500), np.zeros(2500, np.int64), rng.integers(0, n, 4000)])
        dst = np.concatenate([np.zeros(2499, np.int64), np.arange(2500, 5000), rng.integers(0, n, 4000)])
    else:  # two parallel chains of so many levels
        k = int(shape[6:])
        n = 2 * k + 1
        a = np.arange(k)
        src = np.concatenate([a, [0], k + a[1:]])
        dst = np.concatenate([a + 1, [k + 1], k + a[1:] + 1])
    keep = src != dst
    src, dst = src[keep], dst[keep]
    order = np.lexsort((dst, src))
    row = np.concatenate([[0], np.cumsum(np.bincount(src, minlength=n))]).astype(np.int32)
    col = dst[order].astype(np.int32)
    g = gdb.CSR(n, row, col, np.ones_like(col))
    gt = g.transpose()
    sources = np.concatenate([[0], rng.integers(0, n, nsrc - 1)]).astype(np.int32)
    got, _ = gdb.bc(ctx, gdb.DeviceCSR(g), gdb.DeviceCSR(gt), sources,
                    gdb.Opts.make(wgs=wgs, groups=groups, variant=gdb.VARIANT_TUNED))
    bc_close(got, np.asarray(oracle.bc_brandes_tb(row, col, sources), np.float64))


@pytest.mark.parametrize("deg", [15, 16, 17, 63, 64, 65, 128, 129, 192, 193])
@pytest.mark.parametrize("hubs", [1, 3, 4, 5, 64])
def test_rows_walked_by_part_of_a_wave(ctx, deg, hubs):
    """Rows either side of what a lane, a quarter of a wave and a wave walk (16
    edges; 16 for each of 4, 8 or 12 slots a lane), one to 64 of them together."""
    rng = np.random.default_rng(deg + hubs)
    n = 300 + hubs
    a, b = [np.arange(n)], [np.roll(np.arange(n), -1)]
    for h in range(hubs):
        a.append(np.full(deg - 2, h))
        b.append(hubs + 1 + rng.permutation(n - hubs - 2)[:deg - 2])
    a, b = np.concatenate(a), np.concatenate(b)
    key = np.unique(np.concatenate([a * n + b, b * n + a]))
    src, col = key // n, (key % n).astype(np.int32)
    row = np.zeros(n + 1, np.int32)
    row[1:] = np.cumsum(np.bincount(src, minlength=n))
    lo, hi = np.minimum(src, col), np.maximum(src, col)
    w = (1 + (lo * 7919 + hi * 104729) % 97).astype(np.int32)
    g = gdb.DeviceCSR(gdb.CSR(n, row, col, w))
    sources = np.concatenate([[0, n - 1], rng.permutation(n)[:7]]).astype(np.int32)
    assert (np.diff(row)[:hubs] == deg).all()
    want = oracle.bc_brandes_tb(row, col, sources)
    for gt in (g, gdb.DeviceCSR(gdb.CSR(n, row, col, w))):  # as its own transpose, and as a directed graph
        got, _ = gdb.bc(ctx, g, gt, sources, gdb.Opts.make())
        bc_close(got, want)
    want = oracle.dijkstra_tb(row, col, w, n - 1)
    got, _ = gdb.sssp_worklist(ctx, g, n - 1, gdb.Opts.make(wgs=64, groups=2))
    assert (got.astype(np.int64) == want).all()
    want, _ = oracle.sssp_pull_ref(row, col, w, n - 1)
    got, _ = gdb.sssp_pull(ctx, g, n - 1, gdb.Opts.make())
    assert (got == want).all()


@pytest.mark.parametrize("xcd", [0, 3, 7])
@pytest.mark.parametrize("side", [(4, 5), (40, 50), (50, 64)])
@pytest.mark.parametrize("solver", ["bfs", "sssp", "pull", "mis", "mst", "bc"])
def test_small_graphs_on_one_xcd(ctx, solver, side, xcd):
    """Graphs of fewer groups than there are XCDs, on a context restricted to one."""
    g = gdb.gen_grid(*side, 0.0, seed=1, wlo=1, whi=9)
    d = gdb.DeviceCSR(g)
    o = gdb.Opts.make(wgs=0, variant=gdb.VARIANT_TUNED)
    nv = (gdb.permutation(g.n, 2).astype(np.float64) / (g.n + 1)).astype(np.float32)
    src = np.array([0, g.n // 2], np.int32)
    out = gdb.DeviceBuffer.from_numpy(np.full(g.n, -77, np.float32 if solver == "bc" else np.int32))
    ctx.set_xcd_only(xcd)
    try:
        if solver == "mst":
            weight, edges, components, _ = gdb.mst(ctx, d, o)
        elif solver == "bc":
            got, _ = gdb.bc(ctx, d, d, src, o, out=out)
        elif solver == "mis":
            got, _ = gdb.mis(ctx, d, gdb.DeviceBuffer.from_numpy(nv), o, out=out)
        else:
            fn = {"bfs": gdb.bfs_worklist, "sssp": gdb.sssp_worklist, "pull": gdb.sssp_pull}[solver]
            got, _ = fn(ctx, d, 0, o, out=out)
    finally:
        ctx.set_xcd_only(-1)
    if solver == "mst":
        assert (weight, edges, components) == (oracle.mst_kruskal(g.row, g.col, g.w)[0], g.n - 1, 1)
    elif solver == "bc":
        bc_close(got, oracle.bc_brandes_tb(g.row, g.col, src))
    else:
        want = {"bfs": lambda: oracle.bfs_tb(g.row, g.col, 0),
                "sssp": lambda: oracle.dijkstra_tb(g.row, g.col, g.w, 0),
                "pull": lambda: oracle.sssp_pull_ref(g.row, g.col, g.w, 0)[0],
                "mis": lambda: oracle.mis_ref(g.row, g.col, nv)[0]}[solver]()
        assert (got.astype(np.int64) == np.asarray(want).astype(np.int64)).all()


@pytest.mark.parametrize("wgs,groups", [(64, 1), (128, 2), (512, 1), (0, 0)])
def test_bc_rows_walked_by_a_group_in_many_trips(ctx, wgs, groups):
    """Long rows in every few of the trips that a group makes through a level, in the
    forward and in the backward pass."""
    hubs, leaves = 60, 4200
    rng = np.random.default_rng(3)
    # A source that reaches 3000 vertices on one level, hubs spread among them;
    # each hub has the same leaves on the next one.
    first = 1 + rng.permutation(3000)
    a = [np.zeros(3000, np.int64), rng.integers(1, 3001, 9000)]
    b = [np.arange(1, 3001), rng.integers(1, 3001, 9000)]
    n = 3001 + leaves
    for h in first[:hubs]:
        a.append(np.full(leaves, h))
        b.append(np.arange(3001, n))
    a, b = np.concatenate(a), np.concatenate(b)
    key = np.unique(np.concatenate([a * n + b, b * n + a]))
    key = key[key // n != key % n]
    row = np.zeros(n + 1, np.int32)
    row[1:] = np.cumsum(np.bincount(key // n, minlength=n))
    col = (key % n).astype(np.int32)
    assert (np.diff(row) > 4096).sum() == hubs
    sources = np.concatenate([[0], rng.permutation(n)[:10]]).astype(np.int32)
    want = oracle.bc_brandes_mt(row, col, sources)
    d = dev(row, col)
    got, _ = gdb.bc(ctx, d, d, sources, gdb.Opts.make(wgs=wgs, groups=groups, variant=gdb.VARIANT_TUNED))
    bc_close(got, want)


@pytest.mark.parametrize("wgs,groups", [(0, 0), (64, 5), (512, 32)])
@pytest.mark.parametrize("directed", [False, True])
def test_steps_of_a_sparse_graph(ctx, directed, wgs, groups):
    """Levels either side of 256 and 1024 vertices, where a sparse graph's steps change
    how they deal and push vertices, then one whose edges make the next step sweep."""
    rng = np.random.default_rng(8)
    sizes = [1, 16, 256, 257, 1024, 1025, 60000]
    first = np.concatenate([[0], np.cumsum(sizes)])
    a, b = [], []
    for lv in range(1, len(sizes)):
        v = np.repeat(np.arange(first[lv], first[lv + 1]), 3)
        a.append(rng.integers(first[lv - 1], first[lv], v.size))
        b.append(v)
    a, b, n = np.concatenate(a), np.concatenate(b), int(first[-1])
    key = np.unique(a * n + b if directed else np.concatenate([a * n + b, b * n + a]))
    row = np.zeros(n + 1, np.int32)
    row[1:] = np.cumsum(np.bincount(key // n, minlength=n))
    col = (key % n).astype(np.int32)
    w = rng.integers(1, 60, col.size).astype(np.int32)
    assert 100000 + n // 16 < col.size < 6 * n
    g = dev(row, col, w)
    o = gdb.Opts.make(wgs=wgs, groups=groups, variant=gdb.VARIANT_TUNED)
    for source in (0, 20):
        want, rounds = oracle.bfs_worklist_ref(row, col, source)
        got, st = gdb.bfs_worklist(ctx, g, source, o)
        assert (got == want).all() and st.rounds == rounds
        got, _ = gdb.sssp_worklist(ctx, g, source, o)
        assert (got.astype(np.int64) == oracle.dijkstra_tb(row, col, w, source)).all()
    sources = np.array([0, 20, 3, 700, 2000, 1, 500, 9, 30000], np.int32)
    gt = gdb.DeviceCSR(gdb.CSR(n, row, col, w).transpose()) if directed else g
    want = oracle.bc_brandes_mt(row, col, sources)
    for count in (1, sources.size):
        got, _ = gdb.bc(ctx, g, gt, sources[:count], o)
        bc_close(got, want if count > 1 else oracle.bc_brandes_mt(row, col, sources[:1]))


@pytest.mark.parametrize("wgs", [0, 256])
def test_worklist_skips_columns_out_of_range(ctx, wgs):
    """Columns that are no vertex are passed over, also where the graph is sampled."""
    n = 3000
    a = np.repeat(np.arange(n), 3)
    b = np.stack([(np.arange(n) + 1) % n, np.maximum(np.arange(n) - 1, 0), np.arange(n)], 1).ravel()
    col = b.astype(np.int32)
    col[2::30] = -2**31
    col[5::30] = 2**31 - 1
    col[8::30] = -1
    col[11::30] = n
    row = np.arange(0, 3 * n + 1, 3, dtype=np.int32)
    w = (1 + np.arange(3 * n) % 50).astype(np.int32)
    keep = (col >= 0) & (col < n)
    krow = np.concatenate([[0], np.cumsum(np.bincount(a[keep], minlength=n))]).astype(np.int32)
    g = dev(row, b.astype(np.int32), w)
    g.col = gdb.DeviceBuffer.from_numpy(col)  # what a caller of the C ABI may pass
    o = gdb.Opts.make(wgs=wgs, variant=gdb.VARIANT_TUNED)
    for source in (0, n - 1):
        got, _ = gdb.bfs_worklist(ctx, g, source, o)
        assert (got == oracle.bfs_tb(krow, col[keep], source)).all()
        got, _ = gdb.sssp_worklist(ctx, g, source, o)
        assert (got.astype(np.int64) == oracle.dijkstra_tb(krow, col[keep], w[keep], source)).all()


@pytest.mark.parametrize("solver", ["bfs", "sssp"])
def test_worklist_local_graph_under_a_short_wait_bound(ctx, solver):
    """A bound that every iteration's barrier meets with ease, but that a range of the
    owner-partitioned solve, waiting for the first vertex to reach it, does not."""
    g = gdb.gen_grid(1024, 1024, 0.05, seed=2, wlo=1, whi=255)
    d = gdb.DeviceCSR(g)
    fn = gdb.bfs_worklist if solver == "bfs" else gdb.sssp_worklist
    want, _ = fn(ctx, d, 0, gdb.Opts.make(wgs=256, groups=64, variant=gdb.VARIANT_TUNED))
    ctx.set_timeouts(700.0, 20.0)
    try:
        for _ in range(2):  # the bound given up on leaves nothing behind
            got, _ = fn(ctx, d, 0, gdb.Opts.make(wgs=0, variant=gdb.VARIANT_TUNED))
            assert (got == want).all()
    finally:
        ctx.set_timeouts(10e6, 20.0)
    got, _ = fn(ctx, d, 0, gdb.Opts.make(wgs=0, variant=gdb.VARIANT_TUNED))
    assert (got == want).all()


@pytest.mark.parametrize("long_per_mille", [4, 8, 12, 25])
def test_worklist_local_graph_with_long_edges(ctx, long_per_mille):
    """Either side of the shares of long edges up to which BFS and SSSP take the
    owner-partitioned solve (which meets no inter-group barrier)."""
    rng = np.random.default_rng(long_per_mille)
    g = gdb.gen_grid(300, 300, 0.05, seed=2, wlo=1, whi=255)
    src, dst = np.repeat(np.arange(g.n), np.diff(g.row)), np.asarray(g.col, np.int64)
    k = g.m * long_per_mille // 2000
    a = rng.integers(0, g.n, k)
    b = (a + g.n // 2) % g.n
    src, dst = np.concatenate([src, a, b]), np.concatenate([dst, b, a])
    row, col, w = csr_directed(g.n, src, dst, rng, 255)
    d = dev(row, col, w)
    o = gdb.Opts.make(wgs=0, variant=gdb.VARIANT_TUNED)
    got, st = gdb.bfs_worklist(ctx, d, 5, o)
    assert (got == oracle.bfs_tb(row, col, 5)).all() and (st.barriers == 0) == (long_per_mille < 6)
    got, st = gdb.sssp_worklist(ctx, d, 5, o)
    assert (got.astype(np.int64) == oracle.dijkstra_tb(row, col, w, 5)).all()
    assert (st.barriers == 0) == (long_per_mille < 15)


def test_stats_count_samples_and_attempts(ctx):
    """kernel_ms and launches hold all of a solve's device work: the locality sample,
    the level count, and attempts that were given up."""
    o = gdb.Opts.make(wgs=0, variant=gdb.VARIANT_TUNED)
    g = gdb.gen_grid(100, 100, 0.05, seed=3, wlo=1, whi=255)
    local, other = gdb.DeviceCSR(g), gdb.DeviceCSR(g.relabel(gdb.permutation(g.n, 5)))
    assert gdb.bfs_worklist(ctx, local, 0, o)[1].launches == 3
    assert gdb.sssp_worklist(ctx, local, 0, o)[1].launches == 2
    assert gdb.bfs_worklist(ctx, other, 0, o)[1].launches == 2
    assert gdb.bfs_worklist(ctx, other, 0, gdb.Opts.make(wgs=256, variant=gdb.VARIANT_TUNED))[1].launches == 1
    # Equal priorities: the round-free colouring waits 2 ms for progress.
    row, col, _ = csr_from_edges(3, [(0, 1), (1, 2), (0, 2)])
    d, nv = dev(row, col), gdb.DeviceBuffer.from_numpy(np.full(3, 0.5, np.float32))
    out, st = gdb.DeviceBuffer.empty(3, np.int32), gdb.Stats()
    rc = gdb.lib().gdb_color(ctx.h, 3, d.m, d.row.ptr, d.col.ptr, nv.ptr, out.ptr, C.byref(o), C.byref(st))
    assert rc == gdb.GDB_E_TIMEOUT and st.launches == 2 and st.kernel_ms > 2.0
    # Two sources of a directed chain deeper than the level bytes.
    row = np.minimum(np.arange(301), 299).astype(np.int32)
    g = gdb.CSR(300, row, np.arange(1, 300, dtype=np.int32), np.ones(299, np.int32))
    _, st = gdb.bc(ctx, gdb.DeviceCSR(g), gdb.DeviceCSR(g.transpose()), np.array([0, 1], np.int32), o)
    assert st.launches == 2


# The default options of Opts.make are the plain variant's; these run four of the
# tests above on the tuned kernels whose edges they were written for.
@pytest.fixture
def tuned(monkeypatch):
    make = gdb.Opts.make
    monkeypatch.setattr(gdb.Opts, "make", lambda **kw: make(**{"variant": gdb.VARIANT_TUNED, **kw}))


@pytest.mark.parametrize("extra", [0, 1, 31])
@pytest.mark.parametrize("deg", [1, 15, 16, 17, 79, 80, 81, 300])
def test_mis_one_deciding_edge_tuned(ctx, tuned, deg, extra):
    test_mis_one_deciding_edge(ctx, deg, extra)


@pytest.mark.parametrize("n", [1, 255, 256, 257, 1025])
@pytest.mark.parametrize("wgs,groups", [(64, 1), (256, 3), (0, 0)])
def test_bfs_sweep_tuned(ctx, tuned, n, wgs, groups):
    test_bfs_sweep(ctx, n, wgs, groups)


@pytest.mark.parametrize("n", [1023, 1024, 1030])
@pytest.mark.parametrize("directed", [False, True])
@pytest.mark.parametrize("wgs,groups", [(64, 4), (256, 3), (0, 0)])
def test_bc_step_with_many_edges_tuned(ctx, tuned, n, directed, wgs, groups):
    test_bc_step_with_many_edges(ctx, n, directed, wgs, groups)


@pytest.mark.parametrize("deg", [15, 16, 17, 63, 64, 65, 128, 129, 192, 193])
@pytest.mark.parametrize("hubs", [1, 3, 4, 5, 64])
def test_rows_walked_by_part_of_a_wave_tuned(ctx, tuned, deg, hubs):
    test_rows_walked_by_part_of_a_wave(ctx, deg, hubs)
