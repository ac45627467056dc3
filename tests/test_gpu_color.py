"""Colouring parity: every schedule/variant is bit-exact with the oracle's
restatement of the Pannotia max rule."""
import numpy as np
import pytest

import gpu_discovery_barrier_amd as gdb
import oracle
from conftest import csr_from_edges, load_fixtures, values_of

pytestmark = pytest.mark.gpu

FX = load_fixtures()
SCHEDS = [
    dict(schedule=gdb.SCHED_PERSISTENT, variant=gdb.VARIANT_PLAIN),
    dict(schedule=gdb.SCHED_PERSISTENT, variant=gdb.VARIANT_TUNED),
    dict(schedule=gdb.SCHED_RELAUNCH, variant=gdb.VARIANT_PLAIN),
    dict(schedule=gdb.SCHED_RELAUNCH, variant=gdb.VARIANT_PLAIN, relaunch_check=8),
]


@pytest.fixture(scope="module")
def ctx():
    c = gdb.Context()
    yield c
    c.close()


def run(ctx, row, col, nv, **kw):
    g = gdb.DeviceCSR(gdb.CSR(row.size - 1, row, col, np.ones_like(col)), weights=False)
    vals = gdb.DeviceBuffer.from_numpy(nv.astype(np.float32))
    return gdb.color(ctx, g, vals, gdb.Opts.make(**kw))


@pytest.mark.parametrize("sched", SCHEDS, ids=lambda s: "-".join(map(str, s.values())))
@pytest.mark.parametrize("fx", FX["color"], ids=lambda f: f["name"])
def test_color_fixtures(ctx, fx, sched):
    row, col, _ = csr_from_edges(fx["n"], fx["edges"])
    got, st = run(ctx, row, col, values_of(fx), wgs=64, **sched)
    assert got.tolist() == fx["color"]
    assert st.rounds == fx["rounds"]


@pytest.mark.parametrize("sched", SCHEDS, ids=lambda s: "-".join(map(str, s.values())))
@pytest.mark.parametrize("wgs", [64, 256, 1024])
def test_color_c1_rmat14(ctx, sched, wgs):
    g = gdb.gen_rmat(14, 16, seed=1)
    nv = gdb.pannotia_values(g.n)
    want, rounds = oracle.color_ref(g.row, g.col, nv)
    got, st = run(ctx, g.row, g.col, nv, wgs=wgs, **sched)
    print(sched, wgs, st.as_dict())
    assert (got == want).all()
    assert st.rounds == rounds


@pytest.mark.parametrize("bar", [gdb.BARRIER_XF, gdb.BARRIER_COUNTER, gdb.BARRIER_TREE, gdb.BARRIER_AUTO])
def test_color_permutation_values_all_barriers(ctx, bar):
    g = gdb.gen_rmat(13, 16, seed=1)
    nv = gdb.permutation(g.n, 1).astype(np.float32) / np.float32(g.n + 1)
    want, _ = oracle.color_ref(g.row, g.col, nv)
    ctx.configure(gdb.PROTOCOL_LOCKFREE, bar)
    try:
        for variant in (gdb.VARIANT_PLAIN, gdb.VARIANT_TUNED):
            got, _ = run(ctx, g.row, g.col, nv, wgs=256, variant=variant)
            assert (got == want).all()
    finally:
        ctx.configure(gdb.PROTOCOL_LOCKFREE, gdb.BARRIER_AUTO)


def test_color_empty_graph(ctx):
    row = np.zeros(6, np.int32)
    got, st = run(ctx, row, np.zeros(0, np.int32), gdb.pannotia_values(5), wgs=64)
    assert got.tolist() == [1] * 5


def test_color_ties_report_error_not_hang(ctx):
    row, col, _ = csr_from_edges(3, [(0, 1), (1, 2), (0, 2)])
    with pytest.raises(gdb.GdbError):
        run(ctx, row, col, np.full(3, 0.5, np.float32), wgs=64)


def test_color_single_xcd(ctx):
    g = gdb.gen_rmat(14, 16, seed=1)
    nv = gdb.pannotia_values(g.n)
    want, rounds = oracle.color_ref(g.row, g.col, nv)
    ctx.set_xcd_only(0)
    try:
        for variant in (gdb.VARIANT_PLAIN, gdb.VARIANT_TUNED):
            got, st = run(ctx, g.row, g.col, nv, wgs=1024, groups=64, variant=variant)
            print("single-xcd", variant, st.as_dict())
            assert (got == want).all() and st.rounds == rounds
    finally:
        ctx.set_xcd_only(-1)


@pytest.mark.parametrize("order", ["index", "reversed"])
@pytest.mark.parametrize("shape", ["grid", "grid_holes", "rmat"])
def test_color_tuned_blockers(ctx, shape, order):
    # The tuned kernel re-walks a light row only when the neighbour holding
    # its maximum is coloured.  Index-ordered values make a grid colour as a
    # wavefront (a vertex waits on one neighbour for many rounds); R-MAT mixes
    # light rows with chunked heavy rows that can be blockers.
    g = {"grid": lambda: gdb.gen_grid(48, 48, 0.0, seed=1),
         "grid_holes": lambda: gdb.gen_grid(31, 57, 0.15, seed=2),
         "rmat": lambda: gdb.gen_rmat(11, 8, seed=5)}[shape]()
    nv = gdb.pannotia_values(g.n)
    if order == "reversed":
        nv = nv[::-1].copy()
    want, rr = oracle.color_ref(g.row, g.col, nv)
    got, st = run(ctx, np.asarray(g.row), np.asarray(g.col), nv, wgs=128, groups=16,
                  schedule=gdb.SCHED_PERSISTENT, variant=gdb.VARIANT_TUNED)
    assert (got == want).all()
    assert st.rounds == rr


def directed(n, m, seed, hub=0):
    """A random directed CSR (no symmetry, parallel edges kept), with one row
    of `hub` edges."""
    rng = np.random.default_rng(seed)
    src = np.concatenate([rng.integers(0, n, m - hub), np.full(hub, n // 3)])
    dst = rng.integers(0, n, m)
    dst = np.where(dst == src, (dst + 1) % n, dst)
    order = np.lexsort((dst, src))
    row = np.zeros(n + 1, np.int32)
    np.add.at(row, src + 1, 1)
    return np.cumsum(row).astype(np.int32), dst[order].astype(np.int32)


# Launch shapes of the round-free kernels: left open (one group with LDS
# colours up to 8192 vertices and 32768 edges, else 1024-thread groups), and
# fixed ones whose windows of four edges a lane cut rows (the last one covers
# too few edges for most of the graphs, which take the kernel with rounds).
@pytest.mark.parametrize("wgs,groups", [(0, 0), (64, 0), (64, 64), (256, 8)])
@pytest.mark.parametrize("n,m,hub", [(1, 0, 0), (2, 2, 0), (1000, 255, 0), (1000, 256, 0), (3000, 257, 200),
                                     (8192, 32768, 3000), (8193, 32768, 0), (8192, 32769, 5000), (700, 4097, 2500),
                                     (20000, 60000, 700)])
def test_color_flow_edges(ctx, n, m, hub, wgs, groups):
    row, col = directed(n, m, n + m, hub) if n > 1 else (np.zeros(2, np.int32), np.zeros(0, np.int32))
    nv = np.random.default_rng(m).permutation(n).astype(np.float32) / np.float32(n + 1)
    nv[np.argsort(nv)[-3:]] = -2.0  # never coloured (not above -1), and blocking nobody
    want, rr = oracle.color_ref(row, col, nv)
    kw = dict(wgs=wgs, groups=groups, variant=gdb.VARIANT_TUNED)
    if rr < 0:  # neighbours that are never coloured: the loop cannot end
        with pytest.raises(gdb.GdbError) as e:
            run(ctx, row, col, nv, **kw)
        assert e.value.code == gdb.GDB_E_TIMEOUT
        return
    got, st = run(ctx, row, col, nv, **kw)
    assert (got == want).all() and st.rounds == rr


@pytest.mark.parametrize("n", [1, 3, 4, 5, 1023, 1025, 4099])
@pytest.mark.parametrize("per", [7, 9])
def test_color_flow_rounds_of_sparse_and_dense(ctx, n, per):
    """Either side of eight edges a vertex, where the last kernel deals its
    vertices out; sizes that leave its last waves part of a share."""
    m = per * n if n > 1 else 0
    row, col = directed(n, m, n, n // 4) if n > 1 else (np.zeros(2, np.int32), np.zeros(0, np.int32))
    nv = (1 + np.random.default_rng(n).permutation(n).astype(np.float32)) / np.float32(n + 1)
    want, rr = oracle.color_ref(row, col, nv)
    got, st = run(ctx, row, col, nv, wgs=256, variant=gdb.VARIANT_TUNED)
    assert (got == want).all() and st.rounds == rr


@pytest.mark.parametrize("n", [3, 9000])
def test_color_flow_ties_then_clean(ctx, n):
    # A cycle of equal priorities never resolves; the next solve on the same
    # context is unaffected.
    edges = [(i, (i + 1) % n) for i in range(n)]
    row, col, _ = csr_from_edges(n, edges)
    with pytest.raises(gdb.GdbError) as e:
        run(ctx, row, col, np.full(n, 0.5, np.float32), wgs=0, variant=gdb.VARIANT_TUNED)
    assert e.value.code == gdb.GDB_E_TIMEOUT
    nv = gdb.pannotia_values(n)
    want, rr = oracle.color_ref(row, col, nv)
    got, st = run(ctx, row, col, nv, wgs=0, variant=gdb.VARIANT_TUNED)
    assert (got == want).all() and st.rounds == rr


@pytest.mark.parametrize("xcd", [1, 7])
@pytest.mark.parametrize("wgs", [0, 1024])
@pytest.mark.parametrize("shape", ["rmat10", "grid", "pairs"])
def test_color_on_one_xcd_of_any_shape(ctx, shape, wgs, xcd):
    """A restricted context, the shape left open or a group size given: graphs whose
    edges fit fewer groups than there are XCDs, so that a launch of just those groups
    may have none on the chosen one."""
    if shape == "pairs":  # rows of one edge, whose blockers do not count
        n = 20000
        row, col = np.arange(n + 1, dtype=np.int32), (np.arange(n) ^ 1).astype(np.int32)
    else:
        g = gdb.gen_rmat(10, 16, seed=1) if shape == "rmat10" else gdb.gen_grid(100, 90, 0.05, seed=3)
        n, row, col = g.n, np.asarray(g.row), np.asarray(g.col)
    nv = (gdb.permutation(n, 2).astype(np.float64) / (n + 1)).astype(np.float32)
    want, rounds = oracle.color_ref(row, col, nv)
    d = gdb.DeviceCSR(gdb.CSR(n, row, col, np.ones_like(col)), weights=False)
    out = gdb.DeviceBuffer.from_numpy(np.full(n, -77, np.int32))
    ctx.set_xcd_only(xcd)
    try:
        got, st = gdb.color(ctx, d, gdb.DeviceBuffer.from_numpy(nv),
                            gdb.Opts.make(wgs=wgs, variant=gdb.VARIANT_TUNED), out=out)
    finally:
        ctx.set_xcd_only(-1)
    assert (got == want).all() and st.rounds == rounds


@pytest.mark.parametrize("wgs,groups", [(64, 0), (256, 0), (256, 2048), (1024, 0)])
@pytest.mark.parametrize("rows", [513, 514])
def test_color_flow_edge_limit(ctx, rows, wgs, groups):
    """1 M edges (a group of 1024 threads per CU, four edges a lane) end the round-free
    kernel's range for every launch shape; it meets no barrier, the other does."""
    g = gdb.gen_grid(rows, 512, 0.0, seed=1)
    below = g.m <= 256 * 1024 * 4
    assert below == (rows == 513)
    nv = (gdb.permutation(g.n, 2).astype(np.float64) / (g.n + 1)).astype(np.float32)
    d = gdb.DeviceCSR(g, weights=False)
    want, rounds = oracle.color_ref(g.row, g.col, nv)
    got, st = gdb.color(ctx, d, gdb.DeviceBuffer.from_numpy(nv),
                        gdb.Opts.make(wgs=wgs, groups=groups, variant=gdb.VARIANT_TUNED))
    assert (got == want).all() and st.rounds == rounds
    assert (st.barriers == 0) == (below and (groups or 4096) * wgs * 4 >= g.m)


# ---------------------------------------------------------------- max-min colouring
@pytest.mark.parametrize("wgs,groups", [(64, 3), (256, 0), (1024, 16)])
@pytest.mark.parametrize("graph", ["rmat14", "grid", "gnp", "hubs"])
def test_color_maxmin_matches_oracle(ctx, graph, wgs, groups):
    if graph == "rmat14":
        g = gdb.gen_rmat(14, 16, seed=1)  # the C1 graph
    elif graph == "grid":
        g = gdb.gen_grid(120, 90, 0.05, seed=2)
    elif graph == "gnp":
        g = gdb.gen_gnp(20000, 8.0, seed=3)
    else:  # R-MAT with heavy hub rows walked by whole waves
        g = gdb.gen_rmat(12, 64, seed=4)
    nv = (gdb.permutation(g.n, 9).astype(np.float64) / (g.n + 1)).astype(np.float32)
    want, rounds = oracle.color_maxmin_ref(g.row, g.col, nv)
    dg = gdb.DeviceCSR(g, weights=False)
    got, st = gdb.color_maxmin(ctx, dg, gdb.DeviceBuffer.from_numpy(nv), gdb.Opts.make(wgs=wgs, groups=groups))
    print(graph, wgs, groups, st.as_dict())
    assert (got == want).all()
    assert st.rounds == rounds


def test_color_maxmin_fewer_rounds_than_max_rule(ctx):
    g = gdb.gen_rmat(14, 16, seed=1)
    nv = (gdb.permutation(g.n, 1).astype(np.float64) / (g.n + 1)).astype(np.float32)
    dg = gdb.DeviceCSR(g, weights=False)
    d_nv = gdb.DeviceBuffer.from_numpy(nv)
    _, s_mm = gdb.color_maxmin(ctx, dg, d_nv, gdb.Opts.make(wgs=256, groups=64))
    _, s_max = gdb.color(ctx, dg, d_nv, gdb.Opts.make(wgs=256, groups=64, variant=gdb.VARIANT_TUNED))
    print("max-min rounds", s_mm.rounds, "max rounds", s_max.rounds)
    assert s_mm.rounds < s_max.rounds


def test_color_maxmin_ties_report_timeout(ctx):
    row, col, _ = csr_from_edges(4, [(0, 1), (1, 2), (2, 3)])
    dg = gdb.DeviceCSR(gdb.CSR(4, row, col, np.ones_like(col)), weights=False)
    with pytest.raises(gdb.GdbError) as e:
        gdb.color_maxmin(ctx, dg, gdb.DeviceBuffer.from_numpy(np.full(4, 0.5, np.float32)), gdb.Opts.make(wgs=64))
    assert e.value.code == gdb.GDB_E_TIMEOUT
