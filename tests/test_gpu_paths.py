"""Kernels that a size, type or option selects, at the sizes where the selection or a tile ends."""
import numpy as np
import pytest

import accelgraph_amd as ag
import oracle

pytestmark = pytest.mark.gpu

# in-degrees at the ends of the row classes, of a lane group's and a workgroup's chunks, and of
# the rows summed in edge order (8192)
EDGE_DEGREES = [0, 1, 15, 16, 17, 63, 64, 65, 128, 129, 255, 256, 257, 1023, 1024, 1025, 2047,
                2048, 2049, 3072, 4096, 4097, 8191, 8192]


def graph_with_degrees(degrees, n=20011, seed=3):
    """Row i has degrees[i] in-edges from distinct sources; a sparse random part keeps ranks
    moving for a while."""
    rng = np.random.default_rng(seed)
    src = [rng.choice(np.arange(len(degrees), n), d, replace=False) for d in degrees]
    dst = [np.full(d, i) for i, d in enumerate(degrees)]
    src.append(rng.integers(0, n, 4 * n))
    dst.append(rng.integers(len(degrees), n, 4 * n))
    return ag.Graph.from_edges(np.concatenate(src), np.concatenate(dst), n=n)


@pytest.mark.parametrize("init", [ag.INIT_REFERENCE, ag.INIT_UNIFORM])
def test_data_driven_row_classes(device, init):
    """From a built-in start the data-driven pull evaluates every row in edge order: the
    sequential oracle's run bit for bit at every row class's ends, and the run that the same
    start gives as a user start (explicit worklists)."""
    g = graph_with_degrees(EDGE_DEGREES)
    dg = device.upload(g)
    kw = dict(direction=ag.DIR_DATA_DRIVEN, max_iterations=200, epsilon=1e-5, scaled=True)
    run = dg.pagerank(init=init, **kw)
    ref = oracle.pagerank_dd_pull(g.out_degree, g.inv_idx, g.in_degree, g.inv_src, g.edges_idx,
                                  g.out_degree, g.fwd_dest, init=init, max_iterations=200,
                                  epsilon=1e-5)
    assert run.iterations == ref.iterations and run.executed > 5
    np.testing.assert_array_equal(run.hist_active, ref.hist_active)
    np.testing.assert_array_equal(run.scaled.view(np.uint32), ref.scaled.view(np.uint32))
    np.testing.assert_allclose(run.hist_err, ref.hist_err, rtol=1e-9, atol=1e-15)
    start = np.full(g.n, 1.0 if init == ag.INIT_UNIFORM else np.float32(1) - np.float32(0.85),
                    np.float32)
    lists = dg.pagerank(init_ranks=start, **kw)
    np.testing.assert_array_equal(run.scaled.view(np.uint32), lists.scaled.view(np.uint32))
    np.testing.assert_array_equal(run.hist_active, lists.hist_active)
    dg.close()


def acyclic_graphs():
    """A chain, and edges from lower to higher vertices with some in-degrees above a tile's lane
    and wavefront rows."""
    chain = np.arange(49)
    yield ag.Graph.from_edges(chain, chain + 1, n=50)
    rng = np.random.default_rng(17)
    n = 3000
    s, d = rng.integers(0, n, (2, 9 * n))
    keep = s < d
    big = np.arange(2500)
    yield ag.Graph.from_edges(np.concatenate([s[keep], big]),
                              np.concatenate([d[keep], np.full(big.size, n - 3)]), n=n)


@pytest.mark.parametrize("plan", [{}, dict(src_block_bits=8)])
@pytest.mark.parametrize("which", [0, 1])
def test_data_driven_epsilon_zero(device, which, plan):
    """Epsilon 0 updates every listed vertex, and only those: on an acyclic graph the lists run
    empty and the run stops, with the active counts of the oracle and of explicit worklists."""
    g = list(acyclic_graphs())[which]
    dg = device.upload(g, params=ag.plan_params(**plan))
    kw = dict(direction=ag.DIR_DATA_DRIVEN, max_iterations=200, epsilon=0.0, scaled=True)
    ref = oracle.pagerank_dd_pull(g.out_degree, g.inv_idx, g.in_degree, g.inv_src, g.edges_idx,
                                  g.out_degree, g.fwd_dest, max_iterations=200, epsilon=0.0)
    assert ref.executed < 200 and ref.hist_active[-1] == 0
    start = np.full(g.n, np.float32(1) - np.float32(0.85), np.float32)
    for run in (dg.pagerank(**kw), dg.pagerank(init_ranks=start, **kw)):
        assert (run.iterations, run.executed) == (ref.iterations, ref.executed)
        np.testing.assert_array_equal(run.hist_active, ref.hist_active)
        # two orders of a sum of d positive terms: 2 d 2^-24 at most, per rank on a path
        np.testing.assert_allclose(run.scaled, ref.scaled,
                                   rtol=2 * 2.0 ** -24 * float(g.in_degree.max() + ref.executed))
    dg.close()


@pytest.mark.parametrize("degree", [8193, 12288, 12289, 18000])
def test_data_driven_long_rows(device, degree):
    """Rows above 8192 in-edges take one fixed tree in both forms of the data-driven pull."""
    g = graph_with_degrees([degree, 3])
    dg = device.upload(g)
    kw = dict(direction=ag.DIR_DATA_DRIVEN, max_iterations=60, epsilon=1e-5, scaled=True)
    run = dg.pagerank(init=ag.INIT_UNIFORM, **kw)
    lists = dg.pagerank(init_ranks=np.ones(g.n, np.float32), **kw)
    np.testing.assert_array_equal(run.scaled.view(np.uint32), lists.scaled.view(np.uint32))
    np.testing.assert_array_equal(run.hist_active, lists.hist_active)
    dg.close()


@pytest.mark.parametrize("plan", [dict(wave_max_deg=20000, block_max_deg=20000),
                                  dict(group16_max_deg=20000, wave_max_deg=20000,
                                       block_max_deg=30000)])
@pytest.mark.parametrize("degree", [8192, 8193, 18000])
def test_data_driven_long_rows_of_lower_bins(device, plan, degree):
    """Where a row is summed in edge order or in the tree depends on its in-degree alone, not on
    the bin that the plan puts it in: both forms agree, and rows up to 8192 with the oracle."""
    g = graph_with_degrees([degree, 200, 17, 5000])
    dg = device.upload(g, params=ag.plan_params(**plan))
    kw = dict(direction=ag.DIR_DATA_DRIVEN, max_iterations=60, epsilon=1e-5, scaled=True)
    run = dg.pagerank(init=ag.INIT_UNIFORM, **kw)
    lists = dg.pagerank(init_ranks=np.ones(g.n, np.float32), **kw)
    np.testing.assert_array_equal(run.scaled.view(np.uint32), lists.scaled.view(np.uint32))
    np.testing.assert_array_equal(run.hist_active, lists.hist_active)
    if degree <= 8192:
        ref = oracle.pagerank_dd_pull(g.out_degree, g.inv_idx, g.in_degree, g.inv_src, g.edges_idx,
                                      g.out_degree, g.fwd_dest, init=1, max_iterations=60,
                                      epsilon=1e-5)
        np.testing.assert_array_equal(run.scaled.view(np.uint32), ref.scaled.view(np.uint32))
    dg.close()


TILE_PLANS = {"default": {}, "few-workgroups": dict(wg_per_cu=1), "small-tiles": dict(tile_nnz=64),
              # rows above 64 in-edges in the thread bin: still one lane, in stream order
              "long-lanes": dict(thread_max_deg=200, group16_max_deg=300),
              # wave rows that need not fit a tile are left to their groups of lanes
              "wide-waves": dict(wave_max_deg=6000, block_max_deg=6001),
              "wide-groups": dict(group16_max_deg=5000, wave_max_deg=5001, block_max_deg=5002)}


@pytest.mark.parametrize("pname", list(TILE_PLANS))
@pytest.mark.parametrize("n", [20011, 700_001])
def test_row_tiles(device, pname, n):
    """The regular schedule's row tiles at the ends of the row classes, of a tile's in-edges and
    rows and with as many rounds as one workgroup per CU needs: fixed point exact, FP32 rows of
    the thread bin equal to the sequential sum, the others within a reordered sum's bound."""
    degrees = EDGE_DEGREES + [4095, 6000, 6001, 9000, 16384, 16385]
    degrees = [d for d in degrees if d < n - len(degrees)]
    g = graph_with_degrees(degrees, n)
    p = TILE_PLANS[pname]
    dg = device.upload(g, params=ag.plan_params(src_block_bits=ag.SRC_BLOCK_OFF, **p))
    rng = np.random.default_rng(11)
    xq = rng.integers(0, 1 << 20, n, dtype=np.uint32)
    yq, _ = dg.spmv_fixed(xq)
    wc = int(oracle.fixed_encode(32, np.array([0.0001], np.float32))[0])
    np.testing.assert_array_equal(
        yq, oracle.spmv_fixed(g.inv_idx, g.in_degree, g.inv_src, None, wc, xq))
    x = rng.random(n, dtype=np.float32)
    y, _ = dg.spmv(x)
    ref = oracle.spmv_f32(g.inv_idx, g.in_degree, g.inv_src, None, x)
    lane = g.in_degree <= p.get("thread_max_deg", 16)
    np.testing.assert_array_equal(y[lane].view(np.uint32), ref[lane].view(np.uint32))
    d = g.in_degree.astype(np.float64)
    assert np.all(np.abs(y.astype(np.float64) - ref) <= 2 * d * 2.0 ** -24 * np.abs(ref))
    run = dg.pagerank(kind=ag.KIND_FIXED32, max_iterations=6, stop_rule=ag.STOP_NONE)
    want = oracle.pagerank_pull(g.out_degree, g.inv_idx, g.in_degree, g.inv_src, kind=32,
                                max_iterations=6, stop_rule=2)
    np.testing.assert_array_equal(run.ranks.view(np.uint32), want.ranks.view(np.uint32))
    dg.close()


def lanes_sum(v, width):
    """v added by `width` lanes in turn, four accumulators each, then a tree over the lanes."""
    a = np.zeros((4, width), np.float32)
    for k, i in enumerate(range(0, v.size, width)):
        part = v[i:i + width]
        a[k % 4, :part.size] += part
    t = (a[0] + a[1]) + (a[2] + a[3])
    while t.size > 1:
        t = t[:t.size // 2] + t[t.size // 2:]
    return t[0]


@pytest.mark.parametrize("negative", [False, True])
def test_row_tile_sums(device, negative):
    """FP32 rows of a tile above the thread bin keep the partial sums that 16 lanes (up to 64
    in-edges) or a wavefront with four accumulators a lane give them, bit for bit: no longer chain
    of additions, and so no larger error. All values negative zero sum to zero."""
    degrees = list(range(17, 130)) + [192, 193, 255, 256, 257, 511, 512, 513, 2047, 2048]
    g = graph_with_degrees(degrees)
    dg = device.upload(g, params=ag.plan_params(src_block_bits=ag.SRC_BLOCK_OFF))
    x = np.random.default_rng(23).random(g.n, dtype=np.float32)
    if negative:
        x = -x
    y, _ = dg.spmv(x)
    s, _ = dg.spmv_push(x)
    terms = x * np.float32(0.0001)
    for r, d in enumerate(degrees):
        row = g.inv_src[g.inv_idx[r]:g.inv_idx[r] + g.in_degree[r]]
        want = lanes_sum(terms[row], 16 if d <= 64 else 64)
        assert y[r].view(np.uint32) == want.view(np.uint32), d
        assert s[r].view(np.uint32) == want.view(np.uint32), d
    zeros, _ = dg.spmv(np.full(g.n, -0.0, np.float32))
    assert not np.any(zeros[:len(degrees)].view(np.uint32))
    dg.close()


@pytest.mark.parametrize("plan", [{}, dict(src_block_bits=10), dict(src_block_bits=9, piece_nnz=1),
                                  dict(src_block_bits=10, tile_sort=ag.SORT_OFF)])
@pytest.mark.parametrize("form", ["pull", "push"])
def test_weighted_tiles(device, plan, form):
    """Per-edge weights loaded a tile ahead of the gathers: every edge meets its own weight in
    regular and first-pass tiles, full and partly filled (fixed point exact)."""
    g = graph_with_degrees(EDGE_DEGREES + [16385])
    rng = np.random.default_rng(2)
    g.set_weights(rng.random(g.m, dtype=np.float32))
    dg = device.upload(g, weights=True, params=ag.plan_params(**plan))
    if form == "pull":
        xq = rng.integers(0, 1 << 20, g.n, dtype=np.uint32)
        wq = oracle.fixed_encode(32, g.inv_weight).astype(np.uint32)
        want = oracle.spmv_fixed(g.inv_idx, g.in_degree, g.inv_src, wq, 0, xq)
        np.testing.assert_array_equal(dg.spmv_fixed(xq)[0], want)
    else:
        xq = rng.integers(0, 1 << 34, g.n, dtype=np.uint64)
        want = oracle.spmv_push_fixed(g.edges_idx, g.out_degree, g.fwd_dest, g.fwd_weight, xq, 3)
        np.testing.assert_array_equal(dg.spmv_push_fixed(xq, 3)[0], want)
    dg.close()


STEP_RUNS = [dict(kind=ag.KIND_F32), dict(kind=ag.KIND_F32, storage=ag.STORE_BF16, refine_l1=1e-2),
             dict(kind=ag.KIND_FIXED32), dict(kind=ag.KIND_QUANT16),
             dict(kind=ag.KIND_F32, direction=ag.DIR_DATA_DRIVEN)]


@pytest.mark.parametrize("plan", [{}, dict(src_block_bits=8), dict(src_block_bits=8, blocked_min_bin=1),
                                  dict(src_block_bits=8, hot_segments=16),
                                  dict(thread_max_deg=2, group16_max_deg=6, wave_max_deg=20,
                                       block_max_deg=60, segment_nnz=256)])
@pytest.mark.parametrize("run", range(len(STEP_RUNS)))
def test_steps_of_any_length(device, plan, run):
    """An iteration is closed by the next one's first launch, or at the end of its step: the same
    run however many iterations a step queues, past the stop included, with a time for each."""
    g = ag.Graph.rmat(11)
    dg = device.upload(g, params=ag.plan_params(**plan))
    want = None
    for chunk in (32, 1, 2, 3, 7):
        r = dg.pagerank(chunk=chunk, max_iterations=90, epsilon=1e-4, **STEP_RUNS[run])
        if want is None:
            want = r
            assert 5 < r.executed < 90 and r.hist_active[-1] == 0
        assert (r.iterations, r.executed, r.refine_iteration) == (
            want.iterations, want.executed, want.refine_iteration)
        np.testing.assert_array_equal(r.ranks.view(np.uint32), want.ranks.view(np.uint32))
        np.testing.assert_array_equal(r.hist_active, want.hist_active)
        np.testing.assert_allclose(r.hist_err, want.hist_err, rtol=1e-12)
        assert r.hist_ms.size == r.executed and np.all(r.hist_ms > 0) and np.all(r.hist_ms < 50)
        assert abs(r.error_total - want.error_total) <= 1e-12 * want.error_total
    dg.close()


# the data-driven pull of an unblocked plan runs a start of one's own on worklists, whose order varies
@pytest.mark.parametrize("plan,run", [(p, r) for p in ({}, dict(src_block_bits=13))
                                      for r in range(len(STEP_RUNS))
                                      if p or "direction" not in STEP_RUNS[r]])
def test_steps_close_in_one_order(device, plan, run):
    """An iteration of more than two partials a lane (512 workgroups) has the same error to the last
    bit whether the next launch or the step's end closes it, so no stop depends on the steps. One
    huge start value on a vertex without out-edges makes its workgroup's partial so large that the
    others are fractions of its last bit, where the order of a sum shows."""
    g = ag.Graph.rmat(17)
    dg = device.upload(g, params=ag.plan_params(**plan))
    rng = np.random.default_rng(31)
    for sink in rng.choice(np.flatnonzero(g.out_degree == 0), 6, replace=False):
        for e in range(56, 64):
            start = rng.random(g.n, dtype=np.float32)
            start[sink] = 2.0 ** e
            kw = dict(max_iterations=3, stop_rule=ag.STOP_NONE, init_ranks=start, **STEP_RUNS[run])
            a, b = dg.pagerank(chunk=1, **kw), dg.pagerank(chunk=3, **kw)
            np.testing.assert_array_equal(a.hist_err.view(np.uint64), b.hist_err.view(np.uint64))
            np.testing.assert_array_equal(a.hist_active, b.hist_active)
    dg.close()


@pytest.mark.parametrize("n", [1, 1000, (1 << 20) - 1, 1 << 20, (1 << 20) + 1, 4 * (1 << 20) + 3,
                               5 * (1 << 20) + 7])
def test_staged_transfers(device, n):
    """Vectors of less than, exactly and more than one 4 MB chunk of the pinned ring, and of more
    chunks than it has: every value arrives at its place both ways, call after call."""
    chain = np.arange(n - 1, dtype=np.uint32)
    g = ag.Graph.from_edges(chain, chain + 1, n=n)
    dg = device.upload(g)
    rng = np.random.default_rng(n)
    for _ in range(2):
        v = rng.random(n, dtype=np.float32)
        want = np.concatenate([[np.float32(0)], v[:-1]]).astype(np.float32)
        np.testing.assert_array_equal(dg.gather(v, ag.GATHER_F32), want)
        q = rng.integers(0, 1 << 62, n, dtype=np.uint64)
        np.testing.assert_array_equal(dg.gather(q, ag.GATHER_U64),
                                      np.concatenate([np.zeros(1, np.uint64), q[:-1]]))
    dg.close()


@pytest.mark.parametrize("kb", [16, 1024])
@pytest.mark.parametrize("more", [-1, 0, 1])
def test_transfers_at_the_ring_sizes(device, kb, more):
    """Vectors at the sizes where a result leaves the pinned ring (16 KB) and where both ways take it
    (1 MB), of 4- and 8-byte values and of both at once, the ways taking turns."""
    for width in (4, 8):
        n = kb * 1024 // width + more
        chain = np.arange(n - 1, dtype=np.uint32)
        dg = device.upload(ag.Graph.from_edges(chain, chain + 1, n=n))
        rng = np.random.default_rng(n)
        for _ in range(2):
            v = rng.random(n, dtype=np.float32)
            want = np.concatenate([np.zeros(1, np.float32), v[:-1]])
            np.testing.assert_array_equal(dg.gather(v, ag.GATHER_F32), want)
            u = rng.integers(0, 1 << 32, n, dtype=np.uint32)
            np.testing.assert_array_equal(dg.gather(u, ag.GATHER_U32),
                                          np.concatenate([[0], u[:-1]]).astype(np.uint64))
            q = rng.integers(0, 1 << 62, n, dtype=np.uint64)
            np.testing.assert_array_equal(dg.gather(q, ag.GATHER_U64),
                                          np.concatenate([np.zeros(1, np.uint64), q[:-1]]))
        dg.close()


def test_sessions_reuse_parked_buffers(device):
    """Sessions of different kinds, lengths and overlapping lifetimes on one graph take the buffers
    that earlier ones left: the results are those of a fresh graph."""
    g = ag.Graph.rmat(12)
    dg = device.upload(g)
    runs = [dict(kind=ag.KIND_FIXED64), dict(kind=ag.KIND_FIXED8), dict(), dict(max_iterations=300),
            dict(storage=ag.STORE_F16), dict(kind=ag.KIND_QUANT8),
            dict(direction=ag.DIR_DATA_DRIVEN), dict(history=False),
            dict(max_iterations=4000, stop_rule=ag.STOP_L1, l1_tolerance=1e-7)]
    for kw in runs + runs[::-1]:
        fresh = device.upload(g)
        want = fresh.pagerank(**dict(kw))
        fresh.close()
        got = dg.pagerank(**dict(kw))
        np.testing.assert_array_equal(got.ranks.view(np.uint32), want.ranks.view(np.uint32))
        np.testing.assert_array_equal(got.hist_active, want.hist_active)
    a = dg.session(max_iterations=30, stop_rule=ag.STOP_NONE)
    a.step(10)
    b = dg.session(max_iterations=30, stop_rule=ag.STOP_NONE, kind=ag.KIND_FIXED32)
    b.step(30)
    rb, _ = b.end()
    a.step(20)
    ra, _ = a.end()
    np.testing.assert_array_equal(
        ra, dg.pagerank(max_iterations=30, stop_rule=ag.STOP_NONE).ranks)
    np.testing.assert_array_equal(
        rb, dg.pagerank(max_iterations=30, stop_rule=ag.STOP_NONE, kind=ag.KIND_FIXED32).ranks)
    dg.close()


@pytest.mark.parametrize("k", [1, 15, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("storage", [ag.STORE_F32, ag.STORE_BF16, ag.STORE_F16])
def test_ppr_widths(device, k, storage):
    """The column widths the kernels are built for, at their ends: every column is the one a call
    of 64 columns gives (up to the order of long rows' sums) and within the FP64 residual bound;
    one graph serves calls of every width, captured and eager, of any iteration budget."""
    g = graph_with_degrees(EDGE_DEGREES + [16385], seed=5)
    dg = device.upload(g)
    rng = np.random.default_rng(7)
    seeds = rng.integers(0, g.n, 64).astype(np.uint32)
    seeds[0] = ag.PPR_UNIFORM
    kw = dict(max_iterations=200, l1_tolerance=1e-6, storage=storage)
    wide, _, _ = dg.ppr(seeds, **kw)
    ranks, err, res = dg.ppr(seeds[:k], **kw)
    assert ranks.shape == (g.n, k) and res.executed < 200 and np.all(err <= 1e-6)
    np.testing.assert_allclose(ranks, wide[:, :k], rtol=1e-4, atol=1e-9)
    bound, _ = oracle.ppr_residual(g.out_degree, g.inv_idx, g.in_degree, g.inv_src, seeds[:k], ranks)
    assert np.all(bound / 0.15 <= 1e-5)
    eager, _, re = dg.ppr(seeds[:k], use_hip_graph=0, **kw)
    np.testing.assert_array_equal(eager.view(np.uint32), ranks.view(np.uint32))
    assert re.executed == res.executed
    for budget in (1, 16, 17, 31, 33):      # a replay's length, and not a multiple of it
        a, _, ra = dg.ppr(seeds[:k], max_iterations=budget, stop_rule=ag.STOP_NONE, storage=storage)
        b, _, rb = dg.ppr(seeds[:k], max_iterations=budget, stop_rule=ag.STOP_NONE, storage=storage,
                          use_hip_graph=0)
        assert ra.executed == rb.executed == budget
        np.testing.assert_array_equal(a.view(np.uint32), b.view(np.uint32))
    dg.close()


@pytest.mark.parametrize("part_edges", [64, 4096, 16384])
@pytest.mark.parametrize("heavy_deg", [8, 32, 5000])
def test_batch_parts(device, part_edges, heavy_deg):
    """Parts staged in LDS (up to 4096 in-edges) and larger ones, with rows at the ends of both and
    graphs of a single row, no edge and many parts: every graph's run is its own single one."""
    graphs = [graph_with_degrees(EDGE_DEGREES + [9000]), ag.Graph.from_edges([0], [1], n=2),
              ag.Graph.from_edges([], [], n=5), ag.Graph.rmat(13),
              graph_with_degrees([4097, 0, 4096, 1], n=5003)]
    b = ag.Batch(device, graphs)
    for maxit in (7, 100):
        ranks, its, err, _ = b.pagerank(max_iterations=maxit, l1_tolerance=1e-6,
                                        part_edges=part_edges, heavy_deg=heavy_deg)
        assert np.all(np.isfinite(err)) and (maxit < 100 or np.all(err <= 1e-6))
        for g, r, i in zip(graphs, ranks, its):
            want = oracle.pagerank_pull(g.out_degree, g.inv_idx, g.in_degree, g.inv_src, init=1,
                                        stop_rule=1, l1_tolerance=1e-6, max_iterations=maxit)
            assert abs(int(i) - want.iterations) <= 1
            assert np.abs(r - want.ranks).max() <= 1e-5
    b.close()
