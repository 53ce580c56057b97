"""GPU parity of the batched 64-source BFS: every lane's depths equal the
single-source BFS depths from its source (oracle serial BFS), including the
uneven batch (a disjoint union of Kronecker graphs of scales 12..18)."""
import numpy as np
import pytest

from conftest import csr_from_pairs
import dist_mem_gapbs_amd._lib as L

pytestmark = pytest.mark.gpu


def expected(orc, og, srcs):
    out = np.empty((len(srcs), og.n), np.uint8)
    for i, s in enumerate(srcs):
        d = orc.bfs_depth(og, int(s))
        out[i] = np.where(d < 0, 255, d)
    return out


@pytest.mark.parametrize("scale,degree,uniform", [(14, 16, False), (14, 8, True), (17, 16, False)])
def test_batch64_depths(ctx, dmm, orc, graph, scale, degree, uniform):
    g = graph(scale, degree, uniform)
    og = orc.CSR.of(g)
    ctx.upload(g)
    srcs = dmm.pick_sources(g, 64)
    depth, st = ctx.bfs_batch64(srcs)
    assert np.array_equal(depth, expected(orc, og, srcs))
    # GTEPS numerator: sum over lanes of the reached out-degrees
    deg = np.diff(og.oo)
    assert st.reached_edges == int(sum(deg[expected(orc, og, [s])[0] != 255].sum() for s in srcs))


def test_batch64_depths_kept_in_hbm(ctx, dmm, orc, graph):
    """DMM_BATCH_DEPTH_HBM: the run writes the caller-ID depths to HBM with
    no host buffer; dmm_batch_read_depth returns them.  A run that writes no
    depths leaves nothing to read."""
    g = graph(14, 16, False)
    og = orc.CSR.of(g)
    ctx.upload(g)
    srcs = dmm.pick_sources(g, 64)[:40]
    none, st = ctx.bfs_batch64(srcs, want_depth=False, depth_in_hbm=True)
    assert none is None and st.total_ms > 0
    assert np.array_equal(ctx.batch_read_depth(len(srcs)), expected(orc, og, srcs))
    _, st = ctx.bfs_batch64(srcs, want_depth=False, with_stats=False)
    assert st is None
    with pytest.raises(L.DmmError):
        ctx.batch_read_depth(len(srcs))


@pytest.mark.parametrize("td_div", [1, 4, 20, 10 ** 6])
def test_batch64_direction_settings_same_depths(ctx, dmm, orc, graph, td_div):
    g = graph(13, 16, False)
    og = orc.CSR.of(g)
    ctx.upload(g)
    srcs = dmm.pick_sources(g, 64)
    depth, _ = ctx.bfs_batch64(srcs, td_div=td_div, graph_levels=6)
    assert np.array_equal(depth, expected(orc, og, srcs))


def test_batch_partial_and_duplicate_lanes(ctx, dmm, orc, graph):
    g = graph(13, 16, False)
    og = orc.CSR.of(g)
    ctx.upload(g)
    srcs = dmm.pick_sources(g, 5)
    srcs = np.array([srcs[0], srcs[1], srcs[0], srcs[2], srcs[3], srcs[4], srcs[1]], np.int32)
    depth, _ = ctx.bfs_batch64(srcs)
    assert depth.shape == (7, og.n)
    assert np.array_equal(depth, expected(orc, og, srcs))
    d1, _ = ctx.bfs_batch64(srcs[:1])
    assert np.array_equal(d1, expected(orc, og, srcs[:1]))


def test_batch_zero_degree_and_deep(ctx, dmm, orc):
    n = 250  # depths up to 249: within the uint8 depth range (255 = unreached)
    pairs = [[i, i + 1] for i in range(n - 1)]
    g = csr_from_pairs(dmm, pairs, n + 3)  # vertices n..n+2 isolated
    og = orc.CSR.of(g)
    ctx.upload(g)
    srcs = np.array([0, 125, n + 1, n - 1], np.int32)
    depth, st = ctx.bfs_batch64(srcs)
    assert np.array_equal(depth, expected(orc, og, srcs))
    assert st.num_levels >= n - 1


def test_batch_too_deep_is_an_error(ctx, dmm):
    g = csr_from_pairs(dmm, [[i, i + 1] for i in range(299)])
    ctx.upload(g)
    with pytest.raises(dmm.DmmError) as e:
        ctx.bfs_batch64(np.array([0], np.int32))
    assert e.value.code == -5  # DMM_ERR_CAPACITY: depths beyond 254


def test_batch_directed(ctx, dmm, orc):
    rng = np.random.default_rng(11)
    pairs = rng.integers(0, 3000, size=(15000, 2))
    g = dmm.from_edgelist(pairs, 3000, symmetrize=False)
    og = orc.CSR.of(g)
    ctx.upload(g)
    srcs = dmm.pick_sources(g, 64)
    depth, _ = ctx.bfs_batch64(srcs)
    assert np.array_equal(depth, expected(orc, og, srcs))


def test_uneven_batch_disjoint_union(ctx, dmm, orc):
    """32 Kronecker graphs, scales drawn from 12..18 (mt19937(kRandSeed),
    uniform over [12, 18]), graph i relabelled into its own ID range; one
    source per graph (its first SourcePicker draw) in lanes 0..31."""
    import ctypes as C
    lib = dmm.load()
    draws = np.empty(32, np.int64)
    lib.dmm_rng_sequence(0, 27491095, 7, 32, draws.ctypes.data_as(C.POINTER(C.c_int64)))
    scales = (12 + draws).tolist()
    offs, nbrs, srcs = [np.zeros(1, np.int64)], [], []
    base_v, base_e = 0, 0
    for sc in scales:
        gi = dmm.build_graph(sc, 16, False)
        srcs.append(base_v + int(dmm.pick_sources(gi, 1)[0]))
        offs.append(gi.out_offsets[1:] + base_e)
        nbrs.append(gi.out_neighs + base_v)
        base_v += gi.num_nodes
        base_e += int(gi.out_offsets[-1])
    oo = np.concatenate(offs)
    on = np.concatenate(nbrs).astype(np.int32)
    og = orc.CSR(base_v, oo, on)
    ctx.upload(num_nodes=base_v, out_offsets=oo, out_neighs=on, num_edges_directed=base_e)
    srcs = np.array(srcs, np.int32)
    depth, st = ctx.bfs_batch64(srcs)
    assert np.array_equal(depth, expected(orc, og, srcs))


def level_words(depth, level):
    """uint64 words with lane s set where depth[s, v] == level."""
    w = np.zeros(depth.shape[1], np.uint64)
    for s in range(depth.shape[0]):
        w |= (depth[s] == level).astype(np.uint64) << np.uint64(s)
    return w


def test_block_level_equals_full_graph(ctx, dmm, orc, graph):
    """One PE's block (src/partition.h, np = 8, pe = 3): fed the all-gathered
    level words of the oracle's depths (serial BFS per source), each block
    level equals the next level's words restricted to the block.  The
    whole-graph batched run's level words equal the same oracle words.  The
    sparse first levels take the top-down expansion, the dense middle ones
    the bottom-up sweep."""
    hg = graph(14, 16, False)
    g = orc.CSR.of(hg)
    n = g.n
    srcs = dmm.pick_sources(hg, 64)
    odepth = expected(orc, g, srcs)
    words = []
    while True:
        w = level_words(odepth, len(words))
        words.append(w)
        if not w.any():
            break
    assert len(words) >= 4
    ctx.upload(hg)
    ctx.bfs_batch64(srcs, want_depth=False)
    for lv in range(len(words) - 1):
        assert np.array_equal(ctx.batch_read_level(lv), words[lv]), lv
    p = dmm.partition(n, 8, 3)
    b, e = p["start"], p["end"]
    ctx.upload(num_nodes=n, out_offsets=g.oo[b:e + 1] - g.oo[b], out_neighs=g.on[g.oo[b]:g.oo[e]],
               vbegin=b, vend=e, num_edges_directed=g.ned)
    seen = np.zeros(e - b, np.uint64)
    kinds = []
    for lv in range(len(words) - 1):
        seen |= words[lv][b:e]
        nxt, st = ctx.batch_block_level(words[lv], seen)
        assert np.array_equal(nxt, words[lv + 1][b:e]), lv
        assert st.kernel_ms > 0
        assert st.frontier == np.count_nonzero(words[lv])
        assert 0 <= st.edges_examined <= g.oo[e] - g.oo[b]
        kinds.append(st.kind)
    assert kinds[0] == L.DMM_STEP_TD and L.DMM_STEP_BU in kinds


def _or_over_in_neighbours(g, b, e, front):
    """exp[r - b] = OR of front over the in-neighbours of row r."""
    off = g.oo[b:e + 1] - g.oo[b]
    vals = front[g.on[g.oo[b]:g.oo[e]]]
    exp = np.zeros(e - b, np.uint64)
    nonempty = np.flatnonzero(np.diff(off) > 0)
    if len(nonempty):
        exp[nonempty] = np.bitwise_or.reduceat(vals, off[nonempty])
    return exp


def test_block_level_edge_cases(dmm, orc):
    """Empty frontier, a frontier on isolated vertices, a hub whose push list
    is shared by the whole grid, a dense frontier (bottom-up), and blocks at
    the start, in the middle and past the last edge."""
    rng = np.random.default_rng(9)
    n = 40000
    pairs = [[0, i] for i in range(1, 12000)] + rng.integers(0, 30000, size=(60000, 2)).tolist()
    hg = csr_from_pairs(dmm, pairs, n)  # vertices 30000 and above are isolated
    g = orc.CSR.of(hg)
    ctx = dmm.Context(0)
    ctx.set_layout(L.DMM_LAYOUT_NATURAL)
    for (b, e) in ((0, n), (5000, 17000), (35000, n)):
        ctx.upload(num_nodes=n, out_offsets=g.oo[b:e + 1] - g.oo[b], out_neighs=g.on[g.oo[b]:g.oo[e]],
                   vbegin=b, vend=e, num_edges_directed=g.ned)
        kinds = set()
        for front_ids in ([], [0], [0, 7, 123], list(range(30001, 30100)), list(rng.integers(0, n, 20000))):
            front = np.zeros(n, np.uint64)
            for k, v in enumerate(front_ids):
                front[v] |= np.uint64(1) << np.uint64(k % 64)
            seen = front[b:e].copy()
            seen[::7] |= np.uint64(0xF0F0)
            nxt, st = ctx.batch_block_level(front, seen)
            exp = _or_over_in_neighbours(g, b, e, front) & ~seen
            assert np.array_equal(nxt, exp), (b, e, len(front_ids))
            assert st.frontier == np.count_nonzero(front)
            kinds.add(st.kind)
        if b == 0:
            assert kinds == {L.DMM_STEP_TD, L.DMM_STEP_BU}
    ctx.close()


@pytest.mark.parametrize("hub", [511, 512, 4095, 4096, 9000])
@pytest.mark.parametrize("directed", [False, True])
def test_batch_wide_rows_and_dead_lanes(dmm, orc, hub, directed):
    """Rows at the edges of the sweep's row classes (an 8-lane group, a
    wavefront, a workgroup), whose lanes come from few of their many
    in-neighbours, beside small components whose lanes die early: rows out of
    their reach stop looking for them, depths stay exact."""
    rng = np.random.default_rng([hub, directed])
    ring = np.arange(3000)
    pairs = [np.stack((np.arange(3000, 3000 + hub), np.zeros(hub, np.int64)), 1),  # leaves -> hub 0
             np.stack((ring, np.roll(ring, -1)), 1),
             rng.integers(0, 3000, (9000, 2)),
             np.stack((rng.integers(0, 3000, hub), np.arange(3000, 3000 + hub)), 1)]
    base = 3000 + hub
    for k in range(20):  # components of 1 .. 20 edges in a row
        pairs.append(np.stack((np.arange(base, base + k + 1), np.arange(base + 1, base + k + 2)), 1))
        base += k + 2
    g = csr_from_pairs(dmm, np.concatenate(pairs), base, symmetrize=not directed)
    og = orc.CSR.of(g)
    srcs = np.concatenate((rng.integers(0, 3000 + hub, 40), rng.integers(3000 + hub, base, 24))).astype(np.int32)
    with dmm.Context(0) as c:
        c.upload(g)
        for td_div in (1, 1000000):  # pushed and swept levels
            depth, _ = c.bfs_batch64(srcs, td_div=td_div)
            for i, s in enumerate(srcs):
                ref = orc.bfs_depth(og, int(s))
                assert np.array_equal(depth[i], np.where(ref < 0, 255, ref).astype(np.uint8)), (i, s, td_div)


@pytest.mark.parametrize("graph_levels", [1, 6, 17])
@pytest.mark.parametrize("td_div", [1, 1000000])
def test_batch_chain_sized_by_the_last_runs(dmm, orc, graph_levels, td_div):
    """Short and long searches in turn, past the number of runs that size the
    launch chain: the chain grows, shrinks and is continued from either half
    of the loop state, with the same depths and levels every time."""
    n = 160
    g = csr_from_pairs(dmm, np.stack((np.arange(n - 1), np.arange(1, n)), 1), n, symmetrize=False)
    og = orc.CSR.of(g)
    with dmm.Context(0) as c:
        c.upload(g)
        for first in [n - 1, 0, n - 2, n - 3, 100, n - 2] + [n - 4] * 9 + [3, n - 1, 90, 91, 0]:
            srcs = np.array([first, n - 1, min(first + 7, n - 1)], np.int32)
            depth, st = c.bfs_batch64(srcs, td_div=td_div, graph_levels=graph_levels)
            assert np.array_equal(depth, expected(orc, og, srcs)), first
            assert st.num_levels == n - first, first


@pytest.mark.parametrize("n", [(1 << 19) - 1, 1 << 19, 700001])
@pytest.mark.parametrize("directed", [False, True])
def test_batch_words_beyond_l2(dmm, orc, n, directed):
    """The sweep of graphs whose frontier words miss L2, at its size limit:
    rows of every class, and lanes found after any number of rounds."""
    rng = np.random.default_rng([n, directed])
    hub = np.stack((rng.integers(0, n, 6000), np.full(6000, 5)), 1)
    mid = np.stack((rng.integers(0, n, 900), np.full(900, n - 7)), 1)
    g = csr_from_pairs(dmm, np.concatenate((rng.integers(0, n, (6 * n, 2)), hub, mid)), n, symmetrize=not directed)
    og = orc.CSR.of(g)
    srcs = rng.integers(0, n, 64).astype(np.int32)
    with dmm.Context(0) as c:
        c.upload(g)
        for td_div in (1, 20, 1000000):
            depth, _ = c.bfs_batch64(srcs, td_div=td_div)
            for i in (0, 1, 31, 62, 63):
                ref = orc.bfs_depth(og, int(srcs[i]))
                assert np.array_equal(depth[i], np.where(ref < 0, 255, ref).astype(np.uint8)), (i, td_div)


@pytest.mark.parametrize("td_div", [1, 20, 1000000])
@pytest.mark.parametrize("layout", [L.DMM_LAYOUT_NATURAL, L.DMM_LAYOUT_DEGREE])
def test_batch_reached_edges_of_every_source(dmm, orc, td_div, layout):
    """Out-edges of the reached vertices, for sources without in-edges,
    without out-edges and without either, after any kind of last level."""
    n = 3000
    rng = np.random.default_rng(n)
    pairs = rng.integers(100, n - 100, (9000, 2))  # 0 .. 99 and the last 100: no edges
    pairs[:, 0][pairs[:, 0] < 200] += 200           # 100 .. 199: no out-edges
    pairs[:, 1][pairs[:, 1] > n - 200] -= 200       # the 99 before the last 100: no in-edges
    g = csr_from_pairs(dmm, pairs, n, symmetrize=False)
    og = orc.CSR.of(g)
    deg = np.diff(og.oo)
    with dmm.Context(0) as c:
        c.set_layout(layout)
        c.upload(g)
        for srcs in ([5], [150], [n - 150], [n - 5], [1500, 150, n - 150, 7], list(range(90, n - 90, 45))):
            srcs = np.array(srcs, np.int32)
            depth, st = c.bfs_batch64(srcs, td_div=td_div)
            exp = expected(orc, og, srcs)
            assert np.array_equal(depth, exp), srcs
            assert st.reached_edges == sum(int(deg[e != 255].sum()) for e in exp), srcs


@pytest.mark.parametrize("n", [1 << 23, (1 << 23) + 1])
def test_batch_beyond_the_far_sweep(dmm, orc, n):
    """The last size whose sweep probes the frontier's bitmap, and the first
    beyond it: rows of every class, pushed and swept levels."""
    rng = np.random.default_rng(n)
    hub = np.stack((rng.integers(0, n, 6000), np.full(6000, 5)), 1)
    mid = np.stack((rng.integers(0, n, 900), np.full(900, n - 7)), 1)
    pairs = np.concatenate((rng.integers(0, n, (3 * n, 2)), hub, mid)).astype(np.int32)
    srcs = np.concatenate((rng.integers(0, n, 14), [5, n - 1])).astype(np.int32)
    with dmm.Context(0) as c:
        g = c.build_graph(pairs, n)
        del pairs
        og = orc.CSR.of(g)
        c.upload(g)
        refs = {}
        for i in (0, 13, 14, 15):
            ref = orc.bfs_depth(og, int(srcs[i]))
            refs[i] = np.where(ref < 0, 255, ref).astype(np.uint8)
        for td_div in (1, 20, 1000000):
            depth, _ = c.bfs_batch64(srcs, td_div=td_div)
            for i, ref in refs.items():
                assert np.array_equal(depth[i], ref), (i, td_div)


@pytest.mark.parametrize("n", [(7 << 21) - 1, 7 << 21])
def test_batch_wide_rows_of_the_largest_graphs(dmm, orc, n):
    """From 7 * 2^21 vertices on rows are wide from 8192 in-edges on, giant from
    65536: rows around all four limits, below and at that size."""
    rng = np.random.default_rng(n)
    hubs = [511, 512, 513, 4095, 4096, 8191, 8192, 8193, 65535, 65536, 66000]
    pairs = [np.stack((rng.permutation(3 * k)[:k] * 11 % n,
                       np.full(k, n - 1 - 3 * i)), 1) for i, k in enumerate(hubs)]
    pairs = np.concatenate([rng.integers(0, n, (2 * n, 2))] + pairs).astype(np.int32)
    srcs = np.concatenate((rng.integers(0, n, 10), [n - 1 - 3 * i for i in range(len(hubs))])).astype(np.int32)
    with dmm.Context(0) as c:
        g = c.build_graph(pairs, n, symmetrize=False)
        del pairs
        og = orc.CSR.of(g)
        c.upload(g)
        refs = {}
        for i in (0, 9, 10, 20):
            ref = orc.bfs_depth(og, int(srcs[i]))
            refs[i] = np.where(ref < 0, 255, ref).astype(np.uint8)
        for td_div in (1, 1000000):
            depth, _ = c.bfs_batch64(srcs, td_div=td_div)
            for i, ref in refs.items():
                assert np.array_equal(depth[i], ref), (i, td_div)
