"""Results read out through the pinned ring: sizes around one piece, several
pieces, helper threads and the ring's reuse arrive whole, from runs of
different sizes on one context, also into buffers at odd addresses."""
import ctypes as C

import numpy as np
import pytest

import dist_mem_gapbs_amd._lib as L

pytestmark = pytest.mark.gpu


def _graph(dmm, n):
    rng = np.random.default_rng(n)
    return dmm.from_edgelist(rng.integers(0, n, (8 * n, 2)).astype(np.int32), n)


# 64 lanes of n bytes: up to 512 KB in one piece, from 2 MB on with helpers,
# beyond 16 MB with slots used again.
@pytest.mark.parametrize("n", [100, 8191, 8192, 8193, 16384, 16385, 32767, 32769, 262144, 262147, 450001])
def test_batch_depths_arrive_whole(dmm, orc, n):
    g = _graph(dmm, n)
    og = orc.CSR.of(g)
    srcs = dmm.pick_sources(g, 64)
    with dmm.Context(0) as c:
        c.upload(g)
        out = np.empty(64 * n + 3, np.uint8)[3:]  # an odd address
        rc = c._lib.dmm_bfs_batch64(c._h, L.ptr(srcs, C.c_int32), 64, L.ptr(out, C.c_uint8), None, None)
        assert rc == 0
        depth = out.reshape(64, n)
        for i in range(0, 64, 7 if n > 100000 else 1):
            ref = orc.bfs_depth(og, int(srcs[i]))
            assert np.array_equal(depth[i], np.where(ref < 0, 255, ref).astype(np.uint8))
        assert np.array_equal(c.batch_read_depth(64), depth)
        # A smaller and a two-part read behind it.
        parent, d, _ = c.DOBFS(int(srcs[0]))
        ref = orc.bfs_depth(og, int(srcs[0]))
        assert np.array_equal(d, ref)
        assert orc.bfs_verify(og, int(srcs[0]), parent)[0]
        only, none = c.bfs_read(depth=False)
        assert none is None and np.array_equal(only, parent)
        _, only = c.bfs_read(parent=False)
        assert np.array_equal(only, ref)


# Whole pages: allocations of these sizes may follow one another in device
# memory, and a copy must not run from one into the next.
@pytest.mark.parametrize("n", [1024, 2048, 4096, 8192])
def test_parts_of_separate_allocations(dmm, orc, n):
    g = _graph(dmm, n)
    og = orc.CSR.of(g)
    s = int(dmm.pick_sources(g, 1)[0])
    with dmm.Context(0) as c:
        c.set_layout(L.DMM_LAYOUT_NATURAL)
        c.upload(g)
        depth, counts, _, _ = c.bc_forward(s)
        assert np.array_equal(depth, orc.bfs_depth(og, s))
        assert counts[s] == 1 and (counts[depth > 0] > 0).all()
        parent, depth, _ = c.DOBFS(s)
        assert np.array_equal(depth, orc.bfs_depth(og, s)) and orc.bfs_verify(og, s, parent)[0]


# Up to 65536 rows the ring has two slots of 256 KB after the upload: results of
# several parts that fill it, that need more of its quarters than it has, and
# batches (64 bytes a row) that go through it and then enlarge it.
@pytest.mark.parametrize("n", [9000, 21000, 22000, 30000, 33000, 33500, 44000, 65536])
def test_reads_larger_than_the_ring(dmm, orc, n):
    g = _graph(dmm, n)
    og = orc.CSR.of(g)
    srcs = dmm.pick_sources(g, 64)
    s = int(srcs[0])
    counts = orc.bc_forward(og, s)
    depths = np.array([np.where(r < 0, 255, r) for r in (orc.bfs_depth(og, int(x)) for x in srcs[:8])], np.uint8)
    ref = orc.bfs_depth(og, s)
    for first in ("counts", "batch"):
        with dmm.Context(0) as c:
            c.set_layout(L.DMM_LAYOUT_NATURAL)
            c.upload(g)
            for k in range(6):
                if first == "counts" or k > 3:
                    for got, want in zip(c.bc_forward(s)[:3], counts):
                        assert np.array_equal(got, want), (first, k)
                if first == "batch" or k > 3:
                    assert np.array_equal(c.bfs_batch64(srcs)[0][:8], depths), (first, k)
                assert np.array_equal(c.DOBFS(s)[1], ref), (first, k)
