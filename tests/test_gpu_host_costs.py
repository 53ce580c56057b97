"""What the library asks of the HIP runtime on the host: pinned memory of an
upload, waits before a read, launch sizes, graphs instantiated.  Each scenario runs in a process of its own that maps, ahead of the
library, a shared object whose functions count the calls and pass them on."""
import json
import os
import shutil
import subprocess
import sys

import pytest

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")]

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
COUNTS = r"""
#include <atomic>
#include <cstddef>
#include <dlfcn.h>

static void* runtime(const char* name) {
  static void* lib = dlopen("libamdhip64.so.7", RTLD_NOW | RTLD_LOCAL);
  return lib ? dlsym(lib, name) : nullptr;
}
static std::atomic<long> pinned_bytes{0};

extern "C" long count_pinned_bytes() { return pinned_bytes.exchange(0); }
extern "C" int hipHostMalloc(void** p, size_t n, unsigned flags) {
  static auto next = reinterpret_cast<int (*)(void**, size_t, unsigned)>(runtime("hipHostMalloc"));
  pinned_bytes += static_cast<long>(n);
  return next(p, n, flags);
}

struct Dim { unsigned x, y, z; };
static std::atomic<long> queued{0};  // kernels launched since the stream was last waited for
static std::atomic<long> before_last{0};  // ... before the last one

static std::atomic<long> largest{0};  // workgroups of a launch

extern "C" long count_before_last_launch() { return before_last; }
extern "C" long count_largest_grid() { return largest.exchange(0); }
extern "C" int hipLaunchKernel(const void* f, Dim grid, Dim block, void** args, size_t lds, void* stream) {
  static auto next =
      reinterpret_cast<int (*)(const void*, Dim, Dim, void**, size_t, void*)>(runtime("hipLaunchKernel"));
  before_last = queued.fetch_add(1);
  if (grid.x > largest) largest = grid.x;
  return next(f, grid, block, args, lds, stream);
}
extern "C" int hipStreamSynchronize(void* stream) {
  static auto next = reinterpret_cast<int (*)(void*)>(runtime("hipStreamSynchronize"));
  queued = 0;
  return next(stream);
}

static std::atomic<long> graphs{0};
static std::atomic<long> fail_in{-1};  // this many graphs from now on one cannot be had

extern "C" long count_graphs() { return graphs.exchange(0); }
extern "C" void fail_graph(long in) { fail_in = in; }
extern "C" int hipGraphInstantiate(void** exec, void* graph, void** node, char* log, size_t size) {
  static auto next =
      reinterpret_cast<int (*)(void**, void*, void**, char*, size_t)>(runtime("hipGraphInstantiate"));
  if (fail_in.fetch_sub(1) == 0) return 2;  // out of memory
  graphs++;
  return next(exec, graph, node, log, size);
}
"""
PRELUDE = """
import ctypes, json, sys
counts = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
for f in (counts.count_pinned_bytes, counts.count_before_last_launch, counts.count_graphs,
          counts.count_largest_grid):
    f.restype = ctypes.c_long
counts.fail_graph.argtypes = [ctypes.c_long]
sys.path.insert(0, sys.argv[2])
import numpy as np
import dist_mem_gapbs_amd as dmm
def graph(n, degree=8):
    return dmm.from_edgelist(np.random.default_rng(n).integers(0, n, (degree * n, 2)).astype(np.int32), n)
out = []
"""


@pytest.fixture(scope="module")
def counted(tmp_path_factory):
    d = tmp_path_factory.mktemp("counts")
    (d / "counts.cc").write_text(COUNTS)
    so = d / "counts.so"
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", str(d / "counts.cc"), "-o", str(so), "-ldl"],
                   check=True)

    def run(scenario):
        p = subprocess.run([sys.executable, "-c", PRELUDE + scenario + "\nprint(json.dumps(out))", str(so), ROOT],
                           capture_output=True, text=True, timeout=100)
        assert p.returncode == 0, p.stderr
        return json.loads(p.stdout)
    return run


def test_an_upload_pins_what_a_search_reads(counted):
    """The ring for reads: a parent and a depth in at most eight slots, each
    rounded to 64 KB, of 256 KB at least; none for a graph of the same size
    again."""
    sizes = [100, 1000, 32768, 65536, 65537, 131072, 600001]
    got = counted("""
for n in %r:
    g = graph(n, 2)
    with dmm.Context(0) as c:
        counts.count_pinned_bytes()
        c.upload(g)
        first = counts.count_pinned_bytes()
        c.upload(g)
        out.append((n, first, counts.count_pinned_bytes()))
""" % sizes)
    assert [n for n, _, _ in got] == sizes
    for n, first, again in got:
        most = min(16 << 20, max(512 << 10, 8 * n + (1 << 20)))  # eight slots, rounded to 64 KB
        assert 0 < first <= most + 4096, n
        assert again == 0, n


@pytest.mark.parametrize("n", [3000, 400001])
def test_a_block_level_is_waited_for_before_its_read(counted, n):
    """The last kernel of a block's level is the read's, and it is launched
    when the level is done: the read's threads do not poll for the level."""
    got = counted("""
n = %d
g = graph(n)
off = g.out_offsets
b, e = n // 3, n
with dmm.Context(0) as c:
    c.set_layout(0)
    c.upload(num_nodes=n, out_offsets=off[b:] - off[b], out_neighs=g.out_neighs[off[b]:], vbegin=b, vend=e)
    front = np.zeros(n, np.uint64)
    for density in (1, n // 2):  # swept and pushed
        front[:] = 0
        front[::density] = 3
        c.batch_block_level(front, np.zeros(e - b, np.uint64))
        out.append(counts.count_before_last_launch())
""" % n)
    assert got == [0, 0]


RUNS = """
g = dmm.build_graph(14, 16, False)
srcs = dmm.pick_sources(g, 64)
with dmm.Context(0) as c:
    c.upload(g)
    def rank(eps):
        return c.PageRankPull(20, eps, %d)[0]
    def batch(k):
        return c.bfs_batch64(srcs[:k])[0]
"""


@pytest.mark.parametrize("mode", [0, 1, 2])
def test_a_chain_is_captured_when_that_pays(counted, mode):
    """One graph for a first run, none for a second like it; a chain that is
    longer than the runs need is captured anew once, and one that is too short
    not by every run that it is too short for."""
    got = counted(RUNS % mode + """
    for call in [lambda: rank(1e-4)] * 30 + [lambda: batch(64)] * 30:
        counts.count_graphs()
        call()
        out.append(counts.count_graphs())
    counts.count_graphs()
    for eps in [1e-2, 1e-5] * 20:
        rank(eps)
    out.append(counts.count_graphs())
""")
    for runs in (got[:30], got[30:60]):
        assert runs[0] == 1 and runs[1] == 0 and sum(runs) <= 2, runs
    assert got[60] <= 8


def test_a_graph_that_cannot_be_had(counted):
    """The call that needs it reports the error; the calls after it are whole."""
    got = counted(RUNS % 2 + """
    want = [rank(eps) for eps in (1e-2, 1e-6)] + [batch(64)]
    for fail in range(4):
        c.upload(g)
        errors = 0
        counts.fail_graph(fail)
        for k in range(40):
            try:
                # Chains of every, of few and of more iterations; of a batch
                # with one length of chain and then another.
                r = [rank(1e-6 if k %% 12 == 11 else 1e-2)] + ([batch(64)] if k %% 3 == 0 else [])
            except RuntimeError:
                errors += 1
                continue
            assert np.array_equal(r[0], want[1 if k %% 12 == 11 else 0]), (fail, k)
            assert len(r) == 1 or np.array_equal(r[1], want[2]), (fail, k)
        counts.fail_graph(-1)
        out.append(errors)
""".replace("%%", "%"))
    assert got[:3] == [1, 1, 1] and got[3] <= 1


def test_a_block_level_fills_the_card_whatever_a_search_is_tuned_to(counted):
    """Workgroups per CU that a search is tuned to (1 to 4, which make no
    difference to a small graph's) are not a block level's."""
    got = counted("""
g = graph(5000)
with dmm.Context(0) as c:
    c.set_layout(0)
    c.upload(g)
    for per_cu in (8, 1, 2, 4):
        t = c.get_tuning()
        t.grid_per_cu = per_cu
        c.set_tuning(t)
        c.batch_block_level(np.ones(5000, np.uint64), np.zeros(5000, np.uint64))
        counts.count_largest_grid()
        c.batch_block_level(np.ones(5000, np.uint64), np.zeros(5000, np.uint64))
        out.append(counts.count_largest_grid())
""")
    assert got[0] > 0 and got == got[:1] * 4
