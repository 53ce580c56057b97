"""Performance cases: what a program that uses this engine has it do.

Each case is one pass through the public Python API on graphs made from a
seed.  Two graph families are used, the ones the engine's own generator makes:
Kronecker (R-MAT A/B/C = .57/.19/.19, IDs permuted) and uniform random
pairs.  They are drawn here with torch, so that every seed is another graph
and the vertex count need not be a power of two.

Kinds of pass:

  bfs     `searches` direction-optimizing searches from picked sources, one
          after the other.  One search: the default call, parents and depths
          on the host.  Several: the benchmark loop, whose trees stay in
          HBM, and the last one read back.  The depths are the output:
          parents are not compared, since any frontier neighbour may win a
          top-down claim.
  batch   one 64-lane batched search, depths of every lane on the host.
  levels  one 64-lane batched search that keeps its level words in HBM, as a
          partitioned run does, and the words of its first three levels.
  rank    a whole PageRank in one of its three arithmetic modes.
  share   one PageRank iteration of one block of a partitioned graph, on
          device buffers (the serving form, which allocates nothing).
  paths   Brandes' forward phase: depths, path counts, successor bits.
"""
import ctypes

import numpy as np
import torch

import dist_mem_gapbs_amd as dmm
from dist_mem_gapbs_amd import _lib as abi

MODES = {"serial": dmm.DMM_PR_FP32_SERIAL, "kahan": dmm.DMM_PR_FP32_KAHAN, "fp64": dmm.DMM_PR_FP64}


def _case(kind, family, n, degree, **more):
    base = {"kind": kind, "family": family, "n": n, "degree": degree, "directed": False}
    base.update(more)
    return base


def listed():
    def named(name, case):
        return dict(case, name=name)
    return [
        # The smallest configuration of the benchmark: 32,768 vertices, 8
        # pairs each; one search, its result read.  Latency and launches.
        named("bfs_uniform15", _case("bfs", "uniform", 1 << 15, 8, searches=1)),
        # An interactive query on a mid-sized graph of ragged size.
        named("bfs_kron18_ragged", _case("bfs", "kron", 200003, 13, searches=1)),
        # The headline workload: 64 sources on Kronecker-22, results in HBM.
        named("bfs_kron22_x64", _case("bfs", "kron", 1 << 22, 16, searches=64)),
        # Links that point one way only, no hubs, most levels wide.
        named("bfs_uniform21_directed_x16", _case("bfs", "uniform", 1900007, 12, searches=16, directed=True)),
        # All depths of 64 sources for a program that goes on with them.
        named("batch_kron17", _case("batch", "kron", 1 << 17, 16, lanes=64)),
        # The partitioned run's batched search: wide frontiers, kept in HBM.
        named("levels_uniform22_ragged", _case("levels", "uniform", 3700001, 16, lanes=64)),
        # The default call: the reference's arithmetic, stopped at 1e-4.
        named("rank_serial_kron14", _case("rank", "kron", 1 << 14, 16, mode="serial", iters=20, eps=1e-4)),
        # The same at a size where it is worth a GPU.
        named("rank_serial_kron21", _case("rank", "kron", 1 << 21, 16, mode="serial", iters=20, eps=1e-4)),
        # The compensated mode, 20 iterations, as the benchmark runs it.
        named("rank_kahan_kron22", _case("rank", "kron", 1 << 22, 16, mode="kahan", iters=20, eps=0.0)),
        # Double precision throughout, a ragged size.
        named("rank_fp64_kron21_ragged", _case("rank", "kron", 1700003, 19, mode="fp64", iters=20, eps=0.0)),
        # Block 3 of 8 of a partitioned graph, one compensated iteration.
        named("share_kahan_kron23", _case("share", "kron", 1 << 23, 16, mode="kahan", parts=8, part=3)),
        # Shortest-path counts of one source, read back.
        named("paths_kron19_ragged", _case("paths", "kron", 480013, 17)),
    ]


def _size(rng, low, high):
    """A vertex count spread over the logarithm of the range, any parity."""
    return int(round(low * (high / low) ** rng.random()))


def draw(rng):
    kind = rng.choice(["bfs", "bfs", "batch", "levels", "rank", "rank", "rank", "share", "paths"])
    family = rng.choice(["kron", "kron", "uniform"])
    degree = rng.randint(6, 16)
    if kind == "bfs":
        searches = rng.choice([1, 1, 4, 16])
        return _case(kind, family, _size(rng, 20000, 2500000), degree, searches=searches, directed=rng.random() < 0.3)
    if kind == "batch":
        return _case(kind, family, _size(rng, 20000, 250000), degree, lanes=rng.randint(1, 64))
    if kind == "levels":
        return _case(kind, family, _size(rng, 50000, 3000000), degree, lanes=64)
    if kind == "rank":
        eps = rng.choice([0.0, 1e-4])
        return _case(kind, family, _size(rng, 16000, 2000000), degree, mode=rng.choice(sorted(MODES)),
                     iters=rng.randint(10, 20), eps=eps, directed=rng.random() < 0.2)
    if kind == "share":
        parts = rng.randint(2, 8)
        return _case(kind, family, _size(rng, 200000, 4000000), degree, mode=rng.choice(["serial", "kahan"]),
                     parts=parts, part=rng.randrange(parts))
    return _case(kind, family, _size(rng, 20000, 450000), degree)


# ---- inputs -----------------------------------------------------------------


def _pairs(case, seed):
    """The edge list (pairs x 2, int32) of the case's graph, a torch tensor
    on the GPU."""
    g = torch.Generator(device="cuda").manual_seed(int(seed) * 1000003 + 17)
    n, count = case["n"], case["n"] * case["degree"]
    if case["family"] == "uniform":
        return torch.randint(0, n, (count, 2), generator=g, device="cuda", dtype=torch.int32)
    scale = max(1, (n - 1).bit_length())
    u = torch.zeros(count, dtype=torch.int32, device="cuda")
    v = torch.zeros(count, dtype=torch.int32, device="cuda")
    for _ in range(scale):
        r = torch.rand(count, generator=g, device="cuda")
        u = 2 * u + (r >= 0.76)
        v = 2 * v + (((r >= 0.57) & (r < 0.76)) | (r >= 0.95))
    order = torch.randperm(1 << scale, generator=g, device="cuda", dtype=torch.int32)
    u, v = order[u], order[v]
    keep = (u < n) & (v < n)
    return torch.stack((u[keep], v[keep]), 1).to(torch.int32)


def _sources(case, seed, degrees, count):
    """`count` sources with an out-edge, as the benchmark picks them."""
    rng = np.random.default_rng([int(seed), 5])
    picked = []
    while len(picked) < count:
        v = rng.integers(0, case["n"], 4 * count)
        picked += [int(x) for x in v[degrees[v] > 0]]
    return picked[:count]


def _block(case):
    p = dmm.partition(case["n"], case["parts"], case["part"])
    return p["start"], p["end"]


def _contributions(case, seed, degrees):
    """Scores of a rank under way (spread over a decade or so) and what each
    vertex hands on; float32."""
    rng = np.random.default_rng([int(seed), 7])
    scores = ((0.15 + rng.exponential(0.85, case["n"])) / case["n"]).astype(np.float32)
    with np.errstate(divide="ignore"):
        return scores, (scores / degrees.astype(np.float32)).astype(np.float32)


def prepare(case, seed):
    kind = case["kind"]
    ctx = dmm.Context(0)
    pairs = _pairs(case, seed).cpu().numpy()
    graph = ctx.build_graph(pairs, case["n"], symmetrize=not case["directed"])
    del pairs
    degrees = np.diff(graph.out_offsets)
    state = {"case": dict(case), "ctx": ctx}
    if kind == "share":
        b, e = _block(case)
        off = graph.out_offsets
        ctx.set_layout(abi.DMM_LAYOUT_NATURAL)
        ctx.upload(num_nodes=case["n"], out_offsets=off[b:e + 1] - off[b], out_neighs=graph.out_neighs[off[b]:off[e]],
                   vbegin=b, vend=e, num_edges_directed=graph.num_edges_directed)
        scores, contrib = _contributions(case, seed, degrees)
        # The block's layout is built by its first allocating iteration.
        ctx.pr_block_iteration(contrib, scores[b:e], MODES[case["mode"]])
        state["contrib"] = torch.from_numpy(contrib).cuda()
        state["scores"] = torch.from_numpy(scores[b:e]).cuda()
        state["contrib_out"] = torch.zeros(e - b, dtype=torch.float32, device="cuda")
        state["error"] = torch.zeros(1, dtype=torch.float64, device="cuda")
    else:
        if kind == "paths":
            ctx.set_layout(abi.DMM_LAYOUT_NATURAL)
        ctx.upload(graph)
        count = {"bfs": case.get("searches"), "batch": case.get("lanes"), "levels": case.get("lanes")}.get(kind, 1)
        state["sources"] = _sources(case, seed, degrees, count)
    if kind == "paths":
        # The program's result buffers, kept from source to source; the
        # successor bits have room for a graph without a duplicate pair.
        state["depth"] = np.zeros(case["n"], np.int32)
        state["counts"] = np.zeros(case["n"], np.uint64)
        state["successors"] = np.zeros((2 * case["n"] * case["degree"] + 63) // 64, np.uint64)
    graph.free()
    torch.cuda.synchronize()
    return state


# ---- one pass ---------------------------------------------------------------


def run(state):
    case, ctx = state["case"], state["ctx"]
    kind = case["kind"]
    if kind == "bfs":
        for source in state["sources"][:-1]:
            ctx.DOBFS(source, read=False, with_stats=False)
        parent, depth, _ = ctx.DOBFS(state["sources"][-1], with_stats=False)
        return depth
    if kind == "batch":
        depth, stats = ctx.bfs_batch64(state["sources"])
        return {"depth": depth, "reached_edges": stats.reached_edges}
    if kind == "levels":
        _, stats = ctx.bfs_batch64(state["sources"], want_depth=False)
        return {"active": list(stats.level_active[:stats.num_levels]),
                "words": [ctx.batch_read_level(k).view(np.int64) for k in range(3)]}
    if kind == "rank":
        scores, stats = ctx.PageRankPull(case["iters"], case["eps"], MODES[case["mode"]])
        return {"scores": scores, "changes": np.array(stats.err[:stats.iters])}
    if kind == "share":
        ctx._check(ctx._lib.dmm_pr_block_iteration_noalloc(
            ctx._h, ctypes.c_void_p(state["contrib"].data_ptr()), ctypes.c_void_p(state["scores"].data_ptr()),
            ctypes.c_void_p(state["contrib_out"].data_ptr()), MODES[case["mode"]],
            ctypes.c_void_p(state["error"].data_ptr())))
        return {"scores": state["scores"], "contrib": state["contrib_out"]}
    levels = ctypes.c_int32()
    ctx._check(ctx._lib.dmm_bc_forward(
        ctx._h, state["sources"][0], abi.ptr(state["depth"], ctypes.c_int32), abi.ptr(state["counts"], ctypes.c_uint64),
        abi.ptr(state["successors"], ctypes.c_uint64), ctypes.byref(levels)))
    return {"depth": state["depth"], "counts": state["counts"].view(np.int64),
            "successors": state["successors"].view(np.int64), "levels": levels.value}


# ---- what a pass cannot do without --------------------------------------------


def work(case):
    """Bytes: each input read once, each output written once.  A search
    needs, of each vertex, its row bounds and one in-neighbour, and writes a
    parent (a depth too where it is read)."""
    n = case["n"]
    m = case["n"] * case["degree"] * (1 if case["directed"] else 2)
    kind = case["kind"]
    if kind == "bfs":
        return {"bytes": case["searches"] * 16 * n + 4 * n, "flops": 0}
    if kind == "batch":
        return {"bytes": 4 * m + 8 * n + case["lanes"] * n, "flops": 0}
    if kind == "levels":
        return {"bytes": 4 * m + 8 * n + 3 * 8 * n, "flops": 0}
    if kind == "rank":
        size = 8 if case["mode"] == "fp64" else 4
        iters = case["iters"] if case["eps"] == 0.0 else min(case["iters"], 7)
        return {"bytes": iters * ((4 + size) * m + (8 + 3 * size) * n), "flops": iters * (m + 3 * n)}
    if kind == "share":
        rows, edges = n // case["parts"], m // case["parts"]
        return {"bytes": 8 * edges + 20 * rows + 4 * n, "flops": edges + 3 * rows}
    return {"bytes": 4 * m + m // 8 + 20 * n, "flops": m}


# ---- the same in 64 bits --------------------------------------------------------


def _csr64(case, seed):
    """(keys, row, column, out-degrees) of the squished graph, rows the
    targets: duplicates and self-loops removed."""
    p = _pairs(case, seed).long()
    u, v = p[:, 0], p[:, 1]
    if not case["directed"]:
        u, v = torch.cat((u, v)), torch.cat((v, u))
    keep = u != v
    keys = torch.unique(v[keep] * case["n"] + u[keep])
    row, col = keys // case["n"], keys % case["n"]
    return row, col, torch.bincount(col, minlength=case["n"])


def exact(case, seed):
    n = case["n"]
    if case["kind"] == "rank":
        row, col, deg = _csr64(case, seed)
        # The constants are the program's: computed in float32.
        damp = float(np.float32(0.85))
        base = float((np.float32(1.0) - np.float32(0.85)) / np.float32(n))
        scores = torch.full((n,), float(np.float32(1.0) / np.float32(n)), dtype=torch.float64, device="cuda")
        changes = []
        for _ in range(case["iters"]):
            contrib = scores / deg
            new = base + damp * torch.zeros_like(scores).index_add_(0, row, contrib[col])
            changes.append(float((new - scores).abs().sum()))
            scores = new
            if changes[-1] < case["eps"]:
                break
        return {"scores": scores, "changes": np.array(changes)}
    if case["kind"] == "share":
        row, col, deg = _csr64(case, seed)
        _, contrib = _contributions(case, seed, deg.cpu().numpy())
        contrib = torch.from_numpy(contrib).cuda().double()
        b, e = _block(case)
        damp = float(np.float32(0.85))
        base = float((np.float32(1.0) - np.float32(0.85)) / np.float32(n))
        scores = (base + damp * torch.zeros(n, dtype=torch.float64, device="cuda").index_add_(0, row, contrib[col]))[b:e]
        return {"scores": scores, "contrib": scores / deg[b:e]}
    return None  # whole numbers
