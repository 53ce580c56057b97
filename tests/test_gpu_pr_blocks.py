"""The compensated iteration of a PE block (propagation layout) at the edges
of its row classes and value ranges.

Every row's new score must be base + damp * (the exact sum of its in-
neighbours' contributions, rounded once to FP32), bit for bit; the row sums
come from dmm_pr_blocks_check, which tests/test_pr_blocks.py holds to
Python-integer sums.  Value ranges: inside the range that is summed in two
doubles (0 or [2^-57, 1/4]), at its ends, and outside it (larger, smaller,
one stray value), where the integers are used."""
import ctypes as C

import numpy as np
import pytest

import dist_mem_gapbs_amd._lib as L

pytestmark = pytest.mark.gpu

# Rows around every class boundary (8, 256) and the bucket sizes (1024, 16384).
LENGTHS = [0, 1, 7, 8, 9, 63, 255, 256, 257, 1023, 1024, 1025, 4000, 16383, 16384, 16385, 40000] + [2] * 2500 + [31] * 90


def _values(kind, n, rng):
    if kind == "ends":
        return rng.choice(np.array([0.25, 2.0 ** -57, 1.5 * 2.0 ** -57, 0.0, -0.25, 0.249], np.float32), n)
    x = np.exp(rng.uniform(np.log(1e-12), np.log(0.2), n)).astype(np.float32)
    if kind == "signed":
        x[rng.random(n) < 0.5] *= -1
    elif kind == "large":
        x *= np.float32(1e6)
    elif kind == "small":
        x *= np.float32(1e-12)  # some below 2^-57, where bits are cut off
    elif kind == "stray":
        x[rng.integers(0, n, 3)] = 0.5
    return x


@pytest.mark.parametrize("kind", ["rank", "signed", "ends", "large", "small", "stray"])
@pytest.mark.parametrize("n_gather", [40003, 300007])
def test_block_sums_exact(dmm, kind, n_gather):
    rng = np.random.default_rng([n_gather, len(kind), ord(kind[0])])
    lengths = rng.permutation(np.array(LENGTHS, np.int64))
    rows = len(lengths)
    off = np.concatenate(([0], np.cumsum(lengths)))
    src = rng.integers(0, n_gather, off[-1]).astype(np.int32)
    contrib = _values(kind, n_gather, rng)
    inc = np.empty(rows, np.float32)
    st = np.zeros(6, np.int64)
    lib = L.load()
    assert lib.dmm_pr_blocks_check(rows, n_gather, L.ptr(off, C.c_int64), L.ptr(src, C.c_int32),
                                   L.ptr(contrib, C.c_float), L.ptr(inc, C.c_float), L.ptr(st, C.c_int64)) == 0
    base = (np.float32(1.0) - np.float32(0.85)) / np.float32(n_gather)
    with np.errstate(all="ignore"):
        expect = (base + (np.float32(0.85) * inc).astype(np.float32)).astype(np.float32)
    begin = 1000
    with dmm.Context(0) as c:
        c.set_layout(L.DMM_LAYOUT_NATURAL)
        c.upload(num_nodes=n_gather, out_offsets=np.arange(rows + 1), out_neighs=np.zeros(rows, np.int32),
                 in_offsets=off, in_neighs=src, vbegin=begin, vend=begin + rows)
        for _ in range(2):  # the first call builds the layout
            got, _, _ = c.pr_block_iteration(contrib, np.zeros(rows, np.float32), L.DMM_PR_FP32_KAHAN)
            assert np.array_equal(got, expect)


def test_coarse_block_sums_exact(dmm):
    """A block of like rows from many windows, which takes coarse buckets: every
    row as the host's replay of the layout, bit for bit."""
    n_gather, m = 1 << 26, 36 << 20
    rng = np.random.default_rng(26)
    rows = m // 32
    lengths = np.full(rows, 32)
    lengths[:4000] = rng.integers(0, 65, 4000)
    lengths[100] = 600000  # in parts
    lengths[-1] += 5
    off = np.concatenate(([0], np.cumsum(lengths)))
    src = rng.integers(0, n_gather, off[-1], dtype=np.int32)
    contrib = (rng.random(n_gather, np.float32) / np.float32(n_gather)).astype(np.float32)
    lib = L.load()
    us, inc, st = np.zeros(2), np.empty(rows, np.float32), np.zeros(6, np.int64)
    assert lib.dmm_pr_blocks_shape(rows, n_gather, L.ptr(off, C.c_int64), L.ptr(src, C.c_int32), 256,
                                   L.ptr(us, C.c_double)) == 0
    assert lib.dmm_pr_blocks_check(rows, n_gather, L.ptr(off, C.c_int64), L.ptr(src, C.c_int32),
                                   L.ptr(contrib, C.c_float), L.ptr(inc, C.c_float), L.ptr(st, C.c_int64)) == 0
    base = (np.float32(1.0) - np.float32(0.85)) / np.float32(n_gather)
    expect = (base + (np.float32(0.85) * inc).astype(np.float32)).astype(np.float32)
    with dmm.Context(0) as c:
        c.set_layout(L.DMM_LAYOUT_NATURAL)
        c.upload(num_nodes=n_gather, out_offsets=np.arange(rows + 1), out_neighs=np.zeros(rows, np.int32),
                 in_offsets=off, in_neighs=src, vbegin=7, vend=7 + rows)
        for _ in range(2):
            got, _, _ = c.pr_block_iteration(contrib, np.zeros(rows, np.float32), L.DMM_PR_FP32_KAHAN)
            assert np.array_equal(got, expect)
