"""The serial mode's sums (src/pr.cc:57-59) at the edges of its row classes:
bundles of light and heavy rows, rows of a wavefront, rows of a workgroup.

One block iteration from given contributions, each row's sum compared bit for
bit with FP32 additions one after another (numpy's cumulative sum in float32).
The contributions are chosen for what composing additions could get wrong:
exact halves of the running sum's unit (small dyadic numbers), sums that stay
in or leave a binade at every place, zeros, subnormals, signs, infinities and
NaN."""
import numpy as np
import pytest

import dist_mem_gapbs_amd._lib as L

pytestmark = pytest.mark.gpu

# Row lengths around every boundary (64, 512, 32768), bundle and step sizes.
LENGTHS = [0, 1, 7, 8, 9, 15, 16, 17, 31, 63, 64, 65, 95, 96, 97, 128, 255, 300, 511, 512, 513, 519, 520, 521, 1023,
           1024, 1025, 5000, 8191, 32767, 32768, 32769, 40961, 70001] + [3] * 70 + [64] * 17 + [200] * 33


def _values(kind, n, rng):
    if kind == "rank":
        return (rng.exponential(1.0, n) / n).astype(np.float32)
    if kind == "halves":  # multiples of 2^-12 below 1: exact halves from sums of 2^11 on
        return (rng.integers(0, 1 << 12, n) * 2.0 ** -12).astype(np.float32)
    if kind == "ones":
        return np.ones(n, np.float32)
    if kind == "big_halves":  # half the unit of 2^24 now and then, after large values
        return np.where(rng.random(n) < 0.01, 2.0 ** 20, rng.integers(1, 8, n) * 0.5).astype(np.float32)
    if kind == "wide":
        return np.exp2(rng.uniform(-100, 20, n)).astype(np.float32)
    if kind == "tiny":
        return (rng.integers(0, 3, n) * np.float32(1e-45)).astype(np.float32)
    if kind == "signed":
        return rng.standard_normal(n).astype(np.float32)
    x = rng.exponential(1.0, n).astype(np.float32)  # special
    x[rng.integers(0, n, 3)] = np.inf
    x[rng.integers(0, n, 2)] = np.nan
    x[rng.integers(0, n, n // 10)] = -0.0
    return x


# 20011 sources: all in the LDS hub.  90001: none of them.
@pytest.mark.parametrize("n", [20011, 90001])
@pytest.mark.parametrize("kind", ["rank", "halves", "ones", "big_halves", "wide", "tiny", "signed", "special"])
def test_serial_sums_bit_exact(dmm, n, kind):
    rng = np.random.default_rng([n, len(kind)])
    lengths = np.zeros(n, np.int64)
    rows = rng.permutation(n)[:len(LENGTHS)]
    lengths[rows] = LENGTHS
    off = np.concatenate(([0], np.cumsum(lengths)))
    src = rng.integers(0, n, off[-1]).astype(np.int32)
    contrib = _values(kind, n, rng)
    with dmm.Context(0) as c:
        c.set_layout(L.DMM_LAYOUT_NATURAL)
        c.upload(num_nodes=n, out_offsets=np.arange(n + 1), out_neighs=np.zeros(n, np.int32), in_offsets=off,
                 in_neighs=src)
        got, _, _ = c.pr_block_iteration(contrib, np.zeros(n, np.float32), L.DMM_PR_FP32_SERIAL)
    base = (np.float32(1) - np.float32(0.85)) / np.float32(n)
    with np.errstate(all="ignore"):
        for r in rows:
            x = contrib[src[off[r]:off[r + 1]]]
            total = np.add.accumulate(np.concatenate((np.zeros(1, np.float32), x)), dtype=np.float32)[-1]
            want = np.float32(base + np.float32(np.float32(0.85) * total))
            assert got[r] == want or (np.isnan(got[r]) and np.isnan(want)), (r, lengths[r], got[r], want)


# Where a workgroup takes over from a wavefront: 32768 in-edges, halved down to
# 2048 while a graph has less than that many edges for each of 256 workgroups.
TAKEOVER = [1026, 1536, 1537, 2047, 2048, 2049, 4095, 4096, 4097, 5003, 8191, 8192, 8193, 16383, 16384, 16385, 20011,
            32767, 32768, 32769, 40961]


@pytest.mark.parametrize("n,edges", [(20011, 500_000), (90001, 2_200_000), (20011, 8_600_000)])
@pytest.mark.parametrize("kind", ["rank", "halves", "ones", "big_halves", "wide", "tiny", "signed", "special"])
def test_serial_rows_around_the_takeover(dmm, n, edges, kind):
    """The same rows in graphs of more and more edges (the rest in short rows):
    the longest go to workgroups from 2048, from 8192 and from 32768 in-edges
    on, those below to a wavefront each."""
    rng = np.random.default_rng([n, edges, len(kind)])
    lengths = np.zeros(n, np.int64)
    fill = max(0, edges - sum(TAKEOVER))
    lengths[:] = rng.integers(0, 2 * fill // n + 1, n)
    rows = rng.permutation(n)[:len(TAKEOVER)]
    lengths[rows] = TAKEOVER
    off = np.concatenate(([0], np.cumsum(lengths)))
    src = rng.integers(0, n, off[-1]).astype(np.int32)
    contrib = _values(kind, n, rng)
    with dmm.Context(0) as c:
        c.set_layout(L.DMM_LAYOUT_NATURAL)
        c.upload(num_nodes=n, out_offsets=np.arange(n + 1), out_neighs=np.zeros(n, np.int32), in_offsets=off,
                 in_neighs=src)
        got, _, _ = c.pr_block_iteration(contrib, np.zeros(n, np.float32), L.DMM_PR_FP32_SERIAL)
    base = (np.float32(1) - np.float32(0.85)) / np.float32(n)
    with np.errstate(all="ignore"):
        for r in np.concatenate((rows, rng.integers(0, n, 60))):
            x = contrib[src[off[r]:off[r + 1]]]
            total = np.add.accumulate(np.concatenate((np.zeros(1, np.float32), x)), dtype=np.float32)[-1]
            want = np.float32(base + np.float32(np.float32(0.85) * total))
            assert got[r] == want or (np.isnan(got[r]) and np.isnan(want)), (r, lengths[r], got[r], want)
