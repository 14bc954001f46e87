"""Unweighted tasks of the uneven batch whose state is in memory (graphs of
more than 1,209,600 vertices): every width of the lane words, graphs whose last
task holds fewer lanes than the others, levels beyond the 16-bit level stage.
Rows bit-exact against the oracle or the closed form."""
import numpy as np
import pytest

from conftest import dawn

pytestmark = pytest.mark.gpu
N = 1_210_001  # a vertex more than a field of one bit each fits in LDS, rounded up


def graph(pairs, seed):
    """A random graph on the first 200,000 vertices, the others isolated."""
    rng = np.random.default_rng(seed)
    u, v = (rng.integers(0, 200_000, pairs).astype(np.int32) for _ in range(2))
    return dawn.HostGraph.from_edges(N, u, v)


# Lanes per task: all of them below 500,000 edges (one task), half of them from
# there on: 19 sources make tasks of 9, 9 and 1 lanes, 35 of 17, 17 and 1.
@pytest.mark.parametrize("pairs,spg,tasks", [
    (150_000, 8, 1), (150_000, 9, 1), (150_000, 17, 1), (150_000, 33, 1),
    (400_000, 3, 3), (400_000, 16, 2), (400_000, 19, 3), (400_000, 35, 3), (400_000, 64, 2)])
def test_lane_widths(orc, pairs, spg, tasks):
    print(f"case: {N} vertices, {pairs} pairs, {spg} sources, beside a small graph", flush=True)
    h, small = graph(pairs, spg), dawn.HostGraph.er(900, 4.0, 9)
    assert (h.m < 500_000) == (pairs < 250_000) and h.m < 2_000_000
    rng = np.random.default_rng(spg)
    src = rng.integers(0, 200_000, spg).astype(np.int32)
    src[-1] = src[0]            # a repeated source
    src[spg // 2] = N - 1       # an isolated one
    src2 = rng.integers(0, 900, spg).astype(np.int32)
    g, g2 = dawn.Graph(h), dawn.Graph(small)
    rows, st = dawn.batch_mssp([g2, g], np.concatenate([src2, src]), spg)
    assert tasks < st["batches"] <= tasks + -(-spg // 16)
    assert np.array_equal(rows[1], orc.mssp(h.row_ptr, h.col, None, src)[0])
    assert np.array_equal(rows[0], orc.mssp(small.row_ptr, small.col, None, src2)[0])
    g.close()
    g2.close()


@pytest.mark.parametrize("spg", [3, 9])
def test_levels_beyond_16_bits(spg):
    """Levels past 65,534 do not fit the stage and go to the rows at once."""
    k = 66_500
    print(f"case: path of {k} vertices and {N - k} isolated ones, {spg} sources", flush=True)
    u = np.arange(k - 1, dtype=np.int32)
    g = dawn.Graph(dawn.HostGraph.from_edges(N, u, u + 1))
    src = np.array([0, k - 1, 400, 65_000, 1, 2, 3, 33_000, N - 1], np.int32)[:spg]
    rows, _ = dawn.batch_mssp([g], src, spg)
    for i, s in enumerate(src):
        want = np.full(N, dawn.INF, np.int32)
        if s < k:
            want[:k] = np.abs(np.arange(k) - s)
        want[s] = 0
        assert np.array_equal(rows[0][i], want), s
    g.close()
