"""The engines of lanes on graphs small enough for a workgroup per source (a
knob set to another value than the library's choice keeps them there), under
the schedules that would take the other route: rows, sums and counts against
the oracle and against the other route."""
import numpy as np
import pytest

from conftest import dawn

pytestmark = pytest.mark.gpu


def lanes(g, **knobs):
    g.set_knobs(dense_blocks=g.knobs()["dense_blocks"] + 1, **knobs)
    return g


def device_rows(g, src, policy):
    out = dawn.DeviceArray((len(src), g.n), np.int32).fill_bytes(0x5A)
    _, sums, st = g.mssp(src, policy=policy, out=out, stats=True)
    return out.download(), sums, st


@pytest.mark.parametrize("n,degree", [(2, 1), (300, 4), (20_000, 10), (66_000, 3)])
@pytest.mark.parametrize("count", [1, 64, 257])
def test_unweighted_routes_agree(n, degree, count):
    print(f"case: {n} vertices, degree {degree}, {count} sources", flush=True)
    rng = np.random.default_rng(n + count)
    u, v = (rng.integers(0, n, n * degree).astype(np.int32) for _ in range(2))
    h = dawn.HostGraph.from_edges(n, u, v, symmetrize=n % 3 != 0)
    g = dawn.Graph(h)
    src = rng.integers(-n, 2 * n, count).astype(np.int32)
    rows, sums, st = device_rows(g, src, "learned")
    assert st["mode_steps"]["pull"] == st["mode_steps"]["bitmap"] == 0  # a workgroup per source
    lanes(g)
    for p in ("fixed", "learned"):
        want, wsums, wst = device_rows(g, src, p)
        assert np.array_equal(rows, want) and np.array_equal(sums, wsums), p
        assert np.array_equal(g.closeness(src, policy=p)[1], wsums), p
        for f in ("vertices_reached", "edges_reached", "skipped_sources", "batches", "steps"):
            assert st[f] == wst[f], (p, f)
    g.close()


@pytest.mark.parametrize("words,count", [(1, 130), (4, 300), (16, 1024 + 100), (16, 2048 + 40)])
def test_unweighted_batches(orc, words, count):
    """Full and partly filled batches, isolated sources, sums alone, every
    vertex a source."""
    print(f"case: RMAT scale 11 ef 8, {count} sources, lane_words={words}", flush=True)
    h = dawn.HostGraph.rmat(11, 8, 41)
    g = lanes(dawn.Graph(h), lane_words=words)
    src = np.random.default_rng(count).integers(0, h.n, count).astype(np.int32)
    odist, osums, skipped, _ = orc.mssp(h.row_ptr, h.col, None, src)
    for p in ("fixed", "learned"):
        rows, sums, st = device_rows(g, src, p)
        assert np.array_equal(rows, odist) and np.array_equal(sums, osums), p
        assert st["mode_steps"]["pull"] + st["mode_steps"]["bitmap"] > 0, p
        assert st["skipped_sources"] == int(skipped.sum()), p
        dist, hsums = g.mssp(src, policy=p)
        assert np.array_equal(dist, odist) and np.array_equal(hsums, osums), p
        assert np.array_equal(g.closeness(src, policy=p)[1], osums), p
    g.close()


@pytest.mark.parametrize("count", [1, 9, 17, 33, 65])
@pytest.mark.parametrize("kind", ["grid", "rmat"])
def test_weighted_batches(orc, kind, count):
    """Every record width under the rule that mixes push and pull steps."""
    print(f"case: weighted {kind}, {count} sources", flush=True)
    h = dawn.HostGraph.grid(60, 0.02, 3, weighted=True) if kind == "grid" else dawn.HostGraph.rmat(12, 16, 4, weighted=True)
    g = lanes(dawn.Graph(h))
    src = np.random.default_rng(count).integers(0, h.n, count).astype(np.int32)
    src[0] = int(np.argmax(h.degrees()))
    odist, osums, _, _ = orc.mssp(h.row_ptr, h.col, h.weight, src)
    for p in ("fixed", "learned"):
        rows, sums, st = device_rows(g, src, p)
        assert np.array_equal(rows, odist) and np.array_equal(sums, osums), p
        assert st["mode_steps"]["pull"] > 0, p
    g.close()


def test_hub_order(orc):
    print("case: RMAT scale 16 ef 8, 130 sources, hub-first order", flush=True)
    h = dawn.HostGraph.rmat(16, 8, 12)
    src = dawn.gen_sources(h.n, 130, 12)
    odist, osums, _, _ = orc.mssp(h.row_ptr, h.col, None, src)
    g = lanes(dawn.Graph(h), hub_order=1)
    for p in ("fixed", "learned"):
        dist, sums = g.mssp(src, policy=p)
        assert np.array_equal(dist, odist) and np.array_equal(sums, osums), p
    g.close()
