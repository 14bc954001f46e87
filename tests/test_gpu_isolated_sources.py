"""Multi-source calls none of whose sources has an out-edge: rows of INF but for
the source, sums of zero, nothing traversed."""
import numpy as np
import pytest

from conftest import dawn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("count", [0, 1, 70])
def test_only_isolated_sources(weighted, count):
    n = 500
    print(f"case: {n} vertices, {count} isolated sources, weighted={weighted}", flush=True)
    u = np.arange(99, dtype=np.int32)  # a path; the vertices from 100 on are isolated
    g = dawn.Graph(dawn.HostGraph.from_edges(n, u, u + 1, np.full(99, 7, np.int32) if weighted else None))
    src = (100 + np.arange(count) * 13 % 400).astype(np.int32)
    want = np.full((count, n), dawn.INF, np.int32)
    want[np.arange(count), src] = 0
    for p in ("fixed", "learned", "push"):
        out = dawn.DeviceArray((max(count, 1), n), np.int32).fill_bytes(0x5A)
        _, sums, st = g.mssp(src, policy=p, out=out, stats=True)
        assert np.array_equal(out.download().reshape(-1, n)[:count], want), p
        assert st["skipped_sources"] == count and st["vertices_reached"] == count and st["edges_reached"] == 0, p
        if not weighted:
            assert st["steps"] == 0 and st["batches"] == 0, p
        dist, sums = g.mssp(src, policy=p)
        assert np.array_equal(dist, want) and not sums.any(), p
        assert not g.closeness(src, policy=p)[1].any(), p
    g.close()
