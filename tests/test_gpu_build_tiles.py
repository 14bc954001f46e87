"""Device-side graph build around the tiles of its sort and its compaction:
the CSR downloaded from the device equals the host build's."""
import numpy as np
import pytest

from conftest import dawn
from test_gpu_build import log, same_csr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("count", [1, 63, 65, 2047, 2048, 2049, 4095, 4097, 8192, 70_001])
@pytest.mark.parametrize("weighted", [False, True])
def test_edge_counts_around_tiles(count, weighted):
    """Edge lists whose entries fill, just miss and just pass the tiles of the
    sort and the compaction (4096 entries), of few rows (long runs of one
    digit) and of many (rows without entries)."""
    for n in (3, 5_000_000):
        log(f"case: {count} edges on {n} vertices, weighted={weighted}")
        rng = np.random.default_rng(count)
        u, v = (rng.integers(0, n, count).astype(np.int32) for _ in range(2))
        w = rng.integers(0, 4, count).astype(np.int32) if weighted else None
        for sym, dedup in ((True, True), (False, False)):
            h = dawn.HostGraph.from_edges(n, u, v, w, symmetrize=sym, dedup=dedup)
            g = dawn.Graph.from_edges_device(n, u, v, w, symmetrize=sym, dedup=dedup)
            same_csr(g.download(), h)
            g.close()
