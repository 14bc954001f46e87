"""Launch knobs and the route of a small graph's multi-source calls: a
workgroup per source (its steps count as push) unless knobs of the engine of
lanes were set to something else than the library's own choice."""
import numpy as np
import pytest

from conftest import dawn

pytestmark = pytest.mark.gpu


def modes(g, weighted):
    src = dawn.gen_sources(g.n, 64, 5)
    want, _ = g.mssp(src, policy="push")
    dist, _, st = g.mssp(src, policy="fixed", stats=True)
    assert np.array_equal(dist, want)
    return st["mode_steps"]


@pytest.mark.parametrize("weighted", [False, True])
def test_knobs_written_back_keep_the_route(weighted):
    print(f"case: directed random graph of 1500 vertices, degree 24, weighted={weighted}", flush=True)
    rng = np.random.default_rng(8)
    u, v = (rng.integers(0, 1500, 36_000).astype(np.int32) for _ in range(2))
    w = rng.integers(1, 900, 36_000).astype(np.int32) if weighted else None
    g = dawn.Graph(dawn.HostGraph.from_edges(1500, u, v, w, symmetrize=False))
    first = modes(g, weighted)
    assert first["pull"] == 0
    own = g.knobs()
    g.set_knobs(**own)
    assert modes(g, weighted) == first
    g.set_knobs(ss_chunk=5)  # a knob of the single-source engine
    assert modes(g, weighted) == first
    g.set_knobs(dense_blocks=own["dense_blocks"] + 1)
    assert modes(g, weighted)["pull"] > 0
    g.set_knobs(**own)
    assert modes(g, weighted) == first
    g.close()


def test_tuned_knobs_keep_the_route():
    """The tuner's choice is the library's own, also when it is written back."""
    print("case: directed random graph of 1500 vertices, degree 50, tuned", flush=True)
    rng = np.random.default_rng(9)
    u, v = (rng.integers(0, 1500, 75_000).astype(np.int32) for _ in range(2))
    g = dawn.Graph(dawn.HostGraph.from_edges(1500, u, v, symmetrize=False))
    dawn.tune(g)
    assert modes(g, False)["pull"] == 0
    g.set_knobs(**g.knobs())
    assert modes(g, False)["pull"] == 0
    g.close()
