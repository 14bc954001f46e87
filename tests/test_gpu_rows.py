"""Distance rows in managed memory: multi-source calls by either route, the
uneven batch and single-source calls write what they write to device memory."""
import ctypes

import numpy as np
import pytest

from conftest import dawn

pytestmark = pytest.mark.gpu


class Managed:
    """int32 managed memory, filled with 7."""

    def __init__(self, count):
        self.p = ctypes.c_void_p()
        if dawn.lib().hipMallocManaged(ctypes.byref(self.p), ctypes.c_size_t(4 * count), 1):
            pytest.skip("no managed memory")
        self.a = np.ctypeslib.as_array(ctypes.cast(self.p, ctypes.POINTER(ctypes.c_int32)), (count,))
        self.a[:] = 7

    def __del__(self):
        if self.p:
            dawn.lib().hipFree(self.p)


def i32(a):
    return a.ctypes.data_as(ctypes.POINTER(ctypes.c_int32))


# Weighted rows that the kernel lowers distances in (more than 37,797 vertices),
# rows that it only writes, and rows of the engine of lanes.
@pytest.mark.parametrize("n,weighted,policy", [(40_000, True, "fixed"), (2000, True, "fixed"), (2000, True, "push"),
                                               (2000, False, "fixed"), (2000, False, "push")])
def test_mssp(orc, n, weighted, policy):
    print(f"case: {n} vertices, weighted={weighted}, {policy}, 65 managed rows", flush=True)
    h = dawn.HostGraph.er(n, 6.0, 3, weighted=weighted)
    g = dawn.Graph(h)
    src = dawn.gen_sources(n, 65, 4).astype(np.int32)
    out = Managed(65 * n + 1)
    assert dawn.lib().dawn_mssp(g.handle, i32(src), 65, out.p, None, dawn.POLICIES[policy], None) == 0
    assert np.array_equal(out.a[:-1].reshape(65, n), orc.mssp(h.row_ptr, h.col, h.weight if weighted else None, src)[0])
    assert out.a[-1] == 7
    g.close()


@pytest.mark.parametrize("weighted", [False, True])
def test_batch_and_single(orc, weighted):
    print(f"case: 2000 and 40,000 vertices, weighted={weighted}, managed rows", flush=True)
    hs = [dawn.HostGraph.er(n, 6.0, n, weighted=weighted) for n in (2000, 40_000)]
    gs = [dawn.Graph(h) for h in hs]
    src = np.array([5, 6, 7, 8], np.int32)
    at = np.array([3, 3 + 2 * 2000 + 11], np.int64)  # what lies between the rows stays
    out = Managed(int(at[1]) + 2 * 40_000 + 5)
    hd = (ctypes.c_void_p * 2)(*[g.handle.value for g in gs])
    assert dawn.lib().dawn_batch_mssp(hd, 2, i32(src), 2, out.p, at.ctypes.data_as(ctypes.POINTER(ctypes.c_int64)),
                                      None) == 0
    keep = np.ones(len(out.a), bool)
    for i, h in enumerate(hs):
        w = h.weight if weighted else None
        end = int(at[i]) + 2 * h.n
        assert np.array_equal(out.a[at[i]:end].reshape(2, h.n), orc.mssp(h.row_ptr, h.col, w, src[2 * i:2 * i + 2])[0])
        keep[at[i]:end] = False
        fn = dawn.lib().dawn_sssp if weighted else dawn.lib().dawn_bfs
        row = Managed(h.n)
        assert fn(gs[i].handle, 9, row.p, 0, None) == 0
        assert np.array_equal(row.a, orc.mssp(h.row_ptr, h.col, w, [9])[0][0])
    assert (out.a[keep] == 7).all()
