"""GPU check of values read back through the pinned ring (from 12 MB) and of
the reached count made on the GPU (from 2^17 values): vertex counts at those
limits, at a ring slot's and with remainders, into a fresh array and into a
kept one that holds other values."""
import numpy as np
import pytest

import thievory_amd as T

pytestmark = pytest.mark.gpu

MB = 1 << 20


@pytest.mark.parametrize("n", [(1 << 17) - 1, 1 << 17, 3 * MB - 1, 3 * MB, 3 * MB + 5,
                               7 * MB + MB // 2 + 1, 8 * MB, 9 * MB + 3])
def test_values_and_reached(n):
    print("case: readback of", n, "values", flush=True)
    # vertex 2 -> every third vertex from 6 on; the rest unreached
    dst = np.arange(6, n, 3, dtype=np.uint32)
    off = np.zeros(n + 1, np.uint64)
    off[3:] = len(dst)
    g = T.Graph.from_arrays(off, dst)
    ref = np.full(n, n + 1, np.uint32)
    ref[dst], ref[2] = 2, 1
    kept = np.arange(n, dtype=np.uint32)
    for out in (None, kept, kept):
        lv, st = g.bfs(2, out=out)
        assert np.array_equal(lv, ref)
        assert st.reached == len(dst) + 1
    lv, st = g.bfs(n - 1, out=kept)  # no edges
    assert st.reached == 1 and lv[n - 1] == 1 and np.all(lv[:n - 1] == n + 1)
    lab, st = g.cc()
    ref = np.arange(n, dtype=np.uint32)
    ref[dst] = 2
    assert np.array_equal(lab, ref) and st.reached == n
