"""GPU check of the compaction's segment scan on both sides of the vertex
count at which its block grows: frontiers spread over all segments."""
import numpy as np
import pytest

import thievory_amd as T

pytestmark = pytest.mark.gpu

LIMIT = 256 * 64 * 4096  # segments x tiles x vertices


@pytest.mark.parametrize("n", [LIMIT, LIMIT + 1, LIMIT + 70000])
def test_levels_over_all_segments(n):
    """Vertex 0 -> 20,000 vertices spread over the ids, each -> its successor."""
    print("case: segments of", n, "vertices", flush=True)
    k = 20000
    a = 1 + np.arange(k, dtype=np.int64) * ((n - 3) // (k - 1))
    off = np.zeros(n + 1, np.uint64)
    off[1] = k
    off[a + 1] += 1
    np.cumsum(off, out=off)
    dst = np.concatenate([a, a + 1]).astype(np.uint32)
    g = T.Graph.from_arrays(off, dst)
    lv, st = g.bfs(0)
    ref = np.full(n, n + 1, np.uint32)
    ref[a + 1], ref[a], ref[0] = 3, 2, 1
    assert a[-1] + 1 < n and np.array_equal(lv, ref)
    assert st.reached == 2 * k + 1 and st.edges_traversed == 2 * k
