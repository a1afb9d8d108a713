"""GPU check of the reached count made by the copy to the caller: vertex
counts at the least size that goes through pinned slots and with every
remainder of a 16-byte load, several copies through one ring, and graphs of
several threads that share the rings."""
import threading

import numpy as np
import pytest

import thievory_amd as T

pytestmark = pytest.mark.gpu

LEAST = (6 << 20) // 4


def _star(n, first, step):
    """Vertex 0 -> every step-th vertex from `first` on, all weights 3."""
    dst = np.arange(first, n, step, dtype=np.uint32)
    off = np.zeros(n + 1, np.uint64)
    off[1:] = len(dst)
    return T.Graph.from_arrays(off, dst, np.full(len(dst), 3, np.uint32)), dst


def _check(g, n, dst, out):
    for fn, val in ((g.bfs, 2), (g.sssp, 4)):
        lv, st = fn(0, out=out)
        ref = np.full(n, n + 1, np.uint32)
        ref[dst], ref[0] = val, 1
        assert np.array_equal(lv, ref)
        assert st.reached == len(dst) + 1, (n, st.reached)
    lv, st = g.bfs(n - 1, out=out)  # no edges
    assert st.reached == 1 and np.count_nonzero(lv != n + 1) == 1


@pytest.mark.parametrize("n", [LEAST - 1, LEAST, LEAST + 1, LEAST + 2, LEAST + 3,
                               (1 << 21) + 2, (12 << 20) // 4 + 1])
def test_count_of_copied_values(n):
    print("case: count of", n, "copied values", flush=True)
    g, dst = _star(n, 5, 7)
    for out in (None, np.arange(n, dtype=np.uint32)):
        _check(g, n, dst, out)


def test_threads_share_rings():
    print("case: rings of several threads", flush=True)
    bad = []

    def run(i):
        try:
            n = LEAST + 1000 * i + i
            g, dst = _star(n, 2 + i, 3 + i)
            for _ in range(4):
                _check(g, n, dst, None)
            g.close()
        except BaseException as e:  # shown by the main thread
            bad.append((i, repr(e)[:300]))

    th = [threading.Thread(target=run, args=(i,)) for i in range(4)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not bad, bad
