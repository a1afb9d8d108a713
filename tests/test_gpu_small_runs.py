"""GPU check of wide levels in the small-frontier kernel, where lanes whose
destinations share a bitmap word send one atomic together: lists of
consecutive and of spread ids, repeated records, lists that end inside a word,
and more vertices than the kernel's queue holds.  Levels equal the oracle's.
A dense list takes no longer than a spread one."""
import numpy as np
import pytest

from oracle import oracle as O
import thievory_amd as T

pytestmark = pytest.mark.gpu


def csr(n, src, dst):
    order = np.lexsort((dst, src))
    off = np.zeros(n + 1, np.uint64)
    off[1:] = np.cumsum(np.bincount(src, minlength=n))
    return O.CSR(off, dst[order].astype(np.uint32), None)


def hub_lists(kind, k, n):
    """Destinations of the hub (vertex 0): k records, sorted."""
    rng = np.random.default_rng(k)
    if kind == "consecutive":
        return 1 + np.arange(k)
    if kind == "repeated":                      # each id one to three times
        return np.sort(1 + np.repeat(np.arange(k), 1 + np.arange(k) % 3)[:k])
    if kind == "strides":                       # 1, 2, 31, 32, 33 in turn
        return 1 + np.cumsum(np.array([1, 2, 31, 32, 33])[np.arange(k) % 5]) % (n - 1)
    return 1 + rng.integers(0, n - 1, k)        # random, repeats among them


@pytest.mark.parametrize("k", [1025, 1087, 4097, 4160, 16385, 32767])
@pytest.mark.parametrize("kind", ["consecutive", "repeated", "strides", "random"])
def test_wide_levels(kind, k):
    """The hub's level, then a level in which two more vertices list the same
    destinations (found already) and the next k (new ones)."""
    print("case: small runs,", kind, k, flush=True)
    n = 1 << 18
    a = np.sort(hub_lists(kind, k, n))
    p, q = int(a[0]), int(a[-1])
    b = np.sort((a + k) % n)
    src = np.concatenate([np.zeros(k, np.int64), np.full(k, p), np.full(k, q)])
    og = csr(n, src, np.concatenate([a, a, b]))
    g = T.Graph.from_arrays(og.off, og.adj)
    for budget in (None, 0):
        g.store_config(budget, 512)
        for s in (0, p, q):
            ref = O.bfs(og, s)
            lv, st = g.bfs(s)
            assert np.array_equal(lv, ref), (budget, s)
            assert st.edges_traversed == int(og.degrees()[ref != n + 1].sum()), (budget, s)
            assert st.reached == int((ref != n + 1).sum())
            assert np.array_equal(g.bfs_noalloc(s)[0], ref), (budget, s)


def test_dense_list_as_fast_as_spread():
    """20,000 leaves on consecutive ids and on every 200th: the kernel's time
    (events) for the dense star is no longer (a sixth less in fact, where an
    atomic a leaf took three times as long)."""
    k, ms = 20000, []
    for stride in (1, 200):
        og = csr(k * 200 + 1, np.zeros(k, np.int64), 1 + stride * np.arange(k))
        g = T.Graph.from_arrays(og.off, og.adj)
        runs = [g.bfs(0)[1].expand_ms for _ in range(15)]
        ms.append(float(np.median(runs[3:])))
    print("dense, spread ms", ms, flush=True)
    assert ms[0] <= 1.25 * ms[1]
