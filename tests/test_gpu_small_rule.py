"""GPU check of which BFS levels the small-frontier kernel leaves to the
general path: host records weigh twice against its 32,768 edges, and on a
symmetric graph in HBM a level that would find more than 16,384 vertices is
left too.  Seen in the number of expansion launches (one for a run of small
levels, one for each other top-down level)."""
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


@pytest.mark.parametrize("k,host_small,hbm_small", [(16384, True, True), (16385, False, True),
                                                    (32768, False, True), (32769, False, False)])
def test_host_records_weigh_twice(k, host_small, hbm_small):
    """A star, from its hub: one small level, then the leaves (no lists)."""
    print("case: star of", k, flush=True)
    og = csr(k + 1, np.zeros(k, np.int64), 1 + np.arange(k))
    ref = O.bfs(og, 0)
    g = T.Graph.from_arrays(og.off, og.adj)
    for budget, small in ((0, host_small), (None, hbm_small)):
        g.store_config(budget, 512)
        lv, st = g.bfs(0)
        assert np.array_equal(lv, ref)
        # the small run and the general level that finds the end, or two of those
        assert st.expand_launches == 2
        assert (st.hbm_bytes - st.topdown_hbm_bytes != 0) == small, (budget, st.as_dict())


def test_level_that_finds_many():
    """Random graph of degree 32: 28 -> 900 -> 29,000 edges; the third level
    finds 22,700 vertices and is not the kernel's, though its edges are fewer
    than 32,768."""
    print("case: level that finds many", flush=True)
    rng = np.random.default_rng(1)
    n = 1 << 16
    u, v = rng.integers(0, n, 16 * n), rng.integers(0, n, 16 * n)
    og = csr(n, np.concatenate([u, v]), np.concatenate([v, u]))
    ref = O.bfs(og, 77)
    e = [int(og.degrees()[ref == k].sum()) for k in (1, 2, 3)]
    assert e[1] < 16384 < e[2] <= 32768 and int((ref == 4).sum()) > 16384
    g = T.Graph.from_arrays(og.off, og.adj)
    g.set_option("symmetric", 1)
    lv, st = g.bfs(77)
    assert np.array_equal(lv, ref)
    print("launches", st.expand_launches, "bottom-up", st.bottom_up_levels, "levels", st.iterations)
    # two small levels, the third, and at the end the last vertices again
    assert st.expand_launches == 2 + (st.iterations - 3 - st.bottom_up_levels > 0)
