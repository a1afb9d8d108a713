"""GPU checks of the small-frontier kernel (many levels per launch) at its
limits: the queue's 4,096 vertices, the edges a level may have (32,768; SSSP
16,384), the levels of one launch (4,096) and the far list's 65,536 entries,
each one below, at and one past.  Values are whole numbers: equal to the
oracle's."""
import numpy as np
import pytest

from oracle import oracle as O
import thievory_amd as T

pytestmark = pytest.mark.gpu


def graph(n, src, dst, w=None):
    order = np.lexsort((dst, src))
    off = np.zeros(n + 1, np.uint64)
    off[1:] = np.cumsum(np.bincount(src, minlength=n))
    ww = None if w is None else w[order].astype(np.uint32)
    return O.CSR(off, dst[order].astype(np.uint32), ww)


def both(og, sources, weighted, cc=True):
    """BFS, CC and SSSP of og, edges in HBM and on the host, as the oracle."""
    g = T.Graph.from_arrays(og.off, og.adj, og.w if weighted else None)
    for budget in (None, 0):
        g.store_config(budget, 512)
        for s in sources:
            lv, st = g.bfs(s)
            ref = O.bfs(og, s)
            assert np.array_equal(lv, ref), (budget, s)
            assert st.edges_traversed == int(og.degrees()[ref != og.n + 1].sum()), (budget, s)
            assert (st.host_bytes > 0) == (budget == 0 and st.edges_traversed > 0)
            assert np.array_equal(g.bfs_noalloc(s)[0], ref), (budget, s)
            if weighted:
                for delta in (0, 16):
                    g.set_option("sssp_delta", delta)
                    assert np.array_equal(g.sssp(s)[0], O.sssp(og, s)), (budget, s, delta)
        if cc:
            assert np.array_equal(g.cc()[0], O.cc(og)), budget
    return g


@pytest.mark.parametrize("k", [1, 63, 64, 65, 1023, 1024, 1025, 4095, 4096, 4097])
def test_frontier_of_k_vertices(k):
    """A hub with k spokes, each with one neighbour and back edges (symmetric,
    so the direction-optimising loop hands its levels over too)."""
    print("case: small frontier of", k, flush=True)
    i = np.arange(1, k + 1)
    u = np.concatenate([np.zeros(k, np.int64), i])
    v = np.concatenate([i, k + i])
    w = np.random.default_rng(k).integers(1, 65, 2 * k)
    og = graph(2 * k + 1, np.concatenate([u, v]), np.concatenate([v, u]), np.concatenate([w, w]))
    g = both(og, (0, 1, 2 * k), True)
    g.set_option("symmetric", 1)
    for budget in (None, 0):
        g.store_config(budget, 512)
        for s in (0, 1, 2 * k):
            lv, st = g.bfs(s)
            assert np.array_equal(lv, O.bfs(og, s)), (budget, s)
            assert st.iterations == int(lv[lv <= og.n].max()), (budget, s)


@pytest.mark.parametrize("k", [16383, 16384, 16385, 32767, 32768, 32769])
def test_level_of_k_edges(k):
    """Two hubs one after the other share k leaves: both levels have k edges
    (the first one more), from a frontier of one vertex."""
    print("case: small level of", k, "edges", flush=True)
    leaf = np.arange(2, k + 2)
    src = np.concatenate([np.zeros(k, np.int64), np.ones(k, np.int64), [0]])
    dst = np.concatenate([leaf, leaf, [1]])
    w = np.random.default_rng(k).integers(1, 65, len(src))
    both(graph(k + 2, src, dst, w), (0, 1, k + 1), True)


@pytest.mark.parametrize("k", [4095, 4096, 4097, 4098, 8200])
def test_path_of_k_levels(k):
    print("case: path of", k, "levels", flush=True)
    v = np.arange(k)
    w = np.random.default_rng(k).integers(1, 65, k)
    both(graph(k + 1, v, v + 1, w), (0, k // 2, k), True, cc=False)


@pytest.mark.parametrize("hubs,leaves", [(7, 9362), (8, 8192), (9, 8000)])
def test_far_list_limit(hubs, leaves):
    """A chain of hubs at distance 1 from each other, every leaf 60 or more
    away: the leaves of all hubs wait in the far list (65,534, 65,536 and
    72,000 of them) before the first of their buckets opens.  Weights of 0
    and equal distances among them."""
    print("case: far list of", hubs * leaves, flush=True)
    n = hubs * (leaves + 1)
    h = np.arange(hubs) * (leaves + 1)
    src = np.concatenate([np.repeat(h, leaves), h[:-1]])
    dst = np.concatenate([np.setdiff1d(np.arange(n), h), h[1:]])
    rng = np.random.default_rng(hubs)
    w = np.concatenate([rng.integers(60, 90, hubs * leaves), np.ones(hubs - 1, np.int64)])
    # some leaves go on to a neighbour at distance 0
    more = np.setdiff1d(rng.choice(n - 1, 500), np.concatenate([h, h - 1]))
    src, dst = np.concatenate([src, more]), np.concatenate([dst, more + 1])
    og = graph(n, src, dst, np.concatenate([w, np.zeros(len(more), np.int64)]))
    both(og, (0, int(h[1])), True)
