"""GPU check of union-find CC on symmetric graphs without hubs, whose parent
hints form no giant tree: the labels equal the oracle's, and the records read
are bounded, since a call that reads every list is right but slow."""
import numpy as np
import pytest

from oracle import oracle as O
import thievory_amd as T

pytestmark = pytest.mark.gpu


def symmetric(n, u, v):
    src, dst = np.concatenate([u, v]), np.concatenate([v, u])
    order = np.lexsort((dst, src))
    off = np.zeros(n + 1, np.uint64)
    off[1:] = np.cumsum(np.bincount(src, minlength=n))
    return O.CSR(off, dst[order].astype(np.uint32), None)


def no_hubs(kind):
    rng = np.random.default_rng(7)
    if kind == "random":
        n = 1 << 17
        u, v = rng.integers(0, n, 4 * n), rng.integers(0, n, 4 * n)
        u, v = u[u != v], v[u != v]
    else:
        s = 362
        n = s * s
        p = rng.permutation(n).reshape(s, s)
        u = np.concatenate([p[:, :-1].ravel(), p[:-1].ravel()])
        v = np.concatenate([p[:, 1:].ravel(), p[1:].ravel()])
    return symmetric(n, u, v)


@pytest.mark.parametrize("hints", [1, 0])
@pytest.mark.parametrize("share", [1.0, 0.6])
@pytest.mark.parametrize("kind", ["random", "grid"])
def test_graphs_without_hubs(kind, share, hints):
    """At most two records a vertex (a list on the host: its hint, when there
    are hints) and a tenth of a record more for the lists that are left; of a
    grid's lists a split store leaves more, since the two records of a vertex
    lead to its two least neighbours."""
    print("case: CC without hubs,", kind, share, hints, flush=True)
    og = no_hubs(kind)
    g = T.Graph.from_arrays(og.off, og.adj)
    g.set_option("symmetric", 1)
    g.set_option("parent_hints", hints)
    g.store_config(None if share == 1.0 else int(share * og.m * 4), 512)
    lab, st = g.cc()
    assert np.array_equal(lab, O.cc(og))
    assert st.iterations == 2
    left = 0.1 if kind == "random" or share == 1.0 else 1.0
    assert st.edges_traversed <= (2 + left) * og.n
    if hints:
        assert st.host_bytes <= 4 * left * og.n


def test_chain_beside_a_hub():
    """Hints are taken (a star holds most lists), and a caterpillar beside it,
    spine ids consecutive and past its leaves', still makes no link walk its
    chain: a guard of a fifth of the spine is not met."""
    print("case: chain beside a hub", flush=True)
    s, k = 100000, 400000
    leaf, spine, hub = np.arange(s), s + np.arange(s), 2 * s + k
    og = symmetric(2 * s + k + 1, np.concatenate([spine[:-1], leaf, np.full(k, hub)]),
                   np.concatenate([spine[1:], spine, 2 * s + np.arange(k)]))
    g = T.Graph.from_arrays(og.off, og.adj)
    g.set_option("symmetric", 1)
    g.set_option("cc_uf_steps", s // 5)
    lab, st = g.cc()
    assert np.array_equal(lab, O.cc(og))
    assert st.iterations == 2
    # a hint a vertex, and the spine's lists (three records, the ends' two) in step 3
    assert st.edges_traversed == og.n + 3 * s - 2
