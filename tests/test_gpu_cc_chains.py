"""GPU check of union-find CC where the parent hints form one long chain: a
path of vertices of one degree with consecutive ids, each with a leaf.  The
labels equal the oracle's, and no link walks the chain."""
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


def caterpillar(spine, first_leaf, first_spine):
    """A path of `spine` vertices with consecutive ids, one leaf on each."""
    sp, leaf = first_spine + np.arange(spine), first_leaf + np.arange(spine)
    return symmetric(2 * spine, np.concatenate([sp[:-1], leaf]), np.concatenate([sp[1:], sp]))


@pytest.mark.parametrize("leaves_first", [True, False])
@pytest.mark.parametrize("spine", [64, 4000, 100000])
def test_chains_of_hints(spine, leaves_first):
    """A link or find of at most a fifth of the spine: the guard is not met,
    so no link walks the chain (half the spine) and CC stays with union-find
    (2 rounds)."""
    print("case: caterpillar", spine, leaves_first, flush=True)
    og = caterpillar(spine, 0 if leaves_first else spine, spine if leaves_first else 0)
    g = T.Graph.from_arrays(og.off, og.adj)
    g.set_option("symmetric", 1)
    if spine == 100000:
        g.set_option("cc_uf_steps", spine // 5)
    lab, st = g.cc()
    assert np.array_equal(lab, O.cc(og))
    assert st.iterations == 2
