"""GPU check of bottom-up batch levels whose lists are all long (scanned by
groups of lanes): queues of fewer vertices than one wave has groups up to
more than a wave's buffer holds, and the direction chosen from the frontier
edges that the level before has summed."""
import numpy as np
import pytest

from oracle import oracle as O
import thievory_amd as T

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,strides,k", [(37, 5, 3), (37, 5, 64), (5003, 20, 64),
                                         (300007, 8, 1), (300007, 5, 64), (2200013, 5, 64)])
def test_every_list_is_long(n, strides, k):
    """Circulant graphs: v is joined to v +- s for each stride s, so every
    list has 2 x strides records and the levels from one source are those of
    vertex 0, shifted."""
    print("case: batch long lists", n, strides, k, flush=True)
    rng = np.random.default_rng(n + k)
    s = rng.choice(np.arange(1, (n - 1) // 2), strides, replace=False)
    adj = (np.arange(n)[:, None] + np.concatenate([s, -s])[None, :]) % n
    adj = np.sort(adj, 1).astype(np.uint32).ravel()
    off = np.arange(n + 1, dtype=np.uint64) * (2 * strides)
    zero = O.bfs(O.CSR(off, adj), 0)
    g = T.Graph.from_arrays(off, adj)
    g.set_option("symmetric", 1)
    srcs = rng.integers(0, n, k).astype(np.uint32)
    r = g.batch("bfs", srcs)
    assert k == 1 or r["stats"].bottom_up_levels > 0
    for i, v in enumerate(srcs):
        want = O.hash_values(np.roll(zero, int(v)), n + 1)
        assert (r["hash"][i], r["reached"][i], r["depth"][i]) == tuple(want), (i, v)
    # every level top-down counts the same edges whichever way it is counted
    g.set_option("direction", 0)
    td = g.batch("bfs", srcs)
    assert np.array_equal(td["hash"], r["hash"]) and np.array_equal(td["depth"], r["depth"])
