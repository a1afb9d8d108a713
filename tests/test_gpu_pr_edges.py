"""GPU check of PageRank's edge kernels where their cases change: vertex
counts around the push mode's 32,768 hub sums (at or below it every vertex is
one), list lengths around a wave (64), a push chunk (512 edges, 128 staged
entries) and a pull chunk (1,024 or 2,048), runs of one-record lists, both
record sizes, edges in HBM, on the host and split.

One iteration with damping 1/2 and out-degrees that are powers of two (for
pull, vertex counts too) has dyadic values of at most 24 bits: the fp32 ranks
are exact in any order of the sums, so the check is equality."""
import numpy as np
import pytest

import thievory_amd as T

pytestmark = pytest.mark.gpu


def lists(n, src, dst):
    order = np.argsort(src, kind="stable")
    off = np.zeros(n + 1, np.uint64)
    off[1:] = np.cumsum(np.bincount(src, minlength=n))
    return off, dst[order].astype(np.uint32)


def push_ranks(n, src, dst):
    deg = np.bincount(src, minlength=n)
    return 0.5 + np.bincount(dst, weights=0.25 / deg[src], minlength=n)


def pull_ranks(n, src, dst):
    deg = np.bincount(src, minlength=n)
    return 0.5 + 0.5 * np.bincount(dst, weights=1.0 / n / deg[src], minlength=n)


def stores(g):
    for budget in (None, 0, int(0.3 * g.m * g.edge_bytes)):
        g.store_config(budget, 512)
        yield budget


def check_push(n, src, dst):
    ref = push_ranks(n, src, dst)
    off, adj = lists(n, src, dst)
    for rec in (4, 8):
        g = T.Graph.from_arrays(off, adj, np.ones(len(adj), np.uint32) if rec == 8 else None)
        for budget in stores(g):
            for rep in range(2):  # the second call finds the first one's sums taken
                r, _ = g.pr("push", damping=0.5, tol=0.0, max_iter=1)
                assert np.array_equal(r, ref), (rec, budget, rep)


def check_pull(n, src, dst, ept=None):
    ref = pull_ranks(n, src, dst)
    off, adj = lists(n, dst, src)
    g = T.Graph.from_arrays(off, adj, outdeg=np.bincount(src, minlength=n).astype(np.uint32))
    for budget in stores(g):
        for rep in range(2):
            r, _ = g.pr("pull", damping=0.5, tol=0.0, max_iter=1)
            assert np.array_equal(r, ref), (budget, rep)


@pytest.mark.parametrize("n", [2, 33, 32767, 32768, 32769, 50001, 65536])
def test_vertices_around_the_hub_table(n):
    print("case: PageRank on", n, "vertices", flush=True)
    rng = np.random.default_rng(n)
    deg = 1 << rng.integers(0, 4, n)
    src = np.repeat(np.arange(n), deg)
    # skewed destinations: some vertices are hubs, most are not
    dst = (n * rng.random(len(src)) ** 3).astype(np.int64)
    check_push(n, src, dst)
    if n & (n - 1) == 0:
        check_pull(n, src, dst)


@pytest.mark.parametrize("shift", [0, 1, 3])
@pytest.mark.parametrize("big", [64, 128, 512, 1024, 2048])
def test_push_list_lengths(big, shift):
    """Lists of `big` records at every alignment that `shift` one-record
    lists before them give, with runs of 127 to 513 one-record lists between."""
    print("case: PageRank push, lists of", big, "after", shift, flush=True)
    lens = ([1] * shift + [big] + [1] * 127 + [big] + [1] * 129 + [2] * 128 + [big, big] +
            [1] * (513 - shift) + [big] + [1] * 511 + [4, big])
    n = 4000
    rng = np.random.default_rng(big + shift)
    src = np.repeat(np.arange(len(lens)), lens)
    check_push(n, src, rng.integers(0, n, len(src)))


@pytest.mark.parametrize("shift", [0, 1, 5])
@pytest.mark.parametrize("big", [62, 63, 64, 65, 127, 1023, 1024, 1025, 2047, 2048, 2049])
def test_pull_list_lengths(big, shift):
    """In-lists of `big` records, next to each other and among short ones."""
    print("case: PageRank pull, lists of", big, "after", shift, flush=True)
    lens = [1] * shift + [big, big, 1, 3, big + 1, 1, 1, big - 1, 2, big] + [1] * 600 + [big]
    n = 4096
    rng = np.random.default_rng(big + shift)
    dst = np.repeat(np.arange(len(lens)), lens)
    src = rng.integers(0, n, len(dst))
    # every vertex's out-degree up to a power of two: more records to the last vertex
    deg = np.bincount(src, minlength=n)
    want = np.where(deg > 0, 1 << np.ceil(np.log2(np.maximum(deg, 1))).astype(np.int64), 0)
    more = np.repeat(np.arange(n), want - deg)
    check_pull(n, np.concatenate([src, more]), np.concatenate([dst, np.full(len(more), n - 1)]))
