"""GPU check of the small-frontier SSSP kernel when its first listed pending
set holds no vertex of the open bucket, so that it starts with the step that
opens the next one: its block must agree on the length of the far list before
that step resets it."""
import numpy as np
import pytest

from oracle import oracle as O
import thievory_amd as T

pytestmark = pytest.mark.gpu

WIDE, FEW = 20000, 5


@pytest.mark.parametrize("far", [1, 63, 64, 65, 1023, 1024, 1025, 4097, 40000])
def test_first_list_without_near_vertices(far):
    """A star: 20,000 leaves at distance 20 (the hub's and their levels have too
    many edges for the kernel), a few at 60 (a small level, but the kernel
    waits one out after it gave up), a few at 100 (a small level again), and
    `far` at 1,000 and more.  With buckets of 16 the listing after the level of
    those at 100 finds only leaves of later buckets."""
    print("case: first listing of", far, "far vertices", flush=True)
    rng = np.random.default_rng(far)
    w = np.concatenate([np.full(WIDE, 20), np.full(FEW, 60), np.full(FEW, 100),
                        1000 + rng.integers(0, 64, far)]).astype(np.uint32)
    k = len(w)
    off = np.concatenate([[0], k + np.arange(k + 1)]).astype(np.uint64)
    adj = np.concatenate([np.arange(1, k + 1), np.zeros(k)]).astype(np.uint32)
    og = O.CSR(off, adj, np.concatenate([w, w]))
    ref = O.sssp(og, 0)
    g = T.Graph.from_arrays(og.off, og.adj, og.w)
    g.set_option("sssp_delta", 16)
    for budget in (None, 0):
        g.store_config(budget, 512)
        assert np.array_equal(g.sssp(0)[0], ref), budget
