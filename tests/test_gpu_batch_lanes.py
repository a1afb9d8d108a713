"""GPU check of SSSP batches of every group size: 8, 16, 32 or 64 lanes relax
an edge, for batches at and beside those limits; chunks of fewer edges than
one step of a wave, and a level wide enough for the large chunks."""
import numpy as np
import pytest

from oracle import oracle as O
import thievory_amd as T

pytestmark = pytest.mark.gpu


def _check(g, og, srcs):
    r = g.batch("sssp", srcs)
    for i, s in enumerate(srcs):
        want = O.hash_values(O.sssp(og, int(s)), og.n + 1)
        assert (r["hash"][i], r["reached"][i], r["depth"][i]) == tuple(want), (len(srcs), i, s)


@pytest.mark.parametrize("k", [1, 2, 7, 8, 9, 15, 16, 17, 31, 32, 33, 34, 47, 62, 63, 64])
def test_lanes_an_edge(k):
    print("case: batch SSSP of", k, flush=True)
    rng = np.random.default_rng(k)
    for scale, ef in ((5, 2), (12, 12)):
        og = O.rmat(scale, ef, seed=k, weights=True)
        g = T.Graph.rmat(scale, ef, seed=k, weights=True)
        srcs = rng.integers(0, og.n, k).astype(np.uint32)
        _check(g, og, srcs)
        g.store_config(int(0.3 * g.m * 8), 1 << 8)
        _check(g, og, srcs[::-1].copy())


@pytest.mark.parametrize("k", [3, 12, 20, 33, 34])
def test_large_chunks(k):
    print("case: batch SSSP large chunks", k, flush=True)
    og = O.rmat(18, 24, seed=9, weights=True)
    g = T.Graph.rmat(18, 24, seed=9, weights=True)
    _check(g, og, np.random.default_rng(k).integers(0, og.n, k).astype(np.uint32))
