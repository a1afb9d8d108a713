"""GPU check of SSSP levels on both sides of the length from which they leave
room for BFS ones: a mixed stream on a graph whose records are all on the host
(the widest levels read some 190 MB over the link), half of them, and none."""
import functools

import numpy as np
import pytest

from oracle import oracle as O
import thievory_amd as T

pytestmark = pytest.mark.gpu


@functools.lru_cache(maxsize=1)
def case():
    og = O.rmat(20, 24, seed=6, weights=True)
    srcs = np.random.default_rng(4).integers(0, og.n, 12)
    want = {(a, int(s)): tuple(O.hash_values((O.bfs if a == "bfs" else O.sssp)(og, int(s)), og.n + 1))
            for s in srcs for a in ("bfs", "sssp")}
    return og.m, want


@pytest.mark.parametrize("share", [0.0, 0.5, 1.0])
@pytest.mark.parametrize("lanes", [5, 64])
def test_mixed_stream_on_long_levels(share, lanes):
    print("case: serving long levels", share, lanes, flush=True)
    m, want = case()
    g = T.Graph.rmat(20, 24, seed=6, weights=True)
    g.store_config(None if share == 1.0 else int(share * m * 8))
    srv = T.Server(g, max_lanes=lanes)
    tk = [(k, srv.submit(*k)) for k in want]
    srv.drain()
    for k, t in tk:
        r = srv.poll(t)
        assert r["status"] == 0 and (r["hash"], r["reached"], r["depth"]) == want[k], k
    srv.stop()
