"""GPU check of SSSP levels that leave room for BFS ones: a server with both
kinds of queries on a graph whose widest levels have more chunks than the
smaller grid has blocks; every answer equals the oracle's."""
import numpy as np
import pytest

from oracle import oracle as O
import thievory_amd as T

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lanes", [5, 64])
def test_mixed_stream_on_wide_levels(lanes):
    print("case: serving with room", lanes, flush=True)
    og = O.rmat(18, 24, seed=6, weights=True)  # some 6,000 chunks of 1,024 edges
    g = T.Graph.rmat(18, 24, seed=6, weights=True)
    srv = T.Server(g, max_lanes=lanes)
    srcs = np.random.default_rng(lanes).integers(0, og.n, 24)
    tk = [(a, int(s), srv.submit(a, int(s))) for s in srcs for a in ("bfs", "sssp")]
    srv.drain()
    for a, s, t in tk:
        r = srv.poll(t)
        want = O.hash_values((O.bfs if a == "bfs" else O.sssp)(og, s), og.n + 1)
        assert r["status"] == 0 and (r["hash"], r["reached"], r["depth"]) == tuple(want), (a, s)
    srv.stop()
