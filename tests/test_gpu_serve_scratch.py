"""GPU check of the server's scratch budget: a budget of exactly the bytes an
engine is priced at holds the engine, one byte less does not.  The price is
part of what a caller's budget was chosen for, so it is written out here."""
import pytest

import thievory_amd as T

pytestmark = pytest.mark.gpu

TILE = 4096


def price(g, sssp_lanes=0):
    """Bytes of a BFS engine (any number of lanes), or of an SSSP engine."""
    n, words = g.n, g.n // 32 + 2
    b = 2 * (words * 4 + (n + 1) * 8) + 2 * ((n + 1) * 12) + 2 * (g.m // 1024 + 2) * 4
    b += (n // TILE + 1) * TILE * 4
    return b + (sssp_lanes * n * 4 if sssp_lanes else (n + 1) * 8 + words * 4)


@pytest.mark.parametrize("short", [0, 1])
@pytest.mark.parametrize("sssp", [False, True])
def test_budget_of_exactly_the_engines(sssp, short):
    print("case: scratch budget,", "BFS and SSSP" if sssp else "BFS", short, "short", flush=True)
    g = T.Graph.rmat(12, 32, seed=5, symmetric=False, weights=sssp)
    budget = price(g) + (price(g, 1) if sssp else 0) - short
    if short and not sssp:
        with pytest.raises(T.ThvError) as e:
            T.Server(g, max_lanes=1, scratch_bytes=budget)
        assert e.value.code == -3
        return
    s = T.Server(g, max_lanes=1, scratch_bytes=budget)
    try:
        s.submit("bfs", 1)
        if sssp and short:
            with pytest.raises(T.ThvError) as e:
                s.submit("sssp", 1)
            assert e.value.code == -7
        elif sssp:
            s.submit("sssp", 1)
        s.drain()
    finally:
        s.stop()
