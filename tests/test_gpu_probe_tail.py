"""GPU check of the bottom-up probe where the graph's last 1,024-vertex region
ends in the middle of a wave's round of 64: the round's few vertices take their
visited and residency bits from lanes that have no vertex of it."""
import numpy as np
import pytest

from oracle import oracle as O
import thievory_amd as T

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rounds", range(16))
def test_last_round_of_a_region(rounds):
    """n = 1024 + 64 rounds + t: t vertices in the last round, whose words are
    those of lanes 2 rounds and 2 rounds + 1."""
    print("case: probe tail,", rounds, "whole rounds", flush=True)
    for t in sorted({1, 2 * rounds, 2 * rounds + 1, 2 * rounds + 2, 31, 33, 63} - {0}):
        n = 1024 + 64 * rounds + t
        rng = np.random.default_rng(n)
        u, v = rng.integers(0, n, 4 * n), rng.integers(0, n, 4 * n)
        u[:t], v[:t] = n - 1 - np.arange(t), rng.integers(0, n, t)  # the tail has edges
        src, dst = np.concatenate([u, v]), np.concatenate([v, u])
        order = np.lexsort((dst, src))
        off = np.zeros(n + 1, np.uint64)
        off[1:] = np.cumsum(np.bincount(src, minlength=n))
        og = O.CSR(off, dst[order].astype(np.uint32), None)
        g = T.Graph.from_arrays(og.off, og.adj)
        g.set_option("symmetric", 1)
        for hints, alpha in ((1, 1e6), (0, 1e6), (1, 14.0)):
            g.set_option("parent_hints", hints)
            g.set_option("do_alpha", alpha)  # 1e6: bottom-up from the first level on
            for budget in (None, int(0.5 * g.m * 4), 0):
                g.store_config(budget, 256)
                for s in (0, n - 1, n // 2):
                    lv, st = g.bfs(s)
                    ref = O.bfs(og, s)
                    assert np.array_equal(lv, ref), (n, t, hints, alpha, budget, s)
                    assert st.edges_traversed == int(og.degrees()[ref != n + 1].sum())
        g.close()
