"""GPU check of PageRank pull under both launch shapes (chunks of 1,024 and of
2,048 edges) and both record sizes, and of runs that end before max_iter: the
iteration launched ahead of the host's look at the counters changes nothing.

Damping 1/2, out-degrees that are powers of two and (for one iteration) a
vertex count that is one make every value dyadic, of at most 24 bits: the fp32
ranks are exact in any order of the sums, so the checks are equality."""
import numpy as np
import pytest

import thievory_amd as T

pytestmark = pytest.mark.gpu


def lists(n, src, dst):
    order = np.argsort(src, kind="stable")
    off = np.zeros(n + 1, np.uint64)
    off[1:] = np.cumsum(np.bincount(src, minlength=n))
    return off, dst[order].astype(np.uint32)


def with_shape(g, ept, path):
    """Leaves g with launch shape `ept` by way of the tuner's cache."""
    g.tune("pr", repeats=1, pr_iterations=1, cache_path=path)
    with open(path) as f:
        key, val = f.read().strip().rsplit("|", 1)
    val = val.split()
    val[1] = str(ept)
    with open(path, "a") as f:
        f.write(key + "|" + " ".join(val) + "\n")
    r = g.tune("pr", repeats=1, pr_iterations=1, cache_path=path)
    assert r["from_cache"] == 1 and r["edges_per_thread"] == ept


@pytest.mark.parametrize("rec", [4, 8])
@pytest.mark.parametrize("ept", [4, 8])
def test_pull_shapes(ept, rec, tmp_path):
    print("case: PageRank pull, shape", ept, "records of", rec, flush=True)
    n = 4096
    rng = np.random.default_rng(ept * rec)
    for i, big in enumerate((63, 65, 1023, 1024, 1025, 2047, 2049)):
        lens = [1] * i + [big, big, 1, 3, big + 1, 1, 1, big - 1, 2, big] + [1] * 600 + [big]
        dst = np.repeat(np.arange(len(lens)), lens)
        src = rng.integers(0, n, len(dst))
        deg = np.bincount(src, minlength=n)  # up to a power of two: records to the last vertex
        want = np.where(deg > 0, 1 << np.ceil(np.log2(np.maximum(deg, 1))).astype(np.int64), 0)
        more = np.repeat(np.arange(n), want - deg)
        src, dst = np.concatenate([src, more]), np.concatenate([dst, np.full(len(more), n - 1)])
        off, adj = lists(n, dst, src)
        g = T.Graph.from_arrays(off, adj, np.ones(len(adj), np.uint32) if rec == 8 else None,
                                outdeg=want.astype(np.uint32))
        assert g.edge_bytes == rec
        g.store_config(None, 512)
        with_shape(g, ept, str(tmp_path / f"tune{i}"))
        ref = 0.5 + 0.5 * np.bincount(dst, weights=1.0 / n / want[src], minlength=n)
        for budget in (None, 0, int(0.3 * g.m * rec)):
            g.store_config(budget, 512)
            for rep in range(2):
                r, _ = g.pr("pull", damping=0.5, tol=0.0, max_iter=1)
                assert np.array_equal(r, ref), (big, budget, rep)


@pytest.mark.parametrize("mode", ["push", "pull"])
@pytest.mark.parametrize("n", [600, 40000])
def test_ends_before_max_iter(n, mode):
    """Four layers, edges from each to the next: the ranks stop moving after
    the last layer has them.  A run with room for more iterations, one that
    ends there, and each again, give the fixed point and the same count."""
    print("case: PageRank", mode, "that ends early on", n, flush=True)
    rng = np.random.default_rng(n)
    w = n // 4
    deg = np.where(np.arange(n) < 3 * w, 1 << rng.integers(0, 3, n), 0)
    src = np.repeat(np.arange(n), deg)
    dst = (src // w + 1) * w + rng.integers(0, w, len(src))
    ref = np.full(n, 0.5)
    for _ in range(4):
        ref = 0.5 + 0.5 * np.bincount(dst, weights=ref[src] / deg[src], minlength=n)
    if mode == "push":
        g = T.Graph.from_arrays(*lists(n, src, dst))
    else:
        g = T.Graph.from_arrays(*lists(n, dst, src), outdeg=deg.astype(np.uint32))
    for budget in (None, int(0.3 * g.m * 4)):
        g.store_config(budget, 512)
        r, st = g.pr(mode, damping=0.5, tol=0.0, max_iter=100)
        k = st.iterations
        assert np.array_equal(r, ref) and 4 <= k <= 6
        for most in (k, k + 1, 100, k):
            r, st = g.pr(mode, damping=0.5, tol=0.0, max_iter=most)
            assert np.array_equal(r, ref), (budget, most)
            assert st.iterations == k, (budget, most)
