"""GPU check of batches on engines kept from earlier ones: batch after batch
of different sizes, algorithms, graphs, stores, directions and launch shapes,
every lane equal to the oracle's single-source answer; levels of fewer and
of more edges than SSSP's small chunks take; the memory of kept engines is
given back when it is asked for and when a graph is closed."""
import threading

import numpy as np
import pytest

from oracle import oracle as O
import thievory_amd as T

pytestmark = pytest.mark.gpu


def expect(og, algo, srcs):
    fn = O.bfs if algo == "bfs" else O.sssp
    return [O.hash_values(fn(og, int(s)), og.n + 1) for s in srcs]


def check(g, og, algo, srcs):
    r = g.batch(algo, srcs)
    got = list(zip(r["hash"].tolist(), r["reached"].tolist(), r["depth"].tolist()))
    assert got == [tuple(x) for x in expect(og, algo, srcs)], (algo, len(srcs))


def test_batch_after_batch():
    print("case: batches on kept engines", flush=True)
    rng = np.random.default_rng(3)
    graphs = [(T.Graph.rmat(s, ef, seed=s, weights=True), O.rmat(s, ef, seed=s, weights=True))
              for s, ef in ((12, 16), (13, 3))]
    for step, k in enumerate((1, 64, 3, 64, 63, 2, 64, 1)):
        for g, og in graphs:
            srcs = rng.integers(0, og.n, k).astype(np.uint32)
            for algo in ("bfs", "sssp"):
                check(g, og, algo, srcs)
        g, og = graphs[step % 2]
        if step == 2:
            g.store_config(int(0.3 * g.m * 8), 1 << 9)
        if step == 3:
            g.set_option("direction", 0)
        if step == 4:
            g.tune("batch-bfs", sources=[1, 2, 3], repeats=1)
        if step == 5:  # whole arrays between two batches of digests
            r = g.batch("sssp", [5, 6], full=True)
            assert np.array_equal(r["full"][1], O.sssp(og, 6))
        if step == 6:
            with pytest.raises(T.ThvError):
                g.batch("bfs", [og.n])


def test_sssp_chunk_sizes():
    """R-MAT 18: levels of a few edges up to some millions (SSSP's small
    chunks below 2M edges, large ones above)."""
    print("case: batch SSSP chunk sizes", flush=True)
    g, og = T.Graph.rmat(18, 24, seed=4, weights=True), O.rmat(18, 24, seed=4, weights=True)
    check(g, og, "sssp", np.array([1, 7, 99], np.uint32))
    check(g, og, "bfs", np.array([1, 7, 99], np.uint32))


def test_kept_memory_is_given_back():
    print("case: kept engine memory", flush=True)
    g = T.Graph.rmat(18, 8, seed=2, weights=True)
    g.store_config(None)
    before = T.device_memory()["free"]
    for _ in range(2):
        g.batch("bfs", [1, 2, 3])
        g.batch("sssp", [1, 2, 3])
    assert abs(T.device_memory()["free"] - before) <= 64 << 20
    g.batch("bfs", [1])
    g.close()


def test_batches_of_several_threads():
    """A graph each, all at once: engines are not shared between them."""
    print("case: batches of several threads", flush=True)
    og = [O.rmat(11, 8, seed=s, weights=True) for s in range(4)]
    bad = []

    def run(i):
        try:
            g = T.Graph.rmat(11, 8, seed=i, weights=True)
            rng = np.random.default_rng(i)
            for _ in range(6):
                srcs = rng.integers(0, og[i].n, int(rng.integers(1, 65))).astype(np.uint32)
                check(g, og[i], "bfs", srcs)
                check(g, og[i], "sssp", srcs)
            g.close()
        except BaseException as e:  # shown by the main thread
            bad.append((i, repr(e)[:300]))

    th = [threading.Thread(target=run, args=(i,)) for i in range(4)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not bad, bad
