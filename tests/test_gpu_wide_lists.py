"""GPU checks of the numbered vertices of a 64-bit-id graph: destinations
without a list of their own, sources with neither list nor in-edge, lists at
the limits of a segment (256 records) and of a wave's append buffer, and more
records than one piece of the loading pass (16M).  The oracle runs on the
compact graph; ids are spread past 2^32."""
import numpy as np
import pytest

from oracle import oracle as O
import thievory_amd as T

pytestmark = pytest.mark.gpu

M64 = (1 << 64) - 1


def mix64(z):
    z = np.asarray(z, np.uint64)
    with np.errstate(over="ignore"):
        z = z + np.uint64(0x9E3779B97F4A7C15)
        z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
        z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
    return z ^ (z >> np.uint64(31))


def digest(ids, vals):
    with np.errstate(over="ignore"):
        return int(np.sum(mix64(mix64(ids) + vals), dtype=np.uint64))


class Spread:
    """Compact edges src -> dst with weights over c vertices, vertex i at id
    name[i] of an n-vertex graph.  The oracle's graph has PAD more vertices,
    without edges: distances stop at the vertex count."""

    PAD = 1 << 14

    def __init__(self, c, src, dst, w, name, n):
        order = np.lexsort((dst, src))
        src, dst, w = src[order], dst[order], w[order].astype(np.uint32)
        off = np.zeros(c + self.PAD + 1, np.uint64)
        off[1:] = np.cumsum(np.bincount(src, minlength=c + self.PAD))
        self.og = O.CSR(off, dst.astype(np.uint32), w)
        self.name, self.n, self.c = name.astype(np.uint64), n, c
        deg = np.diff(off.astype(np.int64))[:c]
        listed = np.flatnonzero(deg)
        loff = np.concatenate([[0], np.cumsum(deg[listed])]).astype(np.uint64)
        self.g = T.Graph64(n, self.name[listed], loff, self.name[dst], w)

    def check(self, algo, s=None):
        og, none = self.og, np.uint64(self.n + 1)
        if algo == "cc":
            r, ref = self.g.cc(), self.name[O.cc(og)[:self.c]]
        else:
            r = getattr(self.g, algo)(int(self.name[s]))
            ref = (O.bfs if algo == "bfs" else O.sssp)(og, s)[:self.c].astype(np.uint64)
            ref = np.where(ref == og.n + 1, none, ref)
        assert np.array_equal(self.g.values(self.name), ref), (algo, s)
        if algo == "cc":
            assert r["reached"] == self.n
        else:
            fin = ref != none
            assert r["reached"] == int(fin.sum()) and r["depth"] == int(ref[fin].max())
            assert r["hash"] == digest(self.name[fin], ref[fin]), (algo, s)
        return r, ref


def names(c, n, seed):
    """c sorted ids below n, the first and last vertex among them."""
    rng = np.random.default_rng(seed)
    x = np.unique(rng.integers(1, n - 1, 2 * c))
    x = np.sort(rng.permutation(x)[:c - 2])
    return np.concatenate([[0], x, [n - 1]]).astype(np.uint64)


@pytest.mark.parametrize("n", [40000, (1 << 33) + 5])
def test_destinations_without_lists(n):
    """Half of the vertices have no list; some are reached only as
    destinations, some not at all; every one is a source once."""
    print("case: wide, destinations without lists, n =", n, flush=True)
    rng = np.random.default_rng(7)
    c = 120
    src = rng.choice(np.arange(0, c, 2), 260)
    dst = rng.integers(0, c - 20, 260)
    x = Spread(c, src, dst, rng.integers(0, 65, 260), names(c, n, 3), n)
    for s in range(c):
        for algo in ("bfs", "sssp"):
            x.check(algo, s)
    r, ref = x.check("cc")
    if n < 1 << 20:  # the whole arrays
        exp = np.arange(n, dtype=np.uint64)
        exp[x.name.astype(np.int64)] = ref
        r = x.g.cc(out=True)
        assert np.array_equal(r["values"], exp)
        assert r["hash"] == digest(np.arange(n, dtype=np.uint64), exp)
        assert r["depth"] == int(exp.max())
        for s in (0, 1, c - 1):
            _, ref = x.check("bfs", s)
            exp = np.full(n, n + 1, np.uint64)
            exp[x.name.astype(np.int64)] = ref
            assert np.array_equal(x.g.bfs(int(x.name[s]), out=True)["values"], exp), s
        lone = int(np.setdiff1d(np.arange(n), x.name.astype(np.int64))[5])
        r = x.g.bfs(lone, out=True)  # neither a list nor an in-edge
        assert r["values"][lone] == 1 and r["reached"] == r["depth"] == 1
        assert r["hash"] == digest(np.array([lone], np.uint64), np.array([1], np.uint64))
        assert x.g.values([lone, lone + 1 if lone + 1 < n else 0])[0] == 1


@pytest.mark.parametrize("k", [1, 63, 64, 65, 255, 256, 257, 511, 512, 513, 131071, 131073])
def test_list_lengths(k):
    """Two lists of k records, the second reached from the first, and a list
    for every 7th leaf: whole, split and many segments, and a vertex whose
    segments overflow a wave's buffer when it is appended."""
    print("case: wide, lists of", k, flush=True)
    rng = np.random.default_rng(k)
    leaf = np.arange(2, k + 2)
    more = leaf[::7]
    src = np.concatenate([np.zeros(k, np.int64), np.ones(k, np.int64), [0], more])
    dst = np.concatenate([leaf, leaf, [1], np.full(len(more), 1)])
    n = 1 << 34
    x = Spread(k + 2, src, dst, rng.integers(1, 65, len(src)), names(k + 2, n, k), n)
    for s in (0, 1, 2, k + 1):
        for algo in ("bfs", "sssp"):
            x.check(algo, s)
    x.check("cc")
    x.g.store_config(int(0.4 * x.g.m * 16), 64)
    x.check("sssp", 0)


def test_more_than_one_loading_piece():
    """17M records in 17 lists, a third of the destinations listed, the others
    not, over two pieces of the loading pass."""
    print("case: wide, two loading pieces", flush=True)
    k, d, c = 17, 1000000, 1500000
    rng = np.random.default_rng(1)
    src = np.repeat(np.arange(k) * 7, d)
    dst = np.concatenate([np.arange(i, i + d) + rng.integers(0, c - d - k) for i in range(k)])
    n = (1 << 33) + 77
    x = Spread(c, src, dst, rng.integers(1, 65, len(src)), names(c, n, 2), n)
    for algo in ("bfs", "sssp"):
        x.check(algo, 0)
    x.check("cc")
