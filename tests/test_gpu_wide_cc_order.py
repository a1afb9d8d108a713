"""GPU check of 64-bit-id CC's first round: it takes the lists in the order of
the ids, so the least label is far spread when the later ones are read.  A
label that has not arrived by the end of the round costs a third reading of the
lists: fewer than half of them may need one."""
import numpy as np
import pytest

from oracle import oracle as O
import thievory_amd as T

pytestmark = pytest.mark.gpu


def test_first_round_in_id_order():
    print("case: wide CC, records read", flush=True)
    n, d = 1 << 20, 16
    rng = np.random.default_rng(1)
    u, v = rng.integers(0, n, n * d), rng.integers(0, n, n * d)
    order = np.argsort(u, kind="stable")
    deg = np.bincount(u, minlength=n)
    off = np.concatenate([[0], np.cumsum(deg)])
    ref = O.cc(O.CSR(off.astype(np.uint64), v[order].astype(np.uint32), None))
    l = np.flatnonzero(deg)
    g = T.Graph64(7 * n + 1, 7 * l, np.concatenate([[0], np.cumsum(deg[l])]), 7 * v[order])
    read = [g.cc()["stats"].edges_traversed / g.m for _ in range(12)]
    print([round(x, 3) for x in read], flush=True)
    assert (g.values(7 * np.arange(n)) == 7 * ref.astype(np.uint64)).all()
    assert max(read) < 2.5  # all once, those found meanwhile (nearly all) again, and the rest
