"""GPU check of the size limit of 64-bit-id graphs: a graph whose n values
would not fit the device's free memory is refused by every algorithm, however
few of its vertices have edges (CC's digest visits every id)."""
import numpy as np
import pytest

import thievory_amd as T

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("over", ["free", 1 << 60, (1 << 64) - 2])
def test_more_ids_than_memory_holds(over):
    # half as much again as is free: a margin for what the graph itself takes
    n = T.device_memory()["free"] * 3 // 2 // 8 if over == "free" else over
    print("case: wide,", n, "ids", flush=True)
    g = T.Graph64(n, [3, n - 1], [0, 1, 2], [n - 1, 3], [1, 2])
    for run in (lambda: g.bfs(3), lambda: g.cc(), lambda: g.sssp(3)):
        with pytest.raises(T.ThvError) as e:
            run()
        assert e.value.code == -3          # THV_ENOMEM
    with pytest.raises(T.ThvError) as e:   # and no values are left behind
        g.values([3])
    assert e.value.code == -8              # THV_ESTATE


def test_as_many_ids_as_memory_holds():
    """An eighth of the free memory: accepted, and every id has its value."""
    n = T.device_memory()["free"] // 8 // 8
    print("case: wide,", n, "ids", flush=True)
    g = T.Graph64(n, [3, n - 1], [0, 1, 2], [n - 1, 3], [1, 2])
    r = g.bfs(3)
    assert (r["reached"], r["depth"]) == (2, 2)
    r = g.cc()
    assert (r["reached"], r["depth"]) == (n, n - 2)
    assert g.values([3, 4, n - 1]).tolist() == [3, 4, 3]
    r = g.sssp(3)
    assert (r["reached"], r["depth"]) == (2, 2)
