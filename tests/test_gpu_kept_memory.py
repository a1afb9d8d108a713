"""GPU check of the memory that batches keep between calls: an engine stays
after its batch (read with a call that does not give it back), is used again
rather than joined by another, and goes when the free memory is asked for, when
the store changes and when the graph is closed."""
import ctypes as C

import numpy as np
import pytest

import thievory_amd as T

pytestmark = pytest.mark.gpu


def hip():
    """The HIP runtime that the engine has loaded."""
    T.device_info()
    with open("/proc/self/maps") as f:
        path = next(l.split()[-1] for l in f if "libamdhip64.so" in l)
    return C.CDLL(path)


def free_bytes(lib):
    f, t = C.c_size_t(), C.c_size_t()
    assert lib.hipMemGetInfo(C.byref(f), C.byref(t)) == 0
    return f.value


def test_kept_engines_go():
    print("case: kept engines", flush=True)
    lib = hip()
    T.device_memory()
    closed = free_bytes(lib)
    g = T.Graph.rmat(20, 8, seed=2, weights=True)
    g.store_config(None)
    g.sssp(1)                                    # its workspace is there
    srcs = np.arange(64, dtype=np.uint32)
    engine = 64 * 4 * g.n                        # the distances of 64 lanes, 268 MB
    slack = engine // 8
    before = free_bytes(lib)

    def kept():
        g.batch("sssp", srcs)
        first = free_bytes(lib)
        g.batch("sssp", srcs)
        assert before - first >= engine          # it stays
        assert abs(first - free_bytes(lib)) <= slack  # and is the one that is used

    kept()
    T.device_memory()
    assert abs(free_bytes(lib) - before) <= slack
    kept()
    g.store_config(None, 1 << 15)
    assert abs(free_bytes(lib) - before) <= slack
    kept()
    g.close()
    assert free_bytes(lib) >= closed - slack
