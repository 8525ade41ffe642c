"""Reading results of an executor: the copy through pinned 768 KiB chunks (reads of 2
MiB and more into ordinary memory) returns what the runtime's own copy does.  The
graph is x + bias with whole-number values, whose sums are exact in fp32."""
from __future__ import annotations

import ctypes
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CHUNK = (768 << 10) // 4   # floats
FIRST = (2 << 20) // 4     # floats of the smallest read in chunks


@pytest.fixture(scope="module")
def G(gpu):
    from mcke_amd import graph
    return graph


def _executor(G, n):
    g = G.Graph()
    x, b = g.add_input((n, 1), "x"), g.add_input((1,), "b")
    y = g.add_bias_act(x, b, "y", act=0, vector_width=1)
    g.mark_output(y)
    ex = G.Executor(g)
    ex.plan()
    ex.set_input(b, np.full(1, 3.0, np.float32))
    return ex, x, y


def _run(ex, x, n, shift):
    a = ((np.arange(n, dtype=np.int64) * 7 + shift) % 65537).astype(np.float32)
    ex.set_input(x, a)
    ex.run_async()           # the read itself waits for the run
    return a + np.float32(3.0)


@pytest.mark.parametrize("n", [1, CHUNK, FIRST - 1, FIRST, 3 * CHUNK, 3 * CHUNK + 1,
                               5 * CHUNK + 17, 16 * CHUNK - 3])
def test_read_whole_and_part(G, n):
    ex, x, y = _executor(G, n)
    for shift in range(3):   # the chunks of one read are reused by the next
        want = _run(ex, x, n, shift)
        assert np.array_equal(ex.read(y, n), want)
        part = max(1, n - CHUNK // 2 - 1)
        assert np.array_equal(ex.read(y, part), want[:part])
    with pytest.raises(Exception):
        ex.read(y, n + 1)


def test_read_into_pinned_memory(G, gpu):
    n = 3 * CHUNK + 5
    ex, x, y = _executor(G, n)
    want = _run(ex, x, n, 11)
    p = ctypes.c_void_p()
    assert gpu.lib().mcke_rt_host_alloc(ctypes.byref(p), n * 4) == 0
    try:
        assert G.host_lib().mcke_executor_read_tensor(ex.h, y, p, n * 4) == 0
        got = np.ctypeslib.as_array(ctypes.cast(p, ctypes.POINTER(ctypes.c_float)), (n,))
        assert np.array_equal(got, want)
        del got
    finally:
        assert gpu.lib().mcke_rt_host_free(p) == 0


def test_reads_from_several_threads(G):
    n = 5 * CHUNK + 3
    ex, x, y = _executor(G, n)
    want = _run(ex, x, n, 5)
    bad = []

    def reader():
        for _ in range(10):
            if not np.array_equal(ex.read(y, n), want):
                bad.append(1)

    threads = [threading.Thread(target=reader) for _ in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
