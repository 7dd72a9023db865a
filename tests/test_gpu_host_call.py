"""Calls on host buffers around the size of the staging buffers (8 MiB): x and
the outputs of a small call move by kernels through both buffers, of a larger
one by copies. The products are exact (identity weights), so outputs are compared
exactly; four threads with a session each share the buffers.
"""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

STAGE = 8 << 20


def identity_call(gpu, rows, n, seed):
    """x through an n x n identity; returns whether all outputs match."""
    rng = np.random.default_rng(seed)
    x = rng.integers(-8, 9, size=(rows, n)).astype(np.float32)
    s = gpu.DenseSession(rows, n, n, 0, 4, 1, np.eye(n, dtype=np.float32) * 240, None)
    good = True
    for k in range(3):
        xk = np.roll(x, k, axis=0)
        pre, post = s.execute(xk)
        good = good and np.array_equal(pre, xk * 240) and np.array_equal(post, np.maximum(xk, 0) * 240)
    s.close()
    return good


@pytest.mark.parametrize("rows,n", [
    (1, 1), (1, 3), (3, 5), (7, 33),        # words left over after the 16-byte vectors
    (8, 256), (1000, 131),
    (STAGE // 8 // 256, 256),               # both outputs fill the buffer exactly
    (STAGE // 8 // 256 + 1, 256),           # one row more: copies
    (STAGE // 4 // 256 + 1, 256),           # x itself does not fit
])
def test_host_call_sizes(gpu, rows, n):
    assert identity_call(gpu, rows, n, rows + n)


def test_host_calls_from_threads(gpu):
    results = [False] * 4

    def work(i):
        results[i] = all(identity_call(gpu, 64 + i, 256, 10 * i + j) for j in range(5))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(60)
    assert results == [True] * 4
