"""Calls on host buffers around the size up to which x and the outputs move by
kernels through a pinned block (8 MiB each); larger ones move by copies. The
products are exact (identity weights), so outputs are compared exactly, also from
as many threads as there are blocks (4) and from more. A short call does not wait
for another session's long one.
"""
import threading
import time

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


def test_host_calls_from_more_threads_than_blocks(gpu):
    results = [0] * 7

    def work(i):  # growing sizes, so that blocks grow too
        results[i] = sum(identity_call(gpu, 8 << (i + j) % 5, 256, 10 * i + j) for j in range(4))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(7)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(60)
    assert results == [4] * 7


def test_short_call_does_not_wait_for_a_long_one(gpu):
    """One thread calls an attention layer of milliseconds whose buffers are
    small and which fills half of the GPU's wave slots; the other counts its Dense
    calls of tens of microseconds meanwhile. Were a lock held over a call, at
    most a call or two would fit beside each long one."""
    S, hd = 6000, 48  # (a head width without the matrix-core kernel)
    rng = np.random.default_rng(1)
    W = [(rng.standard_normal((hd, hd)) / 7).astype(np.float32) for _ in range(4)]
    long_s = gpu.MHASession(1, S, hd, 1, 1, hd, S, 1, 1, 4, 2, *W)
    short_s = gpu.DenseSession(1, 64, 64, -1, 4, 1, np.eye(64, dtype=np.float32) * 240, None)
    x = rng.standard_normal((S, hd)).astype(np.float32)
    small = rng.integers(-8, 9, size=(1, 64)).astype(np.float32)
    want = long_s.execute(x)[1]
    short_s.execute(small)
    calls, spent, same = 12, [], []

    def work():
        for _ in range(calls):
            t = time.perf_counter()
            y = long_s.execute(x)[1]
            spent.append(time.perf_counter() - t)
            same.append(np.array_equal(y, want))

    thread = threading.Thread(target=work)
    thread.start()
    done = 0
    while thread.is_alive():
        pre, _ = short_s.execute(small)
        done += 1
        assert np.array_equal(pre, small * 240)
    thread.join()
    long_s.close()
    short_s.close()
    print(f"{done} short calls beside {calls} long ones of {1e3 * min(spent):.1f} ms")
    assert same == [True] * calls
    assert min(spent) > 5e-4
    assert done >= 4 * calls
