"""Calls whose kernels must not pay for work that their sizes do not have: each
is timed beside an elementwise pass of this backend that moves the same bytes,
and may take a small multiple of it."""
import time

import numpy as np
import pytest

from dragonwing_edge_rs_amd import ops

pytestmark = pytest.mark.gpu


def per_call(backend, f, calls=50):
    """Seconds a call, the least of several batches of calls."""
    f()
    best = np.inf
    for _ in range(8):
        backend.synchronize()
        t = time.perf_counter()
        for _ in range(calls):
            f()
        backend.synchronize()
        best = min(best, (time.perf_counter() - t) / calls)
    return best


def relu_time(backend, values):
    x, y = backend.from_numpy(np.ones(values, np.float32)), backend.alloc(values * 4)
    return per_call(backend, lambda: ops.relu_f32(backend, x, y, values))


# with 16 threads a row, whatever its length: 15, 7 and 3.5 times as long as the relu
@pytest.mark.parametrize("rows,n", [(2000000, 1), (1000000, 4), (500000, 16)])
def test_softmax_of_short_rows(backend, rows, n):
    x = np.random.default_rng(n).normal(0, 2, (rows, n)).astype(np.float32)
    bx, by = backend.from_numpy(x), backend.alloc(x.nbytes)
    t = per_call(backend, lambda: ops.softmax_f32(backend, bx, by, rows, n))
    assert t < 3 * relu_time(backend, x.size)
    got = backend.to_numpy(by, np.float32, x.shape).astype(np.float64)
    e = np.exp(x.astype(np.float64) - x.max(axis=1, keepdims=True))
    # the subtraction's half ulp of up to 20, exp's 2 ulps, at most 15 additions, two roundings
    np.testing.assert_allclose(got, e / e.sum(axis=1, keepdims=True), rtol=(20 / 2 + 2 + 15 + 2) * 2.0 ** -24)
