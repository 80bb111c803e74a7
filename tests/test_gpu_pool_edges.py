"""Global average pools at the edges of their chunks of pixels (16 loads
ahead; four waves a quarter each for u8) and of their channel groups: every
bit equals the oracle's."""
import numpy as np
import pytest

import oracle
from dragonwing_edge_rs_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(1, 1, 1, 1), (2, 3, 5, 63), (1, 4, 4, 64), (3, 1, 17, 65), (2, 16, 4, 260), (1, 13, 5, 4),
                                   (1, 80, 83, 12)])
def test_pools_bit_exact(backend, shape):
    n, h, w, c = shape
    r = np.random.default_rng(sum(shape))
    x = r.normal(0, 2, shape).astype(np.float32)
    xh = x.astype(np.float16).view(np.uint16)
    xh.ravel()[::5] = 0x0005
    q = r.integers(0, 256, shape).astype(np.uint8)
    by = backend.alloc(n * c * 4)
    ops.global_avg_pool_nhwc(backend, ops.DTYPE_F32, backend.from_numpy(x), by, n, h, w, c)
    np.testing.assert_array_equal(backend.to_numpy(by, np.float32, (n, c)), oracle.global_avg_pool_f32(x))
    by = backend.alloc(n * c * 2)
    ops.global_avg_pool_nhwc(backend, ops.DTYPE_F16, backend.from_numpy(xh), by, n, h, w, c)
    np.testing.assert_array_equal(backend.to_numpy(by, np.uint16, (n, c)), oracle.global_avg_pool_fp16(xh))
    by = backend.alloc(n * c)
    ops.qlinear_global_avg_pool_u8(backend, backend.from_numpy(q), by, n, h, w, c, 0.03, 125, 0.01, 128)
    np.testing.assert_array_equal(backend.to_numpy(by, np.uint8, (n, c)), oracle.qlinear_gap_u8(q, 0.03, 125, 0.01, 128))
