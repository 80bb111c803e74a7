"""Activation values that name none of the activations: a convolution and a
fp32 depthwise layer apply nothing, a fp16 3x3 depthwise layer refuses them."""
import numpy as np
import pytest

from dragonwing_edge_rs_amd import ops
from dragonwing_edge_rs_amd._lib import HipError

pytestmark = pytest.mark.gpu


def values(shape, dtype):
    return np.random.default_rng(sum(shape)).uniform(-1, 1, shape).astype(dtype)


# fp16: 16-byte stores and (c_out % 8 != 0) 8-byte ones
@pytest.mark.parametrize("dtype,f,ci,co", [
    (np.float16, ops.conv2d_bias_act_f16_nhwc, 64, 64), (np.float16, ops.conv2d_bias_act_f16_nhwc, 64, 20),
    (np.float32, ops.conv2d_bias_act_f32_nhwc, 32, 40), (np.float32, ops.conv2d_bias_act_f32_nhwc, 3, 8)])
def test_conv(backend, dtype, f, ci, co):
    x, w, b = values((2, 17, 18, ci), dtype), values((3, 3, ci, co), dtype), values((co,), dtype)
    bufs = [backend.from_numpy(v) for v in (x, w, b)]
    by = backend.alloc(2 * 17 * 18 * co * x.itemsize)
    got = []
    for act in (0, 3, -1):
        f(backend, *bufs, by, 2, 17, 18, ci, co, 3, 3, 1, 1, 1, 1, act)
        got.append(backend.to_numpy(by, dtype, (2, 17, 18, co)))
    assert (got[0] < 0).any()
    np.testing.assert_array_equal(got[1], got[0])
    np.testing.assert_array_equal(got[2], got[0])


@pytest.mark.parametrize("n", [1, 16])  # one row of outputs a thread, and a march
def test_depthwise(backend, n):
    shape = (n, 40, 40, 64)
    x, w, b = values(shape, np.float32), values((3, 3, 64), np.float32), values((64,), np.float32)
    bufs = [backend.from_numpy(v) for v in (x, w, b)]
    by = backend.alloc(x.nbytes)
    got = []
    for act in (0, 3, -1):
        ops.depthwise_conv2d_f32_nhwc(backend, *bufs, by, n, 40, 40, 64, 3, 3, 1, 1, 1, 1, act)
        got.append(backend.to_numpy(by, np.float32, shape))
    assert (got[0] < 0).any()
    np.testing.assert_array_equal(got[1], got[0])
    np.testing.assert_array_equal(got[2], got[0])
    half = [backend.from_numpy(v.astype(np.float16)) for v in (x, w, b)]
    with pytest.raises(HipError, match="activation"):
        ops.depthwise_conv2d_f16_nhwc(backend, *half, backend.alloc(x.nbytes // 2), n, 40, 40, 64, 3, 3, 1, 1, 1, 1, 3)
