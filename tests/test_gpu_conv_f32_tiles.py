"""fp32 convolution on the register-tiled kernel at the edges of its tiles
(32, 64 or 128 pixels, 8 to 40 channels) and chunks of K (32, 64 or 128
steps; whole taps or part of one), every bit equal to the oracle's ordered
sums, with channel-sliced inputs and weights that are not finite."""
import numpy as np
import pytest

import oracle
from dragonwing_edge_rs_amd import ops
from dragonwing_edge_rs_amd.graph import GRAPH_F32, Graph, HipGraphRuntime

pytestmark = pytest.mark.gpu


def run(backend, x, w, b, s, p, act=ops.ACT_NONE):
    n, h, wd, ci = x.shape
    kh, kw, _, co = w.shape
    ho, wo = oracle.out_hw(h, wd, kh, kw, s[0], s[1], p[0], p[1])
    y = backend.alloc(n * ho * wo * co * 4)
    ops.conv2d_bias_act_f32_nhwc(backend, backend.from_numpy(x), backend.from_numpy(w),
                                 None if b is None else backend.from_numpy(b), y, n, h, wd, ci, co, kh, kw, *s, *p, act)
    return backend.to_numpy(y, np.float32, (n, ho, wo, co))


@pytest.mark.parametrize("n,h,w,ci,co,k,s,p", [
    (1, 1, 1, 1, 1, 1, 1, 0),          # one output
    (1, 5, 7, 3, 5, 3, 1, 1),          # several taps a chunk, an odd channel count
    (2, 9, 8, 13, 17, 3, 2, 1),        # a partial quad of K at every tap
    (1, 8, 4, 128, 8, 3, 1, 1),        # whole chunk = one tap; 32 pixels, 8 channels exactly
    (1, 11, 3, 129, 9, 3, 1, 1),       # one channel past it
    (1, 6, 6, 132, 40, 3, 1, 1),       # vector loads, a tap in two chunks
    (3, 20, 21, 64, 41, 3, 1, 1),
    (2, 40, 41, 65, 33, 1, 1, 0),
    (4, 64, 66, 33, 70, 3, 1, 1),      # many pixels: the widest tiles
    (4, 64, 66, 36, 64, 3, 2, 1),
    (1, 12, 13, 6, 24, 5, 1, 2),       # 25 taps
    (1, 7, 30, 20, 12, 3, 3, 0),       # stride 3, no padding
    (1, 4, 5, 16, 8, 3, 1, 4),         # taps that are outside for whole pixels
])
def test_conv_f32_bit_exact(backend, n, h, w, ci, co, k, s, p):
    r = np.random.default_rng(n + 3 * h + 5 * w + 7 * ci + 11 * co + k)
    x = r.uniform(-1, 1, (n, h, w, ci)).astype(np.float32)
    wt = r.uniform(-1, 1, (k, k, ci, co)).astype(np.float32)
    b = r.uniform(-1, 1, co).astype(np.float32)
    ref = oracle.conv2d_f32_nhwc(x, wt, (s, s), (p, p))
    np.testing.assert_array_equal(run(backend, x, wt, None, (s, s), (p, p)), ref)
    np.testing.assert_array_equal(run(backend, x, wt, b, (s, s), (p, p), ops.ACT_RELU), np.maximum(ref + b, 0))


def test_conv_f32_rectangular(backend):
    r = np.random.default_rng(8)
    x, wt = r.normal(0, 1, (2, 17, 9, 10)).astype(np.float32), r.normal(0, 1, (1, 5, 10, 11)).astype(np.float32)
    np.testing.assert_array_equal(run(backend, x, wt, None, (2, 1), (0, 2)), oracle.conv2d_f32_nhwc(x, wt, (2, 1), (0, 2)))


@pytest.mark.parametrize("ci", [5, 64, 200])
def test_conv_f32_weights_not_finite(backend, ci):
    # infinite and NaN weights of taps that lie outside the image for border pixels
    r = np.random.default_rng(ci)
    x, wt = r.normal(0, 1, (1, 6, 9, ci)).astype(np.float32), r.normal(0, 1, (3, 3, ci, 12)).astype(np.float32)
    wt[0, 1, ci // 2, 3], wt[2, 2, 0, 5], wt[1, 0, ci - 1, 7] = np.inf, np.nan, -np.inf
    got, ref = run(backend, x, wt, None, (1, 1), (1, 1)), oracle.conv2d_f32_nhwc(x, wt, (1, 1), (1, 1))
    assert 0 < np.isnan(ref).sum() + np.isinf(ref).sum() < ref.size
    np.testing.assert_array_equal(got, ref)


@pytest.mark.parametrize("c0,c1", [(4, 12), (3, 10)])
def test_conv_f32_channel_slices(backend, c0, c1):
    # the convs read and write channel slices of the concat's output
    r = np.random.default_rng(c0)
    x = r.uniform(-1, 1, (2, 10, 11, c0)).astype(np.float32)
    ws = [r.uniform(-1, 1, (3, 3, c0, c1)).astype(np.float32), r.uniform(-1, 1, (3, 3, c1, 9)).astype(np.float32)]
    g = Graph(GRAPH_F32)
    g.add_tensor("x", x.shape)
    g.add_tensor("r", x.shape)
    g.add_op("relu", "Relu", ["x"], ["r"])
    for i, (src, dst, co) in enumerate((("r", "a", c1), ("a", "b", 9))):
        g.add_initializer(f"w{i}", ws[i])
        g.add_tensor(dst, (2, 10, 11, co))
        g.add_op(f"conv{i}", "Conv", [src, f"w{i}"], [dst], kernel_shape=(3, 3), pads=(1, 1, 1, 1))
    g.add_tensor("y", (2, 10, 11, c0 + c1 + 9))
    g.add_op("cat", "Concat", ["r", "a", "b"], ["y"], axis=3)
    g.set_io(["x"], ["y"])
    rt = HipGraphRuntime(g, backend)
    rt.set_input_f32("x", x)
    rt.run()
    x = np.maximum(x, 0)
    a = oracle.conv2d_f32_nhwc(x, ws[0], (1, 1), (1, 1))
    b = oracle.conv2d_f32_nhwc(a, ws[1], (1, 1), (1, 1))
    want = np.concatenate([x, a, b], 3)
    np.testing.assert_array_equal(rt.get_output_bytes("y").view(np.float32).reshape(want.shape), want)
