"""Calls whose kernels must not pay for work that their sizes do not have: each
is timed beside an elementwise pass of this backend that moves the same bytes,
and may take a small multiple of it."""
import time

import numpy as np
import pytest

import oracle
from dragonwing_edge_rs_amd import ops
from dragonwing_edge_rs_amd.graph import GRAPH_F16, GRAPH_F32, Graph, HipGraphRuntime

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


# in tiles of 256 steps of K, whatever K is: 3.5 to 5 times as long as the relu of as many values
@pytest.mark.parametrize("f16", [False, True])
@pytest.mark.parametrize("m,n,k", [(1024, 1024, 8), (1, 100000, 3), (4097, 257, 5)])
def test_gemm_of_few_steps(backend, m, n, k, f16):
    r = np.random.default_rng(m + n + k)
    a, b = r.normal(0, 1, (m, k)).astype(np.float32), r.normal(0, 0.2, (k, n)).astype(np.float32)
    f, want = ops.gemm_f32, oracle.gemm_f32
    if f16:
        a, b = a.astype(np.float16).view(np.uint16), b.astype(np.float16).view(np.uint16)
        f, want = ops.gemm_fp16, oracle.gemm_fp16
    ba, bb, bc = backend.from_numpy(a), backend.from_numpy(b), backend.alloc(m * n * a.itemsize)
    t = per_call(backend, lambda: f(backend, ba, bb, bc, m, n, k))
    assert t < 2.5 * relu_time(backend, m * n)
    np.testing.assert_array_equal(backend.to_numpy(bc, a.dtype, (m, n)), want(a, b))


# (10 steps: in tiles 7 times as long)
@pytest.mark.parametrize("f16", [False, True])
@pytest.mark.parametrize("m,n,k,limit", [(1500, 700, 4, 3), (523, 2525, 10, 6)])
def test_transposed_gemm_of_few_steps(backend, m, n, k, limit, f16):
    from oracle.cpu_graph import CpuGraph
    r = np.random.default_rng(k + f16)
    dt, cast = ("f16", lambda v: v.astype(np.float16).view(np.uint16)) if f16 else ("f32", lambda v: v.astype(np.float32))
    x, w, b = cast(r.normal(0, 1, (m, k))), cast(r.normal(0, 0.2, (n, k))), cast(r.normal(0, 1, n))
    g = Graph(GRAPH_F16 if f16 else GRAPH_F32)
    g.add_tensor("x", x.shape, dt)
    g.add_initializer("w", w, dt)
    g.add_initializer("b", b, dt)
    g.add_tensor("y", (m, n), dt)
    g.add_op("fc", "Gemm", ["x", "w", "b"], ["y"], trans_b=1)
    g.set_io(["x"], ["y"])
    rt = HipGraphRuntime(g, backend)
    rt.set_input_bytes("x", x)
    assert per_call(backend, rt.run) < limit * relu_time(backend, m * n)
    cg = CpuGraph(g.to_dict(), g.initializer)
    cg.set_input("x", x)
    np.testing.assert_array_equal(rt.get_output_bytes("y").view(x.dtype).reshape(m, n), cg.run()["y"])


def conv_f32(backend, bx, bw, by, x_shape, w_shape, s, p):
    n, h, w, ci = x_shape
    ops.conv2d_bias_act_f32_nhwc(backend, bx, bw, None, by, n, h, w, ci, w_shape[3], *w_shape[:2], s, s, p, p)


# on the register-tiled kernel: 4 to 13 times as long as the relu of the input (19 times with 7 x 7 taps)
@pytest.mark.parametrize("x_shape,w_shape,s,limit", [
    ((1, 640, 641, 4), (1, 1, 4, 1), 1, 2),
    ((1, 640, 639, 1), (3, 3, 1, 1), 1, 3),
    ((32, 112, 111, 3), (7, 7, 3, 8), 2, 9),
    ((8, 150, 151, 5), (1, 1, 5, 11), 1, 3),
])
def test_conv_f32_of_few_channels(backend, x_shape, w_shape, s, limit):
    r = np.random.default_rng(x_shape[2])
    x, w = r.uniform(-1, 1, x_shape).astype(np.float32), r.uniform(-1, 1, w_shape).astype(np.float32)
    p = w_shape[0] // 2
    want = oracle.conv2d_f32_nhwc(x, w, (s, s), (p, p))
    bx, bw, by = backend.from_numpy(x), backend.from_numpy(w), backend.alloc(want.nbytes)
    t = per_call(backend, lambda: conv_f32(backend, bx, bw, by, x_shape, w_shape, s, p))
    np.testing.assert_array_equal(backend.to_numpy(by, np.float32, want.shape), want)
    assert t < limit * relu_time(backend, max(x.size, want.size))


# every tap of the filter on maps that few of them meet: 13, 6, 6 and 10 times as long as the relu
@pytest.mark.parametrize("x_shape,w_shape,s,limit", [
    ((18, 1, 1, 47), (7, 7, 47, 99), 1, 5),      # one tap
    ((11, 1, 23, 20), (7, 7, 20, 1), 1, 4),      # one row
    ((14, 40, 1, 20), (7, 7, 20, 40), 1, 6),     # one column
    ((5, 2, 2, 28), (7, 7, 28, 4), 1, 5),        # three rows of three, several taps a chunk
])
def test_conv_f32_of_taps_outside_the_image(backend, x_shape, w_shape, s, limit):
    test_conv_f32_of_few_channels(backend, x_shape, w_shape, s, limit)


# the same cuts where the register-tiled kernel takes them: whole taps and parts of taps a chunk, strides that
# leave taps between unmet, infinite weights in the taps that are cut off
@pytest.mark.parametrize("x_shape,w_shape,s", [
    ((9, 2, 3, 12), (7, 5, 12, 40), 1), ((23, 7, 2, 188), (7, 7, 188, 13), 2), ((3, 1, 5, 40), (5, 9, 40, 33), 2),
    ((4, 6, 1, 300), (9, 7, 300, 20), 3), ((2, 1, 1, 16), (3, 3, 16, 24), 2), ((2, 3, 3, 30), (9, 9, 30, 9), 4),
])
def test_conv_f32_cut_filters(backend, x_shape, w_shape, s):
    r = np.random.default_rng(sum(x_shape))
    (n, h, w, ci), (kh, kw, _, co) = x_shape, w_shape
    ph, pw = kh // 2, kw // 2
    x, wt = r.uniform(-1, 1, x_shape).astype(np.float32), r.uniform(-1, 1, w_shape).astype(np.float32)
    ho, wo = oracle.out_hw(h, w, kh, kw, s, s, ph, pw)
    rows = [k for k in range(kh) if any(0 <= o * s - ph + k < h for o in range(ho))]
    cols = [k for k in range(kw) if any(0 <= o * s - pw + k < w for o in range(wo))]
    unmet = np.ones((kh, kw), bool)
    unmet[np.ix_(rows, cols)] = False
    assert unmet.any()
    wt[unmet] = np.inf
    want = oracle.conv2d_f32_nhwc(x, wt, (s, s), (ph, pw))
    assert np.isfinite(want).all()
    by = backend.alloc(want.nbytes)
    ops.conv2d_bias_act_f32_nhwc(backend, backend.from_numpy(x), backend.from_numpy(wt), None, by, n, h, w, ci, co, kh,
                                 kw, s, s, ph, pw)
    np.testing.assert_array_equal(backend.to_numpy(by, np.float32, want.shape), want)


@pytest.mark.parametrize("x_shape,w_shape", [
    # few channels on the side of the rule that keeps the tiles: odd quads of K and several taps a chunk
    ((1, 20, 21, 13), (5, 5, 13, 17)), ((2, 31, 33, 3), (7, 7, 3, 101)), ((4, 40, 41, 7), (3, 3, 7, 70)),
    ((1, 14, 15, 11), (3, 3, 11, 45)), ((1, 5, 6, 24), (5, 5, 24, 3)), ((1, 20, 20, 65), (3, 3, 65, 2)),
    # on the other: one channel, a 1x1 on 4, many channels from one, the window kernel's 4 output channels
    ((1, 40, 41, 1), (3, 3, 1, 1)), ((2, 33, 34, 4), (1, 1, 4, 24)), ((2, 25, 26, 1), (7, 7, 1, 97)),
    ((4, 90, 91, 48), (3, 3, 48, 1)), ((9, 101, 102, 32), (3, 3, 32, 4)),
])
def test_conv_f32_on_both_sides_of_the_rule(backend, x_shape, w_shape):
    r = np.random.default_rng(x_shape[1])
    x, w = r.uniform(-1, 1, x_shape).astype(np.float32), r.uniform(-1, 1, w_shape).astype(np.float32)
    p = w_shape[0] // 2
    want = oracle.conv2d_f32_nhwc(x, w, (1, 1), (p, p))
    by = backend.alloc(want.nbytes)
    conv_f32(backend, backend.from_numpy(x), backend.from_numpy(w), by, x_shape, w_shape, 1, p)
    np.testing.assert_array_equal(backend.to_numpy(by, np.float32, want.shape), want)


def test_conv_f32_past_the_tiles_offsets(backend):
    # 2 GB of input, past the register tiles' 32-bit offsets: 5 times as long as half of it, which they reach
    # (11 times with 4 channels a thread)
    w_shape, times = (1, 1, 64, 16), []
    r = np.random.default_rng(2)
    block = r.uniform(-1, 1, (1, 5, 16384, 64)).astype(np.float32)
    w = r.uniform(-1, 1, w_shape).astype(np.float32)
    bw = backend.from_numpy(w)
    for h in (255, 510):
        shape = (1, h, 16384, 64)
        bx, by = backend.from_numpy(np.resize(block, shape)), backend.alloc(h * 16384 * 16 * 4)
        times.append(per_call(backend, lambda: conv_f32(backend, bx, bw, by, shape, w_shape, 1, 0), calls=3))
        got = backend.to_numpy(by, np.float32, (h // 5, 5, 16384, 16))
        np.testing.assert_array_equal(got, np.broadcast_to(oracle.conv2d_f32_nhwc(block, w, (1, 1), (0, 0)), got.shape))
    assert times[1] < 8 * times[0]


# in workgroups of one wave with 16 loads a value, whatever there is to load: 2.2 to 2.5 times as long as the relu
@pytest.mark.parametrize("dtype", [ops.DTYPE_F32, ops.DTYPE_F16])
@pytest.mark.parametrize("n,h,w,c", [(4096, 1, 1, 1024), (4096, 2, 1, 1021), (2500, 3, 1, 1030)])
def test_pool_of_few_pixels(backend, n, h, w, c, dtype):
    f16 = dtype == ops.DTYPE_F16
    x = np.random.default_rng(c).normal(0, 2, (n, h, w, c)).astype(np.float16 if f16 else np.float32)
    bx, by = backend.from_numpy(x), backend.alloc(n * c * x.itemsize)
    t = per_call(backend, lambda: ops.global_avg_pool_nhwc(backend, dtype, bx, by, n, h, w, c))
    assert t < 1.6 * relu_time(backend, n * c * (h * w + 1) // 2)
    if f16:
        x = x.view(np.uint16)
    want = (oracle.global_avg_pool_fp16 if f16 else oracle.global_avg_pool_f32)(x)
    np.testing.assert_array_equal(backend.to_numpy(by, x.dtype, (n, c)), want)


# byte a thread (up to 4 pixels, or channels in no fours) in both workgroup sizes, and a dword
@pytest.mark.parametrize("n,h,w,c", [(4096, 2, 2, 67), (70, 1, 3, 260), (4099, 5, 1, 65), (5, 5, 1, 64)])
def test_quantized_pool_of_few_pixels(backend, n, h, w, c):
    x = np.random.default_rng(c).integers(0, 256, (n, h, w, c)).astype(np.uint8)
    by = backend.alloc(n * c)
    ops.qlinear_global_avg_pool_u8(backend, backend.from_numpy(x), by, n, h, w, c, 0.03, 125, 0.01, 128)
    np.testing.assert_array_equal(backend.to_numpy(by, np.uint8, (n, c)), oracle.qlinear_gap_u8(x, 0.03, 125, 0.01, 128))


# four columns of outputs a thread, whatever the map's width: 1.4 and 1.7 times as long as the map on its side (f16)
@pytest.mark.parametrize("shape,s", [((32, 200, 1, 512), 2), ((26, 58, 2, 712), 2), ((19, 126, 1, 136), 1), ((3, 7, 2, 24), 2),
                                     ((2, 5, 1, 8), 1), ((40, 200, 2, 256), 1)])
@pytest.mark.parametrize("f16", [False, True])
def test_depthwise_of_narrow_maps(backend, shape, s, f16):
    n, h, w, c = shape
    r = np.random.default_rng(c)
    x, k = r.uniform(-1, 1, shape).astype(np.float32), r.uniform(-1, 1, (3, 3, c)).astype(np.float32)
    fn, ref = ops.depthwise_conv2d_f32_nhwc, oracle.depthwise_f32
    if f16:
        x, k = x.astype(np.float16).view(np.uint16), k.astype(np.float16).view(np.uint16)
        fn, ref = ops.depthwise_conv2d_f16_nhwc, oracle.depthwise_fp16
    bx, bk = backend.from_numpy(x), backend.from_numpy(k)
    want = ref(x, k, (s, s), (1, 1))
    by = backend.alloc(want.nbytes)
    if f16 and n > 20 and s == 2:
        t = [per_call(backend, lambda: fn(backend, bx, bk, None, by, n, hh, ww, c, 3, 3, s, s, 1, 1))
             for hh, ww in ((w, h), (h, w))]
        assert t[1] < 1.3 * t[0]
    fn(backend, bx, bk, None, by, n, h, w, c, 3, 3, s, s, 1, 1)
    np.testing.assert_array_equal(backend.to_numpy(by, x.dtype, want.shape), want)


# in tiles of 64 anchors with the loads of 160 channels: 46 and 4.5 times as long as the relu
@pytest.mark.parametrize("f16", [False, True])
@pytest.mark.parametrize("n,hw,nc,reg_max,limit", [(20000, [(1, 2), (1, 1)], 2, 2, 12),
                                                   (32, [(80, 80), (40, 40), (20, 20)], 2, 1, 3)])
def test_tail_of_few_channels(backend, n, hw, nc, reg_max, limit, f16):
    from test_gpu_detect_edges import f64_tail
    r = np.random.default_rng(n)
    strides = [8.0 * 2 ** i for i in range(len(hw))]
    A, chans = sum(h * w for h, w in hw), 4 * reg_max + nc
    lv = [r.normal(0, 3, (n, h, w, chans)).astype(np.float16 if f16 else np.float32) for h, w in hw]
    bl, out = [backend.from_numpy(x) for x in lv], backend.alloc(n * (4 + nc) * A * 4)
    t = per_call(backend, lambda: ops.yolo_detect_tail(backend, bl, hw, strides, n, out, nc=nc, reg_max=reg_max,
                                                       dtype=ops.DTYPE_F16 if f16 else ops.DTYPE_F32))
    assert t < limit * relu_time(backend, n * A * chans)
    got = backend.to_numpy(out, np.float32, (n, 4 + nc, A)).astype(np.float64)
    ref = f64_tail([x.astype(np.float64) for x in lv], strides, nc, reg_max)
    assert (np.abs(got - ref) <= 1e-5 * np.abs(ref).max(axis=(0, 2), keepdims=True)).all()  # as test_tail_tiles


# the widest tile of at least 512 workgroups, which wider ones were chosen over: 1.19 to 1.36 times as long
@pytest.mark.parametrize("f16,x_shape,w_shape,s,tile", [
    (True, (27, 158, 30, 352), (5, 5, 352, 32), 1, "32,2"), (True, (1, 156, 128, 216), (1, 1, 216, 532), 2, "128,1"),
    (True, (14, 30, 77, 16), (3, 3, 16, 204), 1, "128,1"), (False, (16, 13, 151, 384), (1, 1, 384, 428), 2, "128,1"),
    (False, (25, 14, 85, 608), (5, 5, 608, 36), 1, "48,1")])
def test_chosen_tile_is_not_slower(backend, monkeypatch, f16, x_shape, w_shape, s, tile):
    (n, h, w, ci), (k, _, _, co) = x_shape, w_shape
    ho, wo = oracle.out_hw(h, w, k, k, s, s, k // 2, k // 2)
    bx, bw = (backend.from_numpy(np.ones(sh, np.float16 if f16 else np.int8)) for sh in (x_shape, w_shape))
    by = backend.alloc(n * ho * wo * co * (2 if f16 else 4))
    geo = (by, n, h, w, ci, co, k, k, s, s, k // 2, k // 2)

    def conv():
        if f16:
            ops.conv2d_bias_act_f16_nhwc(backend, bx, bw, None, *geo)
        else:
            ops.conv2d_i8_nhwc(backend, bx, bw, *geo)

    times = [np.inf, np.inf]
    for _ in range(2):
        for i in (0, 1):
            if i:
                monkeypatch.setenv("DW_IGEMM_TILE", tile)
            else:
                monkeypatch.delenv("DW_IGEMM_TILE", raising=False)
            times[i] = min(times[i], per_call(backend, conv, calls=20))
    assert times[0] < 1.15 * times[1]


def test_download_of_64_kib(backend):
    # through a kernel: little longer than 4 bytes, also where HIP's copies took 10 times as long, after a
    # large allocation was freed
    backend.from_numpy(np.ones(1 << 29, np.float32)).free()
    times = []
    for size in (4, 64 << 10):
        buf, dst = backend.alloc(size), np.zeros(size, np.uint8)
        times.append(per_call(backend, lambda: backend.download(buf, dst)))
    assert times[1] < 2 * times[0]
