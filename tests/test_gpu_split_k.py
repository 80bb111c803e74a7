"""The split-K int8 kernel: every tile it is built for, at pixel counts and
k-steps that do not fill its 16-pixel tiles, waves and batches of loads, byte
for byte against the oracle; with the table, the shortcut and a fused upsample
inside graphs."""
import numpy as np
import pytest

import oracle
from dragonwing_edge_rs_amd import ops, yolo
from dragonwing_edge_rs_amd.graph import HipGraphRuntime

pytestmark = pytest.mark.gpu

SHAPES = [  # n, h, w, c_in, c_out, k, s, p
    (1, 1, 1, 256, 4, 1, 1, 0), (1, 5, 7, 16, 20, 5, 1, 2), (2, 9, 7, 48, 36, 3, 1, 1), (1, 20, 20, 128, 128, 3, 1, 1),
    (1, 17, 3, 144, 64, 3, 2, 1), (3, 4, 5, 1040, 52, 1, 1, 0), (1, 6, 6, 640, 16, 3, 1, 1), (1, 3, 4, 32, 32, 5, 1, 4),
]


@pytest.mark.parametrize("bc,waves", [(16, 4), (16, 8), (16, 16), (32, 4), (32, 8), (32, 16)])
def test_split_k_bit_exact(backend, monkeypatch, bc, waves):
    monkeypatch.setenv("DW_IGEMM_TILE", f"{bc},{waves},-6")
    for shape in SHAPES:
        n, h, w, ci, co, k, s, p = shape
        r = np.random.default_rng(sum(shape))
        ho, wo = oracle.out_hw(h, w, k, k, s, s, p, p)
        x = r.integers(0, 256, (n, h, w, ci)).astype(np.uint8)
        wt = r.integers(-128, 128, (k, k, ci, co)).astype(np.int8)
        b = r.integers(-4096, 4097, co).astype(np.int32)
        ws = np.exp(r.uniform(np.log(1e-3), np.log(1e-2), co)).astype(np.float32)
        ys = float(0.02 * 4e-3 * 5400 * np.sqrt(ci * k * k) / 40)
        by = backend.alloc(n * ho * wo * co)
        bx, bw, bb = backend.from_numpy(x), backend.from_numpy(wt), backend.from_numpy(b)
        ops.qlinearconv_u8s8(backend, bx, bw, bb, by, n, h, w, ci, co, k, k, s, s, p, p, 0.02, 131, ws, ys, 120)
        ref = oracle.qlinearconv_u8s8(x, wt, b, (s, s), (p, p), 0.02, 131, ws, ys, 120)
        np.testing.assert_array_equal(backend.to_numpy(by, np.uint8, ref.shape), ref, err_msg=str(shape))
        xs = x.view(np.int8)
        acc = backend.alloc(n * ho * wo * co * 4)
        ops.conv2d_i8_nhwc(backend, bx, bw, acc, n, h, w, ci, co, k, k, s, s, p, p)
        np.testing.assert_array_equal(backend.to_numpy(acc, np.int32, ref.shape),
                                      oracle.conv2d_i8_nhwc(xs, wt, (s, s), (p, p)), err_msg=str(shape))


@pytest.mark.parametrize("tile", ["16,4,-6", "32,8,-6", "16,16,-6"])
def test_split_k_graph_same_bytes(backend, monkeypatch, tile):
    # table, shortcut and upsampled-copy epilogues; tensors the graph keeps
    # as channel slices; layers the tile does not take keep their own
    g, info = yolo.int8_graph(backend, batch=2, size=96)
    x = yolo.input_images(2, 96)
    outs = []
    for t in (None, tile):
        if t:
            monkeypatch.setenv("DW_IGEMM_TILE", t)
            monkeypatch.setenv("DW_RESIZE_FUSE", "1")
        rt = HipGraphRuntime(g, backend)
        rt.set_input_f32(info["input"], x)
        rt.run()
        outs.append([rt.get_output_bytes(o) for o in info["outputs"]])
        if t:
            assert sum("_ks" in L["kernel"] for L in rt.launches()) >= 8
    for a, b in zip(*outs):
        np.testing.assert_array_equal(a, b)
