"""The in-order fp16 kernel: every tile it is built for, at pixel counts,
channels and k-steps that do not fill its 16-pixel tiles and rings of loads,
one, two and four k-steps to an address.  Its sums are in the staged kernel's
order, so the bits are that kernel's for any input; a whole graph's too."""
import numpy as np
import pytest

from dragonwing_edge_rs_amd import ops, synth, yolo
from dragonwing_edge_rs_amd.graph import HipGraphRuntime

pytestmark = pytest.mark.gpu

SHAPES = [  # n, h, w, c_in, c_out, k, s, p
    (1, 1, 1, 256, 4, 1, 1, 0), (1, 5, 7, 32, 20, 5, 1, 2), (2, 9, 7, 96, 36, 3, 1, 1), (1, 20, 20, 128, 128, 3, 1, 1),
    (1, 17, 3, 64, 72, 3, 2, 1), (3, 4, 5, 1056, 52, 1, 1, 0), (1, 6, 6, 640, 16, 3, 1, 1), (1, 3, 4, 32, 64, 5, 1, 4),
]


@pytest.mark.parametrize("bc", [16, 32, 64])
def test_in_order_f16_bits(backend, monkeypatch, bc):
    for shape in SHAPES:
        n, h, w, ci, co, k, s, p = shape
        r = np.random.default_rng(sum(shape))
        ho, wo = (h + 2 * p - k) // s + 1, (w + 2 * p - k) // s + 1
        bits = lambda sd, *d: synth.f16_bits(r.normal(0, sd, d).astype(np.float32))  # noqa: E731
        bx, bw, bb = (backend.from_numpy(v) for v in (bits(1, n, h, w, ci), bits(0.1, k, k, ci, co), bits(0.1, co)))
        for bias, act in ((bb, ops.ACT_SILU), (None, ops.ACT_RELU)):
            got = []
            for tile in (f"{bc},1,-7", "16,1"):
                monkeypatch.setenv("DW_IGEMM_TILE", tile)
                by = backend.alloc(n * ho * wo * co * 2)
                ops.conv2d_bias_act_f16_nhwc(backend, bx, bw, bias, by, n, h, w, ci, co, k, k, s, s, p, p, act)
                got.append(backend.to_numpy(by, np.uint16, (n, ho, wo, co)))
            np.testing.assert_array_equal(got[0], got[1], err_msg=str(shape))


@pytest.mark.parametrize("tile", ["16,1,-7", "32,1,-7", "64,1,-7"])
def test_in_order_f16_graph_same_bits(backend, monkeypatch, tile):
    # shortcut, upsampled-copy and sibling epilogues, channel slices; layers
    # the tile does not take keep their own
    g, info = yolo.f16_graph(batch=2, size=96)
    x = yolo.input_images(2, 96)
    outs = []
    for t in ("16,1", tile):
        monkeypatch.setenv("DW_IGEMM_TILE", t)
        monkeypatch.setenv("DW_RESIZE_FUSE", "1")
        rt = HipGraphRuntime(g, backend)
        rt.set_input_f32(info["input"], x)
        rt.run()
        outs.append([rt.get_output_bytes(o) for o in info["outputs"]])
        if t == tile:
            assert sum("_fp" in L["kernel"] for L in rt.launches()) >= 8
        rt.close()
    for a, b in zip(*outs):
        np.testing.assert_array_equal(a, b)
