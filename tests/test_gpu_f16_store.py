"""The fp16 implicit GEMM's stores: channel counts that fill whole blocks,
end inside one, or are no multiple of 8 (the 4-channel stores), odd numbers
of channel blocks, pixels that end inside a 16-pixel block, on each kernel
family.  Small integers, so every sum is exact and the bits equal those of
the direct kernel whatever the order."""
import numpy as np
import pytest

from dragonwing_edge_rs_amd import ops, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tile", ["16,1", "32,2", "48,4", "80,1", "128,2", "32,2,2", "128,4,2", "48,1,-1", "64,4,-3"])
def test_f16_store_bits(backend, monkeypatch, tile):
    monkeypatch.setenv("DW_IGEMM_TILE", tile)
    bits = lambda a: synth.f16_bits(a.astype(np.float32))  # noqa: E731
    for c_in, c_out, k in ((16, 4, 1), (64, 20, 1), (64, 24, 3), (32, 72, 1), (64, 80, 1), (64, 128, 3), (64, 152, 1)):
        r = np.random.default_rng(c_in + c_out + k)
        n, h, w, p = 2, 7, 9, k // 2
        x, wt = bits(r.integers(-3, 4, (n, h, w, c_in))), bits(r.integers(-2, 3, (k, k, c_in, c_out)))
        bx, bw, bb = (backend.from_numpy(v) for v in (x, wt, bits(r.integers(-9, 10, c_out))))
        for bias, act in ((bb, ops.ACT_NONE), (None, ops.ACT_RELU)):
            got = []
            for exact in (False, True):
                by = backend.alloc(n * h * w * c_out * 2)
                ops.conv2d_bias_act_f16_nhwc(backend, bx, bw, bias, by, n, h, w, c_in, c_out, k, k, 1, 1, p, p, act,
                                             exact=exact)
                got.append(backend.to_numpy(by, np.uint16, (n, h, w, c_out)))
            np.testing.assert_array_equal(got[0], got[1], err_msg=f"{c_in} {c_out} {k} {act}")
