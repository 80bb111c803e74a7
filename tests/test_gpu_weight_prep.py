"""The packing of HWIO weights into k-step rows and the per-channel values
computed with it, at the edges of its tiles: K that is not a whole number of
64-byte k-steps, more k-steps than waves, channels that do not fill a
16-channel group, more channels than one launch's arguments hold.  Every
byte of the convolution's output equals the oracle's."""
import numpy as np
import pytest

import oracle
from dragonwing_edge_rs_amd import ops, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("c_in,c_out,k", [
    (16, 4, 1),      # one quarter of a k-step, one channel quad
    (16, 20, 3),     # K = 144: a partial third k-step; a group of 16 and one quad
    (48, 84, 3),     # K = 432; 96-channel tile
    (128, 36, 3),    # 18 k-steps: more than the 16 waves of a workgroup
    (16, 896, 1),    # one launch, whole tiles
    (32, 900, 1),    # one launch, padding channels
    (16, 1008, 1),   # exactly one launch's channels, the padding's groups with them
    (48, 1012, 1),   # one quad in a second launch
    (16, 1800, 1),   # two launches
    (80, 2016, 1),   # exactly two
    (16, 2048, 3),   # three, the middle one whole
])
def test_qconv_prep_bit_exact(backend, c_in, c_out, k):
    r = np.random.default_rng(c_in + 7 * c_out + k)
    n, h, w, p = 1, 5, 6, k // 2
    x = r.integers(0, 256, (n, h, w, c_in)).astype(np.uint8)
    wt = r.integers(-128, 128, (k, k, c_in, c_out)).astype(np.int8)
    bias = r.integers(-4096, 4097, c_out).astype(np.int32)
    ws = np.exp(r.uniform(np.log(1e-3), np.log(1e-2), c_out)).astype(np.float32)
    ys = float(0.02 * 4e-3 * 5000 * np.sqrt(c_in * k * k) / 40)
    bx, bw, bb = backend.from_numpy(x), backend.from_numpy(wt), backend.from_numpy(bias)
    by = backend.alloc(n * h * w * c_out)
    for b, zp in ((bb, 131), (None, 3), (bb, 128), (None, 128)):
        ops.qlinearconv_u8s8(backend, bx, bw, b, by, n, h, w, c_in, c_out, k, k, 1, 1, p, p, 0.02, zp, ws, ys, 120)
        ref = oracle.qlinearconv_u8s8(x, wt, bias if b else None, (1, 1), (p, p), 0.02, zp, ws, ys, 120)
        np.testing.assert_array_equal(backend.to_numpy(by, np.uint8, (n, h, w, c_out)), ref)
    assert len(np.unique(ref)) > 20


@pytest.mark.parametrize("c_in,c_out,k", [(8, 4, 1), (8, 20, 3), (24, 52, 3), (64, 132, 1)])
def test_f16_pack_matches_exact_order(backend, c_in, c_out, k):
    # small integers: every sum is exact in f32 and f16 whatever its order
    r = np.random.default_rng(c_in + c_out + k)
    n, h, w, p = 1, 4, 7, k // 2
    bits = lambda a: synth.f16_bits(a.astype(np.float32))  # noqa: E731
    x, wt = bits(r.integers(-3, 4, (n, h, w, c_in))), bits(r.integers(-2, 3, (k, k, c_in, c_out)))
    bx, bw = backend.from_numpy(x), backend.from_numpy(wt)
    got = []
    for exact in (False, True):
        by = backend.alloc(n * h * w * c_out * 2)
        ops.conv2d_bias_act_f16_nhwc(backend, bx, bw, None, by, n, h, w, c_in, c_out, k, k, 1, 1, p, p, exact=exact)
        got.append(backend.to_numpy(by, np.uint16, (n, h, w, c_out)))
    np.testing.assert_array_equal(got[0], got[1])
