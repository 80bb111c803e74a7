"""Convolutions whose tile the op functions choose by expected time: sizes on
both sides of the choices (staged, streamed-weight and wide tiles; 16 to 256
channels; few and many workgroups), every byte against the oracle, and fp16
on integers whose sums are exact in any order."""
import numpy as np
import pytest

import oracle
from dragonwing_edge_rs_amd import ops, synth

pytestmark = pytest.mark.gpu

SHAPES = [  # n, h, w, c_in, c_out, k, s
    (1, 20, 20, 256, 256, 3, 1), (1, 7, 9, 16, 16, 1, 1), (2, 33, 21, 64, 100, 3, 2), (4, 40, 40, 128, 128, 1, 1),
    (8, 20, 20, 256, 64, 1, 1), (3, 13, 17, 48, 84, 3, 1), (2, 80, 80, 16, 32, 3, 1), (9, 31, 30, 128, 256, 3, 2),
    (1, 1, 33, 1280, 1000, 1, 1),
]


@pytest.mark.parametrize("shape", SHAPES)
def test_chosen_tiles(backend, shape):
    n, h, w, ci, co, k, s = shape
    r = np.random.default_rng(sum(shape))
    p = k // 2
    ho, wo = oracle.out_hw(h, w, k, k, s, s, p, p)
    x, wt = r.integers(0, 256, (n, h, w, ci)).astype(np.uint8), r.integers(-127, 128, (k, k, ci, co)).astype(np.int8)
    bias = r.integers(-4096, 4097, co).astype(np.int32)
    ws = np.exp(r.uniform(np.log(1e-3), np.log(1e-2), co)).astype(np.float32)
    ys = float(0.02 * 4e-3 * 5400 * np.sqrt(ci * k * k) / 40)
    by = backend.alloc(n * ho * wo * co)
    ops.qlinearconv_u8s8(backend, backend.from_numpy(x), backend.from_numpy(wt), backend.from_numpy(bias), by, n, h, w,
                         ci, co, k, k, s, s, p, p, 0.02, 128, ws, ys, 128)
    ref = oracle.qlinearconv_u8s8(x, wt, bias, (s, s), (p, p), 0.02, 128, ws, ys, 128)
    np.testing.assert_array_equal(backend.to_numpy(by, np.uint8, (n, ho, wo, co)), ref)
    xs, wss = r.integers(-1, 2, (n, h, w, ci)), r.integers(-1, 2, (k, k, ci, co))
    xs[r.random(xs.shape) < 0.5] = 0  # |sums| stay below 2^11: exact in f16
    bits = lambda a: synth.f16_bits(a.astype(np.float32))  # noqa: E731
    bx, bw, got = backend.from_numpy(bits(xs)), backend.from_numpy(bits(wss)), []
    for exact in (False, True):
        b2 = backend.alloc(n * ho * wo * co * 2)
        ops.conv2d_bias_act_f16_nhwc(backend, bx, bw, None, b2, n, h, w, ci, co, k, k, s, s, p, p, act=ops.ACT_RELU,
                                     exact=exact)
        got.append(backend.to_numpy(b2, np.uint16, (n, ho, wo, co)))
    np.testing.assert_array_equal(got[0], got[1])


@pytest.mark.parametrize("shape", SHAPES[:6])
def test_chosen_tiles_symmetric_int8(backend, shape):
    n, h, w, ci, co, k, s = shape
    r = np.random.default_rng(sum(shape) + 1)
    p = k // 2
    ho, wo = oracle.out_hw(h, w, k, k, s, s, p, p)
    x, wt = (r.integers(-128, 128, sh).astype(np.int8) for sh in ((n, h, w, ci), (k, k, ci, co)))
    by = backend.alloc(n * ho * wo * co * 4)
    ops.conv2d_i8_nhwc(backend, backend.from_numpy(x), backend.from_numpy(wt), by, n, h, w, ci, co, k, k, s, s, p, p)
    acc = oracle.conv2d_i8_nhwc(x, wt, (s, s), (p, p))
    np.testing.assert_array_equal(backend.to_numpy(by, np.int32, (n, ho, wo, co)), acc)
    bq = backend.alloc(n * ho * wo * co)
    ops.conv2d_requant_relu_i8(backend, backend.from_numpy(x), backend.from_numpy(wt), bq, n, h, w, ci, co, k, k, s, s,
                               p, p, 0.001, True)
    q = np.sign(acc) * np.floor(np.abs(np.clip(acc.astype(np.float32) * np.float32(0.001), -128, 127)) + 0.5)
    np.testing.assert_array_equal(backend.to_numpy(bq, np.int8, (n, ho, wo, co)), np.maximum(q, 0).astype(np.int8))
