"""The detect tail at the edges of its 64-anchor tiles and on heads that its
tile kernel does not take, and post-processing at the sizes where its sort and
its download change form, bit for bit against the oracle."""
import numpy as np
import pytest

import oracle
from dragonwing_edge_rs_amd import ops

pytestmark = pytest.mark.gpu


def f64_tail(levels, strides, nc, reg_max):
    out = []
    for x, s in zip(levels, strides):
        n, h, w, _ = x.shape
        b = x[..., :4 * reg_max].reshape(n, h, w, 4, reg_max)
        e = np.exp(b - b.max(-1, keepdims=True))
        d = (e / e.sum(-1, keepdims=True) * np.arange(reg_max)).sum(-1)
        gy, gx = np.meshgrid(np.arange(h) + 0.5, np.arange(w) + 0.5, indexing="ij")
        x1, y1, x2, y2 = gx - d[..., 0], gy - d[..., 1], gx + d[..., 2], gy + d[..., 3]
        rows = [(x1 + x2) / 2 * s, (y1 + y2) / 2 * s, (x2 - x1) * s, (y2 - y1) * s]
        rows += list(np.moveaxis(1 / (1 + np.exp(-x[..., 4 * reg_max:])), -1, 0))
        out.append(np.stack(rows, 1).reshape(n, 4 + nc, h * w))
    return np.concatenate(out, 2)


# (levels, nc, reg_max): one tile, a tile and an anchor, several ragged levels; an odd
# number of channels and too many of them (thread per anchor); bins other than 16
@pytest.mark.parametrize("hw,nc,reg_max", [([(8, 8)], 80, 16), ([(5, 13)], 80, 16), ([(1, 1), (3, 7), (16, 9)], 80, 16),
                                           ([(9, 8), (4, 4)], 3, 16), ([(9, 8)], 200, 16), ([(7, 9), (2, 3)], 10, 8),
                                           ([(11, 12)], 128, 16), ([(6, 11)], 96, 16)])
@pytest.mark.parametrize("f16", [True, False])
def test_tail_tiles(backend, hw, nc, reg_max, f16):
    r = np.random.default_rng(sum(a * b for a, b in hw) + nc)
    strides = [8.0 * 2 ** i for i in range(len(hw))]
    n, chans = 3, 4 * reg_max + nc
    lv = [r.normal(0, 3, (n, h, w, chans)).astype(np.float16 if f16 else np.float32) for h, w in hw]
    A = sum(h * w for h, w in hw)
    out = backend.alloc(n * (4 + nc) * A * 4)
    ops.yolo_detect_tail(backend, [backend.from_numpy(x) for x in lv], hw, strides, n, out, nc=nc, reg_max=reg_max,
                         dtype=ops.DTYPE_F16 if f16 else ops.DTYPE_F32)
    got = backend.to_numpy(out, np.float32, (n, 4 + nc, A)).astype(np.float64)
    ref = f64_tail([x.astype(np.float64) for x in lv], strides, nc, reg_max)
    scale = np.abs(ref).max(axis=(0, 2), keepdims=True)
    # f32: the expectation of up to 16 bins sums to within 24 half ulps of 16, a box row four such
    assert (np.abs(got - ref) / scale).max() <= 1e-5


# candidates per image: none, one, around a wave, the register sort's last size, the LDS sort's
# first, and more kept than the first download holds
@pytest.mark.parametrize("counts", [[0, 1, 63, 64, 65], [1023, 1024, 1025], [300, 2500, 0]])
@pytest.mark.parametrize("agnostic", [False, True])
def test_postprocess_sizes(backend, counts, agnostic):
    r = np.random.default_rng(sum(counts))
    n, A, nc = len(counts), 3000, 80
    raw = np.zeros((n, 4 + nc, A), np.float32)
    raw[:, :2] = r.uniform(0, 640, (n, 2, A))
    raw[:, 2:4] = r.uniform(4, 40, (n, 2, A))
    raw[:, 4:] = r.uniform(0, 0.2, (n, nc, A))
    for b, k in enumerate(counts):
        at = r.permutation(A)[:k]
        raw[b, 4 + r.integers(0, nc, k), at] = np.round(r.uniform(0.3, 1, k), 2)  # ties among them
    got = ops.yolo_postprocess(backend, backend.from_numpy(raw), n, nc, A, 640, 640, 0.25, 0.45, agnostic=agnostic)
    ref = oracle.yolo_postprocess(raw, 640, 640, 0.25, 0.45, agnostic=agnostic)
    for g, e in zip(got, ref):
        assert g.tobytes() == e.tobytes()


@pytest.mark.parametrize("nc", [1, 15, 16, 17, 91])
def test_postprocess_class_counts(backend, nc):
    r = np.random.default_rng(nc)
    raw = r.uniform(0, 0.5, (2, 4 + nc, 700)).astype(np.float32)
    raw[:, :2] *= 1200
    raw[:, 2:4] = r.uniform(4, 60, (2, 2, 700))
    got = ops.yolo_postprocess(backend, backend.from_numpy(raw), 2, nc, 700, 640, 480, 0.4, 0.5)
    for g, e in zip(got, oracle.yolo_postprocess(raw, 640, 480, 0.4, 0.5)):
        assert g.tobytes() == e.tobytes()
