"""Row and column counts whose launches would pass 2^32 threads in one grid
dimension: more softmax rows and Gemm columns than that are split over another
dimension.  Each case's results are known without an oracle run."""
import numpy as np
import pytest

from dragonwing_edge_rs_amd import ops

pytestmark = pytest.mark.gpu


def test_softmax_many_rows(backend):
    # rows of one value: 1 where it is finite, NaN where it is not (inf - inf)
    rows = (1 << 28) + 37
    x = np.zeros(rows, np.float32)
    x[[0, 1 << 27, (1 << 28) - 1, 1 << 28, rows - 2]] = np.inf
    bx = backend.from_numpy(x)
    by = backend.alloc(x.nbytes)
    ops.softmax_f32(backend, bx, by, rows, 1)
    got = backend.to_numpy(by, np.float32, (rows,))
    np.testing.assert_array_equal(np.flatnonzero(got != 1), np.flatnonzero(x))
    assert np.isnan(got[x > 0]).all()


def test_gemm_many_columns(backend):
    # one row of A, one of B: C is B times A's value
    n = (1 << 29) + 21
    b = np.zeros(n, np.float16)
    at = [0, 15, 16, (1 << 27) * 4 - 1, 1 << 29, n - 1]
    b[at] = np.arange(1, 7)
    a = np.full(1, 2, np.float16)
    c = backend.alloc(n * 2)
    ops.gemm_fp16(backend, backend.from_numpy(a.view(np.uint16)), backend.from_numpy(b.view(np.uint16)), c, 1, n, 1)
    got = backend.to_numpy(c, np.uint16, (n,))
    want = np.zeros(n, np.uint16)
    want[at] = (2 * np.arange(1, 7)).astype(np.float16).view(np.uint16)
    np.testing.assert_array_equal(got, want)
