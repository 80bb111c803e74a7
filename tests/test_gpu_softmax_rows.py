"""Softmax over rows at the edges of its thread groups (16, 64 or 256 threads
a row, rows in registers or walked), f32 against an f64 softmax and the
special values against the oracle."""
import numpy as np
import pytest

import oracle
from dragonwing_edge_rs_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 16, 17, 128, 129, 512, 513, 2048, 2049, 5000])
@pytest.mark.parametrize("rows", [1, 5, 67])
def test_softmax_group_edges(backend, rows, n):
    x = np.random.default_rng(n + rows).normal(0, 4, (rows, n)).astype(np.float32)
    bx, by = backend.from_numpy(x), backend.alloc(x.nbytes)
    ops.softmax_f32(backend, bx, by, rows, n)
    got = backend.to_numpy(by, np.float32, (rows, n)).astype(np.float64)
    e = np.exp(x.astype(np.float64) - x.max(axis=1, keepdims=True))
    # f32: the subtraction's half ulp of up to 40, exp's 2 ulps, a tree sum of at most 32 levels
    np.testing.assert_allclose(got, e / e.sum(axis=1, keepdims=True), rtol=(40 / 2 + 2 + 32 + 2) * 2.0 ** -24,
                               atol=1e-37)


@pytest.mark.parametrize("n", [16, 200, 1000, 3000])
def test_softmax_special_rows(backend, n):
    x = np.random.default_rng(n).normal(0, 2, (6, n)).astype(np.float32)
    x[0] = -np.inf
    x[1, n // 2] = np.inf
    x[2, 3] = np.nan
    x[3] = np.finfo(np.float32).min
    x[4, 1:] = -np.inf
    bx, by = backend.from_numpy(x), backend.alloc(x.nbytes)
    ops.softmax_f32(backend, bx, by, 6, n)
    got, ref = backend.to_numpy(by, np.float32, (6, n)), oracle.softmax_f32(x)
    np.testing.assert_array_equal(np.isnan(got), np.isnan(ref))
    np.testing.assert_allclose(np.nan_to_num(got), np.nan_to_num(ref), rtol=1e-5, atol=1e-30)
