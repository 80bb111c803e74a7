"""Gemm (f32, f16; plain and transposed B) at the edges of its 8 x 16 tiles
and 256-step chunks of K: every bit equals the oracle's, which walks each sum
in the reference's order."""
import numpy as np
import pytest

import oracle
from dragonwing_edge_rs_amd import ops
from dragonwing_edge_rs_amd.graph import GRAPH_F16, GRAPH_F32, Graph, HipGraphRuntime

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 1), (16, 16, 256), (17, 15, 257), (1, 33, 255), (33, 1, 511), (5, 40, 513), (2, 1003, 3), (65, 31, 1030), (7, 16, 300),
          (8, 17, 256), (9, 15, 258)]


@pytest.mark.parametrize("mnk", SHAPES)
def test_gemm_tile_edges_bit_exact(backend, mnk):
    m, n, k = mnk
    r = np.random.default_rng(m + 3 * n + 5 * k)
    a, b = r.normal(0, 1, (m, k)).astype(np.float32), r.normal(0, 0.2, (k, n)).astype(np.float32)
    c = backend.alloc(m * n * 4)
    ops.gemm_f32(backend, backend.from_numpy(a), backend.from_numpy(b), c, m, n, k)
    np.testing.assert_array_equal(backend.to_numpy(c, np.float32, (m, n)), oracle.gemm_f32(a, b))
    ah, bh = a.astype(np.float16).view(np.uint16), b.astype(np.float16).view(np.uint16)
    ah.ravel()[::7] = 0x0003  # subnormals, which the reference decodes at half value
    c = backend.alloc(m * n * 2)
    ops.gemm_fp16(backend, backend.from_numpy(ah), backend.from_numpy(bh), c, m, n, k)
    np.testing.assert_array_equal(backend.to_numpy(c, np.uint16, (m, n)), oracle.gemm_fp16(ah, bh))


@pytest.mark.parametrize("f16", [False, True])
@pytest.mark.parametrize("mnk", SHAPES[1:])
def test_gemm_transposed_tile_edges_bit_exact(backend, mnk, f16):
    from oracle.cpu_graph import CpuGraph
    m, n, k = mnk
    r = np.random.default_rng(m + 3 * n + 5 * k + f16)
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
    rt.run()
    cg = CpuGraph(g.to_dict(), g.initializer)
    cg.set_input("x", x)
    np.testing.assert_array_equal(rt.get_output_bytes("y").view(x.dtype).reshape(m, n), cg.run()["y"])


def test_gemm_infinities_and_nan(backend):
    # products past the end of K are +0 * +0, never 0 * inf
    m, n, k = 18, 20, 259
    r = np.random.default_rng(1)
    a, b = r.normal(0, 1, (m, k)).astype(np.float32), r.normal(0, 1, (k, n)).astype(np.float32)
    a[3, 258], a[4, 0], b[258, 5], b[0, 6] = np.inf, np.nan, -np.inf, np.inf
    c = backend.alloc(m * n * 4)
    ops.gemm_f32(backend, backend.from_numpy(a), backend.from_numpy(b), c, m, n, k)
    got, ref = backend.to_numpy(c, np.float32, (m, n)), oracle.gemm_f32(a, b)
    np.testing.assert_array_equal(np.isnan(got), np.isnan(ref))
    np.testing.assert_array_equal(np.nan_to_num(got), np.nan_to_num(ref))
