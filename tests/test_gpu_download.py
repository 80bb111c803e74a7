"""Downloads at the edges of their chunks and thread shares, and graph outputs
that are channel slices of another tensor: the bytes on the host are the
device's."""
import numpy as np
import pytest

from dragonwing_edge_rs_amd._lib import HipError, check, load
from dragonwing_edge_rs_amd.graph import GRAPH_F16, GRAPH_F32, Graph, HipGraphRuntime

pytestmark = pytest.mark.gpu

MIB = 1 << 20
DW_ERR_INVALID = -4


@pytest.mark.parametrize("n", [1, 4095, 16384, 16385, 131073, MIB, MIB + 1, 4 * MIB - 1, 4 * MIB, 9 * MIB + 77,
                               33 * MIB + 65537])
def test_download_sizes(backend, n):
    src = np.random.default_rng(n).integers(0, 256, n).astype(np.uint8)
    buf = backend.from_numpy(src)
    for _ in range(2):
        np.testing.assert_array_equal(backend.to_numpy(buf, np.uint8, (n,)), src)


def test_empty_download(backend):
    assert backend.to_numpy(backend.alloc(0), np.uint8, (0,)).size == 0


@pytest.mark.parametrize("dtype,pixels", [("f16", 1), ("f16", 90000), ("f32", 7)])
def test_sliced_tensors(backend, dtype, pixels):
    # the concat's inputs are channel slices of its output: one from channel 0, one from channel 8
    np_t, kind = (np.float16, GRAPH_F16) if dtype == "f16" else (np.float32, GRAPH_F32)
    r = np.random.default_rng(pixels)
    xs = [r.choice([-1, 1], (1, pixels, 1, c)) * r.uniform(0.01, 2, (1, pixels, 1, c)) for c in (8, 16)]
    xs = [x.astype(np_t) for x in xs]
    g = Graph(kind)
    for i, x in enumerate(xs):
        g.add_tensor(f"x{i}", x.shape, dtype)
        g.add_tensor(f"r{i}", x.shape, dtype)
        g.add_op(f"relu{i}", "Relu", [f"x{i}"], [f"r{i}"])
    g.add_tensor("y", (1, pixels, 1, 24), dtype)
    g.add_op("cat", "Concat", ["r0", "r1"], ["y"], axis=3)
    g.set_io(["x0", "x1"], ["y"])
    rt = HipGraphRuntime(g, backend)
    for i, x in enumerate(xs):
        rt.set_input_bytes(f"x{i}", x)
    want = [np.maximum(x, 0) for x in xs]
    want.append(np.concatenate(want, 3))
    for _ in range(2):
        rt.run()
        for name, w in zip(("r0", "r1", "y"), want):
            np.testing.assert_array_equal(rt.get_output_bytes(name).view(np_t).reshape(w.shape), w)
            np.testing.assert_array_equal(rt.get_output_f32(name, w.size).reshape(w.shape), w.astype(np.float32))


def test_slice_off_16_byte_addresses(backend):
    # one pixel of a slice is dense, from an address of its own: 6 bytes into the concat's output
    xs = [np.random.default_rng(c).uniform(0.01, 2, (1, 1, 1, c)).astype(np.float16) for c in (3, 5000)]
    g = Graph(GRAPH_F16)
    for i, x in enumerate(xs):
        g.add_tensor(f"x{i}", x.shape, "f16")
        g.add_tensor(f"r{i}", x.shape, "f16")
        g.add_op(f"relu{i}", "Relu", [f"x{i}"], [f"r{i}"])
    g.add_tensor("y", (1, 1, 1, 5003), "f16")
    g.add_op("cat", "Concat", ["r0", "r1"], ["y"], axis=3)
    g.set_io(["x0", "x1"], ["y"])
    rt = HipGraphRuntime(g, backend)
    for i, x in enumerate(xs):
        rt.set_input_bytes(f"x{i}", x)
    rt.run()
    for name, w in (("r0", xs[0]), ("r1", xs[1]), ("y", np.concatenate(xs, 3))):
        np.testing.assert_array_equal(rt.get_output_bytes(name).view(np.float16), w.ravel())


def test_null_destinations_are_refused(backend):
    buf = backend.alloc(24)
    with pytest.raises(HipError, match="null") as e:
        check(load().dw_hip_download(backend.handle, buf.handle, None, 24))
    assert e.value.code == DW_ERR_INVALID
    g = Graph(GRAPH_F32)
    for name in ("x", "y"):
        g.add_tensor(name, (1, 2, 1, 3))
    g.add_op("relu", "Relu", ["x"], ["y"])
    g.set_io(["x"], ["y"])
    rt = HipGraphRuntime(g, backend)
    rt.set_input_f32("x", np.ones(6, np.float32))
    rt.run()
    for f, size in ((load().dw_hip_graph_get_output_f32, 6), (load().dw_hip_graph_get_output_bytes, 24)):
        with pytest.raises(HipError, match="null") as e:
            check(f(rt._h, b"y", None, size))
        assert e.value.code == DW_ERR_INVALID
    np.testing.assert_array_equal(rt.get_output_f32("y", 6), 1)
