"""Device memory that a graph runtime takes for weights: one copy in the layout
that the layer's kernel reads, beside the HWIO one where they differ."""
import ctypes as C

import numpy as np
import pytest

from dragonwing_edge_rs_amd.graph import GRAPH_F32, Graph, HipGraphRuntime

pytestmark = pytest.mark.gpu

MIB = 1 << 20


def free_memory():
    hip = C.CDLL("libamdhip64.so.7")  # the runtime that the backend has loaded
    free, total = C.c_size_t(), C.c_size_t()
    assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


# (64 -> 64 on 4 x 40 x 40 is past the window kernel's waves, 56 x 56 on one image is not)
@pytest.mark.parametrize("x_shape,w_shape,copies", [
    ((1, 8, 8, 2048), (1, 1, 2048, 2048), 1), ((1, 8, 8, 512), (3, 3, 512, 512), 1),
    ((4, 40, 40, 64), (3, 3, 64, 64), 1), ((1, 56, 56, 64), (3, 3, 64, 64), 2),
])
def test_f32_weights_uploaded_once(backend, x_shape, w_shape, copies):
    # enough layers that the weights outweigh everything else
    wbytes, layers = int(np.prod(w_shape)) * 4, 1
    while layers * wbytes < 64 * MIB:
        layers += 1
    w = np.random.default_rng(0).uniform(-1, 1, w_shape).astype(np.float32)
    g = Graph(GRAPH_F32)
    g.add_tensor("t0", x_shape)
    p = w_shape[0] // 2
    for i in range(layers):
        g.add_initializer(f"w{i}", w)
        g.add_tensor(f"t{i + 1}", x_shape)
        g.add_op(f"c{i}", "Conv", [f"t{i}", f"w{i}"], [f"t{i + 1}"], kernel_shape=w_shape[:2], pads=(p, p, p, p))
    g.set_io(["t0"], [f"t{layers}"])
    before = free_memory()
    rt = HipGraphRuntime(g, backend)
    took = before - free_memory()
    rt.close()
    assert (copies - 0.1) * layers * wbytes < took < (copies + 0.6) * layers * wbytes
