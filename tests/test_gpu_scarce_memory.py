"""Downloads where the runtime refuses more memory: each child process loads,
ahead of the backend, a library whose hipHostMalloc and hipMalloc can be told to
return hipErrorOutOfMemory."""
import subprocess
import sys
from pathlib import Path

import pytest

pytestmark = pytest.mark.gpu

ROOT = Path(__file__).resolve().parent.parent

REFUSE = """
#include <dlfcn.h>
#include <stddef.h>
int refuse_host, refuse_device, refused;
static void* real(const char* name) {
  static void* lib;
  if (!lib) lib = dlopen("libamdhip64.so.7", RTLD_NOW);
  return dlsym(lib, name);
}
static int no(void** p) { *p = 0; ++refused; return 2; }
int hipHostMalloc(void** p, size_t n, unsigned flags) {
  return refuse_host ? no(p) : ((int (*)(void**, size_t, unsigned))real("hipHostMalloc"))(p, n, flags);
}
int hipMalloc(void** p, size_t n) { return refuse_device ? no(p) : ((int (*)(void**, size_t))real("hipMalloc"))(p, n); }
"""

SETUP = """
import ctypes as C
import sys
sys.path.insert(0, {root!r})
lib = C.CDLL({lib!r}, C.RTLD_GLOBAL)
flag = lambda name: C.c_int.in_dll(lib, name)
import numpy as np
import __graft_entry__
__graft_entry__.import_pkg()
import dragonwing_edge_rs_amd as dw
from dragonwing_edge_rs_amd.graph import GRAPH_F32, Graph, HipGraphRuntime
be = dw.Backend(0)
"""

HOST = """
sizes = (5, 300001, (2 << 20) + 3, (9 << 20) + 77)
srcs = [np.random.default_rng(n).integers(0, 256, n).astype(np.uint8) for n in sizes]
bufs = [be.from_numpy(s) for s in srcs]
for refuse in (1, 0, 1):
    flag("refuse_host").value = refuse
    for b, s in zip(bufs, srcs):
        np.testing.assert_array_equal(be.to_numpy(b, np.uint8, s.shape), s)
assert flag("refused").value >= len(sizes)
"""

# a slice of the concat's channels, read back once without memory to gather into and once with it
DEVICE = """
xs = [np.random.default_rng(c).uniform(0.1, 1, (2, 9, 7, c)).astype(np.float32) for c in (12, 20)]
g = Graph(GRAPH_F32)
for i, x in enumerate(xs):
    g.add_tensor(f"x{i}", x.shape)
    g.add_tensor(f"r{i}", x.shape)
    g.add_op(f"relu{i}", "Relu", [f"x{i}"], [f"r{i}"])
g.add_tensor("y", (2, 9, 7, 32))
g.add_op("cat", "Concat", ["r0", "r1"], ["y"], axis=3)
g.set_io(["x0", "x1"], ["y"])
rt = HipGraphRuntime(g, be)
for i, x in enumerate(xs):
    rt.set_input_f32(f"x{i}", x)
rt.run()
before = flag("refused").value
for refuse in (1, 0):
    flag("refuse_device").value = refuse
    for i, x in enumerate(xs):
        np.testing.assert_array_equal(rt.get_output_f32(f"r{i}", x.size).reshape(x.shape), x)
    rt.run()
assert flag("refused").value > before
"""


def run(tmp_path, body):
    lib = tmp_path / "refuse.so"
    (tmp_path / "refuse.c").write_text(REFUSE)
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", str(lib), str(tmp_path / "refuse.c"), "-ldl"], check=True)
    code = SETUP.format(root=str(ROOT), lib=str(lib)) + body
    r = subprocess.run([sys.executable, "-c", code], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True,
                       timeout=60)
    assert r.returncode == 0, r.stdout


def test_download_without_page_locked_memory(tmp_path):
    run(tmp_path, HOST)


def test_sliced_output_without_device_memory(tmp_path):
    run(tmp_path, DEVICE)
