"""The work a user has this backend do, as timed cases.

Three kinds of use are covered, each through the public entry points of the
package: whole graphs on ``HipGraphRuntime`` (detector and classifier, fp16
and u8-quantized), single layers as op functions on device buffers (the
convolutions, the depthwise convolution, the classifier-head ops), and the
detector's tail with its post-processing.

A case is a dict of plain values whose ``"kind"`` names the path:

* ``detector``   the YOLOv8n-shaped graph on images that are on the device
                 (NCHW f32 planes, bound once), head outputs read back;
* ``classifier`` a strided conv / bottleneck backbone with a pooled
                 fully-connected head, logits read back;
* ``qconv``      QLinearConv u8 x s8 -> u8 with per-channel scales;
* ``conv_f16``   fp16 convolution + bias + activation;
* ``conv_f32``   fp32 convolution + bias + ReLU;
* ``dwconv``     depthwise 3x3 + bias + SiLU (fp16) or + ReLU (fp32);
* ``head``       global average pool, Gemm and (fp32) softmax;
* ``qhead``      quantized global average pool and QGemm;
* ``tail``       the detect tail (DFL, boxes, sigmoid), then decode + NMS.
"""
import functools
import math

import numpy as np
import torch
import torch.nn.functional as F

import __graft_entry__

__graft_entry__.import_pkg()

import dragonwing_edge_rs_amd as dw  # noqa: E402
from dragonwing_edge_rs_amd import graph as G  # noqa: E402
from dragonwing_edge_rs_amd import ops, yolo  # noqa: E402

DETECTOR_FLOPS_640 = 8.743e9  # 2 * MACs of the detector's 63 convolutions on one 640x640 image
DETECTOR_PARAMS = 3167776


def listed():
    return [
        # One camera frame through the quantized detector: launches and latency.
        {"name": "detector_int8_b1", "kind": "detector", "dtype": "int8", "batch": 1, "size": 640},
        # The throughput configuration of the benchmark.
        {"name": "detector_int8_b32", "kind": "detector", "dtype": "int8", "batch": 32, "size": 640},
        # The fp16 detector at an odd batch and a smaller frame (13x13 coarsest map).
        {"name": "detector_f16_b5", "kind": "detector", "dtype": "f16", "batch": 5, "size": 416},
        # A quantized classifier on a serving batch: every layer small, almost nothing to read back.
        {"name": "classifier_int8_b16", "kind": "classifier", "dtype": "int8", "batch": 16, "size": 224},
        # The benchmark's QLinearConv: a downsampling layer at full batch.
        {"name": "qconv_b32", "kind": "qconv", "n": 32, "h": 80, "w": 80, "cin": 128, "cout": 256, "k": 3, "s": 2},
        # A deep layer on one frame: little work, many channels.
        {"name": "qconv_b1_20", "kind": "qconv", "n": 1, "h": 20, "w": 20, "cin": 256, "cout": 256, "k": 3, "s": 1},
        # A mid-size fp16 bottleneck conv with SiLU.
        {"name": "conv_f16_b8", "kind": "conv_f16", "n": 8, "h": 80, "w": 80, "cin": 64, "cout": 64, "k": 3, "s": 1,
         "act": 2},
        # fp32 conv on a ragged map with odd channels, as calibration runs it.
        {"name": "conv_f32_odd", "kind": "conv_f32", "n": 2, "h": 53, "w": 75, "cin": 48, "cout": 40, "k": 3, "s": 1},
        # The benchmark's depthwise layer.
        {"name": "dwconv_f16_b32", "kind": "dwconv", "dtype": "f16", "n": 32, "h": 40, "w": 40, "c": 384, "s": 1},
        # A classifier head in fp32: pool, 1280 -> 1000, softmax.
        {"name": "head_f32_b32", "kind": "head", "dtype": "f32", "n": 32, "hw": 7, "cin": 1280, "cout": 1000},
        # The same head quantized.
        {"name": "qhead_b32", "kind": "qhead", "n": 32, "hw": 7, "cin": 1280, "cout": 1000},
        # Detect tail and NMS on a batch of frames.
        {"name": "tail_b8", "kind": "tail", "n": 8, "size": 640},
    ]


def _log_int(rng, lo, hi, step=1):
    """An integer multiple of `step` in [lo, hi], spread over its logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return int(min(max(round(v / step) * step, -(-lo // step) * step), hi // step * step))


def _conv_case(rng, kind, cin_step, cout_step, max_n, cin_lo, max_macs):
    while True:
        c = {"kind": kind, "n": _log_int(rng, 1, max_n), "h": _log_int(rng, 7, 160), "w": _log_int(rng, 7, 160),
             "cin": _log_int(rng, cin_lo, 256, cin_step), "cout": _log_int(rng, 16, 256, cout_step),
             "k": rng.choice((1, 3, 3)), "s": rng.choice((1, 1, 2))}
        ho, wo = _out_hw(c)
        if c["n"] * ho * wo * c["cout"] * c["cin"] * c["k"] ** 2 <= max_macs:
            return c


def draw(rng):
    kind = rng.choice(("detector", "classifier", "qconv", "qconv", "conv_f16", "conv_f32", "dwconv", "head", "qhead",
                       "tail"))
    if kind == "detector":
        size = 32 * rng.randint(8, 20)
        most = 32 * 640 * 640 // (size * size)
        return {"kind": kind, "dtype": rng.choice(("int8", "f16")), "batch": _log_int(rng, 1, min(32, most)),
                "size": size}
    if kind == "classifier":
        return {"kind": kind, "dtype": rng.choice(("int8", "f16")), "batch": _log_int(rng, 1, 48),
                "size": 32 * rng.randint(4, 10)}
    if kind == "qconv":
        return _conv_case(rng, kind, 16, 4, 32, 16, 15.2e9)
    if kind == "conv_f16":
        return dict(_conv_case(rng, kind, 8, 4, 32, 16, 8e9), act=rng.choice((0, 1, 2)))
    if kind == "conv_f32":
        return _conv_case(rng, kind, 1, 1, 4, 3, 1e9)
    if kind == "dwconv":
        while True:
            c = {"kind": kind, "dtype": rng.choice(("f16", "f16", "f32")), "n": _log_int(rng, 1, 32),
                 "h": _log_int(rng, 7, 112), "w": _log_int(rng, 7, 112), "c": _log_int(rng, 16, 960, 8),
                 "s": rng.choice((1, 1, 2))}
            if c["n"] * c["h"] * c["w"] * c["c"] <= 32 * 40 * 40 * 384:
                return c
    if kind == "head":
        return {"kind": kind, "dtype": rng.choice(("f32", "f16")), "n": _log_int(rng, 1, 64), "hw": rng.randint(4, 14),
                "cin": _log_int(rng, 64, 2048), "cout": _log_int(rng, 10, 2000)}
    if kind == "qhead":
        return {"kind": kind, "n": _log_int(rng, 1, 64), "hw": rng.randint(4, 14), "cin": _log_int(rng, 64, 2048, 16),
                "cout": _log_int(rng, 12, 2000, 4)}
    return {"kind": kind, "n": _log_int(rng, 1, 16), "size": 32 * rng.randint(8, 20)}


# ---------------------------------------------------------------------------
# What a program has in hand
# ---------------------------------------------------------------------------

_TYPES = {"f32": (torch.float32, "<f4"), "f16": (torch.float16, "<f2"), "u8": (torch.uint8, "|u1"),
          "i8": (torch.int8, "|i1"), "i32": (torch.int32, "<i4")}


@functools.lru_cache(maxsize=None)
def _backend():
    return dw.Backend(0)


class _Span:
    """A backend buffer as the CUDA array interface shows it to torch."""

    def __init__(self, buf, shape, typestr):
        self.buf = buf
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": typestr, "version": 2,
                                         "data": (buf.device_ptr(), False), "strides": None}


class _Dev:
    """A device buffer of the backend with a torch view of its bytes."""

    def __init__(self, shape, dtype):
        torch_type, typestr = _TYPES[dtype]
        n = int(np.prod(shape)) * torch.empty(0, dtype=torch_type).element_size()
        self.buf = _backend().alloc(n)
        self.t = torch.as_tensor(_Span(self.buf, shape, typestr), device="cuda")

    @classmethod
    def of(cls, t):
        dtype = {v[0]: k for k, v in _TYPES.items()}[t.dtype]
        d = cls(tuple(t.shape), dtype)
        d.t.copy_(t)
        return d


def _gen(seed):
    return torch.Generator("cuda").manual_seed(int(seed))


def _normal(g, shape, std=1.0, mean=0.0, dtype=torch.float32):
    return (torch.randn(shape, generator=g, device="cuda") * std + mean).to(dtype)


def _ints(g, shape, lo, hi, dtype):
    return torch.randint(lo, hi + 1, shape, generator=g, device="cuda", dtype=torch.int32).to(dtype)


def _scales(g, n):
    """Per-channel weight scales, log-uniform in [1e-3, 1e-2], on the host as the entry points take them."""
    u = torch.rand(n, generator=g, device="cuda")
    return torch.exp(math.log(1e-3) + u * math.log(10.0)).float().cpu().numpy()


def _out_hw(c):
    p = c["k"] // 2
    return (c["h"] + 2 * p - c["k"]) // c["s"] + 1, (c["w"] + 2 * p - c["k"]) // c["s"] + 1


def _conv_inputs(case, seed):
    """x NHWC, weights HWIO scaled to keep activations of order one, bias."""
    g = _gen(seed)
    dt = torch.float16 if case["kind"] == "conv_f16" else torch.float32
    x = _normal(g, (case["n"], case["h"], case["w"], case["cin"]), dtype=dt)
    w = _normal(g, (case["k"], case["k"], case["cin"], case["cout"]), 1.0 / math.sqrt(case["cin"] * case["k"] ** 2),
                dtype=dt)
    return x, w, _normal(g, (case["cout"],), 0.1, dtype=dt)


def _dw_inputs(case, seed):
    g = _gen(seed)
    dt = _TYPES[case["dtype"]][0]
    x = _normal(g, (case["n"], case["h"], case["w"], case["c"]), dtype=dt)
    return x, _normal(g, (3, 3, case["c"]), 0.3, dtype=dt), _normal(g, (case["c"],), 0.1, dtype=dt)


def _head_inputs(case, seed):
    """Activations after SiLU (mostly small, some large), weights, as a trained head meets them."""
    g = _gen(seed)
    dt = _TYPES[case["dtype"]][0]
    x = F.silu(_normal(g, (case["n"], case["hw"], case["hw"], case["cin"]), 1.5)).to(dt)
    return x, _normal(g, (case["cin"], case["cout"]), 2.0 / math.sqrt(case["cin"]), dtype=dt)


def _tail_inputs(case, seed):
    """Head outputs of the three levels: box bins of order one, class logits that leave a few hundred
    candidates a frame over the threshold."""
    g = _gen(seed)
    out = []
    for s in (8, 16, 32):
        h = case["size"] // s
        box = _normal(g, (case["n"], h, h, 64), 1.0)
        cls = _normal(g, (case["n"], h, h, 80), 1.5, -6.0)
        out.append(torch.cat([box, cls], 3).half())
    return out


def _images(n, size, seed):
    return torch.rand((n, 3, size, size), generator=_gen(seed), device="cuda")


@functools.lru_cache(maxsize=None)
def _detector_ranges(size):
    """Activation ranges of the detector's (fixed) weights: calibrated once, as a deployment does."""
    gc, info = yolo.calibration_graph(2, size)
    G.calibrate(_backend(), gc, info["input"], yolo.calibration_images(2, size))
    return {n: t["range"] for n, t in gc.to_dict()["tensors"].items() if "range" in t}


# The classifier: (op, channels out, stride) of each stage; "res" is a 3x3 bottleneck with its shortcut.
_STAGES = (("conv", 16, 2), ("conv", 32, 2), ("res", 32, 1), ("conv", 64, 2), ("res", 64, 1), ("res", 64, 1),
           ("conv", 128, 2), ("res", 128, 1), ("res", 128, 1), ("conv", 256, 2), ("res", 256, 1), ("point", 1280, 1))
_CLASSES = 1000


@functools.lru_cache(maxsize=None)
def _classifier_weights():
    r = np.random.default_rng(2024)
    out, c = [], 3
    for op, co, _ in _STAGES:
        k = 1 if op == "point" else 3
        for _ in range(2 if op == "res" else 1):
            w = r.normal(0, 1.6 / math.sqrt(c * k * k), (k, k, c, co)).astype(np.float32)
            out.append((w, r.normal(0, 0.1, co).astype(np.float32)))
            c = co
    return out, r.normal(0, 2.0 / math.sqrt(c), (c, _CLASSES)).astype(np.float32), \
        r.normal(0, 0.1, _CLASSES).astype(np.float32)


def _classifier_graph(batch, size):
    g = G.Graph(G.GRAPH_F32)
    convs, fw, fb = _classifier_weights()
    x, hw, i = "images", size, 0
    g.add_tensor(x, (batch, size, size, 3))

    def conv(x, hw, stride):
        nonlocal i
        w, b = convs[i]
        n, k, co = "c%d" % i, w.shape[0], w.shape[3]
        i += 1
        ho = (hw + 2 * (k // 2) - k) // stride + 1
        g.add_initializer(n + ".w", w)
        g.add_initializer(n + ".b", b)
        for t in (".y", ".s", ".o"):
            g.add_tensor(n + t, (batch, ho, ho, co))
        p = k // 2
        g.add_op(n, "Conv", [x, n + ".w", n + ".b"], [n + ".y"], kernel_shape=(k, k), strides=(stride, stride),
                 pads=(p, p, p, p))
        g.add_op(n + ".sig", "Sigmoid", [n + ".y"], [n + ".s"])
        g.add_op(n + ".mul", "Mul", [n + ".y", n + ".s"], [n + ".o"])
        return n + ".o", ho

    for op, co, stride in _STAGES:
        if op == "res":
            t, _ = conv(x, hw, 1)
            t, _ = conv(t, hw, 1)
            g.add_tensor(t + ".add", (batch, hw, hw, co))
            g.add_op(t + ".add", "Add", [x, t], [t + ".add"])
            x = t + ".add"
        else:
            x, hw = conv(x, hw, stride)
    c = fw.shape[0]
    g.add_tensor("pool", (batch, 1, 1, c))
    g.add_tensor("flat", (batch, c))
    g.add_initializer("fc.w", fw)
    g.add_initializer("fc.b", fb)
    g.add_tensor("logits", (batch, _CLASSES))
    g.add_op("gap", "GlobalAveragePool", [x], ["pool"])
    g.add_op("flatten", "Flatten", ["pool"], ["flat"])
    g.add_op("fc", "Gemm", ["flat", "fc.w", "fc.b"], ["logits"])
    g.set_io(["images"], ["logits"])
    return g


@functools.lru_cache(maxsize=None)
def _classifier_ranges(size):
    g = _classifier_graph(4, size)
    r = np.random.default_rng(7)
    G.calibrate(_backend(), g, "images", r.uniform(0, 1, (4, size, size, 3)).astype(np.float32))
    return {n: t["range"] for n, t in g.to_dict()["tensors"].items() if "range" in t}


def prepare(case, seed):
    kind, be = case["kind"], _backend()
    st = {"case": case}
    if kind in ("detector", "classifier"):
        b, size = case["batch"], case["size"]
        if kind == "detector" and case["dtype"] == "int8":
            g, info = yolo.int8_graph_from_ranges(_detector_ranges(size), b, size)
        elif kind == "detector":
            g, info = yolo.f16_graph(b, size)
        else:
            g = _classifier_graph(b, size)
            if case["dtype"] == "int8":
                for n, (lo, hi) in _classifier_ranges(size).items():
                    g.set_activation_range(n, lo, hi)
                g.quantize_qdq(["c0"])  # the three-channel stem stays fp16
            else:
                g.convert_to_f16()
            info = {"input": "images", "outputs": ["logits"], "out_shapes": [(b, _CLASSES)]}
        st["x"] = _Dev.of(_images(b, size, seed))
        torch.cuda.synchronize()
        st["rt"] = G.HipGraphRuntime(g, be)
        st["rt"].bind_input_nchw_f32(info["input"], st["x"].buf)
        st["out"] = list(zip(info["outputs"], info["out_shapes"]))
        st["type"] = np.uint8 if kind == "classifier" and case["dtype"] == "int8" else np.float16
        return st
    if kind == "qconv":
        g = _gen(seed)
        ho, wo = _out_hw(case)
        st["x"] = _Dev.of(_ints(g, (case["n"], case["h"], case["w"], case["cin"]), 0, 255, torch.uint8))
        st["w"] = _Dev.of(_ints(g, (case["k"], case["k"], case["cin"], case["cout"]), -127, 127, torch.int8))
        st["b"] = _Dev.of(_ints(g, (case["cout"],), -4096, 4096, torch.int32))
        st["ws"] = _scales(g, case["cout"])
        # an output scale that spreads the sums of random products over the 256 levels
        st["ys"] = float(0.02 * 3e-3 * 74 * 73 * math.sqrt(case["cin"] * case["k"] ** 2) / 40)
        st["y"] = _Dev((case["n"], ho, wo, case["cout"]), "u8")
    elif kind in ("conv_f16", "conv_f32"):
        ho, wo = _out_hw(case)
        st["x"], st["w"], st["b"] = (_Dev.of(t) for t in _conv_inputs(case, seed))
        st["y"] = _Dev((case["n"], ho, wo, case["cout"]), kind[5:])
    elif kind == "dwconv":
        s = case["s"]
        st["x"], st["w"], st["b"] = (_Dev.of(t) for t in _dw_inputs(case, seed))
        st["y"] = _Dev((case["n"], (case["h"] - 1) // s + 1, (case["w"] - 1) // s + 1, case["c"]), case["dtype"])
    elif kind == "head":
        st["x"], st["w"] = (_Dev.of(t) for t in _head_inputs(case, seed))
        st["pool"] = _Dev((case["n"], case["cin"]), case["dtype"])
        st["y"] = _Dev((case["n"], case["cout"]), case["dtype"])
        if case["dtype"] == "f32":
            st["p"] = _Dev((case["n"], case["cout"]), "f32")
    elif kind == "qhead":
        g = _gen(seed)
        st["x"] = _Dev.of(_ints(g, (case["n"], case["hw"], case["hw"], case["cin"]), 0, 255, torch.uint8))
        st["w"] = _Dev.of(_ints(g, (case["cin"], case["cout"]), -127, 127, torch.int8))
        st["b"] = _Dev.of(_ints(g, (case["cout"],), -4096, 4096, torch.int32))
        st["ws"] = _scales(g, case["cout"])
        st["ys"] = float(0.004 * 3e-3 * 74 * 74 * math.sqrt(case["cin"]) / 40)
        st["pool"] = _Dev((case["n"], case["cin"]), "u8")
        st["y"] = _Dev((case["n"], case["cout"]), "u8")
    else:
        st["x"] = [_Dev.of(t) for t in _tail_inputs(case, seed)]
        st["hw"] = [(case["size"] // s, case["size"] // s) for s in (8, 16, 32)]
        st["A"] = sum(h * w for h, w in st["hw"])
        st["y"] = _Dev((case["n"], 84, st["A"]), "f32")
    torch.cuda.synchronize()  # the backend's stream is its own
    return st


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------

_MAX_DETECTIONS = 1024


def _padded(dets, field, dtype):
    """One field of every frame's detections as one array, zeros past each frame's count."""
    out = np.zeros((len(dets), _MAX_DETECTIONS) + (4,) * (field == "bbox"), dtype)
    for i, d in enumerate(dets):
        out[i, :d.size] = d[field]
    return out


def run(st):
    c, be = st["case"], _backend()
    kind = c["kind"]
    if kind in ("detector", "classifier"):
        st["rt"].run()
        return {n: st["rt"].get_output_bytes(n).view(st["type"]).reshape(s) for n, s in st["out"]}
    if kind == "qconv":
        p = c["k"] // 2
        ops.qlinearconv_u8s8(be, st["x"].buf, st["w"].buf, st["b"].buf, st["y"].buf, c["n"], c["h"], c["w"], c["cin"],
                             c["cout"], c["k"], c["k"], c["s"], c["s"], p, p, 0.02, 128, st["ws"], st["ys"], 128)
        return st["y"].t
    if kind in ("conv_f16", "conv_f32"):
        p = c["k"] // 2
        args = (be, st["x"].buf, st["w"].buf, st["b"].buf, st["y"].buf, c["n"], c["h"], c["w"], c["cin"], c["cout"],
                c["k"], c["k"], c["s"], c["s"], p, p)
        if kind == "conv_f16":
            ops.conv2d_bias_act_f16_nhwc(*args, act=c["act"])
        else:
            ops.conv2d_bias_act_f32_nhwc(*args, act=ops.ACT_RELU)
        return st["y"].t
    if kind == "dwconv":
        f, act = ((ops.depthwise_conv2d_f16_nhwc, ops.ACT_SILU) if c["dtype"] == "f16" else
                  (ops.depthwise_conv2d_f32_nhwc, ops.ACT_RELU))
        f(be, st["x"].buf, st["w"].buf, st["b"].buf, st["y"].buf, c["n"], c["h"], c["w"], c["c"], 3, 3, c["s"], c["s"],
          1, 1, act=act)
        return st["y"].t
    if kind == "head":
        f16 = c["dtype"] == "f16"
        ops.global_avg_pool_nhwc(be, ops.DTYPE_F16 if f16 else ops.DTYPE_F32, st["x"].buf, st["pool"].buf, c["n"],
                                 c["hw"], c["hw"], c["cin"])
        (ops.gemm_fp16 if f16 else ops.gemm_f32)(be, st["pool"].buf, st["w"].buf, st["y"].buf, c["n"], c["cout"],
                                                 c["cin"])
        out = {"pool": st["pool"].t, "logits": st["y"].t}
        if not f16:
            ops.softmax_f32(be, st["y"].buf, st["p"].buf, c["n"], c["cout"])
            out["p"] = st["p"].t
        return out
    if kind == "qhead":
        ops.qlinear_global_avg_pool_u8(be, st["x"].buf, st["pool"].buf, c["n"], c["hw"], c["hw"], c["cin"], 0.02, 128,
                                       0.004, 128)
        ops.qgemm_u8s8(be, st["pool"].buf, st["w"].buf, st["b"].buf, st["y"].buf, c["n"], c["cout"], c["cin"], 0.004,
                       128, st["ws"], st["ys"], 128)
        return {"pool": st["pool"].t, "logits": st["y"].t}
    ops.yolo_detect_tail(be, [d.buf for d in st["x"]], st["hw"], (8.0, 16.0, 32.0), c["n"], st["y"].buf)
    dets = ops.yolo_postprocess(be, st["y"].buf, c["n"], 80, st["A"], 640, 640, 0.25, 0.45, cap=_MAX_DETECTIONS)
    return {"raw": st["y"].t, "counts": np.array([d.size for d in dets]), "boxes": _padded(dets, "bbox", np.float32),
            "classes": _padded(dets, "class_id", np.int64), "confidence": _padded(dets, "confidence", np.float32)}


# ---------------------------------------------------------------------------
# What one pass cannot do without, and how exactly
# ---------------------------------------------------------------------------

def work(case):
    kind = case["kind"]
    if kind == "detector":
        es, f = (1 if case["dtype"] == "int8" else 2), (case["size"] / 640) ** 2 * case["batch"]
        pixels = case["batch"] * case["size"] ** 2
        outs = sum((case["size"] // s) ** 2 for s in (8, 16, 32)) * 144 * 2 * case["batch"]
        return {"bytes": pixels * 12 + DETECTOR_PARAMS * es + outs, "flops": DETECTOR_FLOPS_640 * f}
    if kind == "classifier":
        es, hw, c, flops, params = (1 if case["dtype"] == "int8" else 2), case["size"], 3, 0, 0
        for op, co, s in _STAGES:
            k = 1 if op == "point" else 3
            hw = (hw + 2 * (k // 2) - k) // s + 1
            for _ in range(2 if op == "res" else 1):
                flops += 2 * hw * hw * co * c * k * k
                params += co * c * k * k
                c = co
        flops, params = flops + 2 * c * _CLASSES, params + c * _CLASSES
        return {"bytes": case["batch"] * (case["size"] ** 2 * 12 + _CLASSES * es) + params * es,
                "flops": flops * case["batch"]}
    if kind in ("qconv", "conv_f16", "conv_f32"):
        es = {"qconv": 1, "conv_f16": 2, "conv_f32": 4}[kind]
        ho, wo = _out_hw(case)
        k2c = case["k"] ** 2 * case["cin"]
        elems = case["n"] * (case["h"] * case["w"] * case["cin"] + ho * wo * case["cout"]) + k2c * case["cout"]
        return {"bytes": elems * es + case["cout"] * (8 if kind == "qconv" else es),
                "flops": 2 * case["n"] * ho * wo * case["cout"] * k2c}
    if kind == "dwconv":
        es = 2 if case["dtype"] == "f16" else 4
        out = ((case["h"] - 1) // case["s"] + 1) * ((case["w"] - 1) // case["s"] + 1)
        return {"bytes": es * case["c"] * (case["n"] * (case["h"] * case["w"] + out) + 10),
                "flops": 18 * case["n"] * out * case["c"]}
    if kind in ("head", "qhead"):
        es = 1 if kind == "qhead" else {"f32": 4, "f16": 2}[case["dtype"]]
        x, k, n = case["n"] * case["hw"] ** 2 * case["cin"], case["cin"], case["cout"]
        return {"bytes": es * (x + k * n + case["n"] * (k + n * (2 if es == 4 else 1))) + (8 * n if es == 1 else 0),
                "flops": 2 * case["n"] * k * n + x}
    a = sum((case["size"] // s) ** 2 for s in (8, 16, 32)) * case["n"]
    return {"bytes": a * (144 * 2 + 84 * 4), "flops": a * (64 * 6 + 80 * 4)}


def tolerance(case):
    """About four times what the paths were seen to differ by when their sums run in another order (the
    exact-order kernels beside the matrix-core ones) or, for whole graphs and fp32, from their 64-bit values."""
    kind, dtype = case["kind"], case.get("dtype")
    if kind in ("qconv", "qhead") or kind == "classifier" and dtype == "int8":
        return "exact"  # whole numbers, defined to the bit
    if kind == "detector":
        # int8: only the last fp16 1x1 convs may sum in another order (1.9e-5, 1.5e-3 seen); fp16: 63 layers
        # of f16 rounding (4.4e-4 from 64 bits)
        return {"rel": 8e-5, "max": 6e-3} if dtype == "int8" else {"rel": 2.5e-3, "max": 0.01}
    if kind == "classifier":
        return {"rel": 2.8e-3, "max": 0.01}  # 7.0e-4, 2.2e-3 from 64 bits
    if kind == "conv_f16":
        return {"rel": 7e-4, "max": 0.01}  # 1.7e-4, 2.5e-3 between the two orders
    if kind == "head" and dtype == "f16":
        return {"rel": 5.5e-4, "max": 0.01}
    if kind == "dwconv" and dtype == "f16":
        return {"rel": 2e-4, "max": 0.01}  # nine-term sums: few results round the other way
    if kind in ("tail", "dwconv"):
        return {"rel": 3e-7, "max": 5e-6}  # 6e-8, 1.1e-6 from 64 bits
    return {"rel": 4e-6, "max": 3e-5}  # f32 sums of up to 2304 products: 1.1e-6, 5.6e-6 from 64 bits


# ---------------------------------------------------------------------------
# The same values in 64 bits
# ---------------------------------------------------------------------------

def _conv64(x, w, b, stride):
    """NHWC convolution in f64, HWIO weights, 'same' padding of an odd kernel: one matrix product per tap."""
    kh, kw, ci, co = w.shape
    n, h, wd, _ = x.shape
    p = kh // 2
    ho, wo = (h + 2 * p - kh) // stride + 1, (wd + 2 * p - kw) // stride + 1
    xp = F.pad(x, (0, 0, p, p, p, p))
    y = torch.zeros((n * ho * wo, co), dtype=torch.float64, device=x.device)
    for i in range(kh):
        for j in range(kw):
            t = xp[:, i:i + (ho - 1) * stride + 1:stride, j:j + (wo - 1) * stride + 1:stride].reshape(-1, ci)
            y += t.contiguous() @ w[i, j].contiguous()
    return y.reshape(n, ho, wo, co) + (0 if b is None else b)


def _eval64(d, get, x):
    """A float NHWC graph (its description and initializers) evaluated in f64."""
    v = {d["inputs"][0]: x}

    def val(n):
        if n not in v:
            t = d["tensors"][n]
            a = get(n).view(np.float16 if t["dtype"] == G.DT["f16"] else np.float32)
            v[n] = torch.from_numpy(a.astype(np.float64)).reshape(t["dims"]).cuda()
        return v[n]

    for op in d["ops"]:
        kind, i, o = op["type"], op["inputs"], op["outputs"]
        if kind == "Conv":
            v[o[0]] = _conv64(val(i[0]), val(i[1]), val(i[2]) if len(i) > 2 and i[2] else None, op["strides"][0])
        elif kind == "SiLU":
            v[o[0]] = F.silu(val(i[0]))
        elif kind == "Sigmoid":
            v[o[0]] = torch.sigmoid(val(i[0]))
        elif kind == "Mul":
            v[o[0]] = val(i[0]) * val(i[1])
        elif kind == "Add":
            v[o[0]] = val(i[0]) + val(i[1])
        elif kind == "Split":
            at = 0
            for n in o:
                c = d["tensors"][n]["dims"][3]
                v[n] = val(i[0])[..., at:at + c]
                at += c
        elif kind == "Concat":
            v[o[0]] = torch.cat([val(n) for n in i], 3)
        elif kind == "MaxPool":
            k = op["kernel_shape"][0]
            v[o[0]] = F.max_pool2d(val(i[0]).permute(0, 3, 1, 2), k, 1, k // 2).permute(0, 2, 3, 1)
        elif kind == "Resize":
            v[o[0]] = val(i[0]).repeat_interleave(2, 1).repeat_interleave(2, 2)
        elif kind == "GlobalAveragePool":
            v[o[0]] = val(i[0]).mean((1, 2), keepdim=True)
        elif kind == "Flatten":
            v[o[0]] = val(i[0]).reshape(val(i[0]).shape[0], -1)
        elif kind == "Gemm":
            v[o[0]] = val(i[0]) @ val(i[1]) + val(i[2])
        else:
            raise ValueError(kind)
    return {n: v[n].cpu() for n in d["outputs"]}


def exact(case, seed):
    kind = case["kind"]
    if kind in ("qconv", "qhead") or case.get("dtype") == "int8":
        return None  # whole numbers throughout (the detector's head reads such numbers)
    if kind in ("detector", "classifier"):
        b, size = case["batch"], case["size"]
        if kind == "detector":
            g, info = yolo.f16_graph(b, size)
        else:
            g = _classifier_graph(b, size)
            g.convert_to_f16()
        x = _images(b, size, seed).half().double().permute(0, 2, 3, 1).contiguous()
        return _eval64(g.to_dict(), g.initializer, x)
    if kind in ("conv_f16", "conv_f32"):
        x, w, b = (t.double() for t in _conv_inputs(case, seed))
        y = _conv64(x, w, b, case["s"])
        act = case.get("act", 1)
        return (F.silu(y) if act == 2 else torch.relu(y) if act == 1 else y).cpu()
    if kind == "dwconv":
        x, w, b = (t.double() for t in _dw_inputs(case, seed))
        s, (n, h, wd, c) = case["s"], x.shape
        ho, wo = (h - 1) // s + 1, (wd - 1) // s + 1
        xp, y = F.pad(x, (0, 0, 1, 1, 1, 1)), torch.zeros((n, ho, wo, c), dtype=torch.float64, device="cuda")
        for i in range(3):
            for j in range(3):
                y += xp[:, i:i + (ho - 1) * s + 1:s, j:j + (wo - 1) * s + 1:s] * w[i, j]
        y += b
        return (F.silu(y) if case["dtype"] == "f16" else torch.relu(y)).cpu()
    if kind == "head":
        x, w = (t.double() for t in _head_inputs(case, seed))
        pool = x.mean((1, 2))
        out = {"pool": pool.cpu(), "logits": (pool @ w).cpu()}
        if case["dtype"] == "f32":
            out["p"] = torch.softmax(pool @ w, 1).cpu()
        return out
    boxes, classes = [], []
    for t, s in zip(_tail_inputs(case, seed), (8.0, 16.0, 32.0)):
        t = t.double()
        n, h, w, _ = t.shape
        side = (torch.softmax(t[..., :64].reshape(n, h, w, 4, 16), 4) *
                torch.arange(16, dtype=torch.float64, device="cuda")).sum(4)
        cy, cx = torch.meshgrid(torch.arange(h, device="cuda") + 0.5, torch.arange(w, device="cuda") + 0.5,
                                indexing="ij")
        x1, y1, x2, y2 = cx - side[..., 0], cy - side[..., 1], cx + side[..., 2], cy + side[..., 3]
        boxes.append((torch.stack([(x1 + x2) / 2, (y1 + y2) / 2, x2 - x1, y2 - y1], 1) * s).reshape(n, 4, -1))
        classes.append(torch.sigmoid(t[..., 64:]).permute(0, 3, 1, 2).reshape(n, 80, -1))
    raw = torch.cat([torch.cat(boxes, 2), torch.cat(classes, 2)], 1).cpu()
    # which detections remain is a matter of order and thresholds
    return {"raw": raw, "counts": None, "boxes": None, "classes": None, "confidence": None}
