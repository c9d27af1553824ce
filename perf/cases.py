"""What a program that runs networks on this framework waits for, as cases that can be timed.

Three ways in, as the package offers them:

* ``network``  -- ``excalibur_amd.pipeline.Pipeline``: a host image batch goes in (``set_input``), the network runs, the
  results come back to the host (``get``). This is how applications use the library: the pipeline's interface takes and
  returns host tensors.
* ``backbone`` -- ``excalibur_amd.resnet18.FusedRunner``: the int8 ResNet-18-shaped stack of the headline benchmark, input
  and output resident on the GPU.
* ``layer``    -- ``excalibur_amd.hip.Ctx``: one convolution through the C ABI on resident NHWC operands.

Only forward passes exist (the library runs inference); float32, half and int8 are its three precisions.
"""
import functools
import os
import tempfile

import numpy as np
import torch

from excalibur_amd import hip, mobilenet, modelfile, resnet18, topologies
from excalibur_amd import pipeline as xp

FACE = dict(width=64, blocks=((2, 64, 2), (1, 64, 2), (1, 64, 2), (2, 128, 4), (1, 128, 2), (1, 128, 2), (2, 128, 4), (1, 128, 2)), embed=128)


def listed():
    return [
        # one cropped face to its embedding: the smallest call, launches and host work are all of it
        dict(name="face-f16-1", kind="network", net="face", dtype="f16", n=1, hw=112),
        # the MobileNet-style stack at its benchmark batch: depthwise + pointwise blocks in half precision
        dict(name="mobilenet-f16-64", kind="network", net="mobilenet", dtype="f16", n=64, hw=224),
        # one camera frame through the int8 detector: latency of a live stream
        dict(name="detector-int8-1", kind="network", net="detector", dtype="int8", n=1, hw=640),
        # the detection configuration at its benchmark batch, both precisions it is quoted in
        dict(name="detector-int8-16", kind="network", net="detector", dtype="int8", n=16, hw=640),
        dict(name="detector-f16-16", kind="network", net="detector", dtype="f16", n=16, hw=640),
        # a few frames in float32 at another resolution: feature maps of 52, 26 and 13
        dict(name="detector-f32-3", kind="network", net="detector", dtype="f32", n=3, hw=416),
        # one page through the shipped text detector, a float32 network
        dict(name="text-f32-1", kind="network", net="text", dtype="f32", n=1, hw=640),
        # a batch of faces through the int8 network the library ships
        dict(name="unicorn-int8-64", kind="network", net="unicorn", dtype="int8", n=64, hw=128),
        # the headline benchmark's batch, and a few images of a ragged size
        dict(name="backbone-int8-32", kind="backbone", n=32, h=640, w=640),
        dict(name="backbone-int8-3", kind="backbone", n=3, h=333, w=500),
        # the single-layer configurations: one float32 image, and a requantized int8 layer on eight
        dict(name="conv-f32-1x56", kind="layer", dtype="f32", n=1, c=64, h=56, w=56, k=64, kernel=3, stride=1),
        dict(name="conv-int8-8x80", kind="layer", dtype="int8", n=8, c=128, h=80, w=80, k=256, kernel=3, stride=1),
    ]


def _log(rng, lo, hi):
    """A whole number between lo and hi, spread evenly over the logarithm."""
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    kind = rng.choice(("network", "network", "network", "backbone", "layer"))
    if kind == "network":
        net = rng.choice(("face", "mobilenet", "detector", "detector", "text", "unicorn"))
        if net == "detector":  # stride-32 topology; float32 batches are kept small
            dtype = rng.choice(("int8", "f16", "f32"))
            hw = 32 * rng.randint(5, 20)
            most = (4 if dtype == "f32" else 16) * 640 * 640 // (hw * hw)
            return dict(kind=kind, net=net, dtype=dtype, n=_log(rng, 1, min(32, most)), hw=hw)
        if net == "text":
            hw = 32 * rng.randint(5, 25)
            return dict(kind=kind, net=net, dtype="f32", n=_log(rng, 1, max(1, min(8, 2 * 640 * 640 // (hw * hw)))), hw=hw)
        if net == "unicorn":  # its last layer fixes the input size
            return dict(kind=kind, net=net, dtype="int8", n=_log(rng, 1, 96), hw=128)
        lo, hi = (80, 160) if net == "face" else (96, 256)
        dtype = rng.choice(("f16", "f16", "f32"))
        return dict(kind=kind, net=net, dtype=dtype, n=_log(rng, 1, 64 if dtype == "f16" else 32), hw=rng.randint(lo, hi))
    if kind == "backbone":
        h, w = _log(rng, 96, 640), _log(rng, 96, 640)
        return dict(kind=kind, n=_log(rng, 1, min(64, 32 * 640 * 640 // (h * w))), h=h, w=w)
    dtype = rng.choice(("int8", "f16", "f32"))
    kernel, stride = rng.choice((1, 3, 3)), rng.choice((1, 1, 2))
    c, k = 32 * _log(rng, 1, 16), rng.choice((32 * _log(rng, 1, 16), _log(rng, 32, 512)))
    h = _log(rng, 10, 160)
    w = h + rng.choice((0, 0, rng.randint(-3, 9)))
    most = int(min(4e10 / (2.0 * h * w * c * k * kernel * kernel), 4e7 / (h * w * max(c, k))))
    return dict(kind=kind, dtype=dtype, n=_log(rng, 1, max(1, min(32, most))), c=c, h=h, w=w, k=k, kernel=kernel, stride=stride if kernel == 3 else 1)


# ---- the models: weights of a deployed network do not change with its input, so each is made once ----
@functools.lru_cache(maxsize=None)
def _model(net, dtype, hw):
    """(topology text, names of the results, weight blobs) of a network."""
    if net in ("face", "mobilenet"):
        m = mobilenet.MobileFaceNetF32(hw=hw, **(FACE if net == "face" else {k: v for k, v in mobilenet.CFG3.items() if k != "hw"}))
        return m.topology(), [m.output], m.blobs
    if net == "detector":
        text, outs = topologies.yolov5s_simp(hw, int8=dtype == "int8")
    elif net == "text":
        text, outs = topologies.det_db_resnet18(hw)
    else:
        text, outs = topologies.unicorn_light_int8(hw)
    # gain 1 keeps the float residual sums of the text network near 1; feature-map scales as a calibration would leave them
    model = modelfile.SeededModel(modelfile.parse_topology(text), 5, default_fs=4.0 if net == "unicorn" else 16.0, gain=1.0 if net == "text" else 2.0)
    return text, outs, model.blobs


@functools.lru_cache(maxsize=None)
def _backbone():
    return resnet18.ResNet18Int8(seed=1234, calib_hw=64)


class _Ctx(hip.Ctx):
    """A context whose arrays are released with it."""

    def __init__(self):
        super().__init__(0)
        self.pointers = []

    def empty(self, shape, dtype):
        a = super().empty(shape, dtype)
        self.pointers.append(a.ptr)
        return a

    def array(self, a, dtype=None):
        a = super().array(a, dtype)
        self.pointers.append(a.ptr)
        return a

    def __del__(self):
        for p in self.pointers:
            hip.lib().exhip_free(self.h, p)
        self.close()


class _Shared:
    """A device array as torch sees it; the tensor made of it keeps the context and its arrays alive."""

    def __init__(self, ctx, a):
        self.owner = ctx
        kind = {1: "|i1", 2: "<f2", 4: "<f4"}[a.dtype.itemsize]
        self.__cuda_array_interface__ = {"shape": a.shape, "typestr": kind, "data": (a.ptr.value, False), "version": 2, "strides": None}


def _tensor(ctx, a):
    return torch.as_tensor(_Shared(ctx, a), device="cuda")


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    if case["kind"] == "network":
        text, outs, blobs = _model(case["net"], case["dtype"], case["hw"])
        half = case["dtype"] == "f16"
        with tempfile.NamedTemporaryFile(suffix=".racy", delete=False) as f:
            path = f.name
        modelfile.write_model(path, blobs)
        pipe = xp.Pipeline(text, path, 0, "f16" if half else "f32")
        os.unlink(path)
        x = rng.integers(0, 256, (case["n"], 3, case["hw"], case["hw"]), dtype=np.uint8)  # camera pixels
        x = x.astype(np.float16).view(np.uint16) if half else x.astype(np.float32)
        return dict(pipe=pipe, x=x, outs=outs, half=half)
    ctx = _Ctx()
    if case["kind"] == "backbone":
        n, h, w = case["n"], case["h"], case["w"]
        run_ = resnet18.FusedRunner(ctx, _backbone(), n, h, w)
        run_.set_input(rng.random((n, 3, h, w), dtype=np.float32) * 2 - 1)
        return dict(forward=run_.forward, out=_tensor(ctx, run_.out))
    n, c, h, w, k, kernel = (case[x] for x in ("n", "c", "h", "w", "k", "kernel"))
    dtype, ks = case["dtype"], hip.pad_to(case["k"], 32)
    d = ctx.conv_desc(n, c, h, w, k, kernel, case["stride"], kernel // 2, 1, c, ks, 0, 16.0 if dtype == "int8" else 0.0)
    oh, ow = ctx.conv_out_hw(d)
    weights, bias = rng.normal(0, 0.05, (k, c, kernel, kernel)).astype(np.float32), rng.normal(0, 0.01, k).astype(np.float32)
    b = ctx.array(bias)
    if dtype == "int8":
        x = ctx.array(rng.integers(-127, 128, (n, h, w, c), dtype=np.int8))
        wp = ctx.pack_conv_weights(d, hip.I8, rng.integers(-127, 128, weights.shape, dtype=np.int8))
        scale = ctx.array((rng.uniform(0.5, 1.5, k) / (16.0 * 73 * np.sqrt(c * kernel * kernel))).astype(np.float32))
        y = ctx.empty((n, oh, ow, ks), np.int8).zero()
        return dict(forward=lambda: ctx.conv2d_i8(d, x, wp, scale, b, None, y), out=_tensor(ctx, y))
    values = rng.random((n, h, w, c), dtype=np.float32) * 2 - 1
    if dtype == "f16":
        x = ctx.array(values.astype(np.float16).view(np.uint16))
        wp = ctx.pack_conv_weights(d, hip.F16, weights.astype(np.float16).view(np.uint16))
        y = ctx.empty((n, oh, ow, ks), np.uint16).zero()
        return dict(forward=lambda: ctx.conv2d_f16(d, x, wp, b, None, y), out=_tensor(ctx, y))
    x = ctx.array(values)
    wp = ctx.pack_conv_weights(d, hip.F32, weights)
    y = ctx.empty((n, k, oh, ow), np.float32)
    return dict(forward=lambda: ctx.conv2d_f32(d, x, wp, b, None, None, y), out=_tensor(ctx, y))


def run(state):
    if "pipe" not in state:
        state["forward"]()
        return state["out"]
    pipe = state["pipe"]
    pipe.set_input(state["x"])
    pipe.run()
    out = [pipe.get(name) for name in state["outs"]]
    return [y.view(np.float16) for y in out] if state["half"] else out


def work(case):
    n = case["n"]
    if case["kind"] == "network":
        net, hw = case["net"], case["hw"]
        text, _, blobs = _model(net, case["dtype"], hw)
        values = {"face": 128, "mobilenet": 128, "text": hw * hw, "unicorn": 256, "detector": 255 * 21 * (hw // 32) ** 2}[net]
        size = 2 if case["dtype"] == "f16" else 4
        return dict(bytes=n * (3 * hw * hw + values) * size + sum(map(len, blobs)) * size // 4, flops=1e9 * n * topologies.algorithmic_gop(text, (3, hw, hw)))
    if case["kind"] == "backbone":
        h, w = case["h"], case["w"]
        oh, ow = -(-h // 32), -(-w // 32)
        return dict(bytes=4 * n * (3 * h * w + 512 * oh * ow) + sum(c.w_i8.size + 8 * c.k for c in _backbone().convs), flops=2e9 * n * _backbone().gmac_per_image(h, w))
    c, k, kernel = case["c"], case["k"], case["kernel"]
    oh, ow = -(-case["h"] // case["stride"]), -(-case["w"] // case["stride"])
    size = {"int8": 1, "f16": 2, "f32": 4}[case["dtype"]]
    return dict(bytes=size * (n * case["h"] * case["w"] * c + n * oh * ow * k + k * c * kernel * kernel), flops=2.0 * n * oh * ow * k * c * kernel * kernel)


def tolerance(case):
    """int8 convolutions accumulate whole numbers and their float steps are fixed operation by operation, so their results are
    the same bytes whatever the implementation; the int8 face network ends in a float layer. Half storage rounds every layer's
    result to 11 bits; float32 sums differ in their order, in networks through up to seventy layers."""
    if case["kind"] == "backbone" or case.get("net") == "detector" and case["dtype"] == "int8" or case["kind"] == "layer" and case["dtype"] == "int8":
        return "exact"
    if case["dtype"] == "f16":
        return {"rel": 2e-3 if case["kind"] == "network" else 5e-4}
    return {"rel": 2e-5 if case["kind"] == "network" and case["dtype"] == "f32" else 1e-5}
