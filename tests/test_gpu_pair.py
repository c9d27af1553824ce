"""Two pointwise layers that do not read each other's results in one launch (exhip_conv2d_i8_pair, exhip_conv2d_f16_pair, exhip_conv2d_f32_pair): the bytes of the layers
run by themselves, whichever forms the two have, and also where they do run by themselves."""
import ctypes

import numpy as np
import pytest

from excalibur_amd import hip, modelfile, topologies
from excalibur_amd import pipeline as xp

pytestmark = pytest.mark.gpu


class CallI8(ctypes.Structure):
    _fields_ = [(name, ctypes.c_void_p) for name in ("d", "x", "w", "scale", "bias", "y_i8", "y_f32")]


class CallF16(ctypes.Structure):
    _fields_ = [(name, ctypes.c_void_p) for name in ("d", "x", "w", "bias", "y")]


@pytest.fixture(scope="module")
def ctx():
    c = hip.Ctx(0)
    yield c
    c.close()


LAYERS = {
    # n, h, w, channels, output channels, kernel: forms of one wave to 64 pixels or to 64 channels, with and without pairs of k-steps, and four waves to a tile
    "narrow": (2, 9, 13, 32, 32, 1),
    "narrow pairs": (1, 24, 11, 128, 32, 1),
    "wide": (1, 7, 5, 64, 96, 1),
    "wide pairs": (3, 30, 31, 256, 64, 1),
    "split": (1, 10, 10, 512, 128, 1),
    "split ragged": (1, 6, 7, 320, 160, 1),
    "filter": (1, 8, 8, 64, 64, 3),
}


def layer(ctx, spec, int8, seed, plain):
    n, h, w, c, k, kernel = spec
    r = np.random.default_rng(seed)
    arrays = [r.normal(0, 1, k).astype(np.float32) for _ in range(3)]
    post = {} if plain else dict(post_op="leakyrelu" if int8 else "hardswish", post_alpha=.1 if int8 else 1 / 6, post_beta=.5)
    bias, a, b = (ctx.array(v) for v in arrays)
    if int8:
        post.update(fs_out=15.0, exact_k=int(kernel == 1 and not plain))
        if kernel == 1 and not plain:
            post.update(post_bn=(a, b))
    d = ctx.conv_desc(n, c, h, w, k, kernel, 1, kernel // 2, c_stride=c, k_stride=k, **post)
    if int8:
        x, wt = r.integers(-127, 128, (n, h, w, c), dtype=np.int8), r.integers(-127, 128, (k, c, kernel, kernel), dtype=np.int8)
        scale = ctx.array(np.full(k, 1 / (127 * 73 * np.sqrt(c * kernel * kernel)), np.float32))
    else:
        x, wt = (v.astype(np.float16).view(np.uint16) for v in (r.normal(0, 1, (n, h, w, c)), r.normal(0, c ** -.5, (k, c, kernel, kernel))))
    xd, wp = ctx.array(x), ctx.pack_conv_weights(d, hip.I8 if int8 else hip.F16, wt)

    def call():
        y = ctx.array(np.full(n * h * w * k + 64, 0x55, np.int8 if int8 else np.uint16))
        if int8:
            return y, CallI8(ctypes.addressof(d), xd.ptr, wp.ptr, scale.ptr, bias.ptr, y.ptr, None)
        return y, CallF16(ctypes.addressof(d), xd.ptr, wp.ptr, bias.ptr, y.ptr)

    def alone():
        y, _ = call()
        if int8:
            ctx.conv2d_i8(d, xd, wp, scale, bias, None, y)
        else:
            ctx.conv2d_f16(d, xd, wp, bias, None, y)
        return y.download()
    call.keep = (d, xd, wp, bias, a, b) + ((scale,) if int8 else ())
    return call, alone


@pytest.mark.parametrize("int8", [True, False], ids=["int8", "fp16"])
@pytest.mark.parametrize("second", LAYERS)
@pytest.mark.parametrize("first", LAYERS)
def test_two_layers(ctx, first, second, int8):
    # int8: both with the BatchNorm and LeakyReLU of a joined Concat behind them, fp16: nothing; then a layer that has something else behind it
    for plain in ((False, False), (False, True)) if int8 else ((True, True), (True, False)):
        made = [layer(ctx, LAYERS[name], int8, seed, p) for name, seed, p in zip((first, second), (1, 2), plain)]
        want = [alone() for _, alone in made]
        (ya, a), (yb, b) = made[0][0](), made[1][0]()
        run = hip.lib().exhip_conv2d_i8_pair if int8 else hip.lib().exhip_conv2d_f16_pair
        hip._check(run(ctx.h, ctypes.byref(a), ctypes.byref(b)))
        ctx.sync()
        for got, expected in zip((ya, yb), want):
            assert np.array_equal(got.download(), expected) and np.unique(expected).size > 10


def test_an_error_of_either_layer_is_reported(ctx):
    call, alone = layer(ctx, LAYERS["wide"], False, 1, True)
    want = alone()
    for bad_first in (True, False):
        (y, good), (_, bad) = call(), call()
        bad.y = None
        pair = (bad, good) if bad_first else (good, bad)
        assert hip.lib().exhip_conv2d_f16_pair(ctx.h, ctypes.byref(pair[0]), ctypes.byref(pair[1])) != 0
        ctx.sync()
        if not bad_first:
            assert np.array_equal(y.download(), want)


class Place(ctypes.Structure):
    _fields_ = [(name, ctypes.c_int) for name in ("layout", "group", "residual_stride", "residual_shift", "bn_relu")]


class CallF32(ctypes.Structure):
    _fields_ = [(name, ctypes.c_void_p) for name in ("d", "place", "x", "w", "bias", "residual", "y", "y_nchw")]


def layer_f32(ctx, spec, seed, shortcut):
    n, h, w, c, k, kernel = spec
    r = np.random.default_rng(seed)
    d = ctx.conv_desc(n, c, h, w, k, kernel, 1, kernel // 2, c_stride=c, k_stride=k, act=seed % 2)
    place = Place(0, 0, k, 0, 0)
    x, bias = (ctx.array(r.normal(0, 1, size).astype(np.float32)) for size in ((n, h, w, c), k))
    res = ctx.array(r.normal(0, 1, (n, h, w, k)).astype(np.float32)) if shortcut else None
    wp = ctx.pack_conv_weights(d, hip.F32, r.normal(0, c ** -.5, (k, c, kernel, kernel)).astype(np.float32))

    def call():
        y = ctx.array(np.full(n * h * w * k + 64, -77, np.float32))
        return y, CallF32(ctypes.addressof(d), ctypes.addressof(place), x.ptr, wp.ptr, bias.ptr, res.ptr if shortcut else None, y.ptr, None)
    call.keep = d, place, x, bias, res, wp
    return call


@pytest.mark.parametrize("second", LAYERS)
@pytest.mark.parametrize("first", LAYERS)
def test_two_float32_layers(ctx, first, second):
    made = [layer_f32(ctx, LAYERS[name], seed, shortcut) for name, seed, shortcut in ((first, 1, False), (second, 2, True))]
    want = []
    for call in made:
        y, c = call()
        hip._check(hip.lib().exhip_conv2d_f32_placed(ctx.h, *(ctypes.c_void_p(getattr(c, name)) for name, _ in c._fields_)))
        want.append(y.download())
    (ya, a), (yb, b) = made[0](), made[1]()
    hip._check(hip.lib().exhip_conv2d_f32_pair(ctx.h, ctypes.byref(a), ctypes.byref(b)))
    ctx.sync()
    for got, expected in zip((ya, yb), want):
        assert np.array_equal(got.download(), expected) and np.ptp(expected[:-64]) > 1


@pytest.mark.parametrize("hw,n", [(128, 3), (96, 1)])
def test_a_float32_detection_network(tmp_path, hw, n):
    text, outs = topologies.yolov5s_simp(hw, int8=False)
    path = str(tmp_path / "net.racy")
    modelfile.write_model(path, modelfile.SeededModel(modelfile.parse_topology(text), 5, default_fs=16.0, gain=2.0).blobs)
    x = np.random.default_rng(4).integers(0, 256, (n, 3, hw, hw)).astype(np.float32)
    got = []
    for fusion in (True, False):
        pipe = xp.Pipeline(text, path, 0, "f32", fusion=fusion)
        for _ in range(2):
            pipe.set_input(x)
            pipe.run()
        assert pipe.stored("465") != fusion  # (a blob that the plan makes in no layout of its own)
        got.append([pipe.get(name) for name in outs])
    for a, b in zip(*got):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32)) and np.ptp(a) > 0


def test_float32_layers_that_read_what_the_layer_in_front_writes(tmp_path):
    """Pointwise layers on neighbouring lines: one reads the other's result, the Concat the other is part of, adds the other's result as its shortcut, or adds it through an
    upsampling: none of them shares a launch with what it reads. The same with nothing read in between."""
    r = np.random.default_rng(17)
    lines, blobs = [], []

    def conv(bottom, top, c, k, kernel=1, stride=1, act=0):
        w = r.normal(0, (c * kernel * kernel) ** -.5, (k, c, kernel, kernel)).astype(np.float32)
        lines.append(modelfile.conv_line("Convolution", top + "_l", bottom, top, k, kernel, stride, kernel // 2, True, w.size, act=act))
        blobs.append(modelfile.conv_blob_f32(w, r.normal(0, .5, k).astype(np.float32)))

    def add(*line):
        lines.append(" ".join(line))

    conv("data", "c0", 3, 32, 3)
    add("Split s0 1 5 c0 c00 c01 c02 c03 c04")
    conv("c00", "a", 32, 64)                        # a and b share a launch
    conv("c01", "b", 32, 32)
    add("Split s1 1 2 b b0 b1")
    add("Concat ab 2 1 a b0 ab 0=-1")
    conv("ab", "d", 96, 32)                         # reads the Concat that b is part of
    add("Split s2 1 2 d d0 d1")
    conv("d0", "e", 32, 32)                         # reads d
    add("Eltwise f_l 2 1 e b1 f 0=1")
    conv("c02", "g", 32, 32, 3, 2)
    add("Interp up 1 1 g gu 0=1 1=2.000000e+00 2=2.000000e+00")
    conv("d1", "h", 32, 32)                         # adds g through the upsampling
    add("BinaryOp i_l 2 1 gu h i 0=0")
    conv("c03", "j", 32, 32)
    conv("c04", "k", 32, 32)
    add("Eltwise l_l 2 1 k j l 0=1")                # adds the layer in front's result
    add("Concat out_l 3 1 f i l out 0=-1")
    conv("out", "m", 96, 48)
    path = str(tmp_path / "net.racy")
    modelfile.write_model(path, blobs)
    pipes = [xp.Pipeline(modelfile.topology(lines, "reads"), path, 0, "f32", fusion=on) for on in (True, False)]
    for seed, n, hw in ((1, 1, 16), (2, 3, 24), (3, 3, 24)):
        x = np.random.default_rng(seed).normal(0, 1, (n, 3, hw, hw)).astype(np.float32)
        got = []
        for pipe in pipes:
            pipe.set_input(x)
            pipe.run()
            got.append(pipe.get("m"))
        assert [pipe.stored("c0") for pipe in pipes] == [False, True]
        assert np.array_equal(got[0].view(np.uint32), got[1].view(np.uint32)) and np.ptp(got[0]) > .5


@pytest.mark.parametrize("int8", [True, False], ids=["int8", "fp16"])
def test_a_detection_network(tmp_path, int8):
    text, outs = topologies.yolov5s_simp(128, int8=int8)
    path = str(tmp_path / "net.racy")
    modelfile.write_model(path, modelfile.SeededModel(modelfile.parse_topology(text), 5, default_fs=16.0, gain=2.0).blobs)
    x = np.random.default_rng(3).integers(0, 256, (3, 3, 128, 128))
    x = x.astype(np.float32) if int8 else x.astype(np.float16).view(np.uint16)
    got = []
    for fusion in (True, False):
        pipe = xp.Pipeline(text, path, 0, "f32" if int8 else "f16", fusion=fusion)
        for _ in range(2):
            pipe.set_input(x)
            pipe.run()
        got.append([pipe.get(name) for name in outs])
    for a, b in zip(*got):
        assert a.tobytes() == b.tobytes() if int8 else np.array_equal(a.view(np.float16), b.view(np.float16))


def test_a_layer_that_reads_the_concat_in_front_is_not_paired_with_its_last_writer(tmp_path):
    conv = lambda name, src, dst, c, k, kernel=1: f"Convolution {name} 1 1 {src} {dst} 0={k} 1={kernel} 11={kernel} 2=1 12=1 3=1 13=1 4={kernel // 2} 14={kernel // 2} 15={kernel // 2} 16={kernel // 2} 5=1 6={c * k * kernel * kernel} 8=2"
    lines = ["Input in 0 1 in 0=24 1=24 2=3 3=0,0,0 4=0.0039215", conv("first", "in", "f", 3, 32, 3), "Split s 1 3 f f0 f1 f2", conv("a", "f0", "a", 32, 32), conv("x", "f1", "x0", 32, 64),
             "HardSwish hx 1 1 x0 x 0=1.666667e-01 1=5.000000e-01", conv("b", "x", "b", 64, 32), "Concat p 2 1 a b p 0=-1", conv("c", "p", "c", 64, 32), conv("d", "f2", "d", 32, 32),
             "Concat q 2 1 c d q 0=-1", conv("e", "q", "e", 64, 32)]
    blobs = sum(int(line.split()[3]) for line in lines)
    text = "glsv1\n%d %d\n%s\n" % (len(lines), blobs, "\n".join(lines))
    path = str(tmp_path / "net.racy")
    modelfile.write_model(path, modelfile.SeededModel(modelfile.parse_topology(text), 5, default_fs=16.0, gain=2.0).blobs)
    x = np.random.default_rng(3).integers(0, 256, (4, 3, 24, 24)).astype(np.float32)
    got = []
    for fusion in (True, False):
        pipe = xp.Pipeline(text, path, 0, "f32", fusion=fusion)
        for _ in range(2):
            pipe.set_input(x)
            pipe.run()
        got.append(pipe.get("e"))
        assert pipe.fused == fusion
    assert np.array_equal(*got) and np.ptp(got[0]) > 0
