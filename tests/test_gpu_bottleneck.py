"""Pointwise + depthwise 3x3 + pointwise blocks of fp16 networks as one kernel (bottleneck.hip): the results are those of the layers run one
after the other, bit for bit, through the C ABI with every option and through the pipeline."""
import ctypes
import os
import tempfile

import numpy as np
import pytest

from excalibur_amd import hip, mobilenet, modelfile
from excalibur_amd import pipeline as xp
from tests.test_gpu_depthwise_pair import Depthwise

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = hip.Ctx(0)
    yield c
    c.close()


@pytest.fixture
def blocks():
    yield lambda value: hip.set_option("bottleneck", value)
    hip.set_option("bottleneck", 1)


SHAPES = [
    # n, h, w, input, wide and output channels, stride, padding (top, bottom, left, right)
    (1, 7, 7, 32, 64, 48, 1, (1, 1, 1, 1)),
    (2, 9, 13, 64, 96, 32, 2, (1, 1, 1, 1)),       # tiles that end outside the map
    (1, 14, 14, 128, 512, 128, 2, (1, 1, 1, 1)),   # sums in runs
    (3, 12, 10, 256, 256, 272, 1, (0, 1, 1, 0)),   # uneven padding, half a block at the end
    (1, 5, 4, 16, 32, 16, 1, (2, 0, 0, 2)),        # the map grows above and on the right
    (1, 7, 7, 512, 1024, 512, 1, (1, 1, 1, 1)),
    (1, 17, 14, 64, 256, 128, 1, (1, 1, 1, 1)),    # sums in runs in the last layer alone
    (5, 6, 33, 48, 256, 80, 2, (0, 0, 1, 1)),
]
LAYERS = [
    # behind the first layer, the depthwise layer's activation, biases, shortcut
    ("prelu", "prelu", True, True),
    ("shared", "shared", False, False),
    ("relu", 3, True, True),
    (None, 1, True, False),
    ("act", 0, False, True),
]


def run_block(ctx, blocks, shape, layers, value):
    n, h, w, c, e, k, stride, pad = shape
    behind, dw_act, with_bias, shortcut = layers
    r = np.random.default_rng(c + e + k + h)
    half = lambda a: ctx.array(a.astype(np.float16).view(np.uint16))
    floats = lambda a: ctx.array(a.astype(np.float32))
    bias = lambda ch: floats(r.normal(0, .3, ch)) if with_bias else None
    x, w9 = half(r.normal(0, 1, (n, h, w, c))), floats(r.normal(0, .4, (e, 9)))
    b1, b2, b3 = bias(e), bias(e), bias(k)
    first = ctx.conv_desc(n, c, h, w, e, 1, act=int(behind == "act"), c_stride=c, k_stride=e, post_relu=int(behind == "relu"))
    slope1 = floats(r.uniform(-.5, .5, 1 if behind == "shared" else e))
    if behind in ("prelu", "shared"):
        first.post_op, first.post_slope, first.post_slope_shared = 16, slope1.ptr, int(behind == "shared")  # EXHIP_POST_PRELU
    wp1 = ctx.pack_conv_weights(first, hip.F16, r.normal(0, c ** -.5, (e, c, 1, 1)).astype(np.float16).view(np.uint16))
    wide = ctx.empty((n, h, w, e), np.uint16)
    blocks(0)
    ctx.conv2d_f16(first, x, wp1, b1, None, wide)
    prelu = dw_act in ("prelu", "shared")
    slope2 = floats(r.uniform(-.5, .5, 1 if dw_act == "shared" else e)) if prelu else None
    if prelu:
        mid = ctx.dwconv3x3_nhwc_f16_prelu(wide, e, w9, b2, slope2, dw_act == "shared", stride, pad)
    else:
        mid = ctx.dwconv3x3_nhwc_f16(wide, e, w9, b2, stride, pad, dw_act)
    _, oh, ow, _ = mid.shape
    last = ctx.conv_desc(n, e, oh, ow, k, 1, c_stride=e, k_stride=k)
    wp3 = ctx.pack_conv_weights(last, hip.F16, r.normal(0, e ** -.5, (k, e, 1, 1)).astype(np.float16).view(np.uint16))
    res = half(r.normal(0, 1, (n, oh, ow, k))) if shortcut else None
    want = ctx.empty((n, oh, ow, k), np.uint16)
    ctx.conv2d_f16(last, mid, wp3, b3, res, want)
    guard = 64 * k
    y = ctx.array(np.full(want.size + guard, 0x7e00, np.uint16))
    ptr = lambda a: a.ptr if a is not None else None
    dw = Depthwise(x.ptr, w9.ptr, ptr(b2), ptr(slope2), int(dw_act == "shared"), 0 if prelu else dw_act, n, h, w, stride, *pad)
    blocks(value)
    rc = hip.lib().exhip_bottleneck_f16(ctx.h, ctypes.byref(first), wp1.ptr, ptr(b1), ctypes.byref(dw), ctypes.byref(last), wp3.ptr, ptr(b3), ptr(res), y.ptr)
    if rc == 10002:
        return False
    hip._check(rc)
    ctx.sync()
    got, want = y.download(), want.download()
    assert (got[-guard:] == 0x7e00).all()
    assert np.array_equal(got[:-guard].reshape(want.shape), want)
    assert np.isfinite(want.view(np.float16)).all() and np.ptp(want.view(np.float16).astype(np.float32)) > .5
    return True


@pytest.mark.parametrize("layers", LAYERS, ids=["prelu", "shared", "relu", "none", "act"])
@pytest.mark.parametrize("shape", SHAPES, ids=["x".join(map(str, s[:6])) for s in SHAPES])
def test_a_block_equals_its_layers(ctx, blocks, shape, layers):
    run_block(ctx, blocks, shape, layers, 1)  # the rule's tile, where it takes the block at all
    taken = [run_block(ctx, blocks, shape, layers, value) for value in (16 * 4 + 4, 16 + 1, 16 * 2 + 8, 16 * 3 + 7, 256 + 16 * 4 + 4, 256 + 16 * 2 + 7, 256 + 16 * 8 + 14)]
    assert taken[1] and sum(taken) >= 2  # (a large tile of many channels does not fit into LDS)


@pytest.mark.parametrize("n,hw,width,net", [(1, 64, 16, ((2, 32, 2), (1, 32, 1), (1, 32, 1), (2, 64, 2), (1, 64, 1))), (3, 90, 32, ((2, 64, 2), (1, 64, 2), (2, 128, 4), (1, 128, 2))),
                                            (2, 49, 32, ((1, 32, 4), (2, 160, 4), (1, 160, 2), (2, 256, 2), (1, 256, 2)))])
def test_networks_equal_their_layers(blocks, n, hw, width, net):
    m = mobilenet.MobileFaceNetF32(hw=hw, width=width, blocks=net)
    with tempfile.NamedTemporaryFile(suffix=".racy", delete=False) as f:
        path = f.name
    modelfile.write_model(path, m.blobs)
    pipe = xp.Pipeline(m.topology(), path, 0, "f16")
    os.unlink(path)
    x = np.random.default_rng(hw).integers(0, 256, (n, 3, hw, hw)).astype(np.float16).view(np.uint16)
    got = {}
    for value in (0, 1, 16 * 2 + 2, 256 + 16 * 2 + 4):
        blocks(value)
        pipe.set_input(x)
        pipe.run()
        got[value] = pipe.get(m.output)
        mid = pipe.get("b1_dw")  # a blob that the one launch does not store
        assert mid.shape[0] == n and np.array_equal(mid, got.setdefault("mid", mid))
    assert all(np.array_equal(got[0], got[v]) for v in got if v != "mid")
    assert np.isfinite(got[0].view(np.float16)).all() and np.count_nonzero(got[0]) > got[0].size // 2
    pipe.close()
