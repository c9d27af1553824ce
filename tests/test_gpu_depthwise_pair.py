"""A depthwise 3x3 layer and the pointwise layer behind it as one kernel (conv_pw.hip, dw_pw_kernel): the results are those of
the two layers run one after the other, bit for bit."""
import ctypes
import os
import tempfile

import numpy as np
import pytest

from excalibur_amd import hip, mobilenet, modelfile
from excalibur_amd import pipeline as xp

pytestmark = pytest.mark.gpu


@pytest.fixture
def pairs():
    yield lambda value: hip.set_option("dw_pw", value)
    hip.set_option("dw_pw", 1)


NETS = [
    # n, hw, width, blocks: maps of even and odd sizes (strips of four, two and one pixel), tiles that end inside an image and
    # behind the last one, channels up to the kernel's 512, the split form's sums, residual sums, one or two tiles a group
    (1, 64, 16, ((2, 32, 2), (1, 32, 1), (1, 32, 1), (2, 64, 2), (1, 64, 1))),
    (3, 90, 32, ((2, 64, 2), (1, 64, 2), (2, 128, 4), (1, 128, 2))),
    (2, 50, 32, ((1, 32, 4), (2, 160, 4), (1, 160, 2), (2, 256, 2), (1, 256, 2))),
    (24, 80, 32, ((2, 32, 2), (1, 32, 2), (1, 64, 1))),
]


@pytest.mark.parametrize("n,hw,width,blocks", NETS, ids=lambda v: str(v) if isinstance(v, int) else "")
def test_pairs_equal_the_two_layers(pairs, n, hw, width, blocks):
    m = mobilenet.MobileFaceNetF32(hw=hw, width=width, blocks=blocks)
    with tempfile.NamedTemporaryFile(suffix=".racy", delete=False) as f:
        path = f.name
    modelfile.write_model(path, m.blobs)
    pipe = xp.Pipeline(m.topology(), path, 0, "f16")
    os.unlink(path)
    x = np.random.default_rng(hw).integers(0, 256, (n, 3, hw, hw)).astype(np.float16).view(np.uint16)
    got = {}
    for value in (0, 2):
        pairs(value)
        pipe.set_input(x)
        pipe.run()
        got[value] = pipe.get(m.output).view(np.float16)
    assert np.array_equal(got[0].view(np.uint16), got[2].view(np.uint16))
    assert np.isfinite(got[0]).all() and np.count_nonzero(got[0]) > got[0].size // 2
    pipe.close()


# ---- the two layers' own options, through the C ABI ----
class Depthwise(ctypes.Structure):
    _fields_ = [("x", ctypes.c_void_p), ("w9", ctypes.c_void_p), ("bias", ctypes.c_void_p), ("slope", ctypes.c_void_p)] + \
               [(k, ctypes.c_int) for k in ("slope_shared", "act", "n", "h", "w", "stride", "pt", "pb", "pl", "pr")]


@pytest.fixture(scope="module")
def ctx():
    c = hip.Ctx(0)
    yield c
    c.close()


FRONT = [
    # stride, pad (top, bottom, left, right), map, activation (or "prelu", "shared"), bias
    (1, (1, 1, 1, 1), (12, 16), 1, True),
    (1, (1, 1, 1, 1), (9, 13), 3, False),
    (1, (2, 0, 0, 1), (11, 10), 0, False),      # uneven padding: the map grows above, shrinks beside
    (1, (0, 0, 0, 0), (9, 7), "shared", True),
    (2, (1, 1, 1, 1), (16, 17), 3, True),
    (2, (0, 1, 0, 1), (15, 14), 1, False),
    (2, (2, 1, 1, 2), (7, 9), "prelu", False),
]
BEHIND = [
    # k, options of the pointwise layer, its shortcut
    (64, {}, False),
    (48, dict(post_relu=1), False),
    (64, dict(post_op="hardswish", post_alpha=1 / 6, post_beta=.5), False),
    (96, dict(post_op="leakyrelu", post_alpha=.1), True),
    (80, dict(post_op="clip", post_alpha=-.5, post_beta=.75, residual_last=1), True),   # an odd number of blocks, run-time epilogue
    (32, dict(act=1), True),
    (64, dict(act=3, post_relu=1, residual_last=1), True),
]


@pytest.mark.parametrize("c", [32, 96])
@pytest.mark.parametrize("k,post,shortcut", BEHIND, ids=[f"behind{i}" for i in range(len(BEHIND))])
@pytest.mark.parametrize("stride,pad,hw,act,with_bias", FRONT, ids=[f"front{i}" for i in range(len(FRONT))])
def test_every_option_of_the_two_layers(ctx, pairs, stride, pad, hw, act, with_bias, k, post, shortcut, c):
    n, (h, w) = 2, hw
    r = np.random.default_rng(c + k + h * w)
    half = lambda a: ctx.array(a.astype(np.float16).view(np.uint16))
    x, w9 = half(r.normal(0, 1, (n, h, w, c))), ctx.array(r.normal(0, .4, (c, 9)).astype(np.float32))
    bias = ctx.array(r.normal(0, .3, c).astype(np.float32)) if with_bias else None
    prelu = act in ("prelu", "shared")
    slope = ctx.array(r.uniform(-.5, .5, 1 if act == "shared" else c).astype(np.float32)) if prelu else None
    if prelu:
        mid = ctx.dwconv3x3_nhwc_f16_prelu(x, c, w9, bias, slope, act == "shared", stride, pad)
    else:
        mid = ctx.dwconv3x3_nhwc_f16(x, c, w9, bias, stride, pad, act)
    _, oh, ow, _ = mid.shape
    d = ctx.conv_desc(n, c, oh, ow, k, 1, c_stride=c, k_stride=k, **post)
    wp = ctx.pack_conv_weights(d, hip.F16, r.normal(0, .2, (k, c, 1, 1)).astype(np.float16).view(np.uint16))
    pw_bias = ctx.array(r.normal(0, .3, k).astype(np.float32)) if with_bias else None
    res = half(r.normal(0, 1, (n, oh, ow, k))) if shortcut else None
    want = ctx.empty((n, oh, ow, k), np.uint16)
    ctx.conv2d_f16(d, mid, wp, pw_bias, res, want)
    guard = 64 * k
    y = ctx.array(np.full(want.size + guard, 0x7e00, np.uint16))
    ptr = lambda a: a.ptr if a is not None else None
    dw = Depthwise(x.ptr, w9.ptr, ptr(bias), ptr(slope), int(act == "shared"), 0 if prelu else act, n, h, w, stride, *pad)
    pairs(2)
    hip._check(hip.lib().exhip_dw_pw_f16(ctx.h, ctypes.byref(dw), ctypes.byref(d), wp.ptr, ptr(pw_bias), ptr(res), y.ptr))
    ctx.sync()
    got, want = y.download(), want.download()
    assert (got[-guard:] == 0x7e00).all()
    assert np.array_equal(got[:-guard].reshape(want.shape), want)
    assert np.isfinite(want.view(np.float16)).all() and np.ptp(want.view(np.float16).astype(np.float32)) > .5


# pixels of a group: fewer than a strip's round and than a block, several blocks, more than the map has. Up to 32 for 512 channels and 128 for 96: beyond
# the 40 KiB that a group's depthwise results may take, the option leaves the number to the rule, whose launch must then come out
@pytest.mark.parametrize("pixels", [4, 8, 16, 32, 64, 128, 256])
@pytest.mark.parametrize("front", [0, 2, 4, 5, 6])
@pytest.mark.parametrize("c,behind", [(16, 0), (96, 4), (512, 1)])
def test_pixels_of_a_group(ctx, pairs, front, behind, c, pixels):
    forced = lambda value: pairs(pixels)
    test_every_option_of_the_two_layers(ctx, forced, *FRONT[front], *BEHIND[behind], c)
