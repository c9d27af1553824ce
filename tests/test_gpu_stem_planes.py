"""The first layer of a network on its planes, with the Input layer in front (conv_pw.hip, stem_planes_kernel): the results are those of the
Input layer, the layout conversion or quantizer and the convolution run one after the other, bit for bit."""
import numpy as np
import pytest

from excalibur_amd import hip

pytestmark = pytest.mark.gpu
POST_PRELU = 16


@pytest.fixture(scope="module")
def ctx():
    c = hip.Ctx(0)
    yield c
    c.close()


SHAPES = [
    # n, c, h, w, k, kernel width, stride, padding, options: rows of whole 16-byte pieces and others, one block of channels, an odd number, more
    # than the waves, ragged channels, several rows a group (stem option below), the last group shorter, padding on every side
    (1, 3, 112, 112, 64, 3, 2, (1, 1, 1, 1), dict(prelu=True)),
    (3, 3, 31, 40, 32, 3, 2, (1, 1, 1, 1), dict(act=1)),
    (2, 1, 17, 23, 16, 3, 1, (1, 1, 1, 1), {}),
    (2, 4, 20, 48, 96, 3, 1, (0, 0, 0, 0), dict(post_relu=1)),
    (5, 3, 9, 8, 40, 4, 2, (2, 1, 3, 2), dict(post_op="hardswish", post_alpha=1 / 6, post_beta=.5)),
    (1, 2, 3, 5, 320, 2, 1, (0, 0, 0, 0), dict(act=3)),
    (2, 3, 64, 640, 24, 3, 2, (0, 1, 0, 1), dict(post_op="leakyrelu", post_alpha=.1)),
    (70, 3, 33, 32, 48, 3, 1, (1, 1, 1, 1), dict(act=1)),
]


@pytest.mark.parametrize("scaled", [False, True], ids=["plain", "input"])
@pytest.mark.parametrize("n,c,h,w,k,kw,stride,pad,post", SHAPES, ids=[f"s{i}" for i in range(len(SHAPES))])
def test_stem_equals_the_layers(ctx, n, c, h, w, k, kw, stride, pad, post, scaled):
    r = np.random.default_rng(h * w + k)
    x = ctx.array(r.integers(0, 256, (n, c, h, w)).astype(np.float16).view(np.uint16)) if scaled else ctx.array(r.normal(0, 1, (n, c, h, w)).astype(np.float16).view(np.uint16))
    mean = ctx.array(r.uniform(100, 150, c).astype(np.float32)) if scaled else None
    factor = ctx.array(r.uniform(.005, .02, c).astype(np.float32)) if scaled else None
    post, ks = dict(post), hip.pad_to(k, 16)
    prelu, slope = post.pop("prelu", False), ctx.array(r.uniform(-.5, .5, k).astype(np.float32))
    d = ctx.conv_desc(n, c, h, w, k, (3, kw), stride, pad, c_stride=4, k_stride=ks, **post)
    if prelu:
        d.post_op, d.post_slope = POST_PRELU, slope.ptr
    oh, ow = ctx.conv_out_hw(d)
    wp = ctx.pack_conv_weights(d, hip.F16, r.normal(0, .3, (k, c, 3, kw)).astype(np.float16).view(np.uint16))
    bias = ctx.array(r.normal(0, .3, k).astype(np.float32))
    seen = ctx.channelwise_f16("input", x, mean, factor) if scaled else x
    pixels = ctx.empty((n, h, w, 4), np.uint16)
    hip._check(hip.lib().exhip_nchw_f16_to_nhwc_f16(ctx.h, seen.ptr, n, c, h, w, 4, pixels.ptr))
    want = ctx.empty((n, oh, ow, ks), np.uint16)
    ctx.conv2d_f16(d, pixels, wp, bias, None, want)
    guard = 64 * ks
    for rows in (1, 2, 4):   # at most so many output rows a group (2 upwards: whatever the launch's size)
        y = ctx.array(np.full(want.size + guard, 0x7e00, np.uint16))
        hip.set_option("stem", rows)
        try:
            assert ctx.stem_f16(d, x, mean, factor, wp, bias, y) == 0
            ctx.sync()
        finally:
            hip.set_option("stem", 1)
        got = y.download()
        assert (got[-guard:] == 0x7e00).all()
        assert np.array_equal(got[:-guard].reshape(want.shape), want.download())
    values = want.download().view(np.float16)[..., :k].astype(np.float32)
    assert np.isfinite(values).all() and np.ptp(values) > .5


@pytest.mark.parametrize("scaled", [False, True], ids=["plain", "input"])
@pytest.mark.parametrize("results", ["int8", "float", "both"])
@pytest.mark.parametrize("n,c,h,w,k,kw,stride,pad,post", SHAPES[1:] + [(3, 3, 26, 24, 64, 7, 2, (3, 3, 3, 3), dict(act=1))],
                         ids=[f"s{i}" for i in range(1, len(SHAPES) + 1)])
def test_int8_stem_equals_the_layers(ctx, n, c, h, w, k, kw, stride, pad, post, results, scaled):
    r = np.random.default_rng(h * w + k)
    x = ctx.array((r.integers(0, 256, (n, c, h, w)) if scaled else r.normal(0, 1, (n, c, h, w))).astype(np.float32))
    mean = ctx.array(r.uniform(100, 150, c).astype(np.float32)) if scaled else None
    factor = ctx.array(r.uniform(.005, .02, c).astype(np.float32)) if scaled else None
    ks, fs_in = hip.pad_to(k, 32), 60.0
    d = ctx.conv_desc(n, c, h, w, k, (3, kw), stride, pad, c_stride=4, k_stride=ks, fs_out=40.0 if results != "float" else 0.0, **post)
    oh, ow = ctx.conv_out_hw(d)
    wp = ctx.pack_conv_weights(d, hip.I8, r.integers(-127, 128, (k, c, 3, kw), dtype=np.int8))
    scale = ctx.array((r.uniform(.5, 1.5, k) / (fs_in * 73 * np.sqrt(9 * c))).astype(np.float32))
    bias = ctx.array(r.normal(0, .3, k).astype(np.float32))
    seen = ctx.channelwise_f32("input", x, mean, factor) if scaled else x
    pixels = ctx.quantize_nchw_to_nhwc_i8(seen, fs_in, 4)
    shape = (n, oh, ow, ks)
    forms = [np.int8] * (results != "float") + [np.float32] * (results != "int8")
    want = {t: ctx.empty(shape, t) for t in forms}
    ctx.conv2d_i8(d, pixels, wp, scale, bias, None, want.get(np.int8), want.get(np.float32))
    for rows in (1, 2, 4):
        got = {t: ctx.array(np.full(want[t].size + 64 * ks, 77, t)) for t in forms}
        hip.set_option("stem", rows)
        try:
            assert ctx.stem_i8(d, x, mean, factor, fs_in, wp, scale, bias, got.get(np.int8), got.get(np.float32)) == 0
            ctx.sync()
        finally:
            hip.set_option("stem", 1)
        for t in forms:
            y = got[t].download()
            assert (y[-64 * ks:] == 77).all()
            assert np.array_equal(y[:-64 * ks].reshape(shape), want[t].download())
    assert all(np.ptp(want[t].download()[..., :k].astype(np.float32)) > .5 for t in forms)


def test_what_the_stem_leaves_to_the_layers(ctx):
    x, w, y = ctx.empty((1, 3, 16, 16), np.uint16).zero(), ctx.empty((64 * 1024,), np.uint8).zero(), ctx.empty((1, 16, 16, 64), np.uint16)
    for c, kernel, c_stride in ((3, 1, 4), (5, 3, 16)):
        d = ctx.conv_desc(1, c, 16, 16, 64, kernel, 1, kernel // 2, c_stride=c_stride, k_stride=64)
        assert ctx.stem_f16(d, x, None, None, w, None, y) == hip.ERR_UNSUPPORTED
    with pytest.raises(hip.ExhipError):
        ctx.stem_f16(ctx.conv_desc(1, 3, 16, 16, 64, 3, 1, 1, c_stride=4, k_stride=64), x, ctx.empty((3,), np.float32).zero(), None, w, None, y)
