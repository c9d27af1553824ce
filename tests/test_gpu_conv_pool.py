"""An int8 convolution with the 2x2 max pooling behind it as one kernel (conv_pw.hip, the Pooled epilogues): the results are those of the
two layers run one after the other, bit for bit."""
import ctypes

import numpy as np
import pytest

from excalibur_amd import hip

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = hip.Ctx(0)
    yield c
    c.close()


SHAPES = [
    # n, c, h, w, k, kernel, stride, pad: 32- and 64-byte pixels (single steps and pairs), one block of channels, an odd number, ragged channels,
    # odd maps whose last row and column no window has, tiles that end inside an image and behind the last one
    (1, 32, 8, 8, 32, 3, 1, 1),
    (3, 16, 13, 11, 24, 3, 1, 0),
    (2, 64, 17, 30, 96, 3, 1, 1),
    (5, 96, 9, 7, 64, 3, 1, 1),
    (2, 128, 21, 19, 130, 3, 2, 1),
    (1, 32, 66, 130, 64, 5, 1, 2),
    (9, 64, 2, 2, 32, 1, 1, 0),
]


def pooled_and_the_two_layers(ctx, n, c, h, w, k, kernel, stride, pad, results, act=0, post_relu=0, **options):
    """Asserts that the one launch gives the bytes of the two layers and writes nothing behind its results; its status."""
    r = np.random.default_rng(h * w + k)
    cs, ks = hip.pad_to(c, 32), hip.pad_to(k, 32)
    d = ctx.conv_desc(n, c, h, w, k, kernel, stride, pad, act, cs, ks, post_relu, 40.0 if results != "float" else 0.0)
    oh, ow = ctx.conv_out_hw(d)
    ph, pw = oh // 2, ow // 2
    x = r.integers(-127, 128, (n, h, w, cs), dtype=np.int8)
    x[..., c:] = 0
    x = ctx.array(x)
    wp = ctx.pack_conv_weights(d, hip.I8, r.integers(-127, 128, (k, c, kernel, kernel), dtype=np.int8))
    scale = ctx.array((r.uniform(.5, 1.5, k) / (73 * 73 * kernel * np.sqrt(c))).astype(np.float32))
    bias = ctx.array(r.normal(0, .3, k).astype(np.float32))
    mid, shape = ctx.empty((n, oh, ow, ks), np.float32), (n, ph, pw, ks)
    plain = ctx.conv_desc(n, c, h, w, k, kernel, stride, pad, act, cs, ks, post_relu, 0.0)
    ctx.conv2d_i8(plain, x, wp, scale, bias, None, None, mid)
    forms = [np.int8] * (results != "float") + [np.float32] * (results != "int8")
    want = {t: ctx.empty(shape, t) for t in forms}
    ptr = lambda a: a.ptr if a is not None else None
    hip._check(hip.lib().exhip_maxpool2d_nhwc_f32(ctx.h, mid.ptr, ptr(want.get(np.float32)), ptr(want.get(np.int8)), ctypes.c_float(40.0), n, ks, oh, ow, ks, ph, pw,
                                                  2, 2, 2, 2, 0, 0))
    got = {t: ctx.array(np.full(want[t].size + 64 * ks, 77, t)) for t in forms}
    defaults = dict(direct=1, pw_tile=0)
    for name in options:
        hip.set_option(name, options[name])
    try:
        rc = ctx.conv2d_i8_maxpool2x2(d, ph, pw, x, wp, scale, bias, got.get(np.int8), got.get(np.float32))
    finally:
        for name in options:
            hip.set_option(name, defaults[name])
    if rc:
        return rc
    for t in forms:
        y = got[t].download()
        assert (y[-64 * ks:] == 77).all()
        assert np.array_equal(y[:-64 * ks].reshape(shape), want[t].download())
    assert all(np.ptp(want[t].download()[..., :k].astype(np.float32)) > .5 for t in forms)
    return 0


@pytest.mark.parametrize("act,post_relu", [(0, 0), (1, 0), (0, 1)], ids=["none", "relu", "relu_layer"])
@pytest.mark.parametrize("results", ["int8", "float", "both"])
@pytest.mark.parametrize("n,c,h,w,k,kernel,stride,pad", SHAPES, ids=[f"s{i}" for i in range(len(SHAPES))])
def test_pooled_equals_the_two_layers(ctx, n, c, h, w, k, kernel, stride, pad, results, act, post_relu):
    assert pooled_and_the_two_layers(ctx, n, c, h, w, k, kernel, stride, pad, results, act, post_relu, direct=2) == 0


# waves of 64 pixels x 64 channels (2048 and more take the larger wave tile where option pw_tile asks for it): 2048 exactly, one less, a layer with an
# odd number of channel blocks, one with single k-steps
@pytest.mark.parametrize("results", ["int8", "float", "both"])
@pytest.mark.parametrize("n,c,h,w,k", [(32, 64, 64, 64, 64), (89, 32, 46, 32, 48), (21, 64, 65, 67, 96), (32, 96, 64, 64, 64)], ids=["most", "fewer", "odd", "single"])
def test_pooled_equals_the_two_layers_whatever_the_tile_option(ctx, n, c, h, w, k, results):
    for tile in (0, 2):
        assert pooled_and_the_two_layers(ctx, n, c, h, w, k, 3, 1, 1, results, direct=2, pw_tile=tile) == 0


def test_what_the_pooled_form_leaves_to_the_layers(ctx):
    x, w, s, y = ctx.empty((1, 8, 8, 64), np.int8).zero(), ctx.empty((64 * 1024,), np.uint8).zero(), ctx.empty((64,), np.float32).zero(), ctx.empty((1, 8, 8, 64), np.int8)
    d = ctx.conv_desc(1, 64, 8, 8, 64, 3, 1, 1, 0, 64, 64, 0, 1.0, post_op="hardswish", post_alpha=1 / 6, post_beta=.5)
    assert ctx.conv2d_i8_maxpool2x2(d, 4, 4, x, w, s, None, y) == hip.ERR_UNSUPPORTED
    with pytest.raises(hip.ExhipError):   # windows beyond the map
        ctx.conv2d_i8_maxpool2x2(ctx.conv_desc(1, 64, 8, 8, 64, 3, 1, 1, 0, 64, 64, 0, 1.0), 5, 4, x, w, s, None, y)
