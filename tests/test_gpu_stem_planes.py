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


@pytest.mark.parametrize("width", [48, 41])
def test_planes_that_begin_anywhere(ctx, width):
    """Planes off 16 bytes are read value by value, whatever their width: the results of the aligned ones."""
    r = np.random.default_rng(width)
    for values in (r.normal(0, 1, (2, 3, 21, width)).astype(np.float16).view(np.uint16), r.normal(0, 1, (2, 3, 21, width)).astype(np.float32)):
        half = values.dtype == np.uint16
        d = ctx.conv_desc(2, 3, 21, width, 64, 3, 2, 1, 1, c_stride=4, k_stride=64, fs_out=0.0 if half else 40.0)
        shape = (2,) + ctx.conv_out_hw(d) + (64,)
        w = r.integers(-127, 128, (64, 3, 3, 3), dtype=np.int8)
        wp = ctx.pack_conv_weights(d, hip.F16 if half else hip.I8, (w / np.float16(400)).astype(np.float16).view(np.uint16) if half else w)
        scale, bias = ctx.array(r.uniform(.5, 1.5, 64).astype(np.float32) / 24000), ctx.array(r.normal(0, .3, 64).astype(np.float32))
        got = []
        for shift in (0, 1, 3):
            x = ctx.array(np.concatenate([np.zeros(shift, values.dtype), values.reshape(-1)]))
            x = x.at(shift * values.itemsize)
            y = ctx.empty(shape, np.uint16 if half else np.int8).zero()
            rc = ctx.stem_f16(d, x, None, None, wp, bias, y) if half else ctx.stem_i8(d, x, None, None, 60.0, wp, scale, bias, y)
            assert rc == 0
            got.append(y.download())
        assert np.count_nonzero(got[0]) > got[0].size // 4
        assert all(np.array_equal(g, got[0]) for g in got)


def test_what_the_stem_leaves_to_the_layers(ctx):
    x, w, y = ctx.empty((1, 3, 16, 16), np.uint16).zero(), ctx.empty((64 * 1024,), np.uint8).zero(), ctx.empty((1, 16, 16, 64), np.uint16)
    for c, kernel, c_stride in ((3, 1, 4), (5, 3, 16)):
        d = ctx.conv_desc(1, c, 16, 16, 64, kernel, 1, kernel // 2, c_stride=c_stride, k_stride=64)
        assert ctx.stem_f16(d, x, None, None, w, None, y) == hip.ERR_UNSUPPORTED
    with pytest.raises(hip.ExhipError):
        ctx.stem_f16(ctx.conv_desc(1, 3, 16, 16, 64, 3, 1, 1, c_stride=4, k_stride=64), x, ctx.empty((3,), np.float32).zero(), None, w, None, y)


@pytest.mark.parametrize("scales", [(40.0, 30.0), (40.0, 30.0, 40.0, 20.0)], ids=["two", "three"])
@pytest.mark.parametrize("channels", [32, 24])
@pytest.mark.parametrize("front", ["Input", "none"])
def test_int8_plan_whose_first_layer_is_read_at_several_scales(tmp_path, front, channels, scales):
    """The first layer's float32 result is quantized again for the readers with other feature-map scales, as any layer's is: the plan takes the
    network, with the first layer as one launch or as a quantizer and a convolution, and gives the separate layers' bytes."""
    from excalibur_amd import modelfile as mf
    from excalibur_amd import pipeline as xp
    r = np.random.default_rng(7)
    lines, blobs = ["Input data 0 1 data 0=40 1=24 2=3 3=104,117,123 4=0.017,0.018,0.017"] if front == "Input" else [], []

    def conv(bottom, top, cin, k, kernel, stride, fs):
        w = r.normal(0, np.sqrt(2.0 / (cin * kernel * kernel)), (k, cin, kernel, kernel)).astype(np.float32)
        ws = (np.float32(127.0) / np.abs(w).reshape(k, -1).max(axis=1)).astype(np.float32)
        wq = np.clip(np.rint(w * ws[:, None, None, None]), -127, 127).astype(np.int8)
        lines.append(mf.conv_line("Convolution", top + "_l", bottom, top, k, kernel, stride, kernel // 2, True, w.size, 1, int8=True))
        blobs.append(mf.conv_blob_i8(wq, r.normal(0, .3, k).astype(np.float32), ws, np.float32(fs)))

    conv("data", "c0", 3, channels, 3, 2, 50.0)
    lines.append("HardSwish hs0 1 1 c0 a0 0=1.666667e-01 1=5.000000e-01")
    readers = [f"a0_{i}" for i in range(len(scales))]
    lines.append(f"Split sp0 1 {len(scales)} a0 " + " ".join(readers))
    outputs = [f"c{i + 1}" for i in range(len(scales))]
    for reader, top, fs in zip(readers, outputs, scales):
        conv(reader, top, channels, 16, 1, 1, fs)
    path = str(tmp_path / "net.racy")
    mf.write_model(path, blobs)
    x = np.random.default_rng(8).uniform(0, 255, (3, 3, 24, 40)).astype(np.float32)
    if front != "Input":
        x = (x - 128) / 64
    got, launches = {}, {}
    for way, fusion, stem in (("layers", False, 1), ("quantizer", True, 0), ("stem", True, 1)):
        hip.set_option("stem", stem)
        try:
            p = xp.Pipeline(mf.topology(lines, "scales"), path, 0, fusion=fusion)
            p.time_fused_span(0)
            p.forward(x)
            assert p.fused == fusion, way
            launches[way] = p.last_span()[1]
            got[way] = {b: p.get(b) for b in outputs}
            p.close()
        finally:
            hip.set_option("stem", 1)
    assert launches["stem"] == launches["quantizer"] - 1
    for b in outputs:
        assert np.ptp(got["layers"][b]) > .5
        for way in ("quantizer", "stem"):
            assert np.array_equal(got[way][b].view(np.uint32), got["layers"][b].view(np.uint32)), (way, b)
