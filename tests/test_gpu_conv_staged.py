"""3x3 fp16 and int8 layers with their input staged in LDS (conv_staged.hip): int8 results are the other kernels' byte for byte, fp16 sums, which run in
another order, stay within the rounding of a sum in float32 and of the halves stored."""
import numpy as np
import pytest

from excalibur_amd import hip

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = hip.Ctx(0)
    yield c
    c.close()


@pytest.fixture
def staged():
    yield lambda value: hip.set_option("staged", value)
    hip.set_option("staged", 1)


SHAPES = [
    # n, channels, h, w, output channels, stride, padding (top, bottom, left, right)
    (1, 64, 9, 13, 64, 1, (1, 1, 1, 1)),      # a map smaller than a run
    (5, 64, 6, 7, 96, 1, (1, 1, 1, 1)),       # runs over several maps, half a pair of channel blocks
    (2, 192, 17, 33, 80, 1, (0, 2, 2, 0)),    # three pieces of 64 bytes and an uneven padding; channels that end inside a block
    (1, 320, 12, 41, 64, 1, (1, 1, 1, 1)),    # pieces that do not fill the last stage
    (3, 64, 1, 5, 64, 1, (1, 1, 1, 1)),       # one row
    (1, 128, 40, 40, 128, 1, (0, 0, 0, 0)),
    (2, 64, 15, 21, 64, 2, (1, 1, 1, 1)),     # odd maps at stride 2
    (1, 128, 24, 50, 96, 2, (0, 1, 0, 1)),
    (7, 96, 5, 4, 64, 2, (1, 1, 1, 1)),       # fp16: the packing's chunks are half a piece
    (1, 32, 33, 70, 72, 2, (1, 1, 1, 1)),
    (2, 160, 11, 9, 96, 1, (1, 1, 1, 1)),     # int8: the last piece of 64 bytes half full
    (1, 32, 20, 31, 64, 1, (1, 1, 1, 1)),
    (1, 288, 5, 23, 64, 1, (2, 0, 1, 1)),
]
KINDS = {
    "none": {}, "act": dict(act=1), "relu": dict(post_relu=1), "hardswish": dict(post_op="hardswish", post_alpha=1 / 6, post_beta=.5),
    "leaky": dict(post_op="leakyrelu", post_alpha=.1), "shortcut": dict(post_relu=1), "last": dict(post_op="hardswish", post_alpha=1 / 6, post_beta=.5, residual_last=1),
    "added": {}, "last_relu": dict(post_relu=1, residual_last=1),
}
SHORTCUT = ("shortcut", "last", "added", "last_relu")


def results(ctx, shape, kind, int8, wider, floats, values):
    """A function that runs the layer and returns its results, and the sums of the products' magnitudes (float64)."""
    n, c, h, w, k, stride, pad = shape
    r = np.random.default_rng(c + 7 * h + 31 * k)
    ks = hip.pad_to(k, 16 if not int8 else 32) + 32 * wider
    d = ctx.conv_desc(n, c, h, w, k, 3, stride, pad, c_stride=c, k_stride=ks, fs_out=30.0 if int8 else 0.0, **KINDS[kind])
    oh, ow = ctx.conv_out_hw(d)
    bias = r.normal(0, .3, k).astype(np.float32)
    b = ctx.array(bias)
    if int8:
        x, wt = r.integers(-127, 128, (n, h, w, c), dtype=np.int8), r.integers(-127, 128, (k, c, 3, 3), dtype=np.int8)
        scale = ctx.array((r.uniform(.5, 1.5, k) / (127 * 73 * np.sqrt(9 * c))).astype(np.float32))
    else:
        x, wt = r.normal(0, 1, (n, h, w, c)).astype(np.float16), r.normal(0, (9 * c) ** -.5, (k, c, 3, 3)).astype(np.float16)
        if values == "infinite":
            x[0, 0, 0, 0], x[-1, -1, -1, -1] = np.inf, np.nan
        x, wt = x.view(np.uint16), wt.view(np.uint16)
    res = None
    if kind in SHORTCUT:
        res = r.normal(0, 1, (n, oh, ow, ks)).astype(np.float32 if int8 else np.float16)
        res = ctx.array(res if int8 else res.view(np.uint16))
    xd, wp = ctx.array(x), ctx.pack_conv_weights(d, hip.I8 if int8 else hip.F16, wt)

    def run():
        guard = 4096
        y = ctx.array(np.full(n * oh * ow * ks + guard, 0x55, np.int8 if int8 else np.uint16))
        yf = ctx.array(np.full(n * oh * ow * ks + guard, -77., np.float32)) if floats else None
        if int8:
            ctx.conv2d_i8(d, xd, wp, scale, b, res, y, yf)
        else:
            ctx.conv2d_f16(d, xd, wp, b, res, y)
        ctx.sync()
        out = [a.download() for a in (y, yf) if a is not None]
        assert (out[0][-guard:] == 0x55).all() and (len(out) == 1 or (out[1][-guard:] == -77).all())
        return [a[:-guard].reshape(n, oh, ow, ks) for a in out]

    magnitude = None
    if not int8:
        xa, wa = np.abs(x.view(np.float16).astype(np.float64)), np.abs(wt.view(np.float16).astype(np.float64))
        xa = np.pad(xa, ((0, 0), pad[:2], pad[2:], (0, 0)))
        magnitude = np.zeros((n, oh, ow, ks))
        for i in range(3):
            for j in range(3):
                part = xa[:, i:i + (oh - 1) * stride + 1:stride, j:j + (ow - 1) * stride + 1:stride]
                magnitude[..., :k] += part.reshape(-1, c).dot(wa[:, :, i, j].T).reshape(n, oh, ow, k)
        magnitude[..., :k] += np.abs(bias) + (0 if res is None else np.abs(res.download().view(np.float16).astype(np.float64))[..., :k])
    return run, magnitude


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("shape", [s for s in SHAPES if s[5] == 1], ids=lambda s: "x".join(map(str, s[:6])))
def test_int8_equals_the_other_kernels(ctx, staged, shape, kind):
    for wider, floats in ((0, False), (1, True)):
        run, _ = results(ctx, shape, kind, True, wider, floats, "")
        staged(0)
        want = run()
        assert np.unique(want[0]).size > 30
        for form in (2, 3, 4, 1):
            staged(form)
            for a, b in zip(run(), want):
                assert np.array_equal(a, b), (wider, form)


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s[:6])))
def test_fp16_within_rounding(ctx, staged, shape, kind):
    for wider in (0, 1):
        run, magnitude = results(ctx, shape, kind, False, wider, False, "")
        staged(0)
        want = run()[0].view(np.float16).astype(np.float64)
        # two sums of K products in float32 differ by at most 2 K 2^-24 of the products' magnitudes; an activation's slope is at most 1.5, and up to three
        # values are stored as halves on the way, each of which may land on the neighbouring one
        bound = 1.5 * (2 * 9 * shape[1] * 2. ** -24 * magnitude + 3 * 2. ** -10 * (magnitude / np.sqrt(9 * shape[1]) * 4 + np.abs(want)))
        for form in (2, 3, 4, 1):
            staged(form)
            got = run()[0].view(np.float16).astype(np.float64)
            assert np.isfinite(got).all() and (np.abs(got - want) <= bound).all(), (wider, form)
            assert np.array_equal(got[..., shape[4]:], want[..., shape[4]:])  # channels beyond the layer's: zeros, or untouched behind the packed blocks
        assert np.ptp(want) > 1


@pytest.mark.parametrize("shape", [SHAPES[0], SHAPES[6]], ids=["stride1", "stride2"])
def test_infinities_and_nan_reach_the_pixels_they_reach(ctx, staged, shape):
    run, _ = results(ctx, shape, "none", False, 0, False, "infinite")
    staged(0)
    want = run()[0].view(np.float16)
    assert not np.isfinite(want).all() and np.isfinite(want).any()
    for form in (2, 3, 4):
        staged(form)
        got = run()[0].view(np.float16)
        assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isinf(got), np.isinf(want))
        assert np.array_equal(got[np.isinf(got)], want[np.isinf(want)])


# layers on either side of the rule's lines: the same bytes whichever kernel it is
@pytest.mark.parametrize("n,c,hw,k,kind", [(8, 128, 40, 128, "hardswish"), (16, 64, 30, 64, "none"), (7, 256, 20, 256, "act"), (9, 256, 20, 256, "act"), (5, 128, 53, 224, "shortcut"),
                                           (3, 192, 31, 96, "last")])
def test_int8_by_its_rule(ctx, staged, n, c, hw, k, kind):
    run, _ = results(ctx, (n, c, hw, hw, k, 1, (1, 1, 1, 1)), kind, True, 0, kind == "last", "")
    staged(0)
    want = run()
    staged(1)
    for a, b in zip(run(), want):
        assert np.array_equal(a, b)
