"""The float32 convolution with bfloat16 thirds (conv_f32_thirds.hip): every form on ragged shapes, against sums in 64 bits; infinities, NaN and
values whose thirds would leave the range; and the placements of its results."""
import ctypes

import numpy as np
import pytest

from excalibur_amd import hip
from tests import cases
from tests import test_gpu_conv_f32 as plain

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = hip.Ctx(0)
    yield c
    c.close()


@pytest.fixture(params=range(6))
def tile(request):
    hip.set_option("f32_tile", request.param)
    yield request.param
    hip.set_option("f32_tile", 0)


def conv64(x, w, pad):
    """NHWC x, OIHW w, padding (top, bottom, left, right), in 64 bits; and the sum of the products' absolute values."""
    xp = np.pad(x.astype(np.float64), ((0, 0), pad[:2], pad[2:], (0, 0)))
    oh, ow = xp.shape[1] - 2, xp.shape[2] - 2
    taps = [(xp[:, i:i + oh, j:j + ow], w[:, :, i, j].T.astype(np.float64)) for i in range(3) for j in range(3)]
    return sum(a @ b for a, b in taps), sum(np.abs(a) @ np.abs(b) for a, b in taps)


def run(ctx, x, w, pad, bias=None, res=None, ks=None, **kw):
    n, h, wd, c = x.shape
    k = w.shape[0]
    ks = ks or hip.pad_to(k, 32)
    d = ctx.conv_desc(n, c, h, wd, k, 3, 1, pad, kw.pop("act", 0), c, ks, **kw)
    oh, ow = ctx.conv_out_hw(d)
    rd = None
    if res is not None:
        rd = np.zeros((n, oh, ow, ks), np.float32)
        rd[..., :k] = res
        rd = ctx.array(rd)
    y = ctx.array(np.full(n * oh * ow * ks + 64, 7.0, np.float32))
    flat = ctx.array(np.full(n * oh * ow * k + 64, 7.0, np.float32))
    both = bias if bias is None else ctx.array(bias)
    for rows, planes in ((y, None), (None, flat)):  # rows and planes are finished in different orders
        ctx.conv2d_f32(d, ctx.array(x), ctx.pack_conv_weights(d, hip.F32, w), both, rd, rows, planes)
    ctx.sync()
    got, planar = y.download(), flat.download()
    assert (got[-64:] == 7.0).all() and (planar[-64:] == 7.0).all()
    got = got[:-64].reshape(n, oh, ow, ks)
    assert not got[..., k:].any()
    assert np.array_equal(planar[:-64].reshape(n, k, oh, ow), got[..., :k].transpose(0, 3, 1, 2), equal_nan=True)
    return got[..., :k]


SHAPES = [
    # n, h, w, c, k, padding
    (1, 1, 1, 16, 1, (1, 1, 1, 1)),        # one pixel, one step: most waves have nothing to do
    (70, 1, 1, 32, 33, (1, 1, 1, 1)),      # every pixel a map of its own, nine staged for each
    (1, 2, 300, 16, 32, (1, 1, 1, 1)),     # long rows: strips
    (3, 13, 13, 80, 96, (1, 1, 1, 1)),     # runs across images, five steps: chunks that are not full
    (2, 9, 31, 48, 40, (0, 0, 0, 0)),      # no padding, strips of a ragged width
    (1, 40, 7, 144, 70, (2, 0, 1, 2)),     # uneven padding, a third chunk of one step
    (2, 17, 19, 272, 32, (1, 1, 1, 1)),
    (18, 1, 1, 80, 33, (1, 1, 1, 1)),      # maps of a pixel and more channels than are staged at a time: two buffers
    (70, 1, 1, 272, 40, (1, 1, 1, 1)),
    (32, 3, 3, 96, 64, (0, 0, 0, 0)),
]


@pytest.mark.parametrize("shape", SHAPES, ids=["x".join(map(str, s[:5])) for s in SHAPES])
def test_every_form_against_64_bits(ctx, tile, shape):
    n, h, w, c, k, pad = shape
    r = np.random.default_rng(c + k)
    x, wt, bias = (r.standard_normal(s).astype(np.float32) for s in ((n, h, w, c), (k, c, 3, 3), k))
    want, scale = conv64(x, wt, pad)
    res = r.standard_normal(want.shape).astype(np.float32)
    # 9 c / 16 sums of sixteen products are each rounded once, and so are a handful of sums behind them; the three products of thirds that
    # are left out are at most 3 * 2^-25 of theirs
    bound = (9 * c / 16 + 16) * 2.0 ** -24 * (scale + np.abs(bias) + np.abs(res))
    assert (np.abs(run(ctx, x, wt, pad, bias) - (want + bias)) <= bound).all()
    got = run(ctx, x, wt, pad, bias, res, ks=k, act=1, post_relu=1)
    assert (np.abs(got - np.maximum(np.maximum(want + bias, 0) + res, 0)) <= bound).all()


def test_errors_are_no_larger_than_those_of_float32_products(ctx):
    """2-norm against 64 bits, over layers whose float32 products (a filter of 3 x 4 with a column of zeros runs on those) add the same numbers."""
    r = np.random.default_rng(1)
    for c in (16, 64, 256, 512):
        for x in (r.standard_normal((1, 12, 20, c)), r.random((1, 12, 20, c))):
            x, wt = x.astype(np.float32), r.normal(0, 0.05, (64, c, 3, 3)).astype(np.float32)
            want, _ = conv64(x, wt, (1, 1, 1, 1))
            d = ctx.conv_desc(1, c, 12, 20, 64, (3, 4), 1, (1, 1, 1, 2), 0, c, 64)
            y = ctx.empty((1, 12, 20, 64), np.float32)
            ctx.conv2d_f32(d, ctx.array(x), ctx.pack_conv_weights(d, hip.F32, np.pad(wt, ((0, 0), (0, 0), (0, 0), (0, 1)))), None, None, y)
            ctx.sync()
            assert np.linalg.norm(run(ctx, x, wt, (1, 1, 1, 1)) - want) <= np.linalg.norm(y.download().reshape(want.shape) - want)


@pytest.mark.parametrize("products", [1, 2, 4])
def test_errors_of_few_products_are_no_larger_than_those_of_float32_products(ctx, tile, products):
    """Pruned filters: `products` weights of each output channel are not zero. One product is rounded once by either, except that a sum of thirds that lies
    within 2^-8 of the middle between two floats may be rounded the other way, by 2^-9 more: less than 1e-3 of the 2-norm. (16 channels: one wave has all of a tile's
    products, so that none of the difference is that of sums in parts.)"""
    r = np.random.default_rng(products)
    mine = theirs = 0
    for _ in range(3):
        x, wt = r.standard_normal((1, 12, 20, 16)).astype(np.float32), np.zeros((64, 144), np.float32)
        for row in wt:
            row[r.permutation(144)[:products]] = r.standard_normal(products)
        wt = wt.reshape(64, 16, 3, 3)
        want, _ = conv64(x, wt, (1, 1, 1, 1))
        d = ctx.conv_desc(1, 16, 12, 20, 64, (3, 4), 1, (1, 1, 1, 2), 0, 16, 64)
        y = ctx.empty((1, 12, 20, 64), np.float32)
        ctx.conv2d_f32(d, ctx.array(x), ctx.pack_conv_weights(d, hip.F32, np.pad(wt, ((0, 0), (0, 0), (0, 0), (0, 1)))), None, None, y)
        ctx.sync()
        mine += np.sum((run(ctx, x, wt, (1, 1, 1, 1)) - want) ** 2)
        theirs += np.sum((y.download().reshape(want.shape) - want) ** 2)
    assert np.sqrt(mine) <= 1.001 * np.sqrt(theirs)


@pytest.mark.parametrize("c,k", [(16, 1), (48, 40), (64, 64), (512, 130)])
def test_weights_packed_on_the_device_are_the_hosts(ctx, c, k):
    r = np.random.default_rng(c + k)
    w = (r.standard_normal((k, c, 3, 3)) * np.exp2(r.integers(-150, 120, (k, c, 3, 3)))).astype(np.float32)
    at = r.random(w.shape)
    w[at < .02], w[(at > .02) & (at < .04)], w[(at > .04) & (at < .06)], w[(at > .06) & (at < .08)] = np.inf, -np.nan, 0., np.float32(-3.4028235e38)
    d = ctx.conv_desc(1, c, 20, 20, k, 3, 1, 1, 0, c, hip.pad_to(k, 32))
    want = ctx.pack_conv_weights(d, hip.F32, w).download().view(np.uint8)
    got = ctx.array(np.full(want.size + 64, 0xa5, np.uint8))
    assert hip.lib().exhip_conv_packs_on_device(ctypes.byref(d), hip.F32) == 1
    hip._check(hip.lib().exhip_conv_pack_weights_device(ctx.h, ctypes.byref(d), hip.F32, ctx.array(w).ptr, got.ptr))
    ctx.sync()
    got = got.download()
    assert (got[-64:] == 0xa5).all() and np.array_equal(got[:-64], want)


def test_infinities_nan_and_the_largest_floats(ctx, tile):
    r = np.random.default_rng(3)
    x, wt = r.standard_normal((2, 9, 11, 32)).astype(np.float32), (r.integers(1, 9, (40, 32, 3, 3)) / 8).astype(np.float32)
    x[0, 4, 4, 3], x[1, 0, 0, 31], x[1, 8, 9, 7] = np.inf, -np.inf, np.nan
    wt[:, 5] *= np.float32(2.0 ** -100)
    x[0, 7, 9, 5] = np.float32(3.4028235e38)  # as a bfloat16 it would be an infinity
    want, scale = conv64(x, wt, (1, 1, 1, 1))
    got = run(ctx, x, wt, (1, 1, 1, 1))
    ok = np.isfinite(want)
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(got[~ok], want[~ok].astype(np.float32), equal_nan=True)
    assert (np.abs(got[ok] - want[ok]) <= 288 * 2.0 ** -24 * scale[ok]).all()


def tiny(r, shape, e):
    return np.ldexp(r.choice([-1., 1.], shape) * r.uniform(1, 2, shape), e).astype(np.float32)


@pytest.mark.parametrize("kind", ["pixels", "one pixel", "weights", "one weight", "products"])
def test_values_that_thirds_do_not_hold(ctx, tile, kind):
    """Operands below 2^-103, the smallest ones no normal numbers, and products of that size: float32 sums, as many as products, in any order."""
    r = np.random.default_rng(11)
    n, h, w, c, k = 2, 9, 11, 80, 40
    x, wt = r.standard_normal((n, h, w, c)), r.standard_normal((k, c, 3, 3))
    if kind == "pixels":
        x, wt = tiny(r, x.shape, r.integers(-146, -100, x.shape)), np.ldexp(wt, 60)
    elif kind == "one pixel":
        x, wt = np.zeros_like(x), np.ldexp(wt, 60)
        x[1, 4, 5, 33] = np.ldexp(1 + 2. ** -12 + 2. ** -23, -118)
    elif kind == "weights":
        x, wt = np.ldexp(x, 60), tiny(r, wt.shape, r.integers(-146, -100, wt.shape))
    elif kind == "one weight":
        x, wt = np.ldexp(x, 60), np.zeros_like(wt)
        wt[7, 70, 1, 2] = np.ldexp(1 + 2. ** -12 + 2. ** -23, -118)
    else:
        x, wt = np.ldexp(x, -58), np.ldexp(wt, -62)
    x, wt = x.astype(np.float32), wt.astype(np.float32)
    want, scale = conv64(x, wt, (1, 1, 1, 1))
    products = 1 if kind in ("one pixel", "one weight") else 9 * c
    assert np.count_nonzero(want)
    assert (np.abs(run(ctx, x, wt, (1, 1, 1, 1)) - want) <= products * (2. ** -24 * scale + 2. ** -150)).all()


@pytest.mark.parametrize("tiny", [False, True])
def test_results_in_the_place_of_the_shortcut(ctx, tile, tiny):
    r = np.random.default_rng(13)
    n, h, w, c, k = 2, 7, 12, 48, 64
    x, wt = (r.standard_normal(s).astype(np.float32) for s in ((n, h, w, c), (k, c, 3, 3)))
    res = r.standard_normal((n, h, w, k)).astype(np.float32)
    if tiny:  # (a tile that is computed again)
        x[:, 3, 4], wt[5, 6] = 2.0 ** -120, 2.0 ** -115
    want, scale = conv64(x, wt, (1, 1, 1, 1))
    d = ctx.conv_desc(n, c, h, w, k, 3, 1, (1, 1, 1, 1), 0, c, k)
    y = ctx.array(res)
    ctx.conv2d_f32(d, ctx.array(x), ctx.pack_conv_weights(d, hip.F32, wt), None, y, y, None)
    ctx.sync()
    assert (np.abs(y.download().reshape(want.shape) - (want + res)) <= (9 * c + 1) * 2.0 ** -24 * (scale + np.abs(res))).all()


PLACES = [
    (plain.ROWS, 0, 2, 32, 6, 10, 44, 3, 1, True),
    (plain.GROUPED, 85, 3, 32, 5, 7, 255, 3, None, False),
    (plain.GROUPED, 3, 1, 16, 4, 4, 12, 3, None, True),
    (plain.SHUFFLED, 32, 2, 32, 5, 6, 128, 3, None, True),
    (plain.SHUFFLED, 6, 1, 32, 3, 5, 24, 3, None, False),
]


@pytest.mark.parametrize("args", PLACES, ids=["rows", "head", "small-head", "shuffled", "shuffled-odd"])
def test_placements(ctx, tile, args):
    """288 products at most, of those that the test of the float32 products has 360 of."""
    plain.test_placements_for_every_tile_and_split(ctx, tile, args)


@pytest.mark.parametrize("act", [3, 4, 5])
def test_activations_of_the_layer_itself(ctx, act):

    case = cases.conv_f32_case(77, 1, 32, 9, 8, 48, 3, 1, 1, act=act)
    d = ctx.conv_desc(1, 32, 9, 8, 48, 3, 1, 1, act, 32, 64)
    y = ctx.empty((1, 9, 8, 64), np.float32)
    x = np.ascontiguousarray(case["x"].transpose(0, 2, 3, 1))
    ctx.conv2d_f32(d, ctx.array(x), ctx.pack_conv_weights(d, hip.F32, case["wt"]), ctx.array(case["bias"]), None, y)
    ctx.sync()
    assert cases.check_value(y.download().reshape(1, 9, 8, 64)[..., :48].transpose(0, 3, 1, 2), cases.oracle_eval(case), 1e-5) == 0
