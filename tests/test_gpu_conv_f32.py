"""The float32 convolution kernel (conv_f32.hip): every wave tile and split of its list on ragged shapes, against the CPU
oracle's layers; and what surrounds the products -- pad channels, odd channel strides, four-channel pixels, the shortcut."""
import ctypes

import numpy as np
import pytest

from excalibur_amd import hip
from oracle import port
from tests import cases

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = hip.Ctx(0)
    yield c
    c.close()


@pytest.fixture(params=range(9))
def tile(request):
    hip.set_option("f32_tile", request.param)
    yield request.param
    hip.set_option("f32_tile", 0)


SHAPES = [
    # seed, n, c, h, w, k, kernel, stride, pad, c_stride, k_stride, shortcut
    (900, 1, 8, 1, 1, 1, 1, 1, 0, 8, 1, False),             # one pixel, one step, one channel: splits find too few steps
    (901, 2, 24, 9, 7, 33, 3, 1, 1, 24, 33, True),          # ragged pixels and channels, rows without 16-byte alignment
    (902, 1, 3, 17, 19, 40, 3, 2, 1, 4, 64, False),         # 16-byte pixels (two taps a step), a pad block and pad channels
    (903, 1, 4, 12, 11, 32, (1, 4), 1, 0, 4, 32, False),    # the same with an even row of taps
    (904, 3, 40, 13, 13, 255, 1, 1, 0, 48, 256, True),      # a head: one pad channel
    (905, 2, 72, 10, 14, 96, 1, 2, 0, 72, 96, False),       # strided 1x1: single taps, never outside
    (906, 1, 64, 20, 21, 64, 3, 1, 1, 64, 64, True),        # 72 steps
    (907, 1, 16, 15, 15, 32, 9, 2, 4, 16, 32, False),       # 81 taps
    (908, 1, 136, 6, 5, 160, (2, 3), 1, (0, 1, 2, 0), 136, 160, True),  # uneven padding
]


@pytest.mark.parametrize("args", SHAPES, ids=[f"s{a[0]}" for a in SHAPES])
def test_conv_f32_tiles_and_splits(ctx, tile, args):
    seed, n, c, h, w, k, kernel, stride, pad, cs, ks, shortcut = args
    case = cases.conv_f32_case(seed, n, c, h, w, k, kernel, stride, pad, act=0)
    want = cases.oracle_eval(case)
    r = np.random.default_rng(seed)
    res = r.uniform(-1, 1, want.shape).astype(np.float32)
    d = ctx.conv_desc(n, c, h, w, k, kernel, stride, pad, 0, cs, ks, int(shortcut))
    oh, ow = ctx.conv_out_hw(d)
    x = np.zeros((n, h, w, cs), np.float32)
    x[..., :c] = case["x"].transpose(0, 2, 3, 1)
    guard = 64  # floats behind the tensor that must keep their value
    y = ctx.array(np.full(n * oh * ow * ks + guard, 7.0, np.float32))
    planar = ctx.array(np.full(want.size + guard, 7.0, np.float32))
    rd = None
    if shortcut:
        padded = np.zeros((n, oh, ow, ks), np.float32)
        padded[..., :k] = res.transpose(0, 2, 3, 1)
        rd = ctx.array(padded)
        want = port.relu(port.binaryop_add(want, res))
    ctx.conv2d_f32(d, ctx.array(x), ctx.pack_conv_weights(d, hip.F32, case["wt"]), ctx.array(case["bias"]), rd, y, planar)
    ctx.sync()
    got, flat = y.download(), planar.download()
    assert (got[-guard:] == 7.0).all() and (flat[-guard:] == 7.0).all()
    got = got[:-guard].reshape(n, oh, ow, ks)
    assert cases.check_value(got[..., :k].transpose(0, 3, 1, 2), want, 1e-5) == 0
    assert not got[..., k:].any()
    assert np.array_equal(flat[:-guard].reshape(want.shape), got[..., :k].transpose(0, 3, 1, 2))


class Place(ctypes.Structure):
    _fields_ = [(name, ctypes.c_int) for name in ("layout", "group", "residual_stride", "residual_shift", "bn_relu")]


ROWS, GROUPED, SHUFFLED = range(3)
PLACES = [
    # layout, group, n, c, h, w, k, kernel, shift of the shortcut's map (None: no shortcut), BatchNorm
    (ROWS, 0, 2, 40, 6, 10, 44, 3, 1, True),        # written into 44 of 64 channels
    (GROUPED, 85, 3, 72, 5, 7, 255, 1, None, False),  # a detection head, blocks that cross groups
    (GROUPED, 3, 1, 256, 4, 4, 12, 1, None, True),
    (SHUFFLED, 32, 2, 64, 5, 6, 128, 1, None, True),  # whole blocks per position
    (SHUFFLED, 6, 1, 136, 3, 5, 24, 1, None, False),
]


@pytest.mark.parametrize("args", PLACES, ids=["rows", "head", "small-head", "shuffled", "shuffled-odd"])
def test_placements_for_every_tile_and_split(ctx, tile, args):
    """Results in their groups, as an upsampled map or inside a wider tensor, against the definition in 64 bits. The layers sum at most
    360 float32 products of at most 1 each to results of order 1: 360 roundings of 2^-24 are 2.2e-5."""
    layout, group, n, c, h, w, k, kernel, shift, bn = args
    r = np.random.default_rng(k + c)
    x, wt = r.uniform(-1, 1, (n, h, w, c)).astype(np.float32), r.normal(0, 0.1, (k, c, kernel, kernel)).astype(np.float32)
    bias, slope = (r.normal(0, 0.5, k).astype(np.float32) for _ in range(2))
    a, b = (r.normal(0, 1, k).astype(np.float32) for _ in range(2))
    ks = 64 if layout == ROWS else group if layout == SHUFFLED else 256
    pd = kernel // 2
    d = ctx.conv_desc(n, c, h, w, k, kernel, 1, pd, 1, c, ks, residual_last=1, exact_k=int(layout == ROWS))
    da, db, ds = ctx.array(a), ctx.array(b), ctx.array(slope)
    if bn:
        d.post_bn_a, d.post_bn_b = da.ptr, db.ptr
    d.post_op, d.post_slope = 16, ds.ptr  # EXHIP_POST_PRELU
    xp = np.pad(x.astype(np.float64), ((0, 0), (pd, pd), (pd, pd), (0, 0)))
    want = sum(xp[:, i:i + h, j:j + w] @ wt[:, :, i, j].T.astype(np.float64) for i in range(kernel) for j in range(kernel)) + bias
    want = np.maximum(want, 0)
    if bn:
        want = b * want + a.astype(np.float64)
    want = np.where(want >= 0, want, slope * want)
    res = None
    if shift is not None:
        small = r.uniform(-1, 1, (n, h >> shift, w >> shift, 48)).astype(np.float32)
        res = ctx.array(small)
        want = want + small[..., :k].repeat(1 << shift, 1).repeat(1 << shift, 2)
    if layout == ROWS:
        expect = np.full((n, h, w, ks), 7.0)
        expect[..., :k] = want
    elif layout == GROUPED:
        expect = want.reshape(n, h * w, k // group, group).transpose(0, 2, 1, 3)
    else:
        expect = want.reshape(n, h, w, 2, 2, group).transpose(0, 1, 3, 2, 4, 5)
    y = ctx.array(np.full(expect.size + 64, 7.0, np.float32))
    place = Place(layout, group, 48, shift or 0, 0)
    wp = ctx.pack_conv_weights(d, hip.F32, wt)
    hip._check(hip.lib().exhip_conv2d_f32_placed(ctx.h, ctypes.byref(d), ctypes.byref(place), ctx.array(x).ptr, wp.ptr, ctx.array(bias).ptr,
                                                 res.ptr if res else None, y.ptr, None))
    ctx.sync()
    got = y.download()
    assert (got[-64:] == 7.0).all()
    assert np.abs(got[:-64].reshape(expect.shape) - expect).max() < 2.2e-5 * max(1.0, np.abs(want).max())


PAIRS = [  # 1x1 layers that take the pixels two steps at a time
    (910, 1, 16, 9, 5, 40, 1, 1, 0, 16, 64, False),      # a single pair for all waves
    (911, 3, 48, 13, 13, 96, 1, 1, 0, 48, 96, True),     # three pairs
    (912, 2, 80, 11, 7, 33, 1, 2, 0, 96, 33, False),     # every other pixel, five pairs of a wider pixel, unaligned rows
    (913, 1, 272, 7, 7, 64, 1, 1, 0, 272, 64, True),     # 34 steps: runs of eight and ten
]


@pytest.mark.parametrize("args", PAIRS, ids=[f"s{a[0]}" for a in PAIRS])
def test_conv_f32_pairs_of_steps(ctx, tile, args):
    test_conv_f32_tiles_and_splits(ctx, tile, args)


def test_the_plain_entry_refuses_what_only_the_placed_one_does(ctx):
    """A BatchNorm in the epilogue and writes limited to the layer's own channels: refused, nothing written."""
    c, k, hw = 32, 32, 5
    x, w = ctx.array(np.ones((1, hw, hw, c), np.float32)), np.ones((k, c, 1, 1), np.float32)
    a, b = ctx.array(np.zeros(k, np.float32)), ctx.array(np.ones(k, np.float32))
    y = ctx.array(np.full((1, hw, hw, k), 7.0, np.float32))
    plain = ctx.conv_desc(1, c, hw, hw, k, 1)
    wp = ctx.pack_conv_weights(plain, hip.F32, w)
    for d in (ctx.conv_desc(1, c, hw, hw, k, 1, post_bn=(a, b)), ctx.conv_desc(1, c, hw, hw, k, 1, exact_k=1)):
        with pytest.raises(hip.ExhipError, match="10002"):
            ctx.conv2d_f32(d, x, wp, None, None, y)
    ctx.sync()
    assert (y.download() == 7.0).all()
    ctx.conv2d_f32(plain, x, wp, None, None, y)
    ctx.sync()
    assert (y.download() == c).all()


def test_the_fp16_entry_refuses_them_too(ctx):
    c, k, hw = 32, 32, 5
    x, w = ctx.array(np.ones((1, hw, hw, c), np.float16).view(np.uint16)), np.ones((k, c, 1, 1), np.float16).view(np.uint16)
    a, b = ctx.array(np.zeros(k, np.float32)), ctx.array(np.ones(k, np.float32))
    y = ctx.array(np.full((1, hw, hw, k), 0x4700, np.uint16))
    wp = ctx.pack_conv_weights(ctx.conv_desc(1, c, hw, hw, k, 1), hip.F16, w)
    for d in (ctx.conv_desc(1, c, hw, hw, k, 1, post_bn=(a, b)), ctx.conv_desc(1, c, hw, hw, k, 1, exact_k=1)):
        with pytest.raises(hip.ExhipError, match="10002"):
            ctx.conv2d_f16(d, x, wp, None, None, y)
    ctx.sync()
    assert (y.download() == 0x4700).all()
