"""The split form of the kernel without staging (conv_pw.hip: four waves share a tile's k-steps): int8 results are those of the
unsplit kernels byte for byte, fp16 sums run in another fixed order."""
import numpy as np
import pytest

from excalibur_amd import hip
from tests import cases, gpueval

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = hip.Ctx(0)
    yield c
    c.close()


@pytest.fixture
def options():
    defaults = dict(pw_split=1, direct=1, pw=1)
    yield lambda name, value: hip.set_option(name, value)
    for name, value in defaults.items():
        hip.set_option(name, value)


SHAPES = [
    # seed, n, c, h, w, k, kernel, stride, pad
    (950, 1, 32, 3, 5, 64, 1, 1, 0),       # one k-step for four waves
    (951, 1, 96, 7, 9, 96, 1, 1, 0),       # three: a wave without one; a half-empty channel pair
    (952, 2, 256, 13, 11, 255, 1, 1, 0),   # a head; ragged last tile
    (953, 1, 1056, 6, 6, 64, 1, 1, 0),     # 33 steps: runs of 8 and 9, around what is in flight at once
    (954, 1, 64, 12, 13, 64, 3, 1, 1),     # two steps a tap
    (955, 2, 96, 11, 10, 160, 3, 2, 1),    # 32-byte chunks for int8
    (956, 1, 256, 20, 20, 256, 3, 1, 1),   # 72 / 144 steps, runs that begin in the middle of a row
    (957, 1, 128, 9, 8, 64, (1, 3), 1, (0, 0, 1, 1)),
    (958, 1, 64, 10, 10, 64, 5, 1, 0),     # 25 taps, no padding
]


@pytest.mark.parametrize("shortcut", [0, 1])
@pytest.mark.parametrize("args", SHAPES, ids=[f"s{a[0]}" for a in SHAPES])
def test_int8_split_equals_unsplit(ctx, options, args, shortcut):
    seed, n, c, h, w, k, kernel, stride, pad = args
    case = cases.conv_i8_case(seed, n, c, h, w, k, kernel, stride, pad, act=0)
    d = ctx.conv_desc(n, c, h, w, k, kernel, stride, pad)
    oh, ow = ctx.conv_out_hw(d)
    res = np.random.default_rng(seed).uniform(-2, 2, (n, oh, ow, hip.pad_to(k, 32))).astype(np.float32) if shortcut else None
    kw = dict(fs_out=np.float32(9.7), residual=res, post_relu=shortcut, want=("nhwc",), post_op=None if shortcut else "hardswish", post_alpha=1 / 6, post_beta=.5)
    options("pw_split", 0)
    want = gpueval.conv_i8(ctx, case, **kw)
    options("pw_split", 2)
    got = gpueval.conv_i8(ctx, case, **kw)
    for name in ("nhwc", "i8"):
        assert np.array_equal(got[name], want[name]), name
    assert np.count_nonzero(got["i8"]) > got["i8"].size // 8


@pytest.mark.parametrize("args", SHAPES, ids=[f"s{a[0]}" for a in SHAPES])
def test_fp16_split_against_the_oracle(ctx, options, args):
    seed, n, c, h, w, k, kernel, stride, pad = args
    case = cases.conv_f32_case(seed, n, c, h, w, k, kernel, stride, pad)
    x16, w16 = case["x"].astype(np.float16), case["wt"].astype(np.float16)
    want = cases.oracle_eval(dict(case, x=x16.astype(np.float32), wt=w16.astype(np.float32)))
    ks = hip.pad_to(k, 32)
    d = ctx.conv_desc(n, c, h, w, k, kernel, stride, pad, case["act"], c, ks)
    oh, ow = ctx.conv_out_hw(d)
    x = ctx.array(np.ascontiguousarray(x16.transpose(0, 2, 3, 1)).view(np.uint16))
    wp, bias = ctx.pack_conv_weights(d, hip.F16, w16.view(np.uint16)), ctx.array(case["bias"])
    options("pw_split", 2)
    options("direct", 2)
    runs = []
    for _ in range(2):
        y = ctx.array(np.full((n, oh, ow, ks), 0x7e00, np.uint16))
        ctx.conv2d_f16(d, x, wp, bias, None, y)
        ctx.sync()
        runs.append(y.download())
    assert np.array_equal(runs[0], runs[1])   # the parts meet in a fixed order
    got = runs[0].view(np.float16).astype(np.float32)
    assert cases.check_value(got[..., :k].transpose(0, 3, 1, 2), want, 2e-3) == 0
    assert not got[..., k:].any()


# An odd number of 32-channel blocks leaves the last pair with one: 80 and 144 channels at a stride of their own, maps whose last
# tile holds one or two pixels.
ODD = [
    # seed, c, h, w, k, kernel
    (960, 128, 1, 1, 80, 1),
    (961, 128, 15, 15, 144, 1),    # 225 pixels: 7 * 32 + 1
    (962, 160, 1, 34, 80, 1),
    (963, 32, 3, 11, 80, 3),       # 33 pixels, nine steps or more
    (964, 128, 2, 1, 144, 3),
    (965, 512, 17, 17, 272, 1),
]


def whole_numbers(seed, c, h, w, k, kernel, bound):
    """Inputs and weights whose sums are exact in every precision, and the layer's result [h, w, k] with padding kernel // 2."""
    rng = np.random.default_rng(seed)
    x, wt = rng.integers(-3, 4, (h, w, c)), rng.integers(-3, 4, (k, c, kernel, kernel))
    p = kernel // 2
    padded = np.pad(x, ((p, p), (p, p), (0, 0)))
    y = sum(padded[r:r + h, q:q + w] @ wt[:, :, r, q].T for r in range(kernel) for q in range(kernel))
    assert np.abs(y).max() < bound
    return x, wt, y


def guarded(ctx, shape, dtype, fill):
    """An array in the middle of a larger one: (the operand, a function that returns its values once nothing beside it changed)."""
    size, row = int(np.prod(shape)), int(shape[-1])
    guard = 64 * row
    whole = ctx.array(np.full(size + 2 * guard, fill, dtype))

    def read():
        got = whole.download()
        assert (got[:guard] == fill).all() and (got[-guard:] == fill).all()
        return got[guard:-guard].reshape(shape)

    return whole.at(guard * np.dtype(dtype).itemsize), read


@pytest.mark.parametrize("shortcut", [0, 1])
@pytest.mark.parametrize("split", [0, 1, 2])
@pytest.mark.parametrize("args", ODD, ids=[f"s{a[0]}" for a in ODD])
def test_fp16_split_of_an_odd_number_of_blocks(ctx, options, args, split, shortcut):
    seed, c, h, w, k, kernel = args
    x, wt, want = whole_numbers(seed, c, h, w, k, kernel, 1900)   # whole numbers up to 2048 are halves
    d = ctx.conv_desc(1, c, h, w, k, kernel, 1, kernel // 2, 0, c, k)
    res = np.random.default_rng(seed + 1).integers(-99, 100, (h, w, k)) if shortcut else None
    options("pw_split", split)
    options("direct", 2)
    y, read = guarded(ctx, (h, w, k), np.uint16, 0x7e00)
    xd, wp = ctx.array(x.astype(np.float16).view(np.uint16)), ctx.pack_conv_weights(d, hip.F16, wt.astype(np.float16).view(np.uint16))
    rd = ctx.array(res.astype(np.float16).view(np.uint16)) if shortcut else None
    ctx.conv2d_f16(d, xd, wp, None, rd, y)
    ctx.sync()
    assert np.array_equal(read().view(np.float16).astype(np.int64), want + res if shortcut else want)


@pytest.mark.parametrize("shortcut", [0, 1])
@pytest.mark.parametrize("split", [0, 1, 2])
@pytest.mark.parametrize("args", ODD, ids=[f"s{a[0]}" for a in ODD])
def test_int8_split_of_an_odd_number_of_blocks(ctx, options, args, split, shortcut):
    seed, c, h, w, k, kernel = args
    x, wt, want = whole_numbers(seed, c, h, w, k, kernel, 1 << 20)
    d = ctx.conv_desc(1, c, h, w, k, kernel, 1, kernel // 2, 0, c, k, fs_out=0.25)
    res = np.random.default_rng(seed + 1).integers(-99, 100, (h, w, k)) if shortcut else None
    options("pw_split", split)
    options("direct", 2)
    options("pw", 2)
    y_f, read_f = guarded(ctx, (h, w, k), np.float32, np.float32(7))
    y_q, read_q = guarded(ctx, (h, w, k), np.int8, 77)
    xd, wp = ctx.array(x.astype(np.int8)), ctx.pack_conv_weights(d, hip.I8, wt.astype(np.int8))
    rd = ctx.array(res.astype(np.float32)) if shortcut else None
    ctx.conv2d_i8(d, xd, wp, ctx.array(np.ones(k, np.float32)), None, rd, y_q, y_f)
    ctx.sync()
    want = want + res if shortcut else want
    assert np.array_equal(read_f().astype(np.int64), want)
    t = want * 0.25
    assert np.array_equal(read_q().astype(np.int64), np.clip(np.trunc(t + np.copysign(0.5, t)), -128, 127).astype(np.int64))


# Pairs of k-steps: 64 bytes of a pixel's tap at a time, of one packed chunk or (32-byte chunks, even in number) of two.
PAIRS = [
    # seed, n, c, h, w, k, kernel, stride, pad
    (970, 2, 64, 9, 11, 64, 3, 2, 1),              # int8: two chunks, nine pairs
    (971, 1, 128, 14, 9, 96, 3, 2, (0, 1, 1, 0)),  # uneven padding, three blocks
    (972, 1, 192, 8, 8, 64, (2, 3), 2, 1),         # six chunks: waves that begin in the middle of one
    (973, 3, 128, 7, 5, 160, 1, 2, 0),             # one tap, every other pixel
    (974, 1, 64, 1, 3, 64, 1, 1, 0),               # a single pair for four waves (int8)
    (975, 1, 64, 33, 1, 64, 3, 1, 1),              # a column: the outer taps of every row outside; 33 pixels
    (976, 1, 320, 6, 7, 64, 3, 1, 1),              # 90 steps: waves of 22 and 24
]


@pytest.mark.parametrize("shortcut", [0, 1])
@pytest.mark.parametrize("args", PAIRS, ids=[f"s{a[0]}" for a in PAIRS])
def test_int8_pairs_of_steps(ctx, options, args, shortcut):
    options("direct", 2)
    test_int8_split_equals_unsplit(ctx, options, args, shortcut)


@pytest.mark.parametrize("args", PAIRS, ids=[f"s{a[0]}" for a in PAIRS])
def test_fp16_pairs_of_steps(ctx, options, args):
    test_fp16_split_against_the_oracle(ctx, options, args)
