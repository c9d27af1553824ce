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
