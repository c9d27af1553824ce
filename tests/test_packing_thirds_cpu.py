"""The packed weights of float32 3x3 stride-1 layers of whole 16-channel steps: three bfloat16 thirds of each weight."""
import numpy as np
import pytest

from excalibur_amd import hip
from tests.test_packing_cpu import lanes, padded, pack


def value(bits):
    return (bits.astype(np.uint32) << 16).view(np.float32)


@pytest.mark.parametrize("c,k", [(16, 1), (48, 40), (64, 64), (256, 130)])
def test_thirds_add_up_to_the_weight_and_lie_in_fragment_order(c, k):
    r = np.random.default_rng(c + k)
    w = (r.standard_normal((k, c, 3, 3)) * np.exp2(r.integers(-90, 90, (k, c, 3, 3)))).astype(np.float32)
    if k > 1:  # what rounding would carry into an infinity, and what is none of a number
        w[0, :5, 0, 0] = [3.4028235e38, -3.4e38, np.inf, -np.inf, np.nan]
    got = value(pack(hip.Ctx.conv_desc(1, c, 20, 20, k, 3, 1, 1, 0, c, hip.pad_to(k, 32)), hip.F32, w).view(np.uint16))
    blocks = (k + 31) // 32
    got = got.reshape(blocks, c // 16, 9, 3, 64, 8)
    full = padded(w, blocks * 32, c)
    for b in range(blocks):
        for j in range(c // 16):
            for tap in range(9):
                h, m, l = (got[b, j, tap, t].astype(np.float64) for t in range(3))
                want = lanes(full[b * 32:b * 32 + 32, j * 16:j * 16 + 16, tap // 3, tap % 3])
                assert np.array_equal(h + (m + l), want.astype(np.float64), equal_nan=True)
                ok = np.isfinite(want)
                assert (np.abs(m[ok]) <= np.abs(want[ok]) / 128).all() and (np.abs(l[ok]) <= np.abs(want[ok]) / 32768).all()


def test_weights_that_thirds_do_not_hold_are_kept_whole():
    r = np.random.default_rng(3)
    w = r.standard_normal((32, 16, 3, 3)).astype(np.float32)
    at = r.random(w.shape) < .1
    w[at] = np.ldexp(r.uniform(-2, 2, at.sum()), r.integers(-150, -103, at.sum())).astype(np.float32)
    w[1, 1, 1, 1] = np.uint32(0xffffffff).view(np.float32)
    got = pack(hip.Ctx.conv_desc(1, 16, 20, 20, 32, 3, 1, 1, 0, 16, 32), hip.F32, w).view(np.uint16).reshape(9, 3, 64, 8)
    for tap in range(9):
        h, m, l = got[tap]
        want = lanes(w[:, :, tap // 3, tap % 3]).view(np.uint32)
        size = want & 0x7fffffff
        whole = (size > 0) & (size < 0x0c000000) | (size > 0x7f800000)
        assert whole.any() and np.array_equal(h == 0x7fff, whole)
        assert np.array_equal(m[whole].astype(np.uint32) << 16 | l[whole], want[whole])


@pytest.mark.parametrize("kernel,stride,c", [(3, 2, 64), (3, 1, 24), (1, 1, 64), ((1, 3), 1, 64)])
def test_other_layers_keep_whole_floats(kernel, stride, c):
    kh, kw = (kernel, kernel) if np.isscalar(kernel) else kernel
    w = np.ones((32, c, kh, kw), np.float32)
    assert pack(hip.Ctx.conv_desc(1, c, 20, 20, 32, kernel, stride, 0, 0, c, 32), hip.F32, w).size == (c + 7) // 8 * 8 * kh * kw * 32
