"""The convolutions' packed weights (exhip_conv_pack_weights, host code) against the layout written out with numpy."""
import ctypes
import time

import numpy as np
import pytest

from excalibur_amd import hip
from tests import gpueval

KIND = {hip.I8: np.int8, hip.F16: np.uint16, hip.F32: np.float32}


def pack(d, dtype, w):
    L = hip.lib()
    nbytes = L.exhip_conv_packed_bytes(ctypes.byref(d), dtype)
    assert nbytes > 0, L.exhip_last_error()
    out = np.full(nbytes, 0xa5, np.uint8)
    assert L.exhip_conv_pack_weights(ctypes.byref(d), dtype, w.ctypes.data_as(ctypes.c_void_p), out.ctypes.data_as(ctypes.c_void_p)) == 0
    return out.view(w.dtype)


def lanes(block):
    """A block of 32 output channels x [channels of one 32-byte step] as its 64 lanes hold it: lane rr of either half has channel
    16 * (rr / 4 % 2) + 4 * (rr / 8) + rr % 4, the halves the step's two 16-byte halves."""
    rr = np.arange(32)
    rows = block[(rr // 4 % 2) * 16 + rr // 8 * 4 + rr % 4]
    half = rows.shape[1] // 2
    return np.concatenate([rows[:, :half], rows[:, half:]])


def padded(w, k, c):
    out = np.zeros((k, c) + w.shape[2:], w.dtype)
    out[:w.shape[0], :w.shape[1]] = w
    return out


SHAPES = [(64, 64, 1), (80, 130, 1), (33, 70, 3), (96, 96, (1, 3)), (40, 36, 5), (36, 40, (6, 6))]


@pytest.mark.parametrize("c,k,kernel", SHAPES)
@pytest.mark.parametrize("dtype", [hip.I8, hip.F16, hip.F32])
def test_packed_layout(dtype, c, k, kernel):
    kh, kw = (kernel, kernel) if np.isscalar(kernel) else kernel
    es = np.dtype(KIND[dtype]).itemsize
    w = np.random.default_rng(c + k).integers(1, 120, (k, c, kh, kw)).astype(KIND[dtype])
    cs = gpueval.in_stride(c, dtype, kw)
    d = hip.Ctx.conv_desc(1, c, 20, 20, k, kernel, 1, (kh // 2, kh // 2, kw // 2, kw // 2), 0, cs, hip.pad_to(k, 32))
    got = pack(d, dtype, w)
    step = 32 // es
    if dtype == hip.F32:  # [block][tap][step]
        blocks, steps = (k + 31) // 32, (c + 7) // 8
        full = padded(w, blocks * 32, steps * step)
        want = [lanes(full[b * 32:b * 32 + 32, j * step:j * step + step, r, q]) for b in range(blocks) for r in range(kh) for q in range(kw)
                for j in range(steps)]
        assert np.array_equal(got, np.concatenate(want).ravel())
        return
    # [slab][channel chunk][tap][step of the chunk][block of the slab]; slab and chunk as the planner chose them for the layer
    for slab_blocks in (2, 4):
        for chunk in (64, 32):
            slabs, chunks, per = -(-k // (32 * slab_blocks)), cs * es // chunk, chunk // 32
            if cs * es % chunk or slabs * slab_blocks * chunks * per * kh * kw * 1024 != got.nbytes:
                continue
            full = padded(w, slabs * slab_blocks * 32, cs)
            want = [lanes(full[(s * slab_blocks + b) * 32:(s * slab_blocks + b) * 32 + 32, (cc * per + j) * step:(cc * per + j + 1) * step, r, q])
                    for s in range(slabs) for cc in range(chunks) for r in range(kh) for q in range(kw) for j in range(per) for b in range(slab_blocks)]
            if np.array_equal(got, np.concatenate(want).ravel()):
                return
    raise AssertionError("no slab and chunk give these bytes")


@pytest.mark.parametrize("c,k", [(32, 64), (96, 70), (160, 300)])
def test_int8_pixels_that_end_with_half_a_piece_have_zeros_behind_their_weights(c, k):
    w = np.random.default_rng(c).integers(1, 120, (k, c, 3, 3)).astype(np.int8)
    got = pack(hip.Ctx.conv_desc(1, c, 20, 20, k, 3, 1, 1, 0, c, hip.pad_to(k, 32)), hip.I8, w)
    for slab_blocks in (2, 4):
        pad = 9 * slab_blocks * 1024
        if got.size - pad == -(-k // (32 * slab_blocks)) * slab_blocks * 9 * c // 32 * 1024 and not got[-pad:].any() and got[:-pad].any():
            return
    raise AssertionError("no slab gives this size")


def test_a_pointwise_layer_packs_no_slower_than_its_share_of_a_3x3_layer():
    """The same loop packs both: a weight of a 1x1 layer, whose vectors are plain copies, takes at most twice a 3x3 layer's."""
    def best(kernel):
        w = np.ones((512, 512, kernel, kernel), np.int8)
        d = hip.Ctx.conv_desc(1, 512, 20, 20, 512, kernel, 1, kernel // 2, 0, 512, 512)
        times = []
        for _ in range(25):
            t = time.perf_counter()
            pack(d, hip.I8, w)
            times.append(time.perf_counter() - t)
        return min(times)

    # pack() also fills its result beforehand, the same share of both
    assert best(1) < 2 * best(3) / 9
