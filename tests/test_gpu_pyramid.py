"""The fp16 pooling pyramid and the Concat behind it as one launch, and the float32 one: the values of the layers run one after the other."""
import ctypes
import os
import tempfile

import numpy as np
import pytest

from excalibur_amd import hip, modelfile, topologies
from excalibur_amd import pipeline as xp

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = hip.Ctx(0)
    yield c
    c.close()


def run(ctx, x):
    n, h, w, c = x.shape
    guard = 512
    y = ctx.array(np.full(n * h * w * 4 * c + guard, 0x7bff, np.uint16))
    xd = ctx.array(x)
    rc = hip.lib().exhip_maxpool_pyramid_concat_nhwc_f16(ctx.h, xd.ptr, y.ptr, n, c, h, w)
    if rc == 10002:
        return xd, None
    hip._check(rc)
    ctx.sync()
    got = y.download()
    assert (got[-guard:] == 0x7bff).all()
    return xd, got[:-guard].reshape(n, h, w, 4 * c)


@pytest.mark.parametrize("n,c,h,w", [(1, 8, 1, 1), (2, 24, 3, 5), (1, 8, 1, 40), (5, 16, 13, 7), (1, 8, 45, 45), (17, 256, 20, 20), (2, 2048, 32, 32)])
@pytest.mark.parametrize("values", ["finite", "any"])
def test_the_launch_equals_its_layers(ctx, n, c, h, w, values):
    r = np.random.default_rng(h * w + c)
    x = r.normal(0, 2, (n, h, w, c)).astype(np.float16)
    if values == "any":
        at = r.random(x.shape)
        x[at < .2], x[at > .7] = -np.inf, np.nan
        x[(at > .2) & (at < .25)] = np.inf
    xd, got = run(ctx, x.view(np.uint16))
    layers = [x] + [ctx.maxpool_same_nhwc_f16(xd, k).download().reshape(x.shape).view(np.float16) for k in (5, 9, 13)]
    for level, want in enumerate(layers):
        assert np.array_equal(got[..., level * c:(level + 1) * c].view(np.float16), want, equal_nan=True), level


@pytest.mark.parametrize("n,c,h,w,levels", [(1, 8, 1, 1, 3), (2, 24, 3, 5, 2), (1, 4, 1, 40, 3), (5, 16, 13, 7, 3), (1, 8, 45, 45, 2), (17, 256, 20, 20, 3), (2, 2048, 32, 32, 3), (4, 256, 20, 20, 3), (3, 352, 24, 24, 3)])
@pytest.mark.parametrize("values", ["finite", "any"])
def test_the_float32_launch_equals_its_layers(ctx, n, c, h, w, levels, values):
    r = np.random.default_rng(h * w + c)
    x = r.normal(0, 2, (n, h, w, c)).astype(np.float32)
    if values == "any":
        at = r.random(x.shape)
        x[at < .2], x[at > .7] = -np.inf, np.nan
        x[(at > .2) & (at < .25)] = np.inf
        x[(at > .25) & (at < .5)] = r.choice([-0., 0.], np.count_nonzero((at > .25) & (at < .5)))
    # the input with wider pixels than its own channels, the results side by side
    xd, y = ctx.array(np.pad(x, ((0, 0),) * 3 + ((0, 8),))), ctx.array(np.full(n * h * w * 3 * c + 512, -77, np.float32))
    at = lambda level: ctypes.c_void_p(y.ptr.value + level * c * 4)
    hip._check(hip.lib().exhip_maxpool_pyramid_nhwc_f32(ctx.h, xd.ptr, c + 8, at(0), 3 * c, at(1), 3 * c, at(2) if levels == 3 else None, 3 * c, n, c, h, w))
    ctx.sync()
    got, src, stride = y.download(), xd, c + 8
    assert (got[-512:] == -77).all()
    got = got[:-512].reshape(n, h, w, 3 * c)
    for level in range(levels):
        want = ctx.array(np.zeros(x.shape, np.float32))
        hip._check(hip.lib().exhip_pool2d_nhwc_f32(ctx.h, src.ptr, stride, want.ptr, c, n, c, h, w, h, w, 0, 5, 5, 1, 1, 2, 2, 2, 2, 0))
        ctx.sync()
        src, stride = want, c
        assert got[..., level * c:(level + 1) * c].tobytes() == want.download().reshape(x.shape).tobytes(), level
    assert levels == 3 or (got[..., 2 * c:] == -77).all()


def test_what_the_float32_launch_leaves_to_the_layers(ctx):
    x = ctx.array(np.zeros(43 * 48 * 8, np.float32))
    assert hip.lib().exhip_maxpool_pyramid_nhwc_f32(ctx.h, x.ptr, 8, x.ptr, 8, x.ptr, 8, None, 0, 1, 8, 43, 48) == 10002
    assert hip.lib().exhip_maxpool_pyramid_nhwc_f32(ctx.h, x.ptr, 8, x.ptr, 8, x.ptr, 8, None, 0, 1, 6, 4, 4) == 10002


def test_what_it_leaves_to_the_layers(ctx):
    assert run(ctx, np.zeros((1, 4, 4, 12), np.uint16))[1] is None
    assert run(ctx, np.zeros((1, 43, 48, 8), np.uint16))[1] is None


@pytest.mark.parametrize("n,hw", [(1, 96), (2, 160)])
def test_a_detection_network_with_and_without(n, hw):
    text, outs = topologies.yolov5s_simp(hw, int8=False)
    blobs = modelfile.SeededModel(modelfile.parse_topology(text), 5, default_fs=16.0, gain=2.0).blobs
    with tempfile.NamedTemporaryFile(suffix=".racy", delete=False) as f:
        path = f.name
    modelfile.write_model(path, blobs)
    pipes = [xp.Pipeline(text, path, 0, "f16", fusion=fusion) for fusion in (True, False)]
    os.unlink(path)
    x = np.random.default_rng(hw).integers(0, 256, (n, 3, hw, hw)).astype(np.float16).view(np.uint16)
    got = []
    for pipe in pipes:
        pipe.set_input(x)
        pipe.run()
        got.append([pipe.get(name).view(np.float16) for name in ["467"] + list(outs)])
    for a, b in zip(*got):
        assert a.shape == b.shape and np.array_equal(a, b) and np.ptp(a.astype(np.float32)) > 0
    # a blob that the one launch does not store
    assert np.array_equal(pipes[0].get("465"), pipes[1].get("465"))
