"""The fp16 pooling pyramid and the Concat behind it as one launch: the values of the layers run one after the other."""
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
