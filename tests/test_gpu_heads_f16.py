"""fp16 detection heads, 1x1 convolution -> Reshape of its channels into groups -> Transpose, as one launch: against whole numbers (sums of up to 64
products of at most 2 are exact in half); and the chains that stay three layers."""
import os
import tempfile

import numpy as np
import pytest

from excalibur_amd import modelfile as mf
from excalibur_amd import pipeline as xp

pytestmark = pytest.mark.gpu


def head(c, k, groups, hw, act=0):
    return [mf.conv_line("Convolution", "h_l", "x", "h", k, 1, 1, 0, True, k * c, 1, act=act), f"Reshape r_l 1 1 h r 0={hw} 1={k // groups} 2={groups}"]


CASES = {
    # name: images, channels in and out, groups, height, width, lines behind the Reshape, whether one launch does the three
    "pixels of two images in a tile": (2, 32, 18, 3, 5, 7, ["Transpose t_l 1 1 r out 0=1,0,2"], True),
    "ragged blocks": (3, 64, 255, 3, 13, 11, ["Transpose t_l 1 1 r out 0=1,0,2"], True),
    "one group": (1, 16, 40, 1, 9, 33, ["Transpose t_l 1 1 r out 0=1,0,2"], True),
    "groups of one": (2, 48, 32, 32, 8, 8, ["Transpose t_l 1 1 r out 0=1,0,2"], True),
    "a megabyte, layers behind it": (2, 32, 255, 3, 40, 40, ["Transpose t_l 1 1 r out 0=1,0,2", "ReLU a1 1 1 x z1", "ReLU a2 1 1 z1 z2", "ReLU a3 1 1 z2 z3", "ReLU a4 1 1 z3 z4"], True),
    "channels off the step": (1, 24, 18, 3, 6, 6, ["Transpose t_l 1 1 r out 0=1,0,2"], False),
    "another reader of the Reshape": (1, 32, 18, 3, 6, 6, ["Transpose t_l 1 1 r out 0=1,0,2", "ReLU a1 1 1 r z1"], False),
    "another reader of the convolution": (1, 32, 18, 3, 6, 6, ["Transpose t_l 1 1 r out 0=1,0,2", "ReLU a1 1 1 h z1"], False),
    "no transposition": (1, 32, 18, 3, 6, 6, ["Transpose t_l 1 1 r out 0=0,1,2"], False),
}


@pytest.mark.parametrize("name", CASES)
def test_heads_in_one_launch_equal_their_layers(name):
    n, c, k, groups, h, w, behind, one = CASES[name]
    r = np.random.default_rng(k + c)
    lines = ["ReLU x_l 1 1 y x"] + head(c, k, groups, h * w) + behind
    first = mf.conv_line("Convolution", "y_l", "data", "y", c, 1, 1, 0, True, c * c)  # leaves the NHWC blob that the head reads
    wy, wh, bias = np.eye(c, dtype=np.float32).reshape(c, c, 1, 1), r.integers(-1, 2, (k, c, 1, 1)).astype(np.float32), r.integers(-3, 4, k).astype(np.float32)
    with tempfile.NamedTemporaryFile(suffix=".racy", delete=False) as f:
        f.write(mf.conv_blob_f32(wy, np.zeros(c, np.float32)) + mf.conv_blob_f32(wh, bias))
        path = f.name
    try:
        p = xp.Pipeline(mf.topology([first] + lines), path, 0, "f16")
        for seed in (1, 2):
            x = np.random.default_rng(seed).integers(0, 3, (n, c, h, w)).astype(np.float16)
            want = (np.einsum("kc,nchw->nkhw", wh[:, :, 0, 0], x.astype(np.float32)) + bias[:, None, None]).reshape(n, groups, k // groups, h * w)
            p.forward(x.view(np.uint16))
            assert p.stored("h") != one and p.stored("r") != one
            got = p.get("out").view(np.float16)
            assert np.array_equal(got, want if "0=0,1,2" in behind[0] else want.transpose(0, 1, 3, 2))
            for blob in {"r", "h"} if one else ():  # a blob that was not stored comes from the layers by themselves
                assert p.get(blob).size == want.size
            for j in range(1, len(behind)):
                if behind[j].split()[-2] in ("x", "z1", "z2", "z3"):
                    assert np.array_equal(p.get(f"z{j}").view(np.float16), x)
        p.close()
    finally:
        os.unlink(path)


@pytest.mark.parametrize("kernel,dims", [(3, (400, 85, 3)), (1, (1200, 85, 1))], ids=["3x3", "other groups"])
def test_a_head_that_one_launch_cannot_do_runs_as_layers_that_are_none(kernel, dims):
    """With a filter, or a Reshape that is not one of channels into groups: the convolution makes its NCHW result as it does in front of any other layer."""
    c, k = 256, 255
    r = np.random.default_rng(kernel)
    wy, wh = np.eye(c, dtype=np.float32).reshape(c, c, 1, 1), r.normal(0, .05, (k, c, kernel, kernel)).astype(np.float32)
    x = r.normal(0, 1, (1, c, 20, 20)).astype(np.float16).view(np.uint16)
    lines = [mf.conv_line("Convolution", "y_l", "data", "y", c, 1, 1, 0, True, c * c), "ReLU x_l 1 1 y x",
             mf.conv_line("Convolution", "h_l", "x", "h", k, kernel, 1, kernel // 2, True, wh.size, 1), "Reshape r_l 1 1 h r 0=%d 1=%d 2=%d" % dims]
    with tempfile.NamedTemporaryFile(suffix=".racy", delete=False) as f:
        f.write(mf.conv_blob_f32(wy, np.zeros(c, np.float32)) + mf.conv_blob_f32(wh, r.normal(0, 1, k).astype(np.float32)))
        path = f.name
    got = []
    try:
        for perms in ("1,0,2", "0,1,2"):
            for fusion in (True, False):
                p = xp.Pipeline(mf.topology(lines + [f"Transpose t_l 1 1 r out 0={perms}"], "head"), path, 0, "f16", fusion=fusion)
                p.forward(x)
                out = p.get("out").view(np.float16)
                got.append(out if perms == "0,1,2" else out.transpose(0, 1, 3, 2))
                p.close()
    finally:
        os.unlink(path)
    assert np.isfinite(got[0]).all() and np.ptp(got[0].astype(np.float32)) > 1
    for other in got[1:]:
        assert np.array_equal(got[0], other)
