"""A depthwise 3x3 layer and the pointwise layer behind it as one kernel (conv_pw.hip, dw_pw_kernel): the results are those of
the two layers run one after the other, bit for bit."""
import os
import tempfile

import numpy as np
import pytest

from excalibur_amd import hip, mobilenet, modelfile
from excalibur_amd import pipeline as xp

pytestmark = pytest.mark.gpu


@pytest.fixture
def pairs():
    yield lambda value: hip.set_option("dw_pw", value)
    hip.set_option("dw_pw", 1)


NETS = [
    # n, hw, width, blocks: maps of even and odd sizes (strips of four, two and one pixel), tiles that end inside an image and
    # behind the last one, channels up to the kernel's 512, the split form's sums, residual sums, one or two tiles a group
    (1, 64, 16, ((2, 32, 2), (1, 32, 1), (1, 32, 1), (2, 64, 2), (1, 64, 1))),
    (3, 90, 32, ((2, 64, 2), (1, 64, 2), (2, 128, 4), (1, 128, 2))),
    (2, 50, 32, ((1, 32, 4), (2, 160, 4), (1, 160, 2), (2, 256, 2), (1, 256, 2))),
    (24, 80, 32, ((2, 32, 2), (1, 32, 2), (1, 64, 1))),
]


@pytest.mark.parametrize("n,hw,width,blocks", NETS, ids=lambda v: str(v) if isinstance(v, int) else "")
def test_pairs_equal_the_two_layers(pairs, n, hw, width, blocks):
    m = mobilenet.MobileFaceNetF32(hw=hw, width=width, blocks=blocks)
    with tempfile.NamedTemporaryFile(suffix=".racy", delete=False) as f:
        path = f.name
    modelfile.write_model(path, m.blobs)
    pipe = xp.Pipeline(m.topology(), path, 0, "f16")
    os.unlink(path)
    x = np.random.default_rng(hw).integers(0, 256, (n, 3, hw, hw)).astype(np.float16).view(np.uint16)
    got = {}
    for value in (0, 2):
        pairs(value)
        pipe.set_input(x)
        pipe.run()
        got[value] = pipe.get(m.output).view(np.float16)
    assert np.array_equal(got[0].view(np.uint16), got[2].view(np.uint16))
    assert np.isfinite(got[0]).all() and np.count_nonzero(got[0]) > got[0].size // 2
    pipe.close()
