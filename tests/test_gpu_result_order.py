"""Results that run ahead of the file's order (pipeline.cpp, hoist_results), and the topologies that keep it: every result
against the CPU oracle's layers taken in the file's order. Weights and inputs are whole numbers, so that sums are exact."""
import os
import tempfile

import numpy as np
import pytest

from excalibur_amd import modelfile as mf
from excalibur_amd import pipeline as xp
from tests import netref

pytestmark = pytest.mark.gpu
C = 8


def conv(bottom, top, k=C, kernel=3, c=C):
    return mf.conv_line("Convolution", top + "_l", bottom, top, k, kernel, 1, kernel // 2, True, k * c * kernel * kernel)


TRUNK = [conv("x1", "t1"), conv("t1", "t2"), conv("t2", "t3"), conv("t3", "t4"), conv("t4", "t5")]
CASES = {
    # a result of a megabyte read off the first blob, listed last: runs right behind it
    "moved": ["Split x_s 1 2 x x0 x1", *TRUNK, conv("x0", "h", 64, 1), "ReLU h_r 1 1 h head"],
    # two such chains behind one layer
    "two": ["Split x_s 1 3 x x0 x1 x2", *TRUNK, conv("x0", "h", 64, 1), "ReLU h_r 1 1 h head", conv("x2", "g", 64, 1), "ReLU g_r 1 1 g other"],
    # without a Split: two readers of one blob
    "shared": [conv("x", "t1"), conv("t1", "t2"), conv("t2", "t3"), conv("t3", "t4"), conv("t4", "t5"), conv("t1", "h", 64, 1), "ReLU h_r 1 1 h head",
               conv("t1", "g", 64, 1), "ReLU g_r 1 1 g other"],
    # a blob written over: the head reads it as it is at the end
    "over": ["Split x_s 1 1 x x1", conv("x1", "t1"), "ReLU t1_r 1 1 t1 t1", conv("t1", "t2"), conv("t2", "t3"), conv("t3", "t4"), conv("t4", "t5"),
             conv("t1", "h", 64, 1), "ReLU h_r 1 1 h head"],
    # what would be a head is read by a later layer
    "read": ["Split x_s 1 2 x x0 x1", *TRUNK, conv("x0", "h"), "ReLU h_r 1 1 h hr", "Eltwise sum 2 1 hr t5 head 0=1"],
}


@pytest.mark.parametrize("fusion", [True, False])
@pytest.mark.parametrize("name", CASES)
def test_results_are_those_of_the_file_s_order(name, fusion):
    text = mf.topology(["Input data 0 1 data 0=64 1=64 2=3 3=0,0,0 4=1", conv("data", "x", c=3)] + CASES[name], name)
    layers = mf.parse_topology(text)
    model = mf.SeededModel(layers, 3)
    r, blobs = np.random.default_rng(4), []
    for L in layers:  # whole numbers instead of the seeded weights
        if L.kind == "Convolution":
            w = r.integers(-1, 2, model.weights[L.name]["w"].shape).astype(np.float32)
            b = r.integers(-3, 4, w.shape[0]).astype(np.float32)
            model.weights[L.name] = {"w": w, "bias": b}
            blobs.append(mf.conv_blob_f32(w, b))
    with tempfile.NamedTemporaryFile(suffix=".racy", delete=False) as f:
        path = f.name
    mf.write_model(path, blobs)
    p = xp.Pipeline(text, path, 0, fusion=fusion)
    os.unlink(path)
    read = {b for L in layers for b in L.bottoms}
    results = [t for L in layers for t in L.tops if t not in read]
    try:
        for seed in (5, 6):
            x = np.random.default_rng(seed).integers(-2, 3, (1, 3, 64, 64)).astype(np.float32)
            want = netref.evaluate(layers, model.weights, x)
            p.set_input(x)
            p.run()
            for o in sorted(results, reverse=bool(seed % 2)):
                assert np.abs(want[o]).max() < 1 << 24 and np.ptp(want[o]) > 0
                assert np.array_equal(p.get(o), want[o]), o
    finally:
        p.close()
