"""The float32 plan (pipeline.cpp, build_float_plan): NHWC tensors between the layers, Concats written in place, layers folded
into the convolutions around them. Every blob it gives equals the per-layer executor's bit for bit."""
import os
import tempfile

import numpy as np
import pytest

from excalibur_amd import modelfile as mf
from excalibur_amd import pipeline as xp

pytestmark = pytest.mark.gpu


def network(focus):
    r = np.random.default_rng(71)
    lines, blobs = ["Input data 0 1 data 0=32 1=32 2=3 3=3,2,1 4=0.5"], []

    def conv(bottom, top, cin, k, kernel=1, stride=1, groups=1, act=0):
        w = r.normal(0, np.sqrt(2.0 / (cin // groups * kernel * kernel)), (k, cin // groups, kernel, kernel)).astype(np.float32)
        kind = "Convolution" if groups == 1 else "ConvolutionDepthWise"
        lines.append(mf.conv_line(kind, top + "_l", bottom, top, k, kernel, stride, kernel // 2, True, w.size, groups, act=act))
        blobs.append(mf.conv_blob_f32(w, r.normal(0, 0.5, (k,)).astype(np.float32)))

    def batchnorm(bottom, top, c):
        lines.append(f"BatchNorm {top}_l 1 1 {bottom} {top} 0={c}")
        blobs.append(b"".join(mf.floats_blob(v.astype(np.float32)) for v in (r.normal(1, .2, c), r.normal(0, .5, c), r.uniform(.5, 2, c), r.normal(0, .5, c))))

    def prelu(bottom, top, c):
        lines.append(f"PReLU {top}_l 1 1 {bottom} {top} 0={c}")
        blobs.append(mf.floats_blob(r.uniform(-.5, .5, max(1, c)).astype(np.float32)))

    def split(bottom, n):
        lines.append(f"Split {bottom}_sp 1 {n} {bottom} " + " ".join(f"{bottom}{j}" for j in range(n)))

    def add(kind, bottoms, top, params=""):
        lines.append(f"{kind} {top}_l {len(bottoms)} 1 {' '.join(bottoms)} {top} {params}")

    if focus:
        add("YoloV5Focus", ["data"], "front")
        conv("front", "c0", 12, 24, 3)
    else:
        conv("data", "c0", 3, 24, 3, 2)
    prelu("c0", "p0", 24)
    conv("p0", "d1", 24, 24, 3, 1, groups=24)           # depthwise + PReLU, shared slope
    prelu("d1", "p1", 1)
    conv("p1", "d2", 24, 24, 3, 2, groups=24)           # depthwise + ReLU, stride 2
    add("ReLU", ["d2"], "r2")
    split("r2", 3)
    conv("r20", "c3", 24, 20)                            # 20 channels: pad channels travel with the tensor
    add("HardSwish", ["c3"], "a3", "0=1.666667e-01 1=5.000000e-01")
    conv("a3", "c4", 20, 24, 3)
    add("Eltwise", ["r21", "c4"], "s4", "0=1")           # sum behind a plain convolution, ReLU behind the sum
    add("ReLU", ["s4"], "s4r")
    split("s4r", 4)
    conv("s4r0", "y1", 24, 16)                           # Concat -> BatchNorm -> LeakyRelu in two plain producers
    conv("r22", "y2", 24, 32)
    add("Concat", ["y1", "y2"], "cat", "0=-1")
    batchnorm("cat", "catbn", 48)
    add("LeakyRelu", ["catbn"], "cata", "0=1.000000e-01")
    conv("cata", "c5", 48, 32, act=1)
    split("c5", 3)
    for j, k in enumerate((5, 9)):                       # pools of a pool, written into a Concat beside their input's copy
        add("Pooling", ["c50" if j else "c51"], f"mp{k}", f"0=0 1={k} 11={k} 2=1 12=1 3={k // 2} 13={k // 2} 14={k // 2} 15={k // 2} 5=1 4=0")
    add("Concat", ["c52", "mp5", "mp9"], "spp", "0=-1")
    conv("spp", "c6", 96, 24, 3, 2)
    split("c6", 2)
    add("Interp", ["c60"], "up", "0=1 1=2.000000e+00 2=2.000000e+00")
    conv("s4r1", "lat", 24, 24)
    add("BinaryOp", ["up", "lat"], "fpn", "0=0")         # the upsampled map is read through by the sum
    add("Interp", ["c61"], "up2", "0=1 1=2.000000e+00 2=2.000000e+00")
    add("Pooling", ["s4r2"], "av", "0=1 1=3 11=3 2=1 12=1 3=1 13=1 14=1 15=1 5=1 4=0 6=1")
    add("Concat", ["fpn", "up2", "av"], "wide", "0=-1")  # nothing plain about its producers: BatchNorm as a pass over it
    batchnorm("wide", "widebn", 72)
    split("widebn", 3)
    conv("widebn0", "c7", 72, 42, 1)                     # a head: [n][3 x 14] -> [n][3][pixels][14]
    add("Reshape", ["c7"], "hr", "0=64 1=14 2=3")
    add("Transpose", ["hr"], "head", "0=1,0,2")
    wd = r.normal(0, .2, (72, 8, 2, 2)).astype(np.float32)
    lines.append(f"Deconvolution dc1 1 1 widebn1 dc 0=8 1=2 11=2 2=1 12=1 3=2 13=2 4=0 14=0 15=0 16=0 5=1 6={wd.size} 7=1")
    blobs.append(mf.conv_blob_f32(wd, r.normal(0, .5, (8,)).astype(np.float32)))
    batchnorm("dc", "dcbn", 8)
    add("ReLU", ["dcbn"], "dcr")
    w1 = r.normal(0, .5, (8, 1, 2, 2)).astype(np.float32)
    lines.append(f"Deconvolution dc2 1 1 dcr dm 0=1 1=2 11=2 2=1 12=1 3=2 13=2 4=0 14=0 15=0 16=0 5=1 6={w1.size} 7=1")
    blobs.append(mf.conv_blob_f32(w1, r.normal(0, .5, (1,)).astype(np.float32)))
    add("Sigmoid", ["dm"], "map")
    lines.append(mf.pool_line("gap", "widebn2", "gap", 1, global_pool=True))
    wf = r.normal(0, .2, (10, 72)).astype(np.float32)
    lines.append(f"InnerProduct fc 1 1 gap fc 0=10 1=1 2={wf.size}")
    blobs.append(mf.fc_blob_f32(wf, r.normal(0, .5, (10,)).astype(np.float32)))
    return lines, blobs, ["head", "map", "fc", "s4r3"]


@pytest.mark.parametrize("focus", [False, True])
def test_float_plan_equals_the_layers_bit_for_bit(focus):
    lines, blobs, outs = network(focus)
    with tempfile.NamedTemporaryFile(suffix=".racy", delete=False) as f:
        path = f.name
    mf.write_model(path, blobs)
    planned, plain = (xp.Pipeline(mf.topology(lines, "float"), path, 0, fusion=on) for on in (True, False))
    try:
        for n, seed in ((1, 1), (3, 2), (3, 3)):
            x = np.random.default_rng(seed).uniform(-4, 4, (n, 3, 32, 32)).astype(np.float32)
            planned.forward(x)
            plain.forward(x)
            assert planned.stored("head") and not planned.stored("c0") and plain.stored("c0")
            for o in outs:
                got, want = planned.get(o), plain.get(o)
                assert np.isfinite(want).all() and np.ptp(want) > 0
                assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), (o, n)
            assert np.array_equal(planned.get("spp"), plain.get("spp"))  # a blob the plan never made: by the rerun
    finally:
        planned.close()
        plain.close()
        os.unlink(path)


def pooled_slices():
    """Two producers of a Concat whose slices have other readers too: pools of a slice, one of them inside another Concat. No layer
    fixes the input size."""
    r = np.random.default_rng(73)
    lines, blobs = ["Input data 0 1 data 0=32 1=32 2=3 3=0,0,0 4=1"], []

    def conv(bottom, top, cin, k, kernel=1, stride=1, act=0):
        w = r.normal(0, np.sqrt(2.0 / (cin * kernel * kernel)), (k, cin, kernel, kernel)).astype(np.float32)
        lines.append(mf.conv_line("Convolution", top + "_l", bottom, top, k, kernel, stride, kernel // 2, True, w.size, act=act))
        blobs.append(mf.conv_blob_f32(w, r.normal(0, 0.5, (k,)).astype(np.float32)))

    conv("data", "c0", 3, 16, 3, 2)
    lines.append("Split c0_s 1 2 c0 c00 c01")
    conv("c00", "y1", 16, 24, act=1)
    conv("c01", "y2", 16, 40, 3)
    lines.append("Split y1_s 1 3 y1 y10 y11 y12")
    lines.append("Concat cat_l 2 1 y10 y2 cat 0=-1")
    lines.append(mf.pool_line("mp", "y11", "mp", 0, 3, 1, 1))
    lines.append(mf.pool_line("av", "y12", "av", 1, 3, 2, 1, count_include_pad=1))
    conv("cat", "c1", 64, 24)
    lines.append("Concat cat2_l 2 1 c1 mp cat2 0=-1")
    conv("cat2", "c2", 48, 16, 3)
    return lines, blobs, ["c2", "av"]


@pytest.fixture
def pair():
    lines, blobs, outs = pooled_slices()
    with tempfile.NamedTemporaryFile(suffix=".racy", delete=False) as f:
        path = f.name
    mf.write_model(path, blobs)
    pipes = [xp.Pipeline(mf.topology(lines, "slices"), path, 0, fusion=on) for on in (True, False)]
    os.unlink(path)
    yield (*pipes, outs)
    for p in pipes:
        p.close()


def inputs(shape, seed):
    return np.random.default_rng(seed).uniform(-2, 2, shape).astype(np.float32)


def test_float_plan_with_alternating_input_sizes(pair):
    planned, plain, outs = pair
    sizes = [(1, 3, 32, 32), (2, 3, 21, 46), (1, 3, 33, 17), (2, 3, 21, 46), (1, 3, 32, 32), (3, 3, 32, 32)]
    for seed, shape in enumerate(sizes):
        x = inputs(shape, seed)
        planned.forward(x)
        plain.forward(x)
        assert not planned.stored("y2") and plain.stored("y2")
        for o in outs:
            got, want = planned.get(o), plain.get(o)
            assert np.array_equal(got.view(np.uint32), want.view(np.uint32)) and np.ptp(want) > 0, (shape, o)


def test_float_plan_replayed_as_a_graph(pair):
    """Every replay against the eager layers, with their work between the replays; another size in the middle."""
    planned, plain, outs = pair
    planned.set_graphs(True)
    for seed, shape in enumerate([(2, 3, 30, 28)] * 4 + [(1, 3, 32, 32)] * 3 + [(2, 3, 30, 28)] * 3):
        x = inputs(shape, 20 + seed)
        planned.forward(x)
        plain.forward(x)
        for o in outs:
            assert np.array_equal(planned.get(o).view(np.uint32), plain.get(o).view(np.uint32)), (seed, o)


def test_float_plan_results_held_across_forwards(pair):
    planned, plain, outs = pair
    shape, want = (2, 3, 40, 36), []
    for seed in range(4):
        x = inputs(shape, 40 + seed)
        planned.set_input(x)
        planned.run_keeping()
        plain.forward(x)
        want.append({o: plain.get(o).copy() for o in outs})
    for o in outs:
        assert np.array_equal(planned.get(o), want[3][o])
        for back in (1, 2, 3):
            assert np.array_equal(planned.get_kept(back, o), want[3 - back][o]), (back, o)


@pytest.mark.parametrize("activation", [True, False], ids=["activation", "batchnorm"])
@pytest.mark.parametrize("reader", ["convolution", "interp", "concat", "larger pool", "result"])
def test_a_concats_inputs_keep_their_values_behind_its_batchnorm(tmp_path, reader, activation):
    """The producers of a Concat that is no plain convolutions' write into the joined tensor; the BatchNorm and activation behind it leave
    those values to their other readers, which run later."""
    r = np.random.default_rng(91)
    lines, blobs = [], []

    def conv(bottom, top, cin, k, kernel=1):
        w = r.normal(0, np.sqrt(2.0 / (cin * kernel * kernel)), (k, cin, kernel, kernel)).astype(np.float32)
        lines.append(mf.conv_line("Convolution", top + "_l", bottom, top, k, kernel, 1, kernel // 2, True, w.size, 1))
        blobs.append(mf.conv_blob_f32(w, r.normal(0, 0.5, (k,)).astype(np.float32)))

    def joined(bottoms, top, c):
        lines.append(f"Concat {top}_l 2 1 {' '.join(bottoms)} {top}k 0=-1")
        lines.append(f"BatchNorm {top}_bn 1 1 {top}k {top if not activation else top + 'b'} 0={c}")
        blobs.append(mf.floats_blob(r.uniform(.5, 1.5, c), r.normal(0, .5, c), r.uniform(.5, 2, c), r.normal(0, .5, c)))
        if activation:
            lines.append(f"LeakyRelu {top}_a 1 1 {top}b {top} 0=1.000000e-01")

    conv("data", "c0", 3, 16, 3)
    lines.append("HardSwish hs 1 1 c0 a0 0=1.666667e-01 1=5.000000e-01")
    lines.append("Split sp0 1 3 a0 a0x a0y a0z")
    lines.append(mf.pool_line("p1_l", "a0x", "p1", 0, 3, 1, 1))
    lines.append("Split sp1 1 2 p1 p1x p1y")
    joined(["p1x", "a0y"], "s2", 32)
    if reader == "larger pool":   # reads the smaller pool's result in place of its own input
        lines.append(mf.pool_line("p5_l", "a0z", "late", 0, 5, 1, 2))
    elif reader == "convolution":
        conv("p1y", "late", 16, 24, 3)
    elif reader == "interp":
        lines.append("Interp up 1 1 p1y late 0=1 1=2.000000e+00 2=2.000000e+00")
    elif reader == "concat":
        joined(["a0z", "p1y"], "late", 32)
    conv("s2", "c3", 32, 16)
    outputs = ["c3", "p1y" if reader == "result" else "late"]
    path = str(tmp_path / "net.racy")
    mf.write_model(path, blobs)
    planned, plain = (xp.Pipeline(mf.topology(lines, "joined"), path, 0, fusion=on) for on in (True, False))
    for seed in (1, 2):
        x = np.random.default_rng(seed).normal(0, 1, (2, 3, 12, 20)).astype(np.float32)
        planned.forward(x)
        plain.forward(x)
        assert not planned.stored("c0") and plain.stored("c0")
        for o in outputs:
            got, want = planned.get(o), plain.get(o)
            assert np.ptp(want) > .5
            assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), o
    planned.close()
    plain.close()


@pytest.mark.parametrize("wider", [False, True])
def test_a_pool_of_a_concat_is_no_level_over_the_pool_it_begins_with(tmp_path, wider):
    """p = pool(a), q = Concat(p, b), r = pool(q): q lies where p does and has no launch of its own, but r has to pool all of q's channels. `wider`: a
    itself is a slice of a tensor with room for that many channels behind it."""
    r = np.random.default_rng(93)
    lines, blobs = [], []

    def conv(bottom, top, cin, k, kernel=1):
        w = r.normal(0, np.sqrt(2.0 / (cin * kernel * kernel)), (k, cin, kernel, kernel)).astype(np.float32)
        lines.append(mf.conv_line("Convolution", top + "_l", bottom, top, k, kernel, 1, kernel // 2, True, w.size, 1))
        blobs.append(mf.conv_blob_f32(w, r.normal(0, 0.5, (k,)).astype(np.float32)))

    conv("data", "c0", 3, 16, 3)
    lines.append("Split sp0 1 2 c0 c00 c01")
    conv("c00", "a", 16, 16)
    conv("c01", "z", 16, 48)
    lines.append("Split sp1 1 " + ("3 a a0 a1 a2" if wider else "2 a a0 a2"))
    conv("a0", "b", 16, 16)
    if wider:
        lines.append("Concat wide_l 2 1 a1 z wide 0=-1")
    lines.append(mf.pool_line("p_l", "a2", "p", 0, 5, 1, 2))
    lines.append("Concat q_l 2 1 p b q 0=-1")
    lines.append("Split sp2 1 2 q q0 q1")
    lines.append(mf.pool_line("r_l", "q0", "r", 0, 5, 1, 2))
    conv("r", "late", 32, 16)
    conv("q1", "early", 32, 16)
    conv("wide" if wider else "z", "rest", 64 if wider else 48, 16)
    path = str(tmp_path / "net.racy")
    mf.write_model(path, blobs)
    planned, plain = (xp.Pipeline(mf.topology(lines, "pools"), path, 0, fusion=on) for on in (True, False))
    for seed in (1, 2, 3):
        x = np.random.default_rng(seed).normal(0, 1, (2, 3, 12, 20)).astype(np.float32)
        planned.forward(x)
        plain.forward(x)
        assert not planned.stored("c0") and plain.stored("c0")
        for o in ("late", "early", "rest"):
            got, want = planned.get(o), plain.get(o)
            assert np.ptp(want) > .5
            assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), (seed, o)
    planned.close()
    plain.close()
