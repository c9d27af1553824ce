"""No-GPU checks of the drop-in boundary: both shared libraries load and export every symbol their headers
declare, and the operator registry holds the reference's class names."""
import ctypes
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _declared(header):
    text = open(os.path.join(ROOT, "include", header)).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(ex(?:hip|c)_[a-z0-9_]+)\s*\(", text)))


def test_exhip_exports_every_declared_symbol():
    from excalibur_amd import hip
    L = hip.lib()
    names = _declared("exhip.h")
    assert len(names) >= 40
    for n in names:
        assert hasattr(L, n), f"libexhip.so does not export {n}"


def test_capi_exports_every_declared_symbol():
    from excalibur_amd import pipeline
    L = pipeline.lib()
    names = _declared("excalibur_capi.h")
    assert len(names) >= 10
    for n in names:
        assert hasattr(L, n), f"libexcalibur_hip.so does not export {n}"


@pytest.mark.parametrize("dtype", ["f32", "f16"])
def test_registry_holds_the_reference_class_names(dtype):
    from excalibur_amd import pipeline
    got = set(pipeline.registered_operations(dtype))
    want = {"operation_convolution", "operation_convolutiondepthwise", "operation_pooling", "operation_eltwise",
            "operation_binaryop", "operation_relu", "operation_innerproduct", "operation_split"}
    assert want <= got


def test_argument_errors_need_no_gpu():
    """Descriptor validation and output-size arithmetic run on the host."""
    from excalibur_amd import hip
    L = hip.lib()
    d = hip.Ctx.conv_desc(1, 64, 56, 56, 64, 3, 1, 1, c_stride=64)
    assert hip.Ctx.conv_out_hw(d) == (56, 56)
    assert L.exhip_conv_packed_bytes(ctypes.byref(d), hip.I8) == 9 * 64 * 64
    bad = hip.Ctx.conv_desc(1, 20, 8, 8, 8, 3, 1, 1, c_stride=20)
    assert L.exhip_conv_packed_bytes(ctypes.byref(bad), hip.I8) == 0
    assert b"multiple of 32" in L.exhip_last_error()
    assert hip.Ctx.pool_out_hw(20, 20, 3, 3, 2, 2, 1, 1, 1, 1, 1) == (10, 10)
    assert hip.Ctx.pool_out_hw(14, 14, 3, 3, 2, 2, 0, 0, 0, 0, 0) == (7, 7)
    assert hip.Ctx.pool_out_hw(14, 14, 3, 3, 2, 2, 0, 0, 0, 0, 1) == (6, 6)


def test_stream_slots_and_options_need_no_gpu():
    """The slot of a thread is thread-local state of the host library, and unknown option names are refused."""
    import threading

    from excalibur_amd import pipeline
    L = pipeline.lib()
    assert L.exc_set_stream_slot(3) == 0
    assert L.exc_set_stream_slot(8) == -1 and L.exc_set_stream_slot(-1) == -1
    seen = []

    def other():
        seen.append(L.exc_set_stream_slot(5))  # another thread's slot does not move this one's

    t = threading.Thread(target=other)
    t.start()
    t.join()
    assert seen == [0]
    assert L.exc_set_stream_slot(0) == 0
    with pytest.raises(ValueError):
        pipeline.set_option("no_such_option", 1)
    pipeline.set_option("share_gpu", 0)


ERR_ARG = 10001


def _fused_entry(name, change):
    """The status of a fused entry point for operands that are addresses only, in a process without a GPU: a call that its checks let through ends
    in the runtime's own error."""
    from excalibur_amd import hip
    L = hip.lib()
    ctx = ctypes.create_string_buffer(4096)
    at = {n: 0x10000 * (i + 1) for i, n in enumerate(("x", "wp", "scale", "bias", "mean", "factor", "y", "y_f32"))}
    shape = dict(c=3, c_stride=4, h=16, w=16, k=64, k_stride=64, pool=(4, 4)) if name != "exhip_conv2d_i8_maxpool2x2" else \
        dict(c=64, c_stride=64, h=64, w=64, k=64, k_stride=64, pool=(32, 32))
    fields = {}
    for key, value in change.items():
        if key in at: at[key] = at[key] + value if value else 0
        elif key in shape: shape[key] = value
        else: fields[key] = value
    d = hip.Ctx.conv_desc(1, shape["c"], shape["h"], shape["w"], shape["k"], 3, 1, 1, c_stride=shape["c_stride"], k_stride=shape["k_stride"], fs_out=1.0)
    for key, value in fields.items():
        setattr(d, key, value)
    p = {n: ctypes.c_void_p(v) for n, v in at.items()}
    c, d = ctypes.cast(ctx, ctypes.c_void_p), ctypes.byref(d)
    if name == "exhip_stem_f16":
        return L.exhip_stem_f16(c, d, p["x"], p["mean"], p["factor"], p["wp"], p["bias"], p["y"])
    if name == "exhip_stem_i8":
        return L.exhip_stem_i8(c, d, p["x"], p["mean"], p["factor"], ctypes.c_float(1.0), p["wp"], p["scale"], p["bias"], p["y"], p["y_f32"])
    return L.exhip_conv2d_i8_maxpool2x2(c, d, *shape["pool"], p["x"], p["wp"], p["scale"], p["bias"], p["y"], p["y_f32"])


@pytest.mark.parametrize("name,change,says", [
    ("exhip_stem_f16", dict(k_stride=32), b"k_stride 32 < k 64"),
    ("exhip_stem_f16", dict(wp=4), b"16-byte aligned"),
    ("exhip_stem_f16", dict(bias=4), b"16-byte aligned"),
    ("exhip_stem_i8", dict(k_stride=32), b"k_stride 32 < k 64"),
    ("exhip_stem_i8", dict(wp=8), b"16-byte aligned"),
    ("exhip_stem_i8", dict(scale=4), b"16-byte aligned"),
    ("exhip_stem_i8", dict(bias=12), b"16-byte aligned"),
    ("exhip_conv2d_i8_maxpool2x2", dict(k_stride=32), b"k_stride 32 < k 64"),
    ("exhip_conv2d_i8_maxpool2x2", dict(x=8), b"16-byte aligned"),
    ("exhip_conv2d_i8_maxpool2x2", dict(wp=4), b"16-byte aligned"),
    ("exhip_conv2d_i8_maxpool2x2", dict(scale=4), b"16-byte aligned"),
    ("exhip_conv2d_i8_maxpool2x2", dict(bias=4), b"16-byte aligned"),
    ("exhip_conv2d_i8_maxpool2x2", dict(pool=(1 << 30, 32)), b"does not fit"),
])
def test_fused_first_layers_and_pooling_check_their_operands(name, change, says):
    """What exhip_conv2d_* refuses, the entry points that run the same layers in one launch refuse with the same error, before any launch."""
    import torch
    if torch.cuda.is_available():
        pytest.skip("the operands are no memory of a GPU")
    assert _fused_entry(name, {}) not in (0, ERR_ARG)   # past the checks: no GPU to launch on
    assert _fused_entry(name, change) == ERR_ARG
    from excalibur_amd import hip
    assert says in hip.lib().exhip_last_error()


@pytest.mark.parametrize("name", ["exhip_stem_f16", "exhip_stem_i8", "exhip_conv2d_i8_maxpool2x2"])
@pytest.mark.parametrize("change", [dict(exact_k=1), dict(post_bn_a=0x900000, post_bn_b=0xa00000), dict(post_bn_b=0xa00000)], ids=["exact", "bn", "half_bn"])
def test_fused_first_layers_and_pooling_leave_joined_layers_alone(name, change):
    """A BatchNorm in the epilogue and writes limited to the layer's channels are the pointwise layers'."""
    import torch
    if torch.cuda.is_available():
        pytest.skip("the operands are no memory of a GPU")
    from excalibur_amd import hip
    assert _fused_entry(name, change) == hip.ERR_UNSUPPORTED
