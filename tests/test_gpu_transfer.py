"""Host <-> device copies (csrc/transfer.hip): every size class and its edges, unaligned ends, uploads queued without a
wait, several threads at once, and results in pinned blocks of the pool."""
import ctypes
import threading

import numpy as np
import pytest

from excalibur_amd import hip
from excalibur_amd import pipeline as xp

pytestmark = pytest.mark.gpu
KB, MB = 1 << 10, 1 << 20


@pytest.fixture(scope="module")
def ctx():
    c = hip.Ctx(0)
    yield c
    c.close()


@pytest.mark.parametrize("size", [1, 15, 4096, 64 * KB, 64 * KB + 1, 256 * KB, 256 * KB + 1, MB, 2 * MB + 5, 4 * MB, 4 * MB + 1, 19 * MB + 3])
@pytest.mark.parametrize("offset", [0, 3])
def test_bytes_arrive_in_both_directions(ctx, size, offset):
    want = np.random.default_rng(size).integers(0, 256, size, dtype=np.uint8)
    d = ctx.array(np.zeros(size + 64, np.uint8))
    at, L = d.at(offset), hip.lib()
    hip._check(L.exhip_memcpy_h2d(ctx.h, at.ptr, want.ctypes.data_as(ctypes.c_void_p), ctypes.c_size_t(size)))
    got = np.zeros(size, np.uint8)
    hip._check(L.exhip_memcpy_d2h(ctx.h, got.ctypes.data_as(ctypes.c_void_p), at.ptr, ctypes.c_size_t(size)))
    assert np.array_equal(got, want)
    whole = d.download()
    assert np.array_equal(whole[offset:offset + size], want) and not whole[:offset].any() and not whole[offset + size:].any()
    d.free()


@pytest.mark.parametrize("size", [512 * KB, 512 * KB + 16, MB + 1, 2 * MB - 1, 4 * MB + 16, 8 * MB + 512 * KB + 7, 12 * MB])
@pytest.mark.parametrize("offset", [0, 16, 8])
def test_uploads_in_steps(ctx, size, offset):
    """An upload's pieces: half a megabyte twice, then as much again as is on its way up to a chunk, by kernel; or (8) whole chunks by the engine."""
    test_bytes_arrive_in_both_directions(ctx, size, offset)


def test_uploads_do_not_wait_and_the_source_may_change_at_once(ctx):
    """More uploads than the staging ring holds, queued behind each other from one reused host buffer."""
    L, n, size = hip.lib(), 40, 900 * KB + 8
    host, parts = np.empty(size, np.uint8), [ctx.empty((size,), np.uint8) for _ in range(n)]
    for i, p in enumerate(parts):
        host[:] = i + 1
        hip._check(L.exhip_upload(ctx.h, p.ptr, host.ctypes.data_as(ctypes.c_void_p), ctypes.c_size_t(size)))
    for i, p in enumerate(parts):
        assert (p.download() == i + 1).all()
        p.free()


def test_threads_with_a_context_each_copy_at_once():
    bad = []

    def work(seed):
        c = hip.Ctx(0)
        for k in range(6):
            want = np.random.default_rng(seed * 10 + k).integers(0, 256, 9 * MB + seed, dtype=np.uint8)
            d = c.array(want)
            if not np.array_equal(d.download(), want):
                bad.append((seed, k))
            d.free()
        c.close()

    threads = [threading.Thread(target=work, args=(s,)) for s in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


def test_results_in_pool_blocks_stay_their_holder_s(ctx):
    xp.lib()
    d = ctx.array(np.arange(MB, dtype=np.float32))
    first = xp._host_array((MB,), np.float32)
    hip._check(hip.lib().exhip_memcpy_d2h(ctx.h, first.ctypes.data_as(ctypes.c_void_p), d.ptr, ctypes.c_size_t(d.nbytes)))
    second = xp._host_array((MB,), np.float32)   # the first block is still held: another one
    second[:] = -1
    assert np.array_equal(first, np.arange(MB, dtype=np.float32))
    view = first[10:20]
    del first
    third = xp._host_array((MB,), np.float32)    # a view holds it as well
    third[:] = -2
    assert np.array_equal(view, np.arange(10, 20, dtype=np.float32))
    assert hip.lib().exhip_host_alloc((1 << 30) + 1) is None   # beyond the bound: the caller's own memory
    d.free()


@pytest.mark.parametrize("size", [5, 64 * KB, 256 * KB + 1, 5 * MB + 3, 19 * MB])
@pytest.mark.parametrize("pinned", [False, True])
def test_a_marked_result_leaves_while_the_stream_goes_on(ctx, size, pinned):
    """What was written before the mark arrives whatever is queued behind it; a mark is recorded anew for the next result."""
    L = hip.lib()
    xp.lib()
    d, other = ctx.empty((size,), np.uint8), ctx.empty((64 * MB,), np.uint8)
    mark = ctypes.c_void_p()
    out = xp._host_array((max(size, MB),), np.uint8) if pinned else np.empty(size, np.uint8)
    kept = None
    for turn in range(3):
        want = np.random.default_rng(size + turn).integers(0, 256, size, dtype=np.uint8)
        hip._check(L.exhip_upload(ctx.h, d.ptr, want.ctypes.data_as(ctypes.c_void_p), ctypes.c_size_t(size)))
        hip._check(L.exhip_mark(ctx.h, ctypes.byref(mark)))
        assert kept is None or mark.value == kept
        kept = mark.value
        for value in range(40):
            hip._check(L.exhip_memset(ctx.h, other.ptr, value, ctypes.c_size_t(other.nbytes)))
        out[:] = 0
        hip._check(L.exhip_memcpy_d2h_from(ctx.h, mark, out.ctypes.data_as(ctypes.c_void_p), d.ptr, ctypes.c_size_t(size)))
        assert np.array_equal(out[:size], want) and not out[size:].any()
        assert (other.download() == 39).all()
    assert L.exhip_memcpy_d2h_from(ctx.h, None, out.ctypes.data_as(ctypes.c_void_p), d.ptr, ctypes.c_size_t(size)) == 10001
    hip._check(L.exhip_mark_destroy(mark))
    d.free()
    other.free()
