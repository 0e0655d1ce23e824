"""What dispatch_handle keeps, after requests that fail too (marked `gpu`): pinned
memory of a handle and its context, and the next request on the same handle."""
from __future__ import annotations

import struct
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _plan(axc, n_buffers, pc, wg):
    ro, rw = axc.axh.ACCESS_READ_ONLY, axc.axh.ACCESS_READ_WRITE
    return axc.BindingPlan(buffers=[ro] * (n_buffers - 1) + [rw], push_constant_total_bytes=pc,
                           workgroup_size=(wg, 1, 1))


def _address_space():
    """Bytes of address space this process has mapped (pinned memory included)."""
    with open("/proc/self/statm") as f:
        return int(f.read().split()[0]) * 4096


def _widen(ctx, k, h):
    out = ctx.dispatch_handle(k, ((h.size + 255) // 256, 1, 1), [h.tobytes(), b""],
                              [0, 4 * h.size], struct.pack("<I", h.size))
    return np.array_equal(np.frombuffer(out[1], np.float32), h.view(np.float16).astype(np.float32))


def test_refused_launches_keep_nothing(axc):
    """A launch refused on the host after the inputs were staged (push constants
    of 6 bytes, where this library's kernels take whole words): the handle keeps
    one staging buffer however often it happens."""
    print("refused launches", flush=True)
    ctx = axc.HipContext.new()
    h = np.random.default_rng(3).integers(0, 0x7C00, 4 << 20).astype(np.uint16)  # 8 MiB
    good = ctx.prepare_kernel(axc.builtin_code_object(), _plan(axc, 2, 4, 256), 4, "axh_f16_widen")
    bad = ctx.prepare_kernel(axc.builtin_code_object(), _plan(axc, 2, 6, 256), 6, "axh_f16_widen")
    data = h.tobytes()

    def refused():
        with pytest.raises(axc.DispatchError) as e:
            ctx.dispatch_handle(bad, (1, 1, 1), [data, b""], [0, 4], bytes(6))
        assert e.value.variant == "PushConstantSizeMismatch"

    refused()
    assert _widen(ctx, good, h[:4096])
    before = _address_space()
    for _ in range(12):
        refused()
    # every one left 16 MiB of pinned memory behind when it retired its buffer
    assert _address_space() - before < 64 << 20
    assert _widen(ctx, good, h[:4096])
    good.release()
    bad.release()
    ctx.close()


def test_dispatch_after_a_timed_out_one(axc):
    """The same handle, whose first request (a ~10 ms kernel) outlasted the 5 ms
    timeout: its copies may still use the buffer that it was given."""
    print("dispatch after a timeout", flush=True)
    ctx = axc.HipContext.new_with_options(axc.HipContextOptions(fence_timeout_ms=5))
    k = ctx.prepare_kernel(axc.builtin_code_object(), _plan(axc, 1, 4, 64), 4, "axh_spin")
    for _ in range(2):
        with pytest.raises(axc.DispatchError) as e:
            ctx.dispatch_handle(k, (1, 1, 1), [b""], [4], struct.pack("<I", 3000))
        assert e.value.variant == "FenceTimeout"
        ctx.device_synchronize()  # unbounded wait: the bounded kernel ends by itself
        for n in (10, 11):
            out = ctx.dispatch_handle(k, (1, 1, 1), [b""], [4], struct.pack("<I", n))
            assert struct.unpack("<I", out[0])[0] == n
    k.release()
    ctx.close()


def test_buffer_of_a_wait_that_failed(axc):
    """A request made while the stream records a graph cannot wait: its copies are
    recorded or queued, not done, so its buffer is not used again.  The requests
    after it fail before anything is queued (the recording is invalid) and share
    the next buffer."""
    print("dispatch during a capture", flush=True)
    ctx = axc.HipContext.new_with_options(axc.HipContextOptions(fence_timeout_ms=5000))
    h = np.random.default_rng(5).integers(0, 0x7C00, 4 << 20).astype(np.uint16)  # 8 MiB
    k = ctx.prepare_kernel(axc.builtin_code_object(), _plan(axc, 2, 4, 256), 4, "axh_f16_widen")

    def request():
        return ctx.dispatch_handle(k, (1, 1, 1), [h.tobytes(), b""], [0, 1024],
                                   struct.pack("<I", 256))

    want = h[:256].view(np.float16).astype(np.float32).tobytes()
    assert request()[1] == want  # leaves its 16 MiB buffer idle
    with pytest.raises(axc.DispatchError) as e:
        ctx.capture(request)
    assert e.value.variant == "QueueSubmitFailed"
    before = _address_space()
    for _ in range(3):
        with pytest.raises(axc.DispatchError) as e:
            request()
        assert e.value.variant == "StagingCopyFailed"
    grown = _address_space() - before
    print(f"  address space grew by {grown >> 20} MiB", flush=True)
    assert 16 << 20 <= grown < 32 << 20
    k.release()
    ctx.close()


def test_staging_of_a_copy_whose_wait_failed(axc):
    """The same for the staging memory that uploads and downloads share."""
    print("upload during a capture", flush=True)
    ctx = axc.HipContext.new_with_options(axc.HipContextOptions(fence_timeout_ms=5000))
    data = np.random.default_rng(6).integers(0, 256, 8 << 20).astype(np.uint8)
    buf = ctx.alloc(data.nbytes)
    ctx.upload(buf, data)
    with pytest.raises(axc.DispatchError) as e:
        ctx.capture(lambda: ctx.upload(buf, data))
    assert e.value.variant == "QueueSubmitFailed"
    before = _address_space()
    for _ in range(3):
        with pytest.raises(axc.DispatchError) as e:
            ctx.upload(buf, data)
        assert e.value.variant == "StagingCopyFailed"
    grown = _address_space() - before
    print(f"  address space grew by {grown >> 20} MiB", flush=True)
    assert 8 << 20 <= grown < 16 << 20
    buf.close()
    ctx.close()


def test_handles_share_their_pinned_memory(axc):
    """Eight live handles, each with a request of 8 MiB: one staging buffer of 16
    MiB, not one for each (which a handle held for its life)."""
    print("pinned memory of many handles", flush=True)
    ctx = axc.HipContext.new()
    h = np.random.default_rng(4).integers(0, 0x7C00, 4 << 20).astype(np.uint16)
    modes = [axc.axh.ACCESS_READ_ONLY, axc.axh.ACCESS_READ_WRITE]
    handles = [ctx.prepare_kernel(axc.builtin_code_object(),
                                  axc.BindingPlan([a, b], 4, (wg, 1, 1)), 4, "axh_f16_widen")
               for a in modes for b in modes for wg in (128, 256)]
    assert len({k.cache_key for k in handles}) == 8

    def request(k, n):
        ctx.dispatch_handle(k, (1, 1, 1), [h[:n].tobytes(), b""], [0, 4], struct.pack("<I", 256))

    for k in handles:
        request(k, 16)
    before = _address_space()
    for k in handles:
        request(k, h.size)
    grown = _address_space() - before
    print(f"  address space grew by {grown >> 20} MiB", flush=True)
    # eight device buffers of 8 MiB and one staging buffer: 85 MiB; 194 with eight of them
    assert grown < 128 << 20
    for k in handles:
        k.release()
    ctx.close()


def test_concurrent_dispatches_use_buffers_of_their_own(axc):
    print("concurrent dispatches", flush=True)
    ctx = axc.HipContext.new()
    errors = []

    def work(seed):
        try:
            rng = np.random.default_rng(seed)
            # a handle of this thread's own: another access list or launch size
            mode = axc.axh.ACCESS_READ_ONLY if seed & 1 else axc.axh.ACCESS_READ_WRITE
            k = ctx.prepare_kernel(axc.builtin_code_object(),
                                   axc.BindingPlan([mode, axc.axh.ACCESS_READ_WRITE], 4,
                                                   (256, 1, 1)), 4, "axh_f16_widen")
            for _ in range(12):
                n = int(rng.choice([100, 5000, 1 << 17, 3 << 19]))
                assert _widen(ctx, k, rng.integers(0, 0x7C00, n).astype(np.uint16))
            k.release()
        except BaseException as e:  # noqa: BLE001 - reported by the main thread
            errors.append(e)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
    ctx.close()
