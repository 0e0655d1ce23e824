"""dispatch_handle after requests that fail (marked `gpu`): what a handle and its
context hold, and the next request on the same handle."""
from __future__ import annotations

import struct

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
