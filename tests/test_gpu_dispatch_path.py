"""The dispatch surface (marked `gpu`): the single-output reference kernels at
the edges of their iterations, and dispatch_handle's copies at the edges of
its staging layout."""
from __future__ import annotations

import struct

import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _plan(axc, n_buffers, pc, wg):
    ro, rw = axc.axh.ACCESS_READ_ONLY, axc.axh.ACCESS_READ_WRITE
    return axc.BindingPlan(buffers=[ro] * (n_buffers - 1) + [rw], push_constant_total_bytes=pc,
                           workgroup_size=(wg, 1, 1))


def _dot(ctx, axc, entry, q, x, n):
    h = ctx.prepare_kernel(axc.builtin_code_object(), _plan(axc, 3, 4, 64), 4, entry)
    out = ctx.dispatch_handle(h, (1, 1, 1), [q.tobytes(), x.tobytes(), bytes(4)], [0, 0, 4],
                              struct.pack("<I", n))
    h.release()
    return np.frombuffer(out[2], np.float32)


@pytest.mark.parametrize("n", [1, 7, 8, 9, 40, 47, 48, 49, 56, 97, 511])
def test_q4k_single_output_iterations(ctx, axc, n):
    """8 superblocks per iteration, 6 iterations in flight."""
    print(f"q4_k single output {n}", flush=True)
    q, x = O.gen_q4k_weights(300 + n, n), O.gen_normal_f32(301 + n, n * 256)
    y = _dot(ctx, axc, "q4km_dequant_matvec", q, x, n)
    yf, ad = O.q4k_matvec_f64(q, x, 1, n)
    rep = O.matvec_tolerance_report(y, O.q4k_matvec(q, x, 1, n), yf, ad, n * 256, 1e-3)
    assert rep["ok"], rep


@pytest.mark.parametrize("n", [1, 15, 16, 17, 63, 64, 65, 192, 255, 256, 257, 321, 4095])
def test_q4_0_single_output_iterations(ctx, axc, n):
    """64 blocks per iteration in groups of 16, 4 iterations in flight."""
    print(f"q4_0 single output {n}", flush=True)
    q, x = O.gen_q4_0_weights(400 + n, n), O.gen_normal_f32(401 + n, n * 32)
    y = _dot(ctx, axc, "q4_0_dequant_matvec", q, x, n)
    yf, ad = O.q4_0_matvec_f64(q, x, 1, n)
    rep = O.matvec_tolerance_report(y, O.q4_0_matvec(q, x, 1, n), yf, ad, n * 32, 1e-3)
    assert rep["ok"], rep


# f16 words whose binding sizes lie around 16-byte pieces, one 4 KiB workgroup,
# the largest size copied by the kernel (2 MiB: 2 n and 4 n bytes), and the
# 32 MiB of one staged request (8 n bytes in all).
@pytest.mark.parametrize("n", [1, 3, 7, 8, 9, 1023, 1024, 1025, 2048, (1 << 19) - 1, 1 << 19,
                               (1 << 19) + 1, 1 << 20, (1 << 20) + 3, (1 << 22) - 200, 1 << 22])
def test_dispatch_copies(ctx, axc, n):
    """Both directions of every binding: h goes up and comes back, f = widen(h)."""
    print(f"dispatch copies {n}", flush=True)
    h = np.random.default_rng(n).integers(0, 0x7C00, n).astype(np.uint16)
    k = ctx.prepare_kernel(axc.builtin_code_object(), _plan(axc, 2, 4, 256), 4, "axh_f16_widen")
    for _ in range(2):  # the second one reuses the handle's staging buffer
        out = ctx.dispatch_handle(k, ((n + 255) // 256, 1, 1), [h.tobytes(), b""],
                                  [2 * n, 4 * n], struct.pack("<I", n))
        assert out[0] == h.tobytes()
        assert np.array_equal(np.frombuffer(out[1], np.float32),
                              h.view(np.float16).astype(np.float32))
        h = h[::-1].copy()
    k.release()
