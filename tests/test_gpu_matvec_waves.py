"""One-pass matvecs with 9 to 12 waves per workgroup (marked `gpu`): 4105 to
6144 rows, one workgroup per CU.

A row's sum is formed by one half wave in the same order whatever the size of
the workgroup, so every row must equal, bit for bit, the same row computed by
the 8-wave workgroups of a 4096-row call and of a call over the rest."""
from __future__ import annotations

import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


# the first and last row counts of a wave count and of the range, odd counts,
# rows of 1, 8, 9 superblocks and more; Q4_0 units are blocks
@pytest.mark.parametrize("fmt,rows,units", [
    ("q4k", 4097, 1), ("q4k", 4104, 16), ("q4k", 4105, 16), ("q5k", 4105, 17), ("q6k", 4105, 2),
    ("q4_0", 4105, 66), ("q4k", 4609, 9), ("q4k", 6144, 25), ("q4k", 6145, 9), ("q4k", 5000, 16),
    ("q5k", 4097, 8), ("q5k", 5119, 17), ("q5k", 6144, 33), ("q6k", 4098, 16), ("q6k", 5120, 3),
    ("q6k", 6143, 41), ("q4_0", 4097, 64), ("q4_0", 6144, 130)])
def test_rows_equal_those_of_smaller_calls(ctx, axc, fmt, rows, units):
    unit_bytes, elems = {"q4k": (144, 256), "q5k": (176, 256), "q6k": (210, 256),
                         "q4_0": (18, 32)}[fmt]
    call = getattr(ctx, fmt + "_matvec")
    print(f"one pass {fmt} {rows} x {units}", flush=True)
    q = np.random.default_rng(rows + units).integers(0, 256, rows * units * unit_bytes,
                                                     dtype=np.uint8)
    blocks = q.reshape(-1, unit_bytes)  # every f16 scale small and finite
    for at in {"q4k": (1, 3), "q5k": (1, 3), "q6k": (209,), "q4_0": (1,)}[fmt]:
        blocks[:, at] = 0x18 | (blocks[:, at] & 0x83)
    x = O.gen_normal_f32(units, units * elems)
    dq, dx, dy = ctx.alloc(q.nbytes + 16), ctx.alloc(x.nbytes), ctx.alloc(rows * 4)
    ctx.upload(dq, q)
    ctx.upload(dx, x)

    def run(first, n):
        ctx.upload(dy, np.full(n, np.nan, dtype=np.float32))
        call(dq.ptr + first * units * unit_bytes, dx, dy, n, units,
             axc.Variant(family=axc.FAMILY_ONE_PASS))
        ctx.synchronize()
        return np.frombuffer(ctx.download(dy, n * 4), dtype=np.uint32).copy()

    whole = run(0, rows)
    parts = np.concatenate([run(0, 4096), run(4096, rows - 4096)])
    assert not np.isnan(whole.view(np.float32)).any()
    assert np.array_equal(whole, parts)
    for b in (dq, dx, dy):
        b.close()


@pytest.mark.parametrize("fmt,rows,units,one", [
    ("q5k", 4104, 17, False), ("q5k", 4105, 17, True), ("q5k", 6144, 64, True),
    ("q5k", 6145, 17, False), ("q6k", 4104, 16, False), ("q6k", 4105, 16, True),
    ("q6k", 5121, 16, False), ("q6k", 6144, 41, True), ("q6k", 6145, 41, False)])
def test_defaults(axc, fmt, rows, units, one):
    name = getattr(axc, fmt + "_matvec_kernel_name")(rows, units)
    assert name.startswith(f"axh_{fmt}_matvec_{'one_' if one else 'flat_'}")


def test_first_use_while_recording(axc):
    """The wide kernels are a code object of their own: a context that has not
    launched one yet can load it while its stream records."""
    print("wide one-pass kernel first used in a capture", flush=True)
    rows, units = 4999, 3
    c = axc.HipContext.new()
    q = O.gen_q4k_weights(11, rows * units)
    x = O.gen_normal_f32(12, units * 256)
    dq, dx, dy, de = c.alloc(q.nbytes), c.alloc(x.nbytes), c.alloc(rows * 4), c.alloc(rows * 4)
    c.upload(dq, q)
    c.upload(dx, x)
    g = c.capture(lambda: c.q4k_matvec(dq, dx, dy, rows, units))
    for _ in range(3):
        c.upload(dy, np.full(rows, np.nan, dtype=np.float32))
        c.upload(de, np.full(rows, np.nan, dtype=np.float32))
        c.q4k_matvec(dq, dx, de, rows, units)
        c.synchronize()
        g.launch()
        c.synchronize()
        got = c.download(dy, rows * 4)
        assert got == c.download(de, rows * 4)
        assert not np.isnan(np.frombuffer(got, dtype=np.float32)).any()
    g.close()
    for b in (dq, dx, dy, de):
        b.close()
    c.close()
