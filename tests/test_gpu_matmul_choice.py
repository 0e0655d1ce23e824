"""Where 32 x 32 tiles take the place of a batched matmul variant's own kernel, and
where the narrow-step bodies run (marked `gpu`).

A body forms every output from its row's weights and its column's activations
in an order of its own, whatever the size of the grid, so an output equals,
bit for bit, the same output of a smaller call that runs the same body, and
differs in some last bits where the other body runs."""
from __future__ import annotations

import sys

import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


class _Data:
    def __init__(self, ctx, rows, sb, batch):
        self.ctx, self.sb = ctx, sb
        q = O.gen_q4k_weights(rows + sb, rows * sb)
        xh = O.gen_normal_f32(sb + batch, sb * 256 * batch).astype(np.float16)
        self.q, self.x, self.y = (ctx.alloc(n) for n in (q.nbytes, xh.nbytes, rows * batch * 4))
        ctx.upload(self.q, q)
        ctx.upload(self.x, xh)

    def run(self, axc, rows, batch, variant=None):
        print(f"matmul body {rows}x{self.sb * 256} B={batch} "
              f"{axc.q4k_matmul_kernel_name(rows, self.sb, batch, variant)}", flush=True)
        sys.stdout.flush()
        self.ctx.q4k_matmul(self.q, self.x, self.y, rows, self.sb, batch, variant)
        self.ctx.synchronize()
        y = np.frombuffer(self.ctx.download(self.y, rows * batch * 4), dtype=np.uint32)
        return y.reshape(batch, rows).copy()

    def close(self):
        for b in (self.q, self.x, self.y):
            b.close()


# 16 columns: 64 x 16 tiles, the one-column-tile kernel's own
@pytest.mark.parametrize("rows,sb,batch,tiles", [
    (300, 1, 48, False), (300, 7, 64, False), (300, 8, 33, True),      # one round of 32 x 32
    (8224, 7, 17, False), (8224, 12, 64, False), (8224, 15, 32, False),  # more than one
    (8224, 16, 32, True), (8224, 16, 48, False), (4128, 31, 48, False), (4128, 32, 48, True)])
def test_one_column_tile(ctx, axc, rows, sb, batch, tiles):
    v = axc.MatmulVariant(5, 4, 1, 3, 4)
    d = _Data(ctx, rows, sb, batch)
    whole, first = d.run(axc, rows, batch, v), d.run(axc, rows, 16, v)
    d.close()
    assert np.array_equal(whole[:16], first) == (not tiles)


# rows of few superblocks: 64 x 16 tiles while one round of them covers the grid
@pytest.mark.parametrize("rows,sb,batch,kernel", [
    (4097, 7, 48, "kx_r4_n1_k4_p3"), (4097, 8, 48, "kx_r4_n2_k4_p2"),
    (5440, 1, 48, "kx_r4_n1_k4_p3"), (5441, 1, 48, "kx_r4_n2_k4_p2_short"),
    (3264, 4, 77, "kx_r4_n1_k4_p3"), (3265, 4, 77, "kx_r4_n2_k4_p2_short")])
def test_few_superblocks(ctx, axc, rows, sb, batch, kernel):
    assert axc.q4k_matmul_kernel_name(rows, sb, batch) == "axh_q4k_matmul_" + kernel
    d = _Data(ctx, rows, sb, batch)
    whole = d.run(axc, rows, batch)
    first = d.run(axc, rows, 16, axc.MatmulVariant(5, 4, 1, 3, 4))
    d.close()
    # the narrow-step tiles of every width split and sum K alike
    assert np.array_equal(whole[:16], first) == (sb < 8)


# 64 x 32 tiles with two superblocks in flight: the narrow-step form, two to a CU,
# for several rounds of few superblocks
@pytest.mark.parametrize("rows,sb,batch,kernel", [
    (8192, 8, 64, "kx_r4_n2_k4_p2"), (8193, 8, 64, "kx_r4_n2_k4_p2_short"),
    (8193, 23, 33, "kx_r4_n2_k4_p2_short"), (8193, 24, 33, "kx_r4_n2_k4_p2"),
    (8193, 7, 33, "kx_r4_n2_k4_p2_short")])
def test_two_column_tiles_in_rounds(ctx, axc, rows, sb, batch, kernel):
    v = axc.MatmulVariant(5, 4, 2, 2, 4)
    assert axc.q4k_matmul_kernel_name(rows, sb, batch, v) == "axh_q4k_matmul_" + kernel
    d = _Data(ctx, rows, sb, batch)
    whole, narrow = d.run(axc, rows, batch, v), d.run(axc, rows, 16, axc.MatmulVariant(5, 4, 1, 3, 4))
    d.close()
    assert np.array_equal(whole[:16], narrow) == kernel.endswith("_short")


# 4096 rows of up to 32 columns: one 16-row block per CU, the variant's own kernel
@pytest.mark.parametrize("rows,sb,batch,tiles", [
    (4097, 6, 17, True), (5000, 7, 24, False), (5000, 8, 24, True), (5000, 9, 24, False),
    (5000, 12, 24, False), (8192, 15, 17, False), (8192, 16, 32, False)])
def test_streaming_rows_with_one_column_group(ctx, axc, rows, sb, batch, tiles):
    assert axc.q4k_matmul_kernel_name(rows, sb, batch) == "axh_q4k_matmul_sr_w8_s2_n2"
    d = _Data(ctx, rows, sb, batch)
    whole, first = d.run(axc, rows, batch), d.run(axc, 4096, batch)
    d.close()
    assert np.array_equal(whole[:, :4096], first) == (not tiles)
