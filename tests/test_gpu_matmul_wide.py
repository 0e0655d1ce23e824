"""The batched matmul's wide-K-step bodies at the edges of their tiles and K
groups, and the default's choice between their tiles (marked `gpu`).

Every output is compared with the f64 product of the same f16 weights, per
element to 1e-5 of sum |w x| (f32 accumulation: random-sign rounding of at most
K / 16 = 896 sums in a row gives sqrt(896) * 2^-24 = 1.8e-6, and the guard of
5 covers every element of the largest case), with the output poisoned by NaN
before the call."""
from __future__ import annotations

import sys

import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _check(ctx, axc, rows, sb, batch, variant=None):
    print(f"wide matmul {rows}x{sb * 256} B={batch} "
          f"{axc.q4k_matmul_kernel_name(rows, sb, batch, variant)}", flush=True)
    sys.stdout.flush()
    q = O.gen_q4k_weights(rows * 3 + sb * 5 + batch, rows * sb)
    xh = O.gen_normal_f32(rows + sb + batch, sb * 256 * batch).astype(np.float16)
    y = np.full(batch * rows, np.nan, dtype=np.float32)
    bufs = [ctx.alloc(max(a.nbytes, 16)) for a in (q, xh, y)]
    for buf, a in zip(bufs, (q, xh, y)):
        ctx.upload(buf, a)
    ctx.q4k_matmul(*bufs, rows, sb, batch, variant)
    ctx.synchronize()
    y = np.frombuffer(ctx.download(bufs[2], y.nbytes), dtype=np.float32).reshape(batch, rows)
    for buf in bufs:
        buf.close()
    w16 = O.q4k_dequant(q, rows * sb).reshape(rows, sb * 256).astype(np.float16).astype(np.float64)
    x64 = xh.astype(np.float64).reshape(batch, sb * 256)
    assert np.all(np.abs(y - x64 @ w16.T) <= 1e-5 * (np.abs(x64) @ np.abs(w16).T) + 1e-30)


# one row, superblock and column; row remainders of 1, 31 and 33; fewer
# superblocks than K groups, one more, and a ring's worth; column remainders
@pytest.mark.parametrize("rows,sb,batch", [(1, 1, 17), (31, 9, 33), (33, 19, 31), (257, 8, 129),
                                           (65, 3, 64), (130, 4, 32), (300, 17, 260)])
def test_tiles_and_k_groups_at_their_edges(ctx, axc, rows, sb, batch):
    for v in [(5, 4, 1, 3, 4), (5, 4, 2, 2, 4), (5, 4, 2, 3, 4), (5, 4, 4, 2, 4), (5, 4, 8, 2, 4),
              (8, 4, 8, 4, 1), (8, 8, 8, 4, 1)]:
        _check(ctx, axc, rows, sb, batch, axc.MatmulVariant(*v))


# either side of the lines between the default's tiles (256 and 257 workgroups)
@pytest.mark.parametrize("rows,sb,batch,kernel", [
    (8192, 17, 17, "kx_r4_n1_k4_p3"),          # 32 x 32 tiles: 256
    (8193, 17, 17, "kx_r4_n2_k4_p3"),          # 257
    (8193, 17, 16, "kx_r4_n2_k4_p3"),          # past the long-rows kind, 16 columns
    (4096, 5, 33, "sr_w8_s2_n2"),              # two 16-row blocks per CU: 256 of 32 rows
    (2049, 16, 97, "kx_r4_n2_k4_p2"),          # 65 x 4 of 32 rows is one more
    (8192, 7, 33, "kx_r4_n2_k4_p2_short"),     # 128 x 2 of 64 x 32
    (8193, 7, 33, "kx_r4_n4_k4_p2_short"),
    (4097, 17, 128, "kx_r4_n4_k4_p2"),         # 65 x 4 of 64 x 32
    (16385, 8, 64, "kx_r4_n4_k4_p2"),          # none fits one round: the widest filled
    (16385, 7, 65, "kx_r4_n8_k4_p2_short"),
    (16385, 8, 65, "kx_r4_n8_k4_p2"),
    (8192, 16, 256, "kx_r4_n8_k4_p2"),         # 128 x 2 of 64 x 128
    (8193, 16, 256, "rm_w4_r1_p4"),            # 129 x 2: 65 x 2 of 128 x 128
    (8193, 3, 256, "rm_w4_r1_p4_short"),
    (16384, 9, 128, "kx_r4_n8_k4_p2"), (16385, 9, 128, "rm_w4_r1_p4"),
    (16385, 9, 127, "kx_r4_n8_k4_p2"),
    (20352, 9, 128, "rm_w4_r1_p4"),            # 159 of 128 x 128
    (4608, 9, 512, "rm_w4_r1_p4"),
    (32768, 5, 128, "rm_w4_r1_p4_short"),
    (32768, 6, 128, "rm_w4_r1_p4"),
    (32769, 1, 128, "rm_w8_r1_p4"),
])
def test_default_tiles(ctx, axc, rows, sb, batch, kernel):
    assert axc.q4k_matmul_kernel_name(rows, sb, batch) == "axh_q4k_matmul_" + kernel
    _check(ctx, axc, rows, sb, batch)


# either side of the line between the short and the wide K steps
@pytest.mark.parametrize("rows,sb,variant,kernel", [
    (300, 7, (5, 4, 8, 2, 4), "kx_r4_n8_k4_p2_short"), (300, 8, (5, 4, 8, 2, 4), "kx_r4_n8_k4_p2"),
    (300, 7, (5, 4, 2, 2, 4), "kx_r4_n2_k4_p2_short"), (300, 8, (5, 4, 2, 2, 4), "kx_r4_n2_k4_p2"),
    (300, 5, (8, 4, 8, 4, 1), "rm_w4_r1_p4_short"), (300, 6, (8, 4, 8, 4, 1), "rm_w4_r1_p4"),
    (16400, 7, (8, 4, 8, 4, 1), "rm_w4_r1_p4_short"), (16400, 8, (8, 4, 8, 4, 1), "rm_w4_r1_p4"),
])
def test_short_and_wide_steps(ctx, axc, rows, sb, variant, kernel):
    v = axc.MatmulVariant(*variant)
    assert axc.q4k_matmul_kernel_name(rows, sb, 130, v) == "axh_q4k_matmul_" + kernel
    _check(ctx, axc, rows, sb, 130, v)


def test_streaming_rows_second_body_line(ctx, axc):
    """One 16-row block per CU stays with the variant's own kernel; a second block per CU
    goes to 32-row tiles while those are one round, in every K remainder (4097
    rows of 32 columns, one column group: only where K splits evenly)."""
    for rows, sb, batch in [(4096, 16, 32), (4097, 16, 32), (2064, 7, 64), (1024, 1, 250)]:
        _check(ctx, axc, rows, sb, batch, axc.MatmulVariant(7, 8, 2, 1))


def test_partial_variants_keep_their_holes(axc):
    """Holes a caller leaves 0 beside others do not follow the default's lines."""
    name = axc.q4k_matmul_kernel_name
    assert name(28672, 16, 256) == "axh_q4k_matmul_rm_w8_r1_p4"
    assert name(28672, 16, 256, axc.MatmulVariant(row_tiles=2)) == "axh_q4k_matmul_rm_w4_r2_p4"
    assert name(5000, 43, 128) == "axh_q4k_matmul_kx_r4_n4_k4_p2"
    assert name(5000, 43, 128, axc.MatmulVariant(col_tiles=1)) == "axh_q4k_matmul_kx_r4_n1_k4_p3"
