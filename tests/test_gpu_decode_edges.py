"""Whole-tensor decode kernels at the edges of their workgroups (marked `gpu`):
unit counts around what one workgroup takes (16 Q4_K / Q5_K and 32 Q6_K
superblocks, 128 Q4_0 blocks) and its second unit per thread, bit-exact
against the oracle, with the words after the tensor left alone."""
from __future__ import annotations

import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

Q5, Q6 = 13, 14
GUARD = 64  # words after the tensor
GEN = {"q4_k": lambda n: O.gen_q4k_weights(70 + n, n), "q4_0": lambda n: O.gen_q4_0_weights(70 + n, n),
       "q5_k": lambda n: O.gen_kq_weights(Q5, 70 + n, n), "q6_k": lambda n: O.gen_kq_weights(Q6, 70 + n, n)}
REF = {"q4_k": O.q4k_dequant, "q4_0": O.q4_0_dequant,
       "q5_k": lambda q, n: O.kq_dequant(Q5, q, n), "q6_k": lambda q, n: O.kq_dequant(Q6, q, n)}


@pytest.mark.parametrize("fmt", list(GEN))
@pytest.mark.parametrize("n", [1, 7, 8, 9, 15, 16, 17, 31, 32, 33, 63, 97, 127, 128, 129, 1025])
def test_decode_unit_counts(ctx, fmt, n):
    print(f"decode {fmt} {n} units", flush=True)
    elems = 32 if fmt == "q4_0" else 256
    q = GEN[fmt](n)
    guard = np.full(n * elems + GUARD, 0xA5A5A5A5, np.uint32)
    dq, dw = ctx.alloc(q.nbytes), ctx.alloc(guard.nbytes)
    ctx.upload(dq, q)
    ctx.upload(dw, guard)
    {"q4_k": ctx.q4k_dequant, "q4_0": ctx.q4_0_dequant, "q5_k": ctx.q5k_dequant,
     "q6_k": ctx.q6k_dequant}[fmt](dq, dw, n)
    ctx.synchronize()
    w = np.frombuffer(ctx.download(dw, guard.nbytes), dtype=np.uint32)
    dq.close()
    dw.close()
    assert np.array_equal(w[:n * elems], REF[fmt](q, n).view(np.uint32))
    assert (w[n * elems:] == 0xA5A5A5A5).all()


@pytest.mark.parametrize("fmt", ["q4_0", "q6_k"])
def test_decode_at_the_least_alignment(ctx, fmt):
    """Weights 2 bytes and output 4 bytes past a 16-byte boundary."""
    print(f"decode {fmt} unaligned", flush=True)
    n, elems = 77, 32 if fmt == "q4_0" else 256
    q = GEN[fmt](n)
    dq, dw = ctx.alloc(q.nbytes + 16), ctx.alloc(n * elems * 4 + 16)
    ctx.upload(dq, np.concatenate([np.zeros(2, np.uint8), q.view(np.uint8).reshape(-1)]))
    (ctx.q4_0_dequant if fmt == "q4_0" else ctx.q6k_dequant)(dq.ptr + 2, dw.ptr + 4, n)
    ctx.synchronize()
    w = np.frombuffer(ctx.download(dw, n * elems * 4 + 16), dtype=np.uint32)
    dq.close()
    dw.close()
    assert np.array_equal(w[1:1 + n * elems], REF[fmt](q, n).view(np.uint32))
