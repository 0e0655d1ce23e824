"""The waits of the long-rows and the wide-K-step matmul kernels, checked on the
built code (no GPU needed).

A wave loads X into LDS for every wave of its workgroup and passes a barrier
once its own loads have landed, which it tells from the load counter: loads
return in the order they were issued, so after `s_waitcnt vmcnt(n)` all but the
last n have.  Whether n is right depends on which loads the compiler kept and
where it put them, so it is checked on the instructions: at every barrier no
more loads of X may be in flight than those of the chunks requested ahead of
the one that is read next."""
from __future__ import annotations

import ctypes
import re
import shutil
import subprocess

import pytest

OBJDUMP = shutil.which("llvm-objdump") or "/opt/rocm/llvm/bin/llvm-objdump"


@pytest.fixture(scope="module")
def kernels(axc, tmp_path_factory):
    """name -> instructions of every kernel of the matmul code object."""
    if not shutil.which(OBJDUMP):
        pytest.skip("llvm-objdump is not installed")
    lib = axc.load_library()
    begin, end = (ctypes.addressof(ctypes.c_char.in_dll(lib, f"axh_q4_matmul_co_{n}"))
                  for n in ("begin", "end"))
    co = tmp_path_factory.mktemp("co") / "q4_matmul.co"
    co.write_bytes(ctypes.string_at(begin, end - begin))
    text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", str(co)], check=True, text=True,
                          stdout=subprocess.PIPE).stdout
    out: dict = {}
    for line in text.splitlines():
        if m := re.match(r"^[0-9a-f]+ <(\w+)>:", line):
            out[m.group(1)] = body = []
        elif line.startswith("\t"):
            body.append(line.split("//")[0].strip())
    return out


def _barriers(body):
    """(index, loads of X in flight, LDS reads in flight) at every barrier,
    along the instructions in address order (prologue, one turn of the loop, the
    steps after it: a branch back enters where the fall-through does)."""
    loads, reads, out = [], 0, []
    for i, ins in enumerate(body):
        op = ins.split()[0]
        if op.startswith("buffer_load"):
            loads.append(ins.endswith("lds"))
        elif op.startswith("ds_read"):
            reads += 1
        elif op == "s_waitcnt":
            if m := re.search(r"vmcnt\((\d+)\)", ins):
                n = int(m.group(1))
                loads = loads[len(loads) - n:] if n and n < len(loads) else loads if n else []
            if m := re.search(r"lgkmcnt\((\d+)\)", ins):
                reads = min(reads, int(m.group(1)))
        elif op == "s_barrier":
            out.append((i, sum(loads), reads))
    return out


LK = [("axh_q4k_matmul_lk_c16_x1_w3", 16, 1), ("axh_q4k_matmul_lk_c16_x1_w3_r2", 16, 1),
      ("axh_q4k_matmul_lk_c8_x1_w3", 8, 1), ("axh_q4k_matmul_lk_c8_x2_w2", 8, 2),
      ("axh_q4k_matmul_lk_c8_x2_w2_r2", 8, 2), ("axh_q4k_matmul_lk_c4_x2_w2", 4, 2)]


@pytest.mark.parametrize("name,cols,ahead", LK)
def test_x_has_landed_at_every_barrier(kernels, name, cols, ahead):
    at = _barriers(kernels[name])
    assert len(at) >= ahead + 3  # the steps of a round, those after it, and the sum
    per_chunk = cols * 4 // 8  # loads of X per wave and chunk
    for i, in_flight, _ in at:
        assert in_flight <= (ahead - 1) * per_chunk, (name, i)


@pytest.mark.parametrize("name,cols,ahead", LK)
def test_x_is_read_before_its_buffer_is_refilled(kernels, name, cols, ahead):
    """The loads after a barrier refill the buffer read before it."""
    for i, _, reads in _barriers(kernels[name]):
        assert reads == 0, (name, i)


def test_every_long_rows_kernel_is_listed(kernels):
    assert {n for n in kernels if "_lk_" in n} == {n for n, _, _ in LK}


# X loads per wave and step, steps ahead, weight loads and header loads per superblock
WK = [("t32", 4, 3, 4, 1), ("kx_r4_n2_k4_p2", 2, 5, 5, 0), ("kx_r4_n2_k4_p3", 2, 5, 5, 0),
      ("kx_r4_n4_k4_p2", 4, 3, 4, 1), ("kx_r4_n8_k4_p2", 8, 2, 4, 1),
      ("rm_w4_r1_p4", 4, 3, 4, 1), ("rm_w8_r1_p4", 2, 5, 5, 0)]


@pytest.mark.parametrize("name,n_x,ahead,n_w,n_h", WK)
def test_wide_steps_wait_for_x_and_weights(kernels, name, n_x, ahead, n_w, n_h):
    """The loop's four steps, each behind a barrier: X of the next step was issued
    `ahead` steps before that one, the next weights in the step of chunk 3.  The
    waits may leave no more in flight than the loads that came after those."""
    steps, cur = [], []
    for ins in kernels["axh_q4k_matmul_" + name]:
        op = ins.split()[0]
        if op == "s_barrier":
            steps.append(cur)
            cur = []
        elif op.startswith("buffer_load"):
            cur.append("lds" if ins.endswith("lds") else "h")
        elif op == "s_waitcnt" and (m := re.search(r"vmcnt\((\d+)\)", ins)):
            cur.append(int(m.group(1)))
    steps.append(cur)
    # the loop is the last four that issue loads (first ones for what K groups leave over
    # come before it), and the wait of its first barrier ends what is before that
    at = [i for i, s in enumerate(steps) if "lds" in s][-4:]
    assert at == list(range(at[0], at[0] + 4))
    loop = [steps[i] for i in at]
    loads = []  # of each step: (X or weights or header) in the order of issue
    for e, s in enumerate(loop):
        lds = [v for v in s if v == "lds"]
        assert len(lds) == n_x + (n_w if e == 3 else 0) and s.count("h") == (n_h if e == 0 else 0)
        kinds, k = [], 0
        for v in s:
            if v == "lds":
                kinds.append("x" if k < n_x else "w")
                k += 1
            elif v == "h":
                kinds.append("h")
        loads.append(kinds)
    for e in range(4):
        wait = [v for v in steps[at[e] - 1] if isinstance(v, int)][-1]
        first = loads[(e + 1 - ahead) % 4]  # the step that issued X of the next one
        after = len(first) - 1 - max(i for i, v in enumerate(first) if v == "x")
        after += sum(len(loads[(e - b) % 4]) for b in range(1, ahead - 1))
        assert wait <= after, (e, wait, after)
    seen = 0  # of step 2's loads before its wait for the weights
    waits = []
    for v in loop[2]:
        if v in ("lds", "h"):
            seen += 1
        elif isinstance(v, int):
            waits.append((v, seen))
    wait, seen = waits[0]
    assert wait <= len(loads[0]) + len(loads[1]) + seen, (wait, seen)
