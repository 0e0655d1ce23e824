"""Performance cases of the quantised matvec / matmul path.

Each case is one call (or one recorded sequence of calls) that a program
serving or inspecting GGUF weights makes through the public entry points of
the package: single-token decode over every supported format, batched decode,
prefill, whole-tensor decoding, and the host-buffer dispatch surface.

Weights are random bytes in the formats' own layouts with f16 scales of the
size that real checkpoints hold; activations are N(0, 1).
"""
import numpy as np
import torch

from __graft_entry__ import load_package

# format -> (elements per block, bytes per block, ggml type id)
FORMATS = {
    "q4_0": (32, 18, 2),
    "q4_k": (256, 144, 12),
    "q5_k": (256, 176, 13),
    "q6_k": (256, 210, 14),
}

# The largest shapes of the ranges: the output head of a 128256-token
# vocabulary, and 512 prompt tokens against a 14336 x 4096 projection.
MAX_MATVEC_BYTES = 128256 * 16 * 210
MAX_MATMUL_FLOPS = 2.0 * 14336 * 4096 * 512

_ctx = None


def context():
    """The program's one device context."""
    global _ctx
    if _ctx is None:
        _ctx = load_package().HipContext.new()
    return _ctx


# ---- cases -------------------------------------------------------------------
def listed():
    return [
        # The reference's own GPU benchmark: one dot product of 512 superblocks,
        # host buffers in, host result out, on a prepared kernel handle.
        {"name": "dispatch q4_k 512 sb", "kind": "dispatch", "fmt": "q4_k", "units": 512},
        # The smallest resident-buffer call: a key/value-sized Q4_0 projection,
        # where the latency of one launch counts.
        {"name": "matvec q4_0 256x4096", "kind": "matvec", "fmt": "q4_0", "rows": 256,
         "units": 128},
        # Single-token decode, the down projection of an 8B-class model.
        {"name": "matvec q4_k 4096x14336", "kind": "matvec", "fmt": "q4_k", "rows": 4096,
         "units": 56},
        # A ragged projection: rows no tile divides, an odd superblock count.
        {"name": "matvec q5_k 4999x5376", "kind": "matvec", "fmt": "q5_k", "rows": 4999,
         "units": 21},
        # The output head, the largest matrix of a decode step.
        {"name": "matvec q6_k 128256x4096", "kind": "matvec", "fmt": "q6_k", "rows": 128256,
         "units": 16},
        # One transformer block of a Q4_K_M checkpoint at decode (attn_v and
        # ffn_down in Q6_K), recorded once and replayed per token.
        {"name": "block q4_k 4096/1024/14336", "kind": "block", "fmt": "q4_k", "hidden": 4096,
         "kv": 1024, "ffn": 14336},
        # Whole-tensor decoding to f32 (inspection, conversion), bit-exact.
        {"name": "dequant q4_k 4096x14336", "kind": "dequant", "fmt": "q4_k",
         "units": 4096 * 56},
        # Batched decode: 8 sequences against the down projection.
        {"name": "matmul f16 4096x14336 b8", "kind": "matmul", "x": "f16", "rows": 4096,
         "units": 56, "batch": 8},
        # Batched decode: 32 sequences against the up projection.
        {"name": "matmul f16 14336x4096 b32", "kind": "matmul", "x": "f16", "rows": 14336,
         "units": 16, "batch": 32},
        # A ragged prompt of 77 tokens, f32 activations, an odd superblock count.
        {"name": "matmul f32 5000x11008 b77", "kind": "matmul", "x": "f32", "rows": 5000,
         "units": 43, "batch": 77},
        # A short prompt.
        {"name": "matmul f16 14336x4096 b128", "kind": "matmul", "x": "f16", "rows": 14336,
         "units": 16, "batch": 128},
        # Prefill of a full 512-token chunk from f32 activations.
        {"name": "matmul f32 14336x4096 b512", "kind": "matmul", "x": "f32", "rows": 14336,
         "units": 16, "batch": 512},
    ]


def _log(rng, lo, hi):
    """A whole number in [lo, hi], spread over its logarithm."""
    v = int(round(lo * (hi / lo) ** rng.random()))
    return min(hi, max(lo, v))


def draw(rng):
    kind = rng.choices(["dispatch", "matvec", "block", "dequant", "matmul"], [1, 4, 1, 1, 5])[0]
    if kind == "dispatch":
        fmt = rng.choice(["q4_k", "q4_0"])
        return {"kind": kind, "fmt": fmt,
                "units": _log(rng, 16, 512) if fmt == "q4_k" else _log(rng, 128, 4096)}
    if kind == "matvec":
        fmt = rng.choice(list(FORMATS))
        elems, nbytes, _ = FORMATS[fmt]
        units = _log(rng, 1024 // elems, 28672 // elems)
        rows = _log(rng, 1, min(131072, MAX_MATVEC_BYTES // (units * nbytes)))
        return {"kind": kind, "fmt": fmt, "rows": rows, "units": units}
    if kind == "block":
        hidden = 256 * _log(rng, 4, 20)
        return {"kind": kind, "fmt": rng.choice(["q4_k", "q4_0", "q5_k"]), "hidden": hidden,
                "kv": hidden // rng.choice([1, 4, 8]),
                "ffn": 256 * int(hidden * rng.uniform(2.5, 4.0) // 256)}
    if kind == "dequant":
        fmt = rng.choice(list(FORMATS))
        elems = FORMATS[fmt][0]
        return {"kind": kind, "fmt": fmt,
                "units": _log(rng, 262144 // elems, 4096 * 14336 // elems)}
    units = _log(rng, 4, 56)
    rows = _log(rng, 256, 28672)
    batch = _log(rng, 1, max(1, min(512, int(MAX_MATMUL_FLOPS / (2.0 * rows * 256 * units)))))
    return {"kind": "matmul", "x": rng.choice(["f16", "f32"]), "rows": rows, "units": units,
            "batch": batch}


# ---- inputs ------------------------------------------------------------------
def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _scales(g, n, mean):
    """n f16 block scales, uniform in [0.5, 1.5] * mean, as byte pairs."""
    s = (torch.rand(n, generator=g, device="cuda") + 0.5) * mean
    return s.half().view(torch.uint8).reshape(n, 2)


def _weights(g, fmt, n):
    """n random blocks of a format, one row of bytes each."""
    raw = torch.randint(0, 256, (n, FORMATS[fmt][1]), dtype=torch.uint8, generator=g,
                        device="cuda")
    if fmt == "q4_0":
        raw[:, 0:2] = _scales(g, n, 4e-3)
    elif fmt == "q6_k":
        raw[:, 208:210] = _scales(g, n, 1.5e-5)
    else:
        raw[:, 0:2] = _scales(g, n, 1.2e-4 if fmt == "q4_k" else 6e-5)
        raw[:, 2:4] = _scales(g, n, 9e-4)
    return raw


def _normal(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda")


def _block_matrices(case):
    """The block's matrices: name -> (format, rows, columns)."""
    fmt, hidden, kv, ffn = case["fmt"], case["hidden"], case["kv"], case["ffn"]
    return {"q": (fmt, hidden, hidden), "k": (fmt, kv, hidden), "v": ("q6_k", kv, hidden),
            "o": (fmt, hidden, hidden), "gate": (fmt, ffn, hidden), "up": (fmt, ffn, hidden),
            "down": ("q6_k", hidden, ffn)}


def _inputs(case, seed):
    """The case's tensors, from the seed alone."""
    g = _generator(seed)
    kind = case["kind"]
    if kind == "block":
        d = {n: _weights(g, f, r * (c // FORMATS[f][0]))
             for n, (f, r, c) in _block_matrices(case).items()}
        d["x"] = _normal(g, case["hidden"])       # the normalised hidden state
        d["attn"] = _normal(g, case["hidden"])    # the attention's output
        d["x_ffn"] = _normal(g, case["hidden"])   # the normalised residual
        return d
    if kind == "matmul":
        x = _normal(g, case["batch"], case["units"] * 256)
        return {"w": _weights(g, "q4_k", case["rows"] * case["units"]),
                "x": x.half() if case["x"] == "f16" else x}
    fmt = case["fmt"]
    n = case["units"] * (case["rows"] if kind == "matvec" else 1)
    d = {"w": _weights(g, fmt, n)}
    if kind != "dequant":
        d["x"] = _normal(g, case["units"] * FORMATS[fmt][0])
    return d


def prepare(case, seed):
    ctx = context()
    t = _inputs(case, seed)
    kind = case["kind"]
    state = {"case": case, "ctx": ctx, "t": t}
    if kind == "dispatch":
        pkg = load_package()
        entry = "q4km_dequant_matvec" if case["fmt"] == "q4_k" else "q4_0_dequant_matvec"
        access = [pkg.axh.ACCESS_READ_ONLY, pkg.axh.ACCESS_READ_ONLY, pkg.axh.ACCESS_READ_WRITE]
        plan = pkg.axh.BindingPlan(access, 4, (64, 1, 1))
        state["handle"] = ctx.prepare_kernel(pkg.axh.builtin_code_object(), plan, 4, entry)
        state["inputs"] = [t["w"].cpu().numpy().tobytes(), t["x"].cpu().numpy().tobytes(),
                           bytes(4)]
        state["pc"] = int(case["units"]).to_bytes(4, "little")
    elif kind == "matvec":
        state["y"] = torch.zeros(case["rows"], device="cuda")
    elif kind == "dequant":
        state["y"] = torch.zeros(case["units"] * FORMATS[case["fmt"]][0], device="cuda")
    elif kind == "matmul":
        state["y"] = torch.zeros(case["batch"], case["rows"], device="cuda")
        if case["x"] == "f32":
            state["x16"] = torch.zeros(t["x"].shape, dtype=torch.half, device="cuda")
    else:
        state["y"] = {n: torch.zeros(r, device="cuda")
                      for n, (_, r, _) in _block_matrices(case).items() if n not in ("gate", "up")}
        state["y"]["ffn"] = torch.zeros(case["ffn"], device="cuda")
        torch.cuda.synchronize()
        _block_step(state)  # every operation runs once before it is recorded
        ctx.synchronize()
        state["graph"] = ctx.capture(lambda: _block_step(state))
    return state


# ---- one pass ----------------------------------------------------------------
def _block_step(state):
    """The projections of one transformer block for one token."""
    ctx, t, y, case = state["ctx"], state["t"], state["y"], state["case"]
    mats = _block_matrices(case)

    def project(name, x):
        fmt, rows, cols = mats[name]
        ctx.matvec_ggml(FORMATS[fmt][2], t[name], x, y[name], rows, cols)

    for name in ("q", "k", "v"):
        project(name, t["x"])
    project("o", t["attn"])
    gate_up = {"q4_k": ctx.q4k_gate_up, "q4_0": ctx.q4_0_gate_up, "q5_k": ctx.q5k_gate_up}
    gate_up[case["fmt"]](t["gate"], t["up"], t["x_ffn"], y["ffn"], case["ffn"],
                         case["hidden"] // FORMATS[case["fmt"]][0])
    project("down", y["ffn"])


def run(state):
    case, ctx, t = state["case"], state["ctx"], state["t"]
    kind = case["kind"]
    if kind == "dispatch":
        out = ctx.dispatch_handle(state["handle"], (1, 1, 1), state["inputs"], [0, 0, 4],
                                  state["pc"])
        return np.frombuffer(out[2], dtype=np.float32)
    if kind == "matvec":
        elems, _, ggml = FORMATS[case["fmt"]]
        ctx.matvec_ggml(ggml, t["w"], t["x"], state["y"], case["rows"], case["units"] * elems)
        return state["y"]
    if kind == "dequant":
        decode = {"q4_0": ctx.q4_0_dequant, "q4_k": ctx.q4k_dequant, "q5_k": ctx.q5k_dequant,
                  "q6_k": ctx.q6k_dequant}
        decode[case["fmt"]](t["w"], state["y"], case["units"])
        return state["y"]
    if kind == "matmul":
        shape = case["rows"], case["units"], case["batch"]
        if case["x"] == "f16":
            ctx.q4k_matmul(t["w"], t["x"], state["y"], *shape)
            return state["y"]
        ctx.q4k_matmul_f32(t["w"], t["x"], state["x16"], state["y"], *shape)
        return {"y": state["y"], "x16": state["x16"]}
    state["graph"].launch()
    return state["y"]


def work(case):
    kind = case["kind"]
    if kind == "block":
        mats = _block_matrices(case).values()
        nbytes = sum(r * (c // FORMATS[f][0]) * FORMATS[f][1] for f, r, c in mats)
        nbytes += 4 * (3 * case["hidden"] + 2 * case["kv"] + 3 * case["hidden"] + case["ffn"])
        return {"bytes": nbytes, "flops": sum(2 * r * c for _, r, c in mats)}
    if kind == "matmul":
        rows, cols, batch = case["rows"], case["units"] * 256, case["batch"]
        per_x = 2 if case["x"] == "f16" else 6  # f32 in, f16 copy out
        return {"bytes": rows * case["units"] * 144 + per_x * batch * cols + 4 * batch * rows,
                "flops": 2 * rows * cols * batch}
    elems, nbytes, _ = FORMATS[case["fmt"]]
    n = case["units"]
    if kind == "dequant":
        return {"bytes": n * (nbytes + 4 * elems), "flops": 2 * n * elems}
    rows = case["rows"] if kind == "matvec" else 1
    return {"bytes": rows * n * nbytes + 4 * n * elems + 4 * rows, "flops": 2 * rows * n * elems}


# ---- 64-bit results ----------------------------------------------------------
def _decode(fmt, raw):
    """The weights of raw blocks (n x bytes) in 64 bits, n x elements."""
    raw = raw.contiguous()
    n = raw.shape[0]

    def half(at):
        return raw[:, at:at + 2].contiguous().view(torch.half).double()

    if fmt == "q4_0":
        qs = raw[:, 2:18]
        return (torch.cat([qs & 15, qs >> 4], 1).double() - 8) * half(0)
    if fmt == "q6_k":
        ql = raw[:, 0:128].reshape(n, 2, 2, 32)
        qh = raw[:, 128:192].reshape(n, 2, 1, 32)
        lo = torch.cat([ql & 15, ql >> 4], 2)  # four parts of 32 weights per half
        shift = torch.tensor([0, 2, 4, 6], dtype=torch.uint8, device=raw.device).view(1, 1, 4, 1)
        q = (lo | (((qh >> shift) & 3) << 4)).double() - 32
        sc = raw[:, 192:208].contiguous().view(torch.int8).double()
        sc = sc.reshape(n, 2, 4, 2, 1).expand(n, 2, 4, 2, 16).reshape(n, 256)
        return q.reshape(n, 256) * sc * half(208)
    s = raw[:, 4:16]
    a, b, c = s[:, 0:4], s[:, 4:8], s[:, 8:12]
    sc = torch.cat([a & 63, (c & 15) | ((a >> 6) << 4)], 1).double()
    m = torch.cat([b & 63, (c >> 4) | ((b >> 6) << 4)], 1).double()
    qs = raw[:, 16:144] if fmt == "q4_k" else raw[:, 48:176]
    qs = qs.reshape(n, 4, 1, 32)
    q = torch.cat([qs & 15, qs >> 4], 2).reshape(n, 8, 32)
    if fmt == "q5_k":
        bit = torch.arange(8, dtype=torch.uint8, device=raw.device).view(1, 8, 1)
        q = q | (((raw[:, 16:48].reshape(n, 1, 32) >> bit) & 1) << 4)
    d, dmin = half(0).view(n, 1, 1), half(2).view(n, 1, 1)
    return (d * sc.view(n, 8, 1) * q.double() - dmin * m.view(n, 8, 1)).reshape(n, 256)


def _exact_product(fmt, raw, rows, x, f16_weights=False):
    """x (batch x columns, f64) against the rows of a matrix: batch x rows."""
    units = raw.shape[0] // rows
    step = max(1, (1 << 25) // (units * FORMATS[fmt][0]))
    out = []
    for r in range(0, rows, step):
        w = _decode(fmt, raw[r * units:(r + step) * units])
        if f16_weights:  # the matmul's stated weights: RN_f16(RN_f32(w))
            w = w.float().half().double()
        out.append(torch.mm(x, w.reshape(-1, x.shape[1]).t().contiguous()))
    return torch.cat(out, 1)


def exact(case, seed):
    t = _inputs(case, seed)
    kind = case["kind"]
    if kind == "dequant":
        step = (1 << 25) // FORMATS[case["fmt"]][0]
        return torch.cat([_decode(case["fmt"], t["w"][i:i + step]).reshape(-1)
                          for i in range(0, case["units"], step)])
    if kind == "matmul":
        x16 = t["x"].half()
        y = _exact_product("q4_k", t["w"], case["rows"], x16.double(), True)
        return y if case["x"] == "f16" else {"y": y, "x16": x16.double()}
    if kind == "block":
        mats = _block_matrices(case)

        def project(name, x):
            fmt, rows, _ = mats[name]
            return _exact_product(fmt, t[name], rows, x.double().reshape(1, -1)).reshape(-1)

        y = {name: project(name, t["x"]) for name in ("q", "k", "v")}
        y["o"] = project("o", t["attn"])
        gate, up = project("gate", t["x_ffn"]), project("up", t["x_ffn"])
        y["ffn"] = gate / (1 + torch.exp(-gate)) * up
        y["down"] = project("down", y["ffn"])
        return y
    rows = case["rows"] if kind == "matvec" else 1
    y = _exact_product(case["fmt"], t["w"], rows, t["x"].double().reshape(1, -1)).reshape(-1)
    return y if kind == "matvec" else y.cpu().numpy()


def tolerance(case):
    """f32 sums in another order; decoded weights are exact.

    Measured against 64 bits: 1.5e-7 to 5.4e-7 relative over the listed and
    some drawn cases; another order of these sums (one after the other over
    14336 columns) gives up to about 2e-6.  A single dot product (dispatch,
    few rows) can cancel, so its error stands over a result that may be
    small."""
    kind = case["kind"]
    if kind == "dequant":
        return "exact"
    if kind == "dispatch" or (kind == "matvec" and case["rows"] < 32):
        return {"rel": 1e-4, "max": 1e-3}
    return {"rel": 1e-5, "max": 1e-4}
