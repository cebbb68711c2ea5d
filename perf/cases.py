"""Performance cases of the int8 GEMM framework: the calls a program makes, with their sizes.

`listed()` names the cases, `draw(rng)` gives more of the same ranges. Every case goes through the
public entry points of `veritac_amd.specializations.hip_gemm`:

  gemm    `backend.run` on row-major operands, one call or `layers` calls with a weight each
  packed  `backend.run` on weights packed once by `backend.pack_b`, the same way
  graph   the packed calls of one decode step, captured once and replayed as a HIP graph
  replay  `replay.run_commands`: a Gemmini command stream over host data
  nest    a `loopnest.LoopNestKernel`: an emitted loop nest over device buffers

Activations are uniform int8, weights normal with a deviation of 32 clipped to int8, partial sums
uniform in [-2^20, 2^20]; "adversarial" operands are half -128 or 127 and half uniform. All GEMM
results are whole numbers and compared exactly. The loop nest's float64 buffers hold small whole
numbers, whose sums float64 holds exactly.
"""
import math

import numpy as np
import torch

from veritac_amd.specializations.hip_gemm import backend as hg
from veritac_amd.specializations.hip_gemm import loopnest as ln
from veritac_amd.specializations.hip_gemm import replay as rp
from veritac_amd.specializations.hip_gemm import schedules as sc

DEV = "cuda"
MOST_MACS = 2 * 10**11     # largest drawn GEMM; the largest listed one has 5.5e11
MOST_BYTES = 600 * 2**20   # operands and result of a drawn case


def _gemm(m, n, k, d=False, batch=1, shared=False, layers=1, lda_pad=0, data="plain", kind="gemm"):
    return {"kind": kind, "m": m, "n": n, "k": k, "d": d, "batch": batch, "shared": shared,
            "layers": layers, "lda_pad": lda_pad, "data": data}


def listed():
    return [
        # The smallest product: one 64^3 tile, where launch and call costs are everything.
        dict(_gemm(64, 64, 64), name="tile_64"),
        # One K-tiled accumulation step onto an existing int32 partial sum.
        dict(_gemm(256, 256, 256, d=True), name="partial_256"),
        # A small product of unaligned sizes, as the head or the remainder of an odd model gives.
        dict(_gemm(100, 203, 333), name="odd_small"),
        # An ordinary product of odd sizes onto a partial sum: no row of A, B or C is aligned.
        dict(_gemm(1000, 1001, 999, d=True), name="odd_1000"),
        # One token for each of 16 sequences through the up projections of four layers.
        dict(_gemm(16, 14336, 4096, layers=4), name="decode_16"),
        # One sequence's decode step over packed weights, captured in a HIP graph as servers do:
        # gate and up (4096 -> 14336) and down (14336 -> 4096) projections.
        dict(_gemm(1, 14336, 4096, kind="graph"), name="decode_graph"),
        # A larger decode batch (more rows than one 16-row block) through the down projections of
        # two layers: a long K and few columns.
        dict(_gemm(48, 4096, 14336, layers=2), name="batch_48"),
        # 64 activations sharing one weight matrix: batched B reuse.
        dict(_gemm(512, 1024, 1024, batch=64, shared=True), name="reuse_64"),
        # Prefill of a ragged 2000-token prompt through a square projection, onto a residual sum.
        dict(_gemm(2000, 4096, 4096, d=True), name="prefill_2000"),
        # The large compute-bound product, on operands that toggle the most bits.
        dict(_gemm(8192, 8192, 8192, data="adversarial"), name="cube_8192"),
        # A recorded Gemmini program of the certified 64^3 size, executed with its checks.
        {"name": "replay_64", "kind": "replay", "m": 64, "n": 64, "k": 64, "schedule": "reuse_b"},
        # The loop-nest matrix product of the CPU benchmark, float64 in the stride-1000 layout.
        {"name": "nest_500", "kind": "nest", "m": 500, "n": 500, "k": 500, "dtype": "float64"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _to16(v):
    return max(16, (v + 8) // 16 * 16)


def _state_bytes(c):
    b = c["batch"]
    macs_bytes = b * c["m"] * (c["k"] + c["lda_pad"]) + (1 if c["shared"] else b) * c["k"] * c["n"] * c["layers"]
    return macs_bytes + b * c["m"] * c["n"] * (8 if c["d"] else 4) * c["layers"]


def draw(rng):
    kind = rng.choices(("gemm", "packed", "graph", "replay", "nest"), (13, 3, 1, 1, 2))[0]
    if kind == "replay":
        m, n, k = (16 * rng.randint(2, 6) for _ in range(3))
        return {"kind": kind, "m": m, "n": n, "k": k, "schedule": rng.choice(("reuse_b", "baseline"))}
    if kind == "nest":
        m, n, k = (_log_int(rng, 48, 640) for _ in range(3))
        return {"kind": kind, "m": m, "n": n, "k": k, "dtype": rng.choice(("float64", "int8"))}
    if kind == "graph":
        return _gemm(_log_int(rng, 1, 16), _to16(_log_int(rng, 2048, 14336)),
                     _to16(_log_int(rng, 1024, 8192)), kind=kind)
    while True:
        # Decode batches, prefill and square products alike.
        m = _log_int(rng, 1, 64) if rng.random() < 0.35 else _log_int(rng, 33, 8192)
        n, k = _log_int(rng, 64, 16384), _log_int(rng, 64, 16384)
        c = _gemm(m, n, k, d=rng.random() < 0.35, kind=kind)
        if kind == "packed" or rng.random() < 0.6:
            c["n"], c["k"] = _to16(n), _to16(k)
            if rng.random() < 0.2:
                c["lda_pad"] = 64      # A is a column slice of a wider activation
        if rng.random() < 0.2:
            c["batch"] = _log_int(rng, 2, 64)
            c["shared"] = rng.random() < 0.5
        if (c["batch"] * c["m"] * c["n"] * c["k"] <= MOST_MACS and _state_bytes(c) <= MOST_BYTES):
            return c


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _uniform(g, shape, lo, hi, dtype=torch.int8):
    return torch.randint(lo, hi + 1, shape, generator=g, device=DEV, dtype=dtype)


def _adversarial(g, shape):
    x = _uniform(g, shape, -128, 127)
    ends = _uniform(g, shape, 0, 1) * -1 ^ 127          # 127 or -128
    return torch.where(_uniform(g, shape, 0, 1).bool(), ends, x)


def _weights(g, shape, data):
    if data == "adversarial":
        return _adversarial(g, shape)
    w = torch.empty(shape, device=DEV, dtype=torch.float32).normal_(0.0, 32.0, generator=g)
    return w.round_().clamp_(-128, 127).to(torch.int8)


def _operands(case, seed):
    """A, the layers' weights, D: the same for prepare and exact."""
    g = _gen(seed)
    m, n, k, b = case["m"], case["n"], case["k"], case["batch"]
    rows = (m, k + case["lda_pad"]) if b == 1 else (b, m, k + case["lda_pad"])
    x = _adversarial(g, rows) if case["data"] == "adversarial" else _uniform(g, rows, -127, 127)
    cols = (k, n) if (b == 1 or case["shared"]) else (b, k, n)
    ws = [_weights(g, cols, case["data"]) for _ in range(case["layers"])]
    d = None
    if case["d"]:
        d = _uniform(g, (m, n) if b == 1 else (b, m, n), -(1 << 20), 1 << 20, torch.int32)
    return x[..., :k], ws, d


def _graph_operands(case, seed):
    """x, gate, up [k, n] and the n-wide activation with its down projection [n, k]."""
    g = _gen(seed)
    m, n, k = case["m"], case["n"], case["k"]
    return (_uniform(g, (m, k), -127, 127), _weights(g, (k, n), "plain"), _weights(g, (k, n), "plain"),
            _uniform(g, (m, n), -127, 127), _weights(g, (n, k), "plain"))


def _plan(case, variant="auto"):
    return hg.make_plan(case["m"], case["n"], case["k"], batch=case["batch"], b_shared=case["shared"],
                        has_d=case["d"], d_max_abs=(1 << 20) if case["d"] else 0, variant=variant)


def _prepare_graph(case, seed):
    x, gate, up, h, down = _graph_operands(case, seed)
    m, n, k = case["m"], case["n"], case["k"]
    wide = hg.make_plan(m, n, k, variant="skinny_packed")
    narrow = hg.make_plan(m, k, n, variant="skinny_packed")
    calls = [(wide, x, hg.pack_b(gate)), (wide, x, hg.pack_b(up)), (narrow, h, hg.pack_b(down))]
    outs = [torch.empty((m, p["n"]), dtype=torch.int32, device=DEV) for p, _, _ in calls]
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(side):
        for (p, a, w), o in zip(calls, outs):       # the workspaces, before the capture
            hg.run(p, a, w, out=o)
    with torch.cuda.graph(graph, stream=side):
        for (p, a, w), o in zip(calls, outs):
            hg.run(p, a, w, out=o)
    return {"kind": "graph", "graph": graph, "outs": outs, "calls": calls, "side": side}


def _nest_buffers(case, seed):
    """The flat device buffers of a loop nest: stride-1000 float64, or dense int8 with an int32 C."""
    g = _gen(seed)
    m, n, k = case["m"], case["n"], case["k"]
    if case["dtype"] == "int8":
        return {"A": _uniform(g, (m * k,), -128, 127), "B": _weights(g, (k * n,), "plain"),
                "C": torch.zeros(m * n, dtype=torch.int32, device=DEV)}
    flat = {}
    for name, (r, c), hi in (("A", (m, k), 6), ("B", (k, n), 4), ("C", (m, n), 0)):
        t = torch.zeros((r, 1000), dtype=torch.float64, device=DEV)
        t[:, :c] = _uniform(g, (r, c), 0, hi).double()
        flat[name] = t.reshape(-1)
    return flat


def prepare(case, seed):
    kind = case["kind"]
    if kind == "graph":
        return _prepare_graph(case, seed)
    if kind == "replay":
        rng = np.random.default_rng(seed)
        m, n, k = case["m"], case["n"], case["k"]
        plan = sc.make_plan(m, n, k, case["schedule"])
        return {"kind": kind, "plan": plan, "commands": sc.gen_commands(plan),
                "A": rng.integers(-128, 128, m * k, dtype=np.int8),
                "B": rng.integers(-128, 128, k * n, dtype=np.int8)}
    if kind == "nest":
        m, n, k = case["m"], case["n"], case["k"]
        types = ("int8", "int8", "int32") if case["dtype"] == "int8" else ("float64",) * 3
        shapes = ((m, k), (k, n), (m, n))
        decl = {b: {"dtype": t, "shape": s} for b, t, s in zip("ABC", types, shapes)}
        kernel = ln.LoopNestKernel(ln.matmul_stmt(m, k, n), decl, name="matmul",
                                   layout="dense" if case["dtype"] == "int8" else "reference")
        return {"kind": kind, "kernel": kernel, "buffers": _nest_buffers(case, seed)}
    x, ws, d = _operands(case, seed)
    plan = _plan(case, "skinny_packed" if kind == "packed" else "auto")
    if kind == "packed":
        ws = [hg.pack_b(w) for w in ws]
    return {"kind": kind, "plan": plan, "A": x, "B": ws, "D": d}


def run(state):
    kind = state["kind"]
    if kind == "graph":
        state["graph"].replay()
        return state["outs"]
    if kind == "replay":
        c, stats = rp.run_commands(state["commands"], state["plan"], state["A"], state["B"])
        return {"c": np.asarray(c, dtype=np.int32), "stats": stats}
    if kind == "nest":
        state["buffers"]["C"].zero_()
        status = state["kernel"](state["buffers"])
        return {"c": state["buffers"]["C"], "status": status}
    return [hg.run(state["plan"], state["A"], w, state["D"]) for w in state["B"]]


def work(case):
    m, n, k = case["m"], case["n"], case["k"]
    if case["kind"] == "nest":
        a, c = (1, 4) if case["dtype"] == "int8" else (8, 8)
        return {"bytes": a * (m * k + k * n) + c * m * n, "flops": 2.0 * m * n * k}
    if case["kind"] == "replay":
        return {"bytes": m * k + k * n + 4 * m * n, "flops": 2.0 * m * n * k}
    if case["kind"] == "graph":
        return {"bytes": 3 * n * k + m * (k + n) + 4 * m * (2 * n + k), "flops": 6.0 * m * n * k}
    b, layers = case["batch"], case["layers"]
    weights = (1 if case["shared"] else b) * k * n
    out = 4 * b * m * n
    return {"bytes": b * m * k + layers * (weights + out) + (out if case["d"] else 0),
            "flops": 2.0 * b * m * n * k * layers}


def tolerance(case):
    # Whole-number sums (in int32, or in float64 far below 2^53) have one right answer.
    return "exact"


def _product(a, w, d=None):
    c = torch.matmul(a.double(), w.double())
    if d is not None:
        c += d
    return c.to(torch.int64).to(torch.int32)


def exact(case, seed):
    kind = case["kind"]
    if kind == "graph":
        x, gate, up, h, down = _graph_operands(case, seed)
        return [_product(x, gate), _product(x, up), _product(h, down)]
    if kind == "replay":
        rng = np.random.default_rng(seed)
        m, n, k = case["m"], case["n"], case["k"]
        a = rng.integers(-128, 128, m * k, dtype=np.int8).astype(np.int64).reshape(m, k)
        b = rng.integers(-128, 128, k * n, dtype=np.int8).astype(np.int64).reshape(k, n)
        return {"c": (a @ b).astype(np.int32).reshape(-1), "stats": None}
    if kind == "nest":
        m, n, k = case["m"], case["n"], case["k"]
        f = _nest_buffers(case, seed)
        if case["dtype"] == "int8":
            c = _product(f["A"].reshape(m, k), f["B"].reshape(k, n)).reshape(-1)
        else:
            c = f["C"].clone()
            c.reshape(m, 1000)[:, :n] = f["A"].reshape(m, 1000)[:, :k] @ f["B"].reshape(k, 1000)[:, :n]
        return {"c": c, "status": None}
    x, ws, d = _operands(case, seed)
    return [_product(x, w, d) for w in ws]
