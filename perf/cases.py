"""Performance cases: the GEMM work a user of this library runs through its public entry points.

Each case is a dict of plain values. `kind` names the entry point:

  dgemm   phpc_dgemm_device          FP64 product of resident operands
  host    phpc_gemm_cuda             the drop-in host-pointer product (copies included)
  summa   phpc_summa_device          the SUMMA loop on an emulated p x q grid
  split   phpc_dgemm_split_device    FP64-accurate product on the int8 matrix cores
  sgemm   phpc_sgemm_device          FP32 product (FP32 matrix cores, or 3 x BF16)
  grid    phpc_plan_graph_launch     every rank block of an uneven SUMMA as one FP64 plan
  mix     phpc_plan_graph_launch     many unrelated FP32 products as one plan

Every product accumulates (C += A B), as the entry points do, onto a C that starts uniform.
Inputs are uniform[-1, 1) or sign * 2^e with e uniform in [-20, 20], the two input sets the
library is benchmarked on.
"""
import importlib.util
import math
import random
import sys
from pathlib import Path

import numpy as np
import torch

_PKG = Path(__file__).resolve().parent.parent / "hpc-multigpu-matrixmult_amd"


def _phpc():
    """The package's binding (its folder name is not an importable identifier)."""
    mod = sys.modules.get("phpc")
    if mod is None:
        spec = importlib.util.spec_from_file_location("phpc", _PKG / "phpc.py")
        mod = importlib.util.module_from_spec(spec)
        sys.modules["phpc"] = mod
        spec.loader.exec_module(mod)
    return mod


def listed():
    return [
        # the smallest serving request: one product that cannot fill the GPU, latency only
        {"name": "dgemm_256", "kind": "dgemm", "m": 256, "k": 256, "n": 256},
        # the CPU baseline's size, resident operands
        {"name": "dgemm_1024", "kind": "dgemm", "m": 1024, "k": 1024, "n": 1024},
        # odd sizes, so odd leading dimensions: rows that 16-byte loads cannot take in place
        {"name": "dgemm_odd", "kind": "dgemm", "m": 1777, "k": 1999, "n": 1235},
        # the reference's own call on host matrices, as a program ported from it makes it
        {"name": "host_1024", "kind": "host", "m": 1024, "k": 1024, "n": 1024},
        # the headline SUMMA: 4 x 4 ranks, 64 panels of 256, one chain per output
        {"name": "summa_16384", "kind": "summa", "size": 16384, "p": 4, "q": 4, "panel": 256, "mode": "chained"},
        # FP64-accurate products on the int8 matrix cores: the smallest size that the serving
        # loop sends there, on the wide-exponent set, and the headline size
        {"name": "split_4096_wide", "kind": "split", "m": 4096, "k": 4096, "n": 4096, "dist": "wide"},
        {"name": "split_16384", "kind": "split", "m": 16384, "k": 16384, "n": 16384, "dist": "uniform"},
        # FP32 requests of the serving law that cannot fill the GPU: FP32 matrix cores on an
        # uneven shape, and the binding's default (3 x BF16)
        {"name": "sgemm_uneven", "kind": "sgemm", "m": 1500, "k": 1000, "n": 700, "method": "fp32"},
        {"name": "sgemm_x3_1500", "kind": "sgemm", "m": 1500, "k": 1500, "n": 1500, "method": "bf16x3"},
        # the uneven 3 x 3 grid (blocks 3334 / 3333, panels 3333), one captured launch
        {"name": "grid_10000", "kind": "grid", "size": 10000, "p": 3, "q": 3, "panel": 3333},
        # 512 unrelated products, sizes log-uniform in [64, 4096], one captured launch
        {"name": "mix_512_fp32", "kind": "mix", "count": 512, "lo": 64, "hi": 4096, "shapes": 21, "dtype": "fp32"},
        {"name": "mix_512_x3", "kind": "mix", "count": 512, "lo": 64, "hi": 4096, "shapes": 21, "dtype": "bf16x3"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same ranges: single products from the smallest to half the headline
    size with every side drawn by itself, grids and mixes of other sizes."""
    kind = rng.choice(["dgemm", "dgemm", "dgemm", "split", "split", "sgemm", "sgemm", "sgemm", "summa", "grid", "mix",
                       "mix", "host"])
    if kind in ("dgemm", "host"):
        hi = 8192 if kind == "dgemm" else 2048
        return {"kind": kind, "m": _log_int(rng, 96, hi), "k": _log_int(rng, 96, hi), "n": _log_int(rng, 96, hi)}
    if kind == "split":
        return {"kind": kind, "m": _log_int(rng, 768, 10000), "k": _log_int(rng, 768, 10000),
                "n": _log_int(rng, 768, 10000), "dist": rng.choice(["uniform", "wide"])}
    if kind == "sgemm":
        return {"kind": kind, "m": _log_int(rng, 96, 8192), "k": _log_int(rng, 96, 8192), "n": _log_int(rng, 96, 8192),
                "method": rng.choice(["fp32", "bf16x3"])}
    if kind in ("summa", "grid"):
        size = _log_int(rng, 1024, 10000)
        p, q = rng.randint(1, 4), rng.randint(1, 4)
        case = {"kind": kind, "size": size, "p": p, "q": q, "panel": rng.choice([256, 512, max(1, size // math.lcm(p, q))])}
        if kind == "summa":
            case["mode"] = rng.choice(["fused", "chained"])
        return case
    return {"kind": kind, "count": rng.randint(24, 400), "lo": 64, "hi": rng.choice([1024, 2048, 4096]),
            "shapes": rng.randrange(1 << 20), "dtype": rng.choice(["fp32", "bf16x3"])}


# ---------------- inputs ----------------

def _blocks(n, parts):
    """Start of every rank block, and n: the first n % parts blocks are one larger."""
    return [i * (n // parts) + min(i, n % parts) for i in range(parts + 1)]


def _mix_shapes(case):
    rng = random.Random(case["shapes"])
    return [tuple(_log_int(rng, case["lo"], case["hi"]) for _ in range(3)) for _ in range(case["count"])]  # m, n, k


def _matrix(gen, rows, cols, dtype, dist="uniform"):
    if dist == "wide":  # sign * 2^e from its FP64 bits, so that every value is exact
        e = torch.randint(-20, 21, (rows, cols), generator=gen, device="cuda")
        s = torch.randint(0, 2, (rows, cols), generator=gen, device="cuda")
        return ((s << 63) | ((e + 1023) << 52)).view(torch.float64).to(dtype)
    return torch.empty((rows, cols), dtype=dtype, device="cuda").uniform_(-1.0, 1.0, generator=gen)


def _flat(gen, sizes):
    """One buffer of uniform FP32 values holding a matrix of every size, each 256-byte aligned."""
    starts, total = [], 0
    for r, c in sizes:
        starts.append(total)
        total += -(-(r * c) // 64) * 64
    buf = torch.empty(total, dtype=torch.float32, device="cuda").uniform_(-1.0, 1.0, generator=gen)
    return buf, [buf[s:s + r * c].view(r, c) for s, (r, c) in zip(starts, sizes)]


def _inputs(case, seed):
    """The operands of a case, from its seed alone."""
    kind = case["kind"]
    if kind == "host":
        g = np.random.default_rng(seed)
        return tuple(g.uniform(-1.0, 1.0, s) for s in ((case["m"], case["k"]), (case["k"], case["n"]),
                                                       (case["m"], case["n"])))
    gen = torch.Generator(device="cuda").manual_seed(seed)
    if kind == "mix":
        shapes = _mix_shapes(case)
        a = _flat(gen, [(m, k) for m, n, k in shapes])
        b = _flat(gen, [(k, n) for m, n, k in shapes])
        c = _flat(gen, [(m, n) for m, n, k in shapes])
        return a[1], b[1], c[1], c[0]
    if kind in ("summa", "grid"):
        m = k = n = case["size"]
    else:
        m, k, n = case["m"], case["k"], case["n"]
    dtype = torch.float32 if kind == "sgemm" else torch.float64
    dist = case.get("dist", "uniform")
    return _matrix(gen, m, k, dtype, dist), _matrix(gen, k, n, dtype, dist), _matrix(gen, m, n, dtype)


def prepare(case, seed):
    phpc = _phpc()
    phpc.lib()
    kind = case["kind"]
    x = _inputs(case, seed)
    state = {"case": case, "A": x[0], "B": x[1], "C": x[2]}
    if kind in ("grid", "mix"):
        stream = torch.cuda.Stream()
        if kind == "grid":
            rows, cols = _blocks(case["size"], case["p"]), _blocks(case["size"], case["q"])
            items = [(x[0][r0:r1], x[1][:, c0:c1], x[2][r0:r1, c0:c1], case["panel"])
                     for r0, r1 in zip(rows, rows[1:]) for c0, c1 in zip(cols, cols[1:])]
            state["plan"] = phpc.Plan(phpc.F64, items, stream=stream)
        else:
            dtype = phpc.F32 if case["dtype"] == "fp32" else phpc.F32X3
            state["plan"] = phpc.Plan(dtype, list(zip(x[0], x[1], x[2])), stream=stream)
            state["out"] = x[3]
        state["stream"] = stream
    if kind != "host":
        torch.cuda.synchronize()  # the plan's stream starts on finished inputs
    return state


def run(state):
    phpc = _phpc()
    case = state["case"]
    kind = case["kind"]
    A, B, C = state["A"], state["B"], state["C"]
    if kind == "dgemm":
        phpc.dgemm_device(A, B, C)
    elif kind == "host":
        phpc.gemm_cuda(A, B, C)
    elif kind == "summa":
        mode = phpc.SUMMA_CHAINED if case["mode"] == "chained" else phpc.SUMMA_FUSED
        phpc.summa_device(A, B, C, case["p"], case["q"], panel=case["panel"], mode=mode)
    elif kind == "split":
        phpc.dgemm_split_device(A, B, C)
    elif kind == "sgemm":
        phpc.sgemm_device(A, B, C, method=phpc.SGEMM_FP32 if case["method"] == "fp32" else phpc.SGEMM_BF16X3)
    else:
        state["plan"].graph_launch(state["stream"])
    return state.get("out", C)


def work(case):
    """Each operand read once, C read and written once; 2 m n k operations per product."""
    kind = case["kind"]
    if kind == "mix":
        shapes, size = _mix_shapes(case), 4
    elif kind in ("summa", "grid"):
        shapes, size = [(case["size"],) * 3], 8
    else:
        shapes, size = [(case["m"], case["n"], case["k"])], 4 if kind == "sgemm" else 8
    return {"bytes": float(sum(size * (m * k + k * n + 2 * m * n) for m, n, k in shapes)),
            "flops": float(sum(2 * m * n * k for m, n, k in shapes))}


def exact(case, seed):
    """C + A B in 64 bits by torch (numpy for host matrices)."""
    x = _inputs(case, seed)
    if case["kind"] == "host":
        return x[2] + x[0] @ x[1]
    if case["kind"] != "mix":
        return x[2].double() + x[0].double() @ x[1].double()
    out, want = x[3], x[3].double()
    for a, b, c in zip(*x[:3]):
        s = c.data_ptr() // 4 - out.data_ptr() // 4
        want[s:s + c.numel()] += (a.double() @ b.double()).reshape(-1)
    return want
