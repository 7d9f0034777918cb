"""Timed workloads of the reduction / scan path, through the package's public
entry points.

A case is a dict: its `kind` names a way a program uses the library, the other
entries its sizes and options.  `prepare` makes the inputs on the GPU and the
buffers and plans that a program keeps; `run` is one pass.  Kinds:

* vector_step   one power-iteration step on f32 vectors: the small calls of an
                iterative solver, two of which return a scalar to the host.
* axis_batch    prepared axis reductions of one matrix, submitted as a batch.
* reduce        full reductions of a flat buffer (sum, max, argmax), each an
                immediate call.
* rows          prepared fused row sum, max and argmax of fmaf(a, x, b).
* interior      reductions over the inside of a matrix with a border (a slice
                whose rows are padded): residual dot and norm, sum, argmax.
* scan          1-D prefix scans: inclusive or exclusive, forward or reverse.
* axis_scan     prefix scans of a matrix along one axis.
* segmented     segmented sums over CSR offsets.

Every pass goes to the device's own stream, as the package's defaults do.
"""
from __future__ import annotations

import math

import torch

import hephaestus_amd as hx
from hephaestus_amd import Layout, StridedView

import numpy as np

DTYPES = {"f32": np.float32, "u32": np.uint32, "i32": np.int32}
OPS = {"sum": hx.SumOp, "max": hx.MaxOp, "min": hx.MinOp, "mean": hx.MeanOp, "argmax": hx.ArgMaxOp}
PROLOGUE = (0.5, 0.25)
SHIFT = 0.125  # of the power iteration

_device = None


def _dev():
    global _device
    if _device is None:
        _device = hx.RocmDevice.try_default()
    return _device


# ------------------------------------------------------------------ cases
def listed():
    return [
        # The smallest matrices whose axis statistics the reference publishes;
        # launches and latency are all of it.
        {"name": "axis_stats_256", "kind": "axis_batch", "rows": 256, "cols": 256, "axis": 0,
         "ops": "sum,min,max,mean"},
        # A solver on 65536 unknowns (the reference's dot size): host
        # round trips and launches count.
        {"name": "vector_step_65536", "kind": "vector_step", "n": 65536},
        # Statistics of one mid-sized array (the 2^20 of the smallest headline
        # configuration).
        {"name": "stats_f32_2p20", "kind": "reduce", "dtype": "f32", "n": 1 << 20, "ops": "sum,max,argmax"},
        # The headline's full reduction: memory bandwidth alone.
        {"name": "sum_f32_2p28", "kind": "reduce", "dtype": "f32", "n": 1 << 28, "ops": "sum"},
        # The headline's scan, as stream compaction and allocation use it.
        {"name": "scan_u32_2p28", "kind": "scan", "dtype": "u32", "n": 1 << 28, "scan": "exclusive",
         "direction": "forward"},
        # An ordinary running total of a few million integers of odd length.
        {"name": "scan_i32_3m", "kind": "scan", "dtype": "i32", "n": 3_000_017, "scan": "inclusive",
         "direction": "forward"},
        # The largest configuration: 4 GiB in, 4 GiB out.
        {"name": "scan_f32_2p30", "kind": "scan", "dtype": "f32", "n": 1 << 30, "scan": "inclusive",
         "direction": "forward"},
        # Row statistics with the fused prologue (scores of 65536 rows).
        {"name": "rows_65536x4096", "kind": "rows", "rows": 65536, "cols": 4096},
        # Segment sums over long rows of a CSR structure ...
        {"name": "segments_2p27_300", "kind": "segmented", "dtype": "i32", "n": 1 << 27, "mean": 300.0},
        # ... and over a sparse matrix with a handful of entries a row.
        {"name": "segments_2p24_8", "kind": "segmented", "dtype": "i32", "n": 1 << 24, "mean": 8.0},
        # Running totals of 64 channels over a million steps.
        {"name": "cumsum_1048576x64", "kind": "axis_scan", "dtype": "u32", "rows": 1 << 20, "cols": 64, "axis": 0,
         "scan": "inclusive", "direction": "forward"},
        # The inside of a 4096 x 4096 grid with a border of one cell.
        {"name": "interior_4094", "kind": "interior", "rows": 4094, "cols": 4094, "pitch": 4096, "offset": 4097},
    ]


def _log_int(rng, lo, hi):
    """An integer of [lo, hi], even over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _matrix(rng, lo, hi, min_side, max_cols):
    """Rows and columns of a matrix of lo to hi elements."""
    n = _log_int(rng, lo, hi)
    cols = _log_int(rng, min_side, min(max_cols, max(min_side, n // min_side)))
    return max(min_side, n // cols), cols


def draw(rng):
    kind = rng.choice(("axis_batch", "vector_step", "reduce", "reduce", "scan", "scan", "scan", "rows", "segmented",
                       "segmented", "axis_scan", "axis_scan", "interior"))
    if kind == "axis_batch":
        rows, cols = _matrix(rng, 1 << 14, 1 << 27, 16, 16384)
        return {"kind": kind, "rows": rows, "cols": cols, "axis": rng.randrange(2),
                "ops": ",".join(rng.sample(("sum", "min", "max", "mean", "argmax"), 3))}
    if kind == "vector_step":
        return {"kind": kind, "n": _log_int(rng, 1 << 12, 1 << 26)}
    if kind == "reduce":
        dtype = rng.choice(("f32", "f32", "u32", "i32"))
        return {"kind": kind, "dtype": dtype, "n": _log_int(rng, 1 << 14, 1 << 28),
                "ops": rng.choice(("sum", "max", "argmax", "sum,max,argmax"))}
    if kind == "scan":
        return {"kind": kind, "dtype": rng.choice(("f32", "u32", "i32")), "n": _log_int(rng, 1 << 14, 1 << 28),
                "scan": rng.choice(("inclusive", "exclusive")),
                "direction": rng.choice(("forward", "forward", "reverse"))}
    if kind == "rows":
        rows, cols = _matrix(rng, 1 << 16, 1 << 28, 8, 32768)
        return {"kind": kind, "rows": rows, "cols": cols}
    if kind == "segmented":
        return {"kind": kind, "dtype": rng.choice(("u32", "i32")), "n": _log_int(rng, 1 << 16, 1 << 27),
                "mean": round(math.exp(rng.uniform(math.log(2.0), math.log(3000.0))), 2)}
    if kind == "axis_scan":
        rows, cols = _matrix(rng, 1 << 16, 1 << 27, 16, 8192)
        return {"kind": kind, "dtype": rng.choice(("f32", "u32", "i32")), "rows": rows, "cols": cols,
                "axis": rng.randrange(2), "scan": rng.choice(("inclusive", "exclusive")),
                "direction": rng.choice(("forward", "forward", "reverse"))}
    rows, cols = _matrix(rng, 1 << 16, 1 << 27, 32, 16384)
    pitch = cols + rng.choice((1, 2, 2, 2, 4, 8, 16, 96))
    return {"kind": kind, "rows": rows, "cols": cols, "pitch": pitch, "offset": rng.choice((0, 1, pitch + 1))}


# ----------------------------------------------------------------- inputs
class _Memory:
    """Device memory of a RocmBuffer as torch takes it, alive with the tensor
    made from it.  32-bit integers of either sign are shown as int32."""

    def __init__(self, buffer, shape):
        self.buffer = buffer
        kind = "<f4" if buffer.dtype == np.float32 else "<i4"
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": kind, "data": (buffer.ptr, False),
                                         "version": 2}


def _tensor(buffer, shape=None):
    return torch.as_tensor(_Memory(buffer, shape or (len(buffer),)), device="cuda")


def _new(dtype, length, shape=None):
    """An output buffer and the tensor over it."""
    buffer = _dev().alloc_zeroed(dtype, length)
    return buffer, _tensor(buffer, shape)


def _upload(values, dtype):
    """A RocmBuffer with the values of a GPU tensor."""
    buffer = _dev().alloc_uninitialized(dtype, values.numel())
    _tensor(buffer).copy_(values.reshape(-1))
    return buffer


def _values(g, dtype, n, lo=-1.0):
    if dtype == "f32":
        return torch.empty(n, device="cuda").uniform_(lo, 1.0, generator=g)
    lo, hi = (0, 256) if dtype == "u32" else (-1000, 1001)
    return torch.randint(lo, hi, (n,), device="cuda", dtype=torch.int32, generator=g)


def _segments(case):
    return max(1, round(case["n"] / case["mean"]))


def _inputs(case, seed):
    """The values of a case's operands, from the seed alone."""
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    kind = case["kind"]
    if kind == "axis_batch":
        return {"x": torch.randn(case["rows"] * case["cols"], device="cuda", generator=g)}
    if kind == "rows":
        return {"x": torch.randn(case["rows"] * case["cols"], device="cuda", generator=g)}
    if kind == "vector_step":  # a start vector and a positive diagonal
        return {"v": torch.randn(case["n"], device="cuda", generator=g),
                "d": torch.empty(case["n"], device="cuda").uniform_(0.5, 1.0, generator=g)}
    if kind == "interior":
        n = (case["rows"] + 2) * case["pitch"]
        return {"x": torch.randn(n, device="cuda", generator=g), "y": torch.randn(n, device="cuda", generator=g)}
    if kind == "segmented":
        # Cut points drawn evenly: lengths are geometric about the mean, with
        # the few empty rows that CSR structures have.
        cuts = torch.randint(0, case["n"] + 1, (_segments(case) - 1,), device="cuda", dtype=torch.int64, generator=g)
        ends = torch.tensor([0, case["n"]], device="cuda")
        offsets = torch.cat((ends[:1], torch.sort(cuts).values, ends[1:])).to(torch.int32)
        return {"x": _values(g, "i32", case["n"]), "offsets": offsets}
    if kind == "reduce":
        return {"x": _values(g, case["dtype"], case["n"])}
    n = case["n"] if kind == "scan" else case["rows"] * case["cols"]
    return {"x": _values(g, case["dtype"], n, lo=0.0)}


# ---------------------------------------------------------------- prepare
def prepare(case, seed):
    dev = _dev()
    kind, values = case["kind"], _inputs(case, seed)
    state = {"case": case, "dev": dev}
    if kind == "axis_batch":
        rows, cols, axis = case["rows"], case["cols"], case["axis"]
        x = StridedView(_upload(values["x"], np.float32), Layout.c_contiguous([rows, cols]))
        shape = [1, cols] if axis == 0 else [rows, 1]
        ops, state["plans"], state["out"] = hx.RocmAxisReductionOps(), [], {}
        for op in case["ops"].split(","):
            buffer, view = _new(np.uint32 if op == "argmax" else np.float32, shape[0] * shape[1])
            state["plans"].append(ops.prepare_reduce_axis_into(
                dev, OPS[op], x, axis, StridedView(buffer, Layout.c_contiguous(shape))))
            state["out"][op] = view
    elif kind == "vector_step":
        ops = hx.RocmDenseVectorOps()
        state.update(ops=ops, v=_upload(values["v"], np.float32), d=_upload(values["d"], np.float32))
        state["w"], _ = _new(np.float32, case["n"])
        state["dot"] = ops.prepare_dot(dev, state["v"], state["w"])
        state["norm"] = ops.prepare_norm_l2(dev, state["w"])
        state["vector"] = _tensor(state["v"])
    elif kind == "reduce":
        x = _upload(values["x"], DTYPES[case["dtype"]])
        state.update(ops=hx.RocmFullReductionOps(), x=StridedView(x, Layout.c_contiguous([case["n"]])), todo=[],
                     out={})
        for op in case["ops"].split(","):
            buffer, view = _new(np.uint32 if op == "argmax" else x.dtype, 1)
            state["todo"].append((op, buffer, StridedView(buffer, Layout.c_contiguous([1]))))
            state["out"][op] = view
    elif kind == "rows":
        rows = case["rows"]
        s, m, i = _new(np.float32, rows), _new(np.float32, rows), _new(np.uint32, rows)
        state["plan"] = hx.RocmAxisReductionOps().prepare_reduce_rows_fused(
            dev, _upload(values["x"], np.float32), rows, case["cols"], prologue=PROLOGUE, out_sum=s[0], out_max=m[0],
            out_argmax=i[0])
        state["out"] = {"sum": s[1], "max": m[1], "argmax": i[1]}
    elif kind == "interior":
        x, y = (_upload(values[k], np.float32) for k in "xy")
        inside = Layout.try_new([case["rows"], case["cols"]], [case["pitch"], 1], case["offset"])
        vx, vy = StridedView(x, inside), StridedView(y, inside)
        total, index, value = _new(np.float32, 1), _new(np.uint32, 1), _new(np.float32, 1)
        full = hx.RocmFullReductionOps()
        one = StridedView(total[0], Layout.c_contiguous([1]))
        dot, norm = hx.prepare_dot(dev, vx, vy), hx.prepare_norm_l2(dev, vx)
        state.update(full=full, plans=[full.prepare_reduce_full(dev, hx.SumOp, vx, one), dot, norm], x=vx,
                     index=index[0], value=value[0])
        state["out"] = {"sum": total[1], "dot": _tensor(dot.output), "norm": _tensor(norm.output),
                        "argmax": index[1], "max": value[1]}
    elif kind == "segmented":
        dtype = DTYPES[case["dtype"]]
        state.update(ops=hx.RocmSegmentedReductionOps(), x=_upload(values["x"], dtype),
                     offsets=_upload(values["offsets"], np.uint32))
        state["y"], state["out"] = _new(dtype, _segments(case))
    else:
        shape = [case["n"]] if kind == "scan" else [case["rows"], case["cols"]]
        dtype, layout = DTYPES[case["dtype"]], Layout.c_contiguous(shape)
        x = _upload(values["x"], dtype)
        y, state["out"] = _new(dtype, len(x), shape)
        state.update(ops=hx.RocmScanOps(), x=StridedView(x, layout), y=StridedView(y, layout),
                     axis=case.get("axis", 0), kind=getattr(hx.ScanKind, case["scan"].capitalize()),
                     direction=getattr(hx.ScanDirection, case["direction"].capitalize()))
    torch.cuda.synchronize()  # torch wrote the operands on a stream of its own
    return state


# -------------------------------------------------------------------- run
def run(state):
    case, dev = state["case"], state["dev"]
    kind = case["kind"]
    if kind == "axis_batch":
        hx.submit_prepared_axis_reduction_batch(dev, state["plans"])
    elif kind == "vector_step":
        # w = (D + SHIFT)·v, the Rayleigh quotient's v·w, then v = w / ‖w‖.
        ops, v, w = state["ops"], state["v"], state["w"]
        ops.multiply_into(dev, state["d"], v, w)
        ops.axpy(dev, w, v, SHIFT)
        vw = ops.dot_prepared(dev, state["dot"], v, w)
        norm = ops.norm_l2_prepared(dev, state["norm"], w)
        ops.copy_vector(dev, w, v)
        ops.scale_vector(dev, v, 1.0 / norm)
        return {"vector": state["vector"], "dot": vw, "norm": norm}
    elif kind == "reduce":
        for op, buffer, view in state["todo"]:
            if op == "argmax":
                state["ops"].argmax_full_into(dev, state["x"], buffer)
            else:
                state["ops"].reduce_full_into(dev, OPS[op], state["x"], view)
    elif kind == "rows":
        state["plan"].dispatch()
    elif kind == "interior":
        hx.submit_prepared_reduction_batch(state["plans"])
        state["full"].argmax_full_into(dev, state["x"], state["index"], state["value"])
    elif kind == "segmented":
        state["ops"].segmented_sum_into(dev, state["x"], state["offsets"], state["y"])
    else:
        state["ops"].scan_axis_into(dev, hx.CumSumOp, state["x"], state["axis"], state["direction"], state["y"],
                                    state["kind"])
    return state["out"]


# ------------------------------------------------------------------- work
def work(case):
    """Bytes that the entry points called in a pass must read and write, each
    operand of a call once, and the arithmetic on its elements."""
    kind = case["kind"]
    n = case["n"] if "n" in case else case["rows"] * case["cols"]
    if kind == "axis_batch":
        calls = len(case["ops"].split(","))
        outputs = case["cols"] if case["axis"] == 0 else case["rows"]
        return {"bytes": calls * (4 * n + 4 * outputs), "flops": calls * n}
    if kind == "vector_step":  # multiply 3, axpy 3, dot 2, norm 1, copy 2, scale 2 vectors
        return {"bytes": 13 * 4 * n, "flops": 8 * n}
    if kind == "reduce":
        calls = len(case["ops"].split(","))
        return {"bytes": calls * (4 * n + 4), "flops": calls * n}
    if kind == "rows":
        return {"bytes": 4 * n + 12 * case["rows"], "flops": 5 * n}
    if kind == "interior":  # sum 1, dot 2, norm 1, argmax 1 operands
        return {"bytes": 5 * 4 * n, "flops": 6 * n}
    if kind == "segmented":
        return {"bytes": 4 * n + 8 * _segments(case) + 4, "flops": n}
    return {"bytes": 8 * n, "flops": n}


# -------------------------------------------------------------- tolerance
def tolerance(case):
    """Integers, max and argmax are exact.  f32 sums are bounded over ranges
    that cancel (uniform about zero) by their terms, not their value, so a
    single total may move more than an element-wise 1e-6."""
    kind = case["kind"]
    if case.get("dtype", "f32") != "f32":
        return "exact"
    if kind in ("scan", "axis_scan"):
        return {"rel": 4e-7, "max": 4e-6}
    if kind == "vector_step":
        return {"rel": 2e-6, "max": 2e-5}
    return {"rel": 1e-5, "max": 1e-4}


# ------------------------------------------------------------------ exact
def _wrap(v):
    """int64 values mod 2^32, as int32."""
    return (((v + 2**31) & 0xFFFFFFFF) - 2**31).to(torch.int32)


def _first_max(x):
    """Lowest index of the maximum along the last axis."""
    top = x.max(dim=-1, keepdim=True).values
    at = torch.arange(x.shape[-1], device=x.device, dtype=torch.int32)
    return torch.where(x == top, at, torch.iinfo(torch.int32).max).min(dim=-1).values.to(torch.int32)


def exact(case, seed):
    kind, values = case["kind"], _inputs(case, seed)
    if kind == "vector_step":
        v, d = values["v"].double(), values["d"].double()
        w = (d + SHIFT) * v
        norm = w.square().sum().sqrt()
        return {"vector": w / norm, "dot": (v * w).sum(), "norm": norm}
    if kind == "axis_batch":
        x = values["x"].view(case["rows"], case["cols"])
        x = (x.t().contiguous() if case["axis"] == 0 else x).double()
        found = {"sum": lambda: x.sum(1), "mean": lambda: x.mean(1), "min": lambda: x.min(1).values,
                 "max": lambda: x.max(1).values, "argmax": lambda: _first_max(x)}
        return {op: found[op]() for op in case["ops"].split(",")}
    if kind == "reduce":
        x = values["x"]
        found = {"sum": lambda: x.double().sum() if case["dtype"] == "f32" else _wrap(x.long().sum()),
                 "max": lambda: x.max().double() if case["dtype"] == "f32" else x.max(),
                 "argmax": lambda: _first_max(x)}
        return {op: found[op]().reshape(1) for op in case["ops"].split(",")}
    if kind == "rows":
        # The prologue's single rounding is part of the operation: max and
        # argmax are of the rounded values.  x / 2 is exact, and the sum
        # with 1/4 rounds once.
        y = values["x"].view(case["rows"], case["cols"]) * PROLOGUE[0] + PROLOGUE[1]
        return {"sum": y.sum(1, dtype=torch.float64), "max": y.max(1).values.double(), "argmax": _first_max(y)}
    if kind == "interior":
        at = (case["rows"], case["cols"]), (case["pitch"], 1), case["offset"]
        x, y = (torch.as_strided(values[k], *at).contiguous() for k in "xy")
        return {"sum": x.sum(dtype=torch.float64).reshape(1), "dot": (x.double() * y.double()).sum().reshape(1),
                "norm": x.double().square().sum().sqrt().reshape(1), "argmax": _first_max(x.view(-1)).reshape(1),
                "max": x.max().double().reshape(1)}
    if kind == "segmented":
        total = torch.zeros(case["n"] + 1, device="cuda", dtype=torch.int64)
        torch.cumsum(values["x"].long(), 0, out=total[1:])
        ends = total[values["offsets"].long()]
        return _wrap(ends[1:] - ends[:-1])
    x = values["x"].view([case["n"]] if kind == "scan" else [case["rows"], case["cols"]])
    axis = case.get("axis", 0)
    x = x.double() if case["dtype"] == "f32" else x.long()
    if case["direction"] == "reverse":
        x = x.flip(axis)
    y = torch.cumsum(x, axis)
    if case["scan"] == "exclusive":
        # Shifted, not subtracted: the first of a line is 0.
        y = y.roll(1, axis)
        y.select(axis, 0).zero_()
    if case["direction"] == "reverse":
        y = y.flip(axis)
    return y if case["dtype"] == "f32" else _wrap(y)
