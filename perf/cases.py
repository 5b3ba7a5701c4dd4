"""The work that is timed: calls of the sparse hot path as a user's program
makes them, through the package's public entry points.

A case is a dict of plain values.  ``listed`` gives the fixed ones, ``draw``
more of the same ranges, ``prepare`` what a program holds before the call
(operands in device memory, descriptors, and the plan, batch or generated
module that it keeps), ``run`` one pass, ``work`` the traffic and arithmetic
a pass cannot do without, ``exact`` the same outputs in 64 bits by plain
torch and ``tolerance`` what another correct order of the sums may differ by.

Kinds of case:
  spmv       y = A x with the default schedule (no schedule argument)
  plan       y = A x through a slab plan kept for the matrix
  spmm       C = A B with the default schedule; bf16 operands go to the
             matrix cores, as the schedule selector sends them
  spgemm     C = A B, all CSR: assemble, then compute
  batch      many CSR instances in one captured launch, SpMV or SpMM
  generated  a module printed by the code generator for one of the
             reference's GPU schedules, or for the merge path

Structures: "uniform" has the same number of entries in every row at random
columns; "powerlaw" has Zipf(2) row lengths on [1, 1e5] scaled to the mean;
"banded" has 2 .. 2*mean - 2 entries a row within 64 columns of the diagonal
(a discretised operator).  Batches mix uniform, banded and 8x8 block-diagonal
instances with 2 .. 64 entries a row.
"""
import ctypes
import math

import numpy as np
import torch

from taco_amd import _lib
from taco_amd import batch as BT
from taco_amd import codegen
from taco_amd import descriptors as D

DEV = "cuda"
BAND = 64
DTYPES = {"f64": torch.float64, "f32": torch.float32, "bf16": torch.bfloat16}
SIZE = {"f64": 8, "f32": 4, "bf16": 2}


# ------------------------------------------------------------------ cases --

def listed():
    return [
        # A small operator applied in a host loop: launches and latency.
        {"name": "spmv_f64_1k", "kind": "spmv", "dtype": "f64", "structure": "uniform",
         "rows": 1000, "mean": 10},
        # The benchmark's uniform matrix: one that fits in the caches.
        {"name": "spmv_f64_uniform_100k", "kind": "spmv", "dtype": "f64", "structure": "uniform",
         "rows": 100000, "mean": 10},
        # One product with a large graph's matrix: no time for a plan.
        {"name": "spmv_f32_powerlaw_2m", "kind": "spmv", "dtype": "f32",
         "structure": "powerlaw", "rows": 2000003, "mean": 16},
        # The benchmark's headline: an iterative solver on the 2M-row
        # power-law matrix, its slab plan built once.
        {"name": "plan_f64_powerlaw_2m", "kind": "plan", "dtype": "f64", "structure": "powerlaw",
         "rows": 2000000, "mean": 16},
        # A block of 64 right-hand sides on a graph's matrix.
        {"name": "spmm_f64_powerlaw_1m", "kind": "spmm", "dtype": "f64", "structure": "powerlaw",
         "rows": 1000000, "mean": 16, "width": 64},
        # An odd number of right-hand sides on a discretised operator.
        {"name": "spmm_f32_banded_w33", "kind": "spmm", "dtype": "f32", "structure": "banded",
         "rows": 400009, "mean": 24, "width": 33},
        # Graph features in bf16 on the matrix cores, at the benchmark's size.
        {"name": "spmm_bf16_powerlaw_2m", "kind": "spmm", "dtype": "bf16",
         "structure": "powerlaw", "rows": 2000000, "mean": 16, "width": 64},
        # The benchmark's SpGEMM: short rows at random columns.
        {"name": "spgemm_f64_uniform_500k", "kind": "spgemm", "dtype": "f64",
         "structure": "uniform", "rows": 500000, "mean": 8},
        # A discretised operator squared (a coarse-grid product): hundreds of
        # candidates a row, most of them repeats.
        {"name": "spgemm_f64_banded_100k", "kind": "spgemm", "dtype": "f64",
         "structure": "banded", "rows": 100003, "mean": 20},
        # Many uneven systems in one launch, replayed as a graph: the
        # benchmark's instance sizes with the schedule its tuner picks.
        {"name": "batch_spmv_f32", "kind": "batch", "op": "spmv", "instances": 128,
         "rmin": 1000, "rmax": 200000, "lanes": 0, "width": 1},
        {"name": "batch_spmm_f32_w32", "kind": "batch", "op": "spmm", "instances": 128,
         "rmin": 1000, "rmax": 200000, "lanes": 8, "width": 32},
        # The reference's fused, position-split SpMV schedule, compiled.
        {"name": "generated_spmv_nnz_1m", "kind": "generated", "spec": "spmv_nnz_f64",
         "dtype": "f64", "structure": "powerlaw", "rows": 1000000, "mean": 16},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["spmv", "spmv", "plan", "spmm", "spmm", "spgemm", "batch", "generated"])
    structure = rng.choice(["uniform", "powerlaw", "banded"])
    mean = rng.randint(4, 32)
    if kind == "batch":
        op = rng.choice(["spmv", "spmm"])
        rmax = _log_int(rng, 4000, 200000)
        width = 1 if op == "spmv" else rng.choice([16, 20, 32, 48])
        lanes = 0 if op == "spmv" else 8 if width <= 32 else 16
        return {"kind": kind, "op": op, "instances": rng.randint(8, 96), "rmin": 1000,
                "rmax": rmax, "lanes": lanes, "width": width}
    case = {"kind": kind, "dtype": "f64", "structure": structure,
            "rows": _log_int(rng, 1000, 1500000), "mean": mean}
    if kind == "spmv":
        case["dtype"] = rng.choice(["f64", "f32"])
        case["rows"] = min(case["rows"], 32000000 // mean)
    elif kind == "plan":
        case["rows"] = min(_log_int(rng, 100000, 2000000), 32000000 // mean)
    elif kind == "spmm":
        case["dtype"] = rng.choice(["f64", "f32", "bf16"])
        width = _log_int(rng, 3, 256)
        if case["dtype"] == "bf16":
            width = max(4, width // 4 * 4)
        case["width"] = width
        case["rows"] = max(1000, min(case["rows"], 1000000000 // (mean * width)))
    elif kind == "spgemm":
        case["structure"] = structure = rng.choice(["uniform", "banded"])
        case["mean"] = mean = rng.randint(4, 24)
        case["rows"] = _log_int(rng, 1000, 30000000 // (mean * mean))
    else:
        case["spec"] = rng.choice(["spmv_rows_f64", "spmv_nnz_f64", "spmv_merge_f64",
                                   "spmv_nnz_f32", "spmm_merge_f64"])
        if case["spec"].endswith("f32"):
            case["dtype"] = "f32"
        if case["spec"].startswith("spmm"):
            case["width"] = rng.randint(16, 128)
            case["rows"] = min(case["rows"], 250000)
        case["rows"] = min(case["rows"], 16000000 // mean)
    return case


# ----------------------------------------------------------------- inputs --

def _rand(n, g, dtype=torch.float64):
    return torch.rand(n, generator=g, device=DEV, dtype=dtype)


def _values(n, g, dtype):
    """U[-1, 1) in the given type."""
    v = torch.rand(n, generator=g, device=DEV,
                   dtype=torch.float64 if dtype == "f64" else torch.float32)
    return v.mul_(2).sub_(1).to(DTYPES[dtype])


def _counts(m, structure, mean, g):
    if structure == "uniform":
        return torch.full((m,), mean, dtype=torch.int64, device=DEV)
    if structure == "banded":
        return torch.randint(2, 2 * mean - 1, (m,), generator=g, device=DEV)
    u = (torch.randperm(m, generator=g, device=DEV).double() + 0.5) / m
    raw = (1.0 / u).clamp_(max=min(1e5, float(m)))
    return (raw * (mean / raw.mean())).round_().clamp_(1, m // 2 + 1).long()


def _pack(rows, cols, m, bits):
    """pos, crd (int32), and the row of every entry (int64), of the distinct
    (row, column) pairs; columns sorted inside a row."""
    key = torch.unique((rows << bits) | cols)
    r = key >> bits
    pos = torch.zeros(m + 1, dtype=torch.int32, device=DEV)
    pos[1:] = torch.cumsum(torch.bincount(r, minlength=m), 0)
    return pos, (key & ((1 << bits) - 1)).int(), r


def _pattern(m, structure, mean, g):
    rows = torch.repeat_interleave(torch.arange(m, device=DEV),
                                   _counts(m, structure, mean, g))
    if structure == "banded":
        off = torch.randint(-BAND, BAND + 1, rows.shape, generator=g, device=DEV)
        cols = (rows + off).clamp_(0, m - 1)
    else:
        cols = (_rand(rows.numel(), g) * m).long().clamp_(max=m - 1)
    return _pack(rows, cols, m, 31)


def _factor_patterns(case, g):
    """The patterns of an SpGEMM's operands: a fixed pair of matrices under
    a relabelling drawn from g, so that every seed gives other patterns of
    products with one size.  Banded matrices are shifted cyclically, others
    permuted."""
    m = case["rows"]
    base = torch.Generator(device=DEV)
    base.manual_seed(m * 64 + case["mean"])
    pairs = []
    for _ in range(2):
        _, crd, rows = _pattern(m, case["structure"], case["mean"], base)
        pairs.append((rows, crd.long()))
    if case["structure"] == "banded":
        shift = int(torch.randint(0, m, (1,), generator=g, device=DEV))
        return [_pack((r + shift) % m, (c + shift) % m, m, 31) for r, c in pairs]
    p, q, s = (torch.randperm(m, generator=g, device=DEV) for _ in range(3))
    (ra, ca), (rb, cb) = pairs
    return [_pack(p[ra], q[ca], m, 31), _pack(q[rb], s[cb], m, 31)]


def _batch_pattern(case, g):
    """Concatenated instances: m, nnz per instance, row -> instance, local
    pos and crd."""
    n = case["instances"]
    u = (torch.randperm(n, generator=g, device=DEV).double() + 0.5) / n
    md = (case["rmin"] * (case["rmax"] / case["rmin"]) ** u).long()
    m = md.cpu().numpy()
    row_off = torch.cat([torch.zeros(1, dtype=torch.int64, device=DEV), torch.cumsum(md, 0)])
    total = int(row_off[-1])
    inst = torch.repeat_interleave(torch.arange(n, device=DEV), md)
    local = torch.arange(total, device=DEV) - row_off[inst]
    size = md[inst]
    structure = torch.randint(0, 3, (n,), generator=g, device=DEV)
    counts = torch.randint(2, 65, (total,), generator=g, device=DEV)
    counts = torch.where(structure[inst] == 2, torch.full_like(counts, 8), counts)
    rows = torch.repeat_interleave(torch.arange(total, device=DEV), counts)
    first = torch.cumsum(counts, 0) - counts
    rank = torch.arange(rows.numel(), device=DEV) - first[rows]
    here, top = local[rows], size[rows] - 1
    cols = (_rand(rows.numel(), g) * size[rows]).long()
    s = structure[inst][rows]
    off = torch.randint(-BAND, BAND + 1, rows.shape, generator=g, device=DEV)
    cols = torch.where(s == 1, here + off, cols)
    cols = torch.where(s == 2, here // 8 * 8 + rank, cols)
    cols = torch.minimum(cols.clamp_(min=0), top)
    gpos, crd, rows = _pack(rows, cols, total, 20)
    starts = gpos[row_off].long()
    nnz = (starts[1:] - starts[:-1]).cpu().numpy()
    # Local offsets: every instance has m + 1 of them, starting at 0.
    pos = torch.empty(total + n, dtype=torch.int32, device=DEV)
    at = torch.arange(total, device=DEV) + inst
    pos[at] = gpos[:-1] - gpos[row_off[inst]]
    pos[row_off[1:] + torch.arange(n, device=DEV)] = (starts[1:] - starts[:-1]).int()
    return m, nnz, inst, row_off, pos, crd, rows


def _inputs(case, seed):
    """The operands, made from the seed alone."""
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    kind = case["kind"]
    if kind == "batch":
        m, nnz, inst, row_off, pos, crd, rows = _batch_pattern(case, g)
        total, w = int(row_off[-1]), case["width"]
        return {"m": m, "nnz": nnz, "pos": pos, "crd": crd, "rows": rows,
                "cols": (rows, row_off, inst), "vals": _values(crd.numel(), g, "f32"),
                "x": _values(total * w, g, "f32"), "total": total}
    m, dtype = case["rows"], case["dtype"]
    s = {}
    if kind == "spgemm":
        (s["pos"], s["crd"], s["rows"]), (s["pos2"], s["crd2"], _) = _factor_patterns(case, g)
        s["vals"] = _values(s["crd"].numel(), g, dtype)
        s["vals2"] = _values(s["crd2"].numel(), g, dtype)
        return s
    s["pos"], s["crd"], s["rows"] = _pattern(m, case["structure"], case["mean"], g)
    s["vals"] = _values(s["crd"].numel(), g, dtype)
    if "width" in case:
        s["x"] = _values(m * case["width"], g, dtype).view(m, case["width"])
    else:
        s["x"] = _values(m, g, dtype)
    return s


def _bits(t):
    return t.view(torch.int16) if t.dtype == torch.bfloat16 else t


class _Workload:
    """What a batch borrows: the instances' sizes and device buffers."""


class _Block:
    """A device array that the library allocated for an output; freed with
    the last tensor over it."""

    def __init__(self, address, count, typestr):
        self.address = address
        self.__cuda_array_interface__ = {"shape": (count,), "typestr": typestr,
                                         "data": (address, False), "version": 2}

    def __del__(self):
        if _lib is not None and _lib._lib is not None:
            _lib._lib.taco_hip_unified_free(ctypes.c_void_p(self.address))


def _owned(address, count, typestr, dtype):
    if not address:
        return torch.empty(0, dtype=dtype, device=DEV)
    return torch.as_tensor(_Block(address, count, typestr), device=DEV)


def prepare(case, seed):
    s = _inputs(case, seed)
    s["kind"] = kind = case["kind"]
    s.pop("rows")
    if kind == "batch":
        s.pop("cols")
        w = _Workload()
        w.ninst, w.width, w.m, w.nnz = case["instances"], case["width"], s["m"], s["nnz"]
        w.pos, w.crd, w.vals = s["pos"], s["crd"], s["vals"]
        w.x = w.B = s["x"]
        w.y = w.C = s["out"] = torch.zeros(s["total"] * case["width"], device=DEV)
        op = 0 if case["op"] == "spmv" else 1
        s["batch"] = BT.Batch(w, op, np.full(case["instances"], case["lanes"], np.int32))
        s["batch"].capture()
        return s
    m, dtype = case["rows"], case["dtype"]
    s["shape"] = (m, m)
    s["A"] = D.csr(s["pos"], s["crd"], _bits(s["vals"]), (m, m), dtype)
    if kind == "spgemm":
        s["B"] = D.csr(s["pos2"], s["crd2"], s["vals2"], (m, m), dtype)
        return s
    s["in"] = D.dense(_bits(s["x"]), dtype)
    out = "f32" if dtype == "bf16" else dtype
    s["out"] = torch.zeros(s["x"].shape, dtype=DTYPES[out], device=DEV)
    s["y"] = D.dense(s["out"], out)
    s["schedule"] = None
    if kind == "plan":
        s["plan"] = _lib.SpmvPlan(s["A"])
    elif kind == "generated":
        s["kernel"] = codegen.Kernel(codegen.standard(case["spec"]))
    elif dtype == "bf16":
        s["schedule"] = _lib.Schedule()
        s["schedule"].algo = _lib.MFMA
    return s


def run(s):
    kind = s["kind"]
    L = _lib.lib()
    if kind == "spmv":
        _lib.check(L.taco_hip_spmv_compute(s["y"].ptr, s["A"].ptr, s["in"].ptr, None))
    elif kind == "spmm":
        _lib.check(L.taco_hip_spmm_compute(s["y"].ptr, s["A"].ptr, s["in"].ptr, s["schedule"]))
    elif kind == "plan":
        s["plan"].compute(s["y"], s["in"])
    elif kind == "generated":
        s["kernel"].compute(s["y"], s["A"], s["in"])
    elif kind == "batch":
        s["batch"].launch_graph()
    else:
        c = D.csr_empty(s["shape"])
        _lib.check(L.taco_hip_spgemm_assemble(c.ptr, s["A"].ptr, s["B"].ptr), "assemble")
        _lib.check(L.taco_hip_spgemm_compute(c.ptr, s["A"].ptr, s["B"].ptr), "compute")
        m, nnz = s["shape"][0], c.t.vals_size
        return {"pos": _owned(c.level_ptr(1, 0), m + 1, "<i4", torch.int32),
                "crd": _owned(c.level_ptr(1, 1), nnz, "<i4", torch.int32),
                "vals": _owned(c.vals_ptr(), nnz, "<f8", torch.float64)}
    return s["out"]


# ------------------------------------------------------- work and results --

def _distinct(picks, among):
    """Expected distinct values of `picks` draws among `among`."""
    return among * -math.expm1(picks * math.log1p(-1.0 / among)) if among > 1 else 1.0


def _row_entries(case):
    m, mean = case["rows"], case["mean"]
    if case["structure"] == "banded":
        w = 2 * BAND + 1
        return sum(_distinct(k, w) for k in range(2, 2 * mean - 1)) / (2 * mean - 3)
    return _distinct(mean, m) if case["structure"] == "uniform" else float(mean)


def work(case):
    kind = case["kind"]
    if kind == "batch":
        lo, hi, n = case["rmin"], case["rmax"], case["instances"]
        rows = n * (hi - lo) / math.log(hi / lo)
        banded = sum(_distinct(k, 2 * BAND + 1) for k in range(2, 65)) / 63
        nnz = rows * (33 + banded + 8) / 3
        return {"bytes": 4 * (rows + n) + 8 * nnz + 8 * rows * case["width"],
                "flops": 2 * nnz * case["width"]}
    m, v = case["rows"], SIZE[case["dtype"]]
    each = _row_entries(case)
    nnz = m * each
    if kind == "spgemm":
        among = 4 * BAND + 1 if case["structure"] == "banded" else m
        out = m * _distinct(each * each, min(m, among))
        # assemble reads both patterns; compute reads both operands whole
        # and writes the values on the pattern.
        return {"bytes": 2 * 2 * 4 * (m + 1) + 2 * (4 + 4 + v) * nnz + 4 * (m + 1)
                + (4 + v) * out, "flops": 2 * nnz * each}
    w = case.get("width", 1)
    out = 4 if case["dtype"] == "bf16" else v
    return {"bytes": 4 * (m + 1) + (4 + v) * nnz + (v + out) * m * w, "flops": 2 * nnz * w}


def tolerance(case):
    """Sums in another order, at the type the sums are held in (bf16 operands
    are summed in f32): four times what was seen.  Against 64 bits f32 sums
    were 1.1e-7 off (bf16 1.5e-7); two runs of the plan, whose rows of 1e5
    terms are summed in no fixed order, differed by 3.5e-15 in norm and
    7.7e-13 at most, and two runs of the bf16 case by 1.1e-5 at most."""
    if case["kind"] != "batch" and case["dtype"] == "f64":
        return {"rel": 2e-14, "max": 3e-12}
    return {"rel": 5e-7, "max": 5e-5}


def _product(rows, cols, vals, x, m):
    """Sums of vals * x[cols] by row, 64 bits, in chunks of entries."""
    w = x.shape[1]
    out = torch.zeros(m, w, dtype=torch.float64, device=DEV)
    step = max(1, (1 << 27) // w)
    for a in range(0, rows.numel(), step):
        b = a + step
        out.index_add_(0, rows[a:b], vals[a:b, None] * x[cols[a:b]].double())
    return out


def exact(case, seed):
    s = _inputs(case, seed)
    kind = case["kind"]
    vals = s["vals"].double()
    if kind == "batch":
        rows, row_off, inst = s["cols"]
        cols = s["crd"].long() + row_off[inst[rows]]
        return _product(rows, cols, vals, s["x"].view(-1, case["width"]), s["total"]).view(-1)
    m = case["rows"]
    if kind != "spgemm":
        x = s["x"].view(m, -1)
        return _product(s["rows"], s["crd"].long(), vals, x, m).view(s["x"].shape)
    # Every candidate (row of A's entry, column of B's entry) and its product.
    j = s["crd"].long()
    start, end = s["pos2"][j].long(), s["pos2"][j + 1].long()
    entry = torch.repeat_interleave(torch.arange(j.numel(), device=DEV), end - start)
    first = torch.cumsum(end - start, 0) - (end - start)
    at = start[entry] + torch.arange(entry.numel(), device=DEV) - first[entry]
    key = (s["rows"][entry] << 31) | s["crd2"][at].long()
    key, slot = torch.unique(key, return_inverse=True)
    out = torch.zeros(key.numel(), dtype=torch.float64, device=DEV)
    out.index_add_(0, slot, vals[entry] * s["vals2"].double()[at])
    pos = torch.zeros(m + 1, dtype=torch.int32, device=DEV)
    pos[1:] = torch.cumsum(torch.bincount(key >> 31, minlength=m), 0)
    return {"pos": pos, "crd": (key & ((1 << 31) - 1)).int(), "vals": out}
