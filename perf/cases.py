"""Timed workloads of the tcuscan operators.

Each case is a plain dict: an operator, its sizes and its data type.
`listed()` names the fixed ones, `draw(rng)` gives others of the same
operators over the same ranges, `prepare` builds a case's inputs on the GPU
from a seed, `run` makes one pass through the public entry points, `work`
states the bytes and operations that pass cannot do without, and `exact`
computes the same outputs with torch in 64 bits.
"""
from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "pytorch-tcuscan_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import tcuscan  # noqa: E402
from tcuscan import workloads  # noqa: E402

S = 128  # the tile side the reference's benchmarks use

_TORCH = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32,
          "int8": torch.int8, "int16": torch.int16, "int32": torch.int32}
_BYTES = {"fp16": 2, "bf16": 2, "fp32": 4, "int8": 1, "int16": 2, "int32": 4}


def listed():
    return [
        # The plain 1-D scan of 2^20 values: one launch, latency counts.
        {"name": "scan_f16_2p20", "op": "scan", "entry": "single_core", "dtype": "fp16", "n": 1 << 20},
        # The large scan (prefix sums of a whole tensor): the headline workload.
        {"name": "scan_f16_2p28", "op": "scan", "entry": "multi_core", "dtype": "fp16", "n": 1 << 28},
        # Counting scan (offsets from 0/1 or small counts) of a ragged length.
        {"name": "scan_i8_odd", "op": "scan", "entry": "multi_core", "dtype": "int8", "n": 33554467},
        # Many short segments over int8 data, as a batch of indptr seg-sums is laid out.
        {"name": "segsum_i8_2p26", "op": "seg_sum", "dtype": "int8", "rows": 1 << 20, "mean": 64},
        # CSR SpMV on the 2^22 x 2^22 matrix with lognormal row lengths.
        {"name": "spmv_f16_2p22", "op": "spmv", "dtype": "fp16", "rows": 1 << 22, "mean": 16},
        # Compaction of values and indices by a Bernoulli(0.3) mask, the large configuration.
        {"name": "compress_f32_2p28", "op": "compress_ind", "dtype": "fp32", "n": 1 << 28, "p": 0.3},
        # A filter by value on an ordinary, odd-sized column.
        {"name": "filter_f16_10m", "op": "filter", "cmp": "ge", "dtype": "fp16", "n": 10000019, "pivot": 0.5},
        # The large sort of fp16 keys with their positions.
        {"name": "sort_f16_2p28", "op": "sort", "dtype": "fp16", "n": 1 << 28, "descending": False},
        # A small sort of 32-bit keys, where launches count.
        {"name": "sort_i32_100k", "op": "sort", "dtype": "int32", "n": 100003, "descending": False},
        # The 2048 largest of a large tensor.
        {"name": "topk_f16_2p28", "op": "topk", "dtype": "fp16", "n": 1 << 28, "k": 2048},
        # Lookup of random keys in a sorted table.
        {"name": "searchsorted_2p24", "op": "searchsorted", "n": 1 << 24, "needles": 1 << 24},
        # Nucleus filtering of one vocabulary's probabilities in a sampling loop.
        {"name": "top_p_131071", "op": "top_p", "dtype": "fp16", "n": 131071, "p": 0.9},
    ]


def _size(rng, lo, hi):
    """Log-uniform in [2^lo, 2^hi], half of them odd."""
    n = int(2 ** rng.uniform(lo, hi))
    return n | 1 if rng.random() < 0.5 else n & -16


def draw(rng):
    op = rng.choice(["scan", "scan", "seg_sum", "spmv", "compress_ind", "filter", "sort", "sort", "topk",
                     "searchsorted", "top_p"])
    if op == "scan":
        return {"op": op, "entry": rng.choice(["single_core", "multi_core"]),
                "dtype": rng.choice(["fp16", "bf16", "int8"]), "n": _size(rng, 8, 28)}
    if op == "seg_sum":
        return {"op": op, "dtype": rng.choice(["int8", "fp16"]), "rows": _size(rng, 8, 20),
                "mean": rng.choice([8, 16, 64])}
    if op == "spmv":
        return {"op": op, "dtype": rng.choice(["fp16", "fp32"]), "rows": _size(rng, 14, 21.5), "mean": 16}
    if op == "compress_ind":
        return {"op": op, "dtype": rng.choice(["fp32", "fp16"]), "n": _size(rng, 10, 27.5),
                "p": round(rng.uniform(0.05, 0.9), 3)}
    if op == "filter":
        return {"op": op, "cmp": rng.choice(["ge", "le", "where"]), "dtype": rng.choice(["fp16", "fp32"]),
                "n": _size(rng, 10, 27.5), "pivot": round(rng.uniform(-1.5, 1.5), 3)}
    if op == "sort":
        dtype = rng.choice(["fp16", "int16", "fp32", "int32"])
        return {"op": op, "dtype": dtype, "n": _size(rng, 10, 27.5 if _BYTES[dtype] == 2 else 26),
                "descending": rng.random() < 0.3}
    if op == "topk":
        n = _size(rng, 12, 27.5)
        return {"op": op, "dtype": rng.choice(["fp16", "int16", "fp32"]), "n": n,
                "k": max(1, _size(rng, 0, 12))}
    if op == "searchsorted":
        return {"op": op, "n": _size(rng, 10, 24), "needles": _size(rng, 10, 24)}
    return {"op": op, "dtype": "fp16", "n": _size(rng, 12, 20), "p": rng.choice([0.5, 0.9, 0.95])}


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _uniform(n, dtype, g):
    """U[-1, 1] rounded to dtype; integers uniform in [-4, 4]."""
    if dtype == "int8":
        return torch.randint(-4, 5, (n,), generator=g, device="cuda", dtype=torch.int8)
    return (torch.rand(n, generator=g, device="cuda") * 2 - 1).to(_TORCH[dtype])


def _keys(n, dtype, g):
    """Standard normals; integers over the type's whole range."""
    if dtype in ("int16", "int32"):
        i = torch.iinfo(_TORCH[dtype])
        return torch.randint(i.min, i.max + 1, (n,), generator=g, device="cuda", dtype=torch.int64).to(_TORCH[dtype])
    return torch.randn(n, generator=g, device="cuda").to(_TORCH[dtype])


def _kept(case, x):
    pivot = torch.tensor(case["pivot"], dtype=torch.float32).to(x.dtype).to(x.device)
    return x <= pivot if case["cmp"] == "le" else x >= pivot


def _filter_input(case, g):
    """Standard normals, a few of them moved across the pivot so that every
    seed keeps as many: the expected number."""
    x = _keys(case["n"], case["dtype"], g)
    want = round(_kept_share(case) * case["n"])
    keep = _kept(case, x)
    extra = int(keep.sum()) - want
    if extra:
        at = torch.nonzero(keep if extra > 0 else ~keep).flatten()
        at = at[torch.randperm(at.numel(), generator=g, device="cuda")[:abs(extra)]]
        x[at] = case["pivot"] + (1.0 if (extra > 0) == (case["cmp"] == "le") else -1.0)
    return x


def prepare(case, seed):
    g, op = _gen(seed), case["op"]
    st = {"case": case}
    if op == "scan":
        st["x"] = _uniform(case["n"], case["dtype"], g)
    elif op == "seg_sum":
        # Geometric segment lengths of the given mean, at least 1.
        u = torch.rand(case["rows"], generator=g, device="cuda", dtype=torch.float64)
        lens = 1 + torch.floor(torch.log1p(-u) / math.log1p(-1.0 / case["mean"])).long()
        ends = torch.cumsum(lens, 0)
        st["indptr"] = torch.cat([ends.new_zeros(1), ends]).int()
        nnz = int(ends[-1])
        if case["dtype"] == "int8":
            st["x"] = torch.randint(-128, 128, (nnz,), generator=g, device="cuda", dtype=torch.int8)
        else:
            st["x"] = _uniform(nnz, case["dtype"], g)
    elif op == "spmv":
        st["vals"], st["indptr"], st["cols"], st["x"] = workloads.lognormal_csr(
            case["rows"], case["rows"], case["mean"], 1.2, 20000, seed, torch.device("cuda"),
            _TORCH[case["dtype"]])
    elif op == "compress_ind":
        n = case["n"]
        st["x"] = torch.rand(n, generator=g, device="cuda").to(_TORCH[case["dtype"]])
        # round(p * n) ones in random places: every seed keeps as many.
        order = torch.randperm(n, generator=g, device="cuda", dtype=torch.int32)
        st["mask"] = (order < round(case["p"] * n)).to(torch.int8)
        st["idx"] = torch.arange(n, dtype=torch.int32, device="cuda")
    elif op == "filter":
        st["x"] = _filter_input(case, g)
    elif op in ("sort", "topk"):
        st["x"] = _keys(case["n"], case["dtype"], g)
    elif op == "searchsorted":
        st["table"] = torch.sort(_keys(case["n"], "int32", g)).values
        st["needles"] = _keys(case["needles"], "int32", g)
    else:
        # Softmax of normal logits with standard deviation 2.
        logits = torch.randn(case["n"], generator=g, device="cuda") * 2
        st["probs"] = torch.softmax(logits, 0).half()
    return st


def run(state):
    c = state["case"]
    op = c["op"]
    if op == "scan":
        if c["entry"] == "single_core":
            return tcuscan.run_scan_single_core(state["x"], S)
        return tcuscan.run_scan_multi_core(state["x"], S)
    if op == "seg_sum":
        return tcuscan.run_seg_sum_multi_core(state["x"], state["indptr"], S)
    if op == "spmv":
        return tcuscan.run_spmv_v2(state["vals"], state["indptr"], state["cols"], state["x"], S)
    if op == "compress_ind":
        return tcuscan.run_compress_ind(state["x"], state["idx"], state["mask"], S)
    if op == "filter":
        f = {"ge": tcuscan.run_filter_greater_eq, "le": tcuscan.run_filter_less_eq, "where": tcuscan.run_where}
        return f[c["cmp"]](state["x"], c["pivot"], S)
    if op == "sort":
        if c["descending"]:
            return tcuscan.run_radix_sort_ex(state["x"], True)
        return tcuscan.run_radix_sort(state["x"], S)
    if op == "topk":
        if c["dtype"] == "fp16":
            return tcuscan.run_topk_fp16(state["x"], c["k"], -10.0, 10.0, S)
        return tcuscan.run_topk(state["x"], c["k"], True)
    if op == "searchsorted":
        return tcuscan.run_searchsorted(state["table"], state["needles"])
    return tcuscan.top_p_filter(state["probs"], c["p"], S)


def _kept_share(case):
    """Expected share of standard normals a filter keeps."""
    above = 0.5 * math.erfc(case["pivot"] / math.sqrt(2.0))
    return 1.0 - above if case["cmp"] == "le" else above


def work(case):
    op = case["op"]
    n, e = case.get("n", 0), _BYTES.get(case.get("dtype"), 4)
    if op == "scan":
        return {"bytes": n * (e + 4), "flops": n}
    if op == "seg_sum":
        nnz = case["rows"] * case["mean"]
        return {"bytes": nnz * e + case["rows"] * 8, "flops": nnz}
    if op == "spmv":
        nnz = case["rows"] * case["mean"]
        return {"bytes": nnz * (e + 4) + case["rows"] * (e + 8), "flops": 2 * nnz}
    if op == "compress_ind":
        return {"bytes": n * (e + 5) + case["p"] * n * (e + 4), "flops": 0}
    if op == "filter":
        return {"bytes": n * e + _kept_share(case) * n * (4 if case["cmp"] == "where" else e), "flops": 0}
    if op == "sort":
        return {"bytes": n * (2 * e + 4), "flops": 0}
    if op == "topk":
        return {"bytes": n * e + case["k"] * (e + 4), "flops": 0}
    if op == "searchsorted":
        return {"bytes": 4 * n + 8 * case["needles"], "flops": 0}
    return {"bytes": n * (2 + 4 + 4), "flops": 2 * n}  # probabilities in; kept weights and order out


def exact(case, seed):
    st = prepare(case, seed)
    op = case["op"]
    if op == "scan":
        return None if case["dtype"] == "int8" else torch.cumsum(st["x"].double(), 0)
    if op == "seg_sum":
        if case["dtype"] == "int8":
            return None
        sums = torch.cat([torch.zeros(1, dtype=torch.float64, device="cuda"), torch.cumsum(st["x"].double(), 0)])
        return torch.diff(sums[st["indptr"].long()])
    if op == "spmv":
        lens = torch.diff(st["indptr"]).long()
        row = torch.repeat_interleave(torch.arange(lens.numel(), device="cuda"), lens)
        prod = st["vals"].double() * st["x"].double()[st["cols"].long()]
        return torch.zeros(lens.numel(), dtype=torch.float64, device="cuda").index_add_(0, row, prod)
    if op == "compress_ind":
        return st["x"][st["mask"].bool()].double(), None
    if op == "filter":
        if case["cmp"] == "where":
            return None
        return st["x"][_kept(case, st["x"])].double()
    if op == "sort":
        if case["dtype"].startswith("int"):
            return None
        return torch.sort(st["x"], descending=case["descending"]).values.double(), None
    if op == "topk":
        if case["dtype"].startswith("int"):
            return None
        return torch.topk(st["x"], case["k"]).values.double(), None
    if op == "searchsorted":
        return None
    srt = torch.sort(st["probs"], descending=True).values.double()
    mass = torch.cumsum(srt, 0)
    kept = torch.where(mass - srt > float(np.float32(case["p"])), torch.zeros_like(srt), srt)
    return kept / kept.sum(), None
