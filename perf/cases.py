"""The calls this library is used for, as measurable cases: SpMM and SDDMM on GNN-style graphs through
``trspmm.Plan``, and the path of a graph seen for the first time (format, plan, one product).

A case is a plain dict:

    op      "spmm"   C = A B with a plan the program keeps (a layer's aggregation)
            "sddmm"  out[e] = X[row_e] . Y[col_e] with a plan the program keeps (attention scores, and
                     the gradient of the SpMM with respect to its values)
            "fresh"  the format built on the GPU, the plan made and one SpMM (a sampled or changed graph)
    graph   "er"     uniform random edges plus self loops, values D^-1/2 (A + I) D^-1/2
            "rmat"   power law (0.57, 0.19, 0.19, 0.05), symmetric
            "sbm"    communities of 16 nodes, p_in 0.6, plus `degree` random edges per node
            "grid"   4-neighbour grid of `nodes` = side^2 nodes plus 64 hub rows
    nodes, degree, k  the sizes; k is the feature width

The graphs are those of trspmm.graphs (the benchmark's and the tests'), sampled with torch on the GPU.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tr-spmm_zzx_amd"))

import trspmm  # noqa: E402

#: Stored entries times features of the largest listed case: no drawn case has more.
MOST_WORK = 17_000_000 * 256


def listed():
    return [
        # citation-graph size: one GCN layer, where launches and latency count
        {"name": "spmm er 4k k64", "op": "spmm", "graph": "er", "nodes": 4096, "degree": 16, "k": 64},
        # a sampled mini-batch subgraph with hubs, hidden width 64
        {"name": "spmm rmat 16k k64", "op": "spmm", "graph": "rmat", "nodes": 1 << 14, "degree": 16, "k": 64},
        # attention scores on a mid-size graph at an odd head width
        {"name": "sddmm rmat 64k k33", "op": "sddmm", "graph": "rmat", "nodes": 1 << 16, "degree": 16, "k": 33},
        # a graph seen for the first time: format, plan and one layer
        {"name": "fresh rmat 256k k128", "op": "fresh", "graph": "rmat", "nodes": 1 << 18, "degree": 16, "k": 128},
        # class scores of the last layer (an odd width) on a community graph
        {"name": "spmm sbm 250k k41", "op": "spmm", "graph": "sbm", "nodes": 250_000, "degree": 4, "k": 41},
        # the headline: power-law graph of 2^20 nodes and 31M entries, hidden width 128
        {"name": "spmm rmat 1m k128", "op": "spmm", "graph": "rmat", "nodes": 1 << 20, "degree": 16, "k": 128},
        # the same graph at a narrow hidden width
        {"name": "spmm rmat 1m k32", "op": "spmm", "graph": "rmat", "nodes": 1 << 20, "degree": 16, "k": 32},
        # the same graph at an input feature width that is no multiple of 8
        {"name": "spmm rmat 1m k100", "op": "spmm", "graph": "rmat", "nodes": 1 << 20, "degree": 16, "k": 100},
        # dense blocks of 16 rows: the matrix-core windows, wide features
        {"name": "spmm sbm 1m k256", "op": "spmm", "graph": "sbm", "nodes": 1_000_000, "degree": 4, "k": 256},
        # a mesh with a few very long rows
        {"name": "spmm grid 4m k32", "op": "spmm", "graph": "grid", "nodes": 2048 * 2048, "degree": 4, "k": 32},
        # attention scores on the headline graph, one wide head and one narrow head
        {"name": "sddmm rmat 1m k128", "op": "sddmm", "graph": "rmat", "nodes": 1 << 20, "degree": 16, "k": 128},
        {"name": "sddmm rmat 1m k32", "op": "sddmm", "graph": "rmat", "nodes": 1 << 20, "degree": 16, "k": 32},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """Graphs of 4096 to 2^20 nodes (grids to 2048 x 2048), widths 8 to 256, half of them multiples of 8."""
    while True:
        graph = rng.choice(["er", "rmat", "rmat", "sbm", "grid"])
        degree = rng.randint(4, 16)
        if graph == "rmat":
            nodes = 1 << rng.randint(12, 20)
        elif graph == "grid":
            nodes = _log_int(rng, 64, 2048) ** 2
            degree = 4
        else:
            nodes = _log_int(rng, 4096, 1 << 20)
            degree = min(degree, 8) if graph == "sbm" else degree
        k = _log_int(rng, 8, 256)
        if rng.random() < 0.5:
            k = (k + 7) // 8 * 8
        op = rng.choice(["spmm", "spmm", "sddmm", "fresh"] if nodes <= 1 << 18 else ["spmm", "spmm", "sddmm"])
        case = {"op": op, "graph": graph, "nodes": nodes, "degree": degree, "k": k}
        if _entries(case) * k <= MOST_WORK:
            return case


def _hub_degree(nodes):
    return max(64, nodes // 42)


def _sampled(case):
    """Edges that are sampled at random: undirected pairs, or the hub rows' entries of a grid."""
    n, d = case["nodes"], case["degree"]
    return {"er": n * d // 2, "rmat": n * d * 15 // 16, "sbm": n * d, "grid": 64 * _hub_degree(n)}[case["graph"]]


def _fixed(case):
    """Pairs inside the communities; the grid's own entries."""
    n = case["nodes"]
    return {"er": 0, "rmat": 0, "sbm": n // 16 * 72, "grid": 4 * n - 4 * math.isqrt(n)}[case["graph"]]


def _entries(case):
    """Stored entries, the same for every seed."""
    n, e = case["nodes"], _sampled(case) + _fixed(case)
    return e if case["graph"] == "grid" else 2 * e + (n if case["graph"] == "er" else 0)


# ------------------------------------------------------------------------------------------------
# Graphs: canonical CSR on the GPU (int32 rowptr padded to 16 rows, int32 col, float32 val that fp16 holds).

def _rand(shape, gen):
    return torch.rand(shape, generator=gen, device="cuda")


def _randint(hi, shape, gen):
    return torch.randint(hi, shape, generator=gen, device="cuda")


def _perm(n, gen):
    return torch.randperm(n, generator=gen, device="cuda")


def _pairs(u, v, n):
    """Keys u * n + v with u < v of the pairs that are no self loops."""
    keep = u != v
    return torch.minimum(u, v)[keep] * n + torch.maximum(u, v)[keep]


def _rmat_pairs(n, count, gen):
    u = torch.zeros(count, dtype=torch.int64, device="cuda")
    v = torch.zeros_like(u)
    for _ in range(n.bit_length() - 1):
        r = _rand(count, gen)
        u = (u << 1) | (r >= 0.76)
        v = (v << 1) | (((r >= 0.57) & (r < 0.76)) | (r >= 0.95))
    return _pairs(u, v, n)


def _with_sampled(base, sample, count, gen):
    """base (distinct keys) and `count` other distinct keys out of sample(number of draws)."""
    more = torch.empty(0, dtype=torch.int64, device="cuda")
    while more.shape[0] < count:
        more = torch.unique(torch.cat([more, sample((count - more.shape[0]) * 21 // 20 + 64)]))
        if base.shape[0]:
            more = more[~torch.isin(more, base)]
    return torch.cat([base, more[_perm(more.shape[0], gen)[:count]]])


def _keys(case, gen):
    """Distinct keys row * n + col of all stored entries, sorted."""
    n, graph, count = case["nodes"], case["graph"], _sampled(case)
    none = torch.empty(0, dtype=torch.int64, device="cuda")
    if graph == "grid":
        side = math.isqrt(n)
        idx = torch.arange(n, device="cuda")
        r, c = idx // side, idx % side
        base = []
        for dr, dc in ((0, 1), (0, -1), (1, 0), (-1, 0)):
            ok = (r + dr >= 0) & (r + dr < side) & (c + dc >= 0) & (c + dc < side)
            base.append(idx[ok] * n + (r[ok] + dr) * side + c[ok] + dc)
        hubs = _perm(n, gen)[:64]
        keys = _with_sampled(torch.cat(base), lambda q: hubs[_randint(64, (q,), gen)] * n + _randint(n, (q,), gen), count, gen)
        return torch.sort(keys).values
    if graph == "rmat":
        keys = _with_sampled(none, lambda q: _rmat_pairs(n, q, gen), count, gen)
    elif graph == "er":
        keys = _with_sampled(none, lambda q: _pairs(_randint(n, (q,), gen), _randint(n, (q,), gen), n), count, gen)
    else:
        i, j = torch.triu_indices(16, 16, 1, device="cuda")
        pick = _perm(n // 16 * 120, gen)[:_fixed(case)]
        inside = _pairs(pick // 120 * 16 + i[pick % 120], pick // 120 * 16 + j[pick % 120], n)
        keys = _with_sampled(inside, lambda q: _pairs(_randint(n, (q,), gen), _randint(n, (q,), gen), n), count, gen)
    u, v = keys // n, keys % n
    loops = torch.arange(n if graph == "er" else 0, device="cuda")
    return torch.sort(torch.cat([keys, v * n + u, loops * n + loops])).values


def _graph(case, gen):
    n = case["nodes"]
    keys = _keys(case, gen)
    row, col = keys // n, keys % n
    rows = (n + 15) // 16 * 16
    count = torch.bincount(row, minlength=rows)
    rowptr = torch.zeros(rows + 1, dtype=torch.int64, device="cuda")
    rowptr[1:] = count.cumsum(0)
    if case["graph"] == "er":
        val = (count[row] * count[col]).float().rsqrt()
    else:
        val = _rand(keys.shape[0], gen)
    return rowptr.int(), col.int(), val.half().float()


def _dense(rows, k, gen):
    return (_rand((rows, k), gen) * 2 - 1).half()


def _inputs(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    n, k = case["nodes"], case["k"]
    return _graph(case, gen), _dense(n, k, gen), _dense(n, k, gen) if case["op"] == "sddmm" else None


# ------------------------------------------------------------------------------------------------

def prepare(case, seed):
    """The operands on the GPU; for "spmm" and "sddmm" also what a training or serving loop keeps: the plan,
    the output and the workspace."""
    csr, b, y = _inputs(case, seed)
    n, k = case["nodes"], case["k"]
    state = {"op": case["op"], "n": n, "csr": csr, "b": b, "y": y}
    if case["op"] != "fresh":
        fmt = trspmm.build_format_device(*csr)
        if case["op"] == "spmm":
            plan = trspmm.Plan.from_format(fmt, n, n)
            need = plan.workspace_bytes(k)
            state["out"] = torch.empty((n, k), dtype=torch.float32, device="cuda")
        else:
            plan = trspmm.Plan.for_sddmm(fmt, n, n)
            need = plan.sddmm_workspace_bytes(k)
            state["out"] = torch.empty(csr[1].shape[0], dtype=torch.float32, device="cuda")
        state["plan"] = plan
        state["ws"] = torch.empty(max(need, 16), dtype=torch.uint8, device="cuda")
        state["csr"] = None
    return state


def run(state):
    if state["op"] == "spmm":
        return state["plan"].spmm(state["b"], out=state["out"], workspace=state["ws"])
    if state["op"] == "sddmm":
        return state["plan"].sddmm(state["b"], state["y"], out=state["out"], workspace=state["ws"])
    fmt = trspmm.build_format_device(*state["csr"])
    plan = trspmm.Plan.from_format(fmt, state["n"], state["n"])
    return plan.spmm(state["b"])


def work(case):
    """SpMM: column id and fp16 value per entry, row pointers, B and C once.  SDDMM: column id and fp32 output
    per entry, row pointers, X and Y once.  "fresh" reads its values in fp32 and writes no format."""
    n, k, e = case["nodes"], case["k"], _entries(case)
    per_entry = 6 if case["op"] == "spmm" else 8
    dense = 4 * n * k if case["op"] == "sddmm" else 6 * n * k
    return {"bytes": per_entry * e + 4 * (n + 1) + dense, "flops": 2 * e * k}


def tolerance(case):
    """fp16 products are exact in fp32 and the sums are 32-bit: four times the distance seen from the 64-bit result
    (2.1e-7 over all values; 7e-5 at the worst single value, in hub rows of 100,000 entries)."""
    return {"rel": 1e-6, "max": 3e-4}


def exact(case, seed):
    (rowptr, col, val), b, y = _inputs(case, seed)
    n, k = case["nodes"], case["k"]
    col = col.long()
    row = torch.repeat_interleave(torch.arange(rowptr.shape[0] - 1, device="cuda"), rowptr.diff().long())
    total, step = col.shape[0], max(1, (1 << 28) // k)
    if case["op"] == "sddmm":
        out = torch.empty(total, dtype=torch.float64, device="cuda")
        for s in range(0, total, step):
            out[s:s + step] = (b[row[s:s + step]].double() * y[col[s:s + step]].double()).sum(1)
        return out
    out = torch.zeros((n, k), dtype=torch.float64, device="cuda")
    for s in range(0, total, step):
        out.index_add_(0, row[s:s + step], b[col[s:s + step]].double() * val[s:s + step, None].double())
    return out
