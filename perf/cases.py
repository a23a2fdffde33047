"""The work that users of this framework have it do, as measurable cases.

A case is a dict of plain values.  ``prepare`` makes what a program holds
before the call (inputs from a seed, the matrix's ME-TCF, weights), ``run``
is one pass through the public entry points, ``exact`` the same outputs from
plain torch in float64.  Sparse patterns are the families of dtc/graphs.py,
drawn on the GPU so that inputs of another seed cost little.  A seed relabels
a case's pattern (see _relabel) and draws every value, so that the outputs of
all seeds have the same sizes:

  uniform  random columns, rows of about the same length
  rmat     power-law graph (a, b, c = 0.57, 0.19, 0.19), symmetrised
  block    block model, Zipf community sizes, plus hub rows
  band     half-filled band

Kinds of case:

  spmm   C = A B over a prepared matrix (DTCMatrix.spmm, or the operator
         names of the reference's harness: run_DTCSpMM, run_DTCSpMM_balance)
  build  ME-TCF from a CSR (DTCMatrix)
  setup  ME-TCF of a CSR and of its transpose, as training needs
  grad   C = A B and the gradients of A's values and of B
  gcn    H = A (act(X) W): forward only, or with the gradients of the values,
         X and W
"""
import math
import os
import sys

import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "dtc-spmm_asplos24_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from dtc import load_extension  # noqa: E402
from dtc.gcn import gcn_layer  # noqa: E402
from dtc.matrix import DTCMatrix, spmm_autograd  # noqa: E402


def _spmm(name, pattern, rows, degree, n, b="float32", precision="fp32", entry="matrix", values=True):
    return {"name": name, "kind": "spmm", "pattern": pattern, "rows": rows, "degree": degree, "n": n, "b": b,
            "precision": precision, "entry": entry, "values": values}


def listed():
    return [
        # The small plain product: one call is a few microseconds of GPU work,
        # so launches, host work and the length of one wave's chain count.
        _spmm("spmm_uniform_4096_n128", "uniform", 4096, 16, 128),
        # The power-law benchmark matrix at its usual width: gathers of B far
        # beyond the caches, hub rows of tens of thousands of entries.
        _spmm("spmm_rmat_1048576_n256", "rmat", 1048576, 32, 256),
        # The largest matrix: communities plus hub rows, 120M entries.
        _spmm("spmm_block_232965_n128", "block", 232965, 490, 128),
        # The reference's own harness call on an unweighted graph, at a width
        # that no vector load divides and a row count that fills no window.
        _spmm("spmm_balance_100003_n47", "rmat", 100003, 16, 47, entry="balance", values=False),
        # A near-dense band: few columns per window, wide B and C, the split
        # precision that the selector offers beside float32.
        _spmm("spmm_band_200000_n512", "band", 200000, 17, 512, precision="bf16x6"),
        # Inference on stored bfloat16 features.
        _spmm("spmm_uniform_65536_n64_bf16", "uniform", 65536, 32, 64, b="bfloat16"),
        # One training step of a propagation A B with learned edge weights.
        {"name": "grad_rmat_262144_n128", "kind": "grad", "pattern": "rmat", "rows": 262144, "degree": 32, "n": 128},
        # A small graph served: one layer, forward only.
        {"name": "gcn_serve_2048", "kind": "gcn", "pattern": "rmat", "rows": 2048, "degree": 32, "k": 256, "f": 128,
         "x": "bfloat16", "relu": False, "train": False},
        # A hidden layer of a GCN in training: float32 input from the layer
        # before, its ReLU taken with the transform, all three gradients.
        {"name": "gcn_train_262144", "kind": "gcn", "pattern": "rmat", "rows": 262144, "degree": 32, "k": 256, "f": 256,
         "x": "float32", "relu": True, "train": True},
        # A small matrix built for a few products: host and launch latency.
        {"name": "build_uniform_4096", "kind": "build", "pattern": "uniform", "rows": 4096, "degree": 16},
        # The power-law benchmark matrix built.
        {"name": "build_rmat_1048576", "kind": "build", "pattern": "rmat", "rows": 1048576, "degree": 32},
        # A community graph made ready for training: ME-TCF of A and A^T.
        {"name": "setup_block_60000", "kind": "setup", "pattern": "block", "rows": 60000, "degree": 200},
    ]


def _between(rng, lo, hi):
    """Log-uniform integer in [lo, hi]."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _graph(rng, max_rows, max_entries):
    pattern = rng.choice(["uniform", "rmat", "block", "band"])
    rows = _between(rng, 2048, max_rows)
    if rng.random() < 0.5:  # the other half stays odd or ragged
        rows = max(2048, rows // 256 * 256)
    # at least 4 entries per row; block models are the dense family
    top = max(4, min(400 if pattern == "block" else 64, max_entries // rows, rows // 8))
    return {"pattern": pattern, "rows": rows, "degree": _between(rng, min(32, top) if pattern == "block" else 4, top)}


def _width(rng, hi, multiple=1):
    n = _between(rng, 8, hi)
    if multiple == 1 and rng.random() < 0.3:
        return n  # any width, odd ones among them
    step = max(multiple, 16 if n >= 16 else 4)
    return max(step, n // step * step)


def draw(rng):
    kind = rng.choice(["spmm", "spmm", "spmm", "grad", "gcn", "build", "setup"])
    if kind == "spmm":
        c = {"kind": kind, **_graph(rng, 1 << 20, 1 << 24)}
        b = "bfloat16" if rng.random() < 0.25 else "float32"
        widest = max(8, min(512, (1 << 27) // c["rows"], (1 << 31) // (c["rows"] * c["degree"])))
        c["n"] = _width(rng, widest, 4 if b == "bfloat16" else 1)
        c["b"] = b
        c["precision"] = "fp32" if b == "bfloat16" else rng.choice(["fp32", "fp32", "fp32", "bf16x6", "bf16x3", "bf16"])
        c["entry"] = "matrix" if b == "bfloat16" else rng.choice(["matrix", "matrix", "windows", "balance"])
        c["values"] = rng.random() < 0.75
        return c
    if kind == "grad":
        c = {"kind": kind, **_graph(rng, 1 << 18, 1 << 23)}
        c["n"] = _width(rng, 256)
        return c
    if kind == "gcn":
        c = {"kind": kind, **_graph(rng, 1 << 18, 1 << 23)}
        c["k"] = 32 * rng.randint(1, 8)
        c["f"] = 64 * rng.randint(1, 4)
        c["relu"] = rng.random() < 0.5
        c["x"] = rng.choice(["bfloat16", "float32"])
        c["train"] = rng.random() < 0.6
        return c
    return {"kind": kind, **_graph(rng, 1 << 20 if kind == "build" else 1 << 18, 1 << 24)}


# ------------------------------------------------------------------ inputs

def _relabel(rows, g):
    """New id of every node: the groups of 16 consecutive nodes rotated by a
    random distance, and the 16 shuffled inside each (a last group of fewer
    stays).  Row windows keep their sets of columns and the transpose's keep
    theirs, so entries and TC blocks number the same for every seed, and
    neighbours stay near each other."""
    groups = rows // 16
    ids = torch.arange(rows, device="cuda")
    if groups == 0:
        return ids
    turn = torch.randint(0, groups, (1,), generator=g, device="cuda")
    inside = torch.rand(groups, 16, generator=g, device="cuda").argsort(1)
    base = (torch.arange(groups, device="cuda") + turn) % groups * 16
    ids[:groups * 16] = (base[:, None] + inside).reshape(-1)
    return ids


def _csr(row, col, rows, g):
    """int32 rowptr, column and row of every entry of the relabelled pattern."""
    ids = _relabel(rows, g)
    keys = torch.unique(ids[row] * rows + ids[col])
    r = torch.div(keys, rows, rounding_mode="floor")
    rowptr = torch.zeros(rows + 1, dtype=torch.int64, device="cuda")
    rowptr[1:] = torch.cumsum(torch.bincount(r, minlength=rows), 0)
    return rowptr.int(), (keys - r * rows).int(), r


def _pattern(case, g):
    """CSR of the case's pattern, relabelled with the seed's generator g."""
    kind, rows, degree = case["pattern"], case["rows"], case["degree"]
    own = torch.Generator(device="cuda")
    own.manual_seed(rows * 1000 + degree)

    def ints(hi, count):
        return torch.randint(0, hi, (count,), generator=own, device="cuda")

    def rand(count):
        return torch.rand(count, generator=own, device="cuda")

    if kind == "uniform":
        r = torch.arange(rows, device="cuda").repeat_interleave(degree)
        return _csr(r, ints(rows, rows * degree), rows, g)
    if kind == "rmat":
        m = rows * degree // 2
        scale = max(1, (rows - 1).bit_length())
        src = torch.zeros(m, dtype=torch.int64, device="cuda")
        dst = torch.zeros(m, dtype=torch.int64, device="cuda")
        for _ in range(scale):
            u = rand(m)
            src = src * 2 + (u >= 0.76)
            dst = dst * 2 + (((u >= 0.57) & (u < 0.76)) | (u >= 0.95))
        src, dst = src * rows >> scale, dst * rows >> scale
        keep = src != dst
        src, dst = src[keep], dst[keep]
        return _csr(torch.cat([src, dst]), torch.cat([dst, src]), rows, g)
    if kind == "band":
        offs = torch.arange(-degree, degree + 1, device="cuda")
        r = torch.arange(rows, device="cuda").repeat_interleave(2 * degree + 1)
        c = r + offs.repeat(rows)
        keep = (c >= 0) & (c < rows) & (rand(r.numel()) < 0.5)
        return _csr(r[keep], c[keep], rows, g)
    # block: 50 communities of Zipf sizes, 5% of a row's entries anywhere, hub rows
    w = 1.0 / torch.arange(1, 51, dtype=torch.float64) ** 1.1
    sizes = torch.clamp((w / w.sum() * rows).floor().long(), min=1)
    sizes[0] += rows - int(sizes.sum())
    start = torch.cumsum(sizes, 0) - sizes
    of = torch.repeat_interleave(torch.arange(50), sizes).cuda()
    # draws with replacement whose distinct columns number the wanted share
    inside = torch.clamp(0.95 * degree / sizes.double(), max=0.999)
    draws = (-sizes.double() * torch.log1p(-inside)).round().long().clamp(min=1).cuda()
    r = torch.arange(rows, device="cuda").repeat_interleave(draws[of])
    c = start.cuda()[of[r]] + (rand(r.numel()) * sizes.cuda()[of[r]]).long()
    across = torch.arange(rows, device="cuda").repeat_interleave(max(1, degree // 20))
    hubs = torch.randperm(rows, generator=own, device="cuda")[:max(1, rows // 1165)]
    hub = hubs.repeat_interleave(max(1, min(35000, rows // 7)))
    other = torch.cat([across, hub])
    return _csr(torch.cat([r, other]), torch.cat([c.clamp(max=rows - 1), ints(rows, other.numel())]), rows, g)


def _graph_of(case, seed):
    """(rowptr, col, row of every entry, values, generator)."""
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    rowptr, col, row = _pattern(case, g)
    if case["pattern"] == "rmat":  # symmetric normalisation
        deg = torch.diff(rowptr).double().clamp(min=1)
        values = (1.0 / torch.sqrt(deg[row] * deg[col.long()])).float()
    else:
        values = torch.rand(col.numel(), generator=g, device="cuda")
    return rowptr, col, row, values, g


def _normal(g, rows, cols, dtype=torch.float32, scale=1.0):
    return (torch.randn(rows, cols, generator=g, device="cuda") * scale).to(dtype)


def _inputs(case, seed):
    """Everything drawn from the seed, in the order that fixes the stream."""
    rowptr, col, row, values, g = _graph_of(case, seed)
    rows, kind = case["rows"], case["kind"]
    x = {"rowptr": rowptr, "col": col, "row": row, "values": values}
    if kind == "spmm":
        x["B"] = _normal(g, rows, case["n"], getattr(torch, case["b"]))
    elif kind == "grad":
        x["B"] = _normal(g, rows, case["n"])
        x["dC"] = _normal(g, rows, case["n"])
    elif kind == "gcn":
        x["X"] = _normal(g, rows, case["k"], getattr(torch, case["x"]))
        x["W"] = _normal(g, case["k"], case["f"], torch.bfloat16, math.sqrt(2.0 / (case["k"] + case["f"])))
        x["dH"] = _normal(g, rows, case["f"])
    return x


def prepare(case, seed):
    x = _inputs(case, seed)
    del x["row"]
    kind, rows = case["kind"], case["rows"]
    x["case"] = case
    if kind in ("build", "setup"):
        return x
    with_values = case.get("values", True)
    x["A"] = DTCMatrix(x["rowptr"], x["col"], x["values"] if with_values else None, num_rows=rows, num_cols=rows)
    if kind == "grad" or case.get("train"):
        x["A"].transpose()  # part of a training program's setup
    if kind == "grad":
        for k in ("values", "B"):
            x[k].requires_grad_(True)
    elif case.get("train"):
        for k in ("values", "X", "W"):
            x[k].requires_grad_(True)
    return x


def _metcf(A):
    return {"row_window_offset": A.row_window_offset, "tcblock_rowid": A.tcblock_rowid,
            "tcblocktile_id": A.tcblocktile_id, "tcblock_offset": A.tcblock_offset, "sparse_atox": A.sparse_atox,
            "block_count": A.block_count, "values_tc": A.values_tc, "tc_edge": A.tc_edge,
            "block_partition": A.block_partition, "edge_to_column": A.edge_to_column, "edge_to_row": A.edge_to_row}


def run(s):
    case = s["case"]
    kind, rows = case["kind"], case["rows"]
    if kind in ("build", "setup"):
        A = DTCMatrix(s["rowptr"], s["col"], s["values"], num_rows=rows, num_cols=rows)
        if kind == "build":
            return _metcf(A)
        return {"A": _metcf(A), "At": _metcf(A.transpose()), "perm_t": A.perm_t}
    A = s["A"]
    if kind == "spmm":
        if case["entry"] == "matrix":
            return A.spmm(s["B"], precision=case["precision"])
        ext = load_extension()
        if case["entry"] == "windows":
            return ext.run_DTCSpMM(s["B"], A.row_window_offset, A.tcblocktile_id, A.tcblock_offset, A.sparse_atox,
                                   rows, A.nnz, "float4_split", values=A.values_tc, precision=case["precision"])[0]
        return ext.run_DTCSpMM_balance(s["B"], A.tcblock_rowid, A.tcblocktile_id, A.tcblock_offset, A.sparse_atox,
                                       rows, "float4_split", values=A.values_tc, precision=case["precision"])[0]
    if kind == "grad":
        C = spmm_autograd(s["values"], s["B"], A)
        dvalues, dB = torch.autograd.grad(C, (s["values"], s["B"]), s["dC"])
        return {"C": C.detach(), "dvalues": dvalues, "dB": dB}
    if not case["train"]:
        with torch.no_grad():
            return gcn_layer(s["values"], s["X"], s["W"], A, input_relu=case["relu"])
    H = gcn_layer(s["values"], s["X"], s["W"], A, input_relu=case["relu"])
    dvalues, dX, dW = torch.autograd.grad(H, (s["values"], s["X"], s["W"]), s["dH"])
    return {"H": H.detach(), "dvalues": dvalues, "dX": dX, "dW": dW}


# --------------------------------------------------------------- yardsticks

def _entries(case):
    """Expected entries of the pattern."""
    rows, degree = case["rows"], case["degree"]
    if case["pattern"] == "band":
        return rows * (2 * degree + 1) // 2
    hubs = max(1, rows // 1165) * max(1, min(35000, rows // 7)) if case["pattern"] == "block" else 0
    return rows * degree + hubs


def work(case):
    rows, nnz, kind = case["rows"], _entries(case), case["kind"]
    csr = 4 * (rows + 1) + 4 * nnz
    if kind == "spmm":
        n = case["n"]
        b = 2 if case["b"] == "bfloat16" else 4
        return {"bytes": csr + (4 * nnz if case["values"] else 0) + rows * n * (b + 4), "flops": 2 * nnz * n}
    if kind == "grad":
        n = case["n"]  # values, B, dC in; C, dvalues, dB out
        return {"bytes": csr + 8 * nnz + 16 * rows * n, "flops": 6 * nnz * n}
    if kind == "gcn":
        k, f = case["k"], case["f"]
        xb = 2 if case["x"] == "bfloat16" else 4
        forward = csr + 4 * nnz + rows * (k * xb + f * 4) + 2 * k * f
        flops = 2 * rows * k * f + 2 * nnz * f
        if not case["train"]:
            return {"bytes": forward, "flops": flops}
        return {"bytes": forward + 4 * nnz + rows * (k * xb + f * 4) + 2 * k * f, "flops": 3 * flops}
    # rowptr, columns and values in; edgeToColumn, edgeToRow, tile ids, values
    # and edge order out, plus the windows' and blocks' arrays (a block per
    # 8 to 16 entries on these patterns; the fewest are counted)
    build = csr + 4 * nnz + 17 * nnz + 8 * (rows // 16) + 40 * (nnz // 16)
    if kind == "build":
        return {"bytes": build, "flops": 0}
    return {"bytes": 2 * build + 2 * csr + 4 * nnz, "flops": 0}


_CHUNK = 1 << 21  # entries per step of the float64 products


def _product64(row, col, values, B, rows):
    """A B in float64, a slice of entries at a time."""
    out = torch.zeros(rows, B.shape[1], dtype=torch.float64, device="cuda")
    step = max(1, _CHUNK * 128 // B.shape[1])
    for i in range(0, row.numel(), step):
        j = slice(i, i + step)
        out.index_add_(0, row[j], B[col[j]].double() * values[j, None])
    return out


def _dots64(row, col, X, Y):
    out = torch.empty(row.numel(), dtype=torch.float64, device="cuda")
    step = max(1, _CHUNK * 64 // X.shape[1])
    for i in range(0, row.numel(), step):
        j = slice(i, i + step)
        out[j] = (X[row[j]].double() * Y[col[j]].double()).sum(1)
    return out


def exact(case, seed):
    kind, rows = case["kind"], case["rows"]
    if kind in ("build", "setup"):
        return None  # indices, and values that are moved only
    x = _inputs(case, seed)
    row, col = x["row"], x["col"].long()
    values = x["values"].double()
    if kind == "spmm":
        return _product64(row, col, values if case["values"] else torch.ones_like(values), x["B"], rows)
    if kind == "grad":
        return {"C": _product64(row, col, values, x["B"], rows), "dvalues": _dots64(row, col, x["dC"], x["B"]),
                "dB": _product64(col, row, values, x["dC"], rows)}
    X, W = x["X"].double(), x["W"].double()
    if case["relu"]:
        X = torch.relu(X)
    XW = X @ W
    H = _product64(row, col, values, XW, rows)
    if not case["train"]:
        return H
    dXW = _product64(col, row, values, x["dH"], rows)
    dX = dXW @ W.t().contiguous()
    if case["relu"]:
        dX = dX * (x["X"] > 0)
    return {"H": H, "dvalues": _dots64(row, col, x["dH"], XW), "dX": dX, "dW": X.t().contiguous() @ dXW}
