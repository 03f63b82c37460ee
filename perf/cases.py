"""The sparse products and conversions whose time counts: what a program that uses this library has it do.

Every listed case is one of the workloads of the repository's benchmark (bench.py: c1 - c5 and its further modes), at
its sizes or, where a round power of two would be a special case, at odd sizes next to them.  `draw` takes more cases
from the ranges that these stand for: from a few thousand entries, where a call is its launches, to tens of millions.

  spmv      y = alpha * op(A) * x + beta * y     a Krylov or power iteration's product; one call a pass
  spmvop    z = alpha * A * x + beta * y         the same through the SpMVOp descriptor / plan API
  spmm      C = alpha * A * B                    several right-hand sides, block methods, feature matrices
  train     C = A * B and dB = A^T * dC          a graph layer forward and backward; A^T is kept as a matrix
  assemble  unsorted triples or unsorted rows -> sorted CSR, its values, and its CSC form

Matrices: `mesh5` / `mesh9` (2-D), `mesh7` / `mesh27` (3-D) stencils with varying coefficients, `band` (random columns
near the diagonal), `uniform` (a fixed number of random columns a row), `graph` (power-law row lengths, random columns).
"""
import ctypes
import importlib.util
import itertools
import math
import os
import sys

import torch


def _package():
    """The package's folder has a hyphen in its name: it is loaded by path, as ops_sparse_amd."""
    if "ops_sparse_amd" not in sys.modules:
        folder = os.path.join(os.getcwd(), "ops-sparse_amd")
        spec = importlib.util.spec_from_file_location("ops_sparse_amd", os.path.join(folder, "__init__.py"),
                                                      submodule_search_locations=[folder])
        module = importlib.util.module_from_spec(spec)
        sys.modules["ops_sparse_amd"] = module
        spec.loader.exec_module(module)
    return sys.modules["ops_sparse_amd"]


osa = _package()
wl = importlib.import_module("ops_sparse_amd.workloads")

DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
BYTES = {"f32": 4, "f16": 2, "bf16": 2}
BOX2 = list(itertools.product((-1, 0, 1), repeat=2))
BOX3 = list(itertools.product((-1, 0, 1), repeat=3))
STENCILS = {"mesh5": [o for o in BOX2 if abs(o[0]) + abs(o[1]) <= 1], "mesh9": BOX2,
            "mesh7": [o for o in BOX3 if sum(map(abs, o)) <= 1], "mesh27": BOX3}


# ------------------------------------------------------------------ the cases

def listed():
    return [
        # c1: a small system; the call is launch latency
        {"name": "spmv_small", "path": "spmv", "matrix": "uniform", "rows": 4096, "per_row": 16, "dtype": "f32",
         "out": "f32", "op": "n", "alg": "default", "alpha": 1.0, "beta": 0.0},
        # c2, the headline: 5-point Laplacian, one product of an iterative solver
        {"name": "spmv_mesh5", "path": "spmv", "matrix": "mesh5", "nx": 2048, "ny": 2048, "dtype": "f32", "out": "f32",
         "op": "n", "alg": "default", "alpha": 1.0, "beta": 0.5},
        # the stencils mode: 27 couplings a point on a 3-D mesh of odd extents
        {"name": "spmv_mesh27", "path": "spmv", "matrix": "mesh27", "nx": 131, "ny": 127, "nz": 129, "dtype": "f32",
         "out": "f32", "op": "n", "alg": "default", "alpha": 1.0, "beta": 0.5},
        # c3: a power-law graph, values free to change between calls
        {"name": "spmv_graph", "path": "spmv", "matrix": "graph", "rows": 8388608, "exponent": 2.0, "longest": 200000,
         "mean": 0.0, "dtype": "f32", "out": "f32", "op": "n", "alg": "default", "alpha": 1.0, "beta": 0.0},
        # c3 with the values frozen at Preprocess (ACL_SPARSE_SPMV_CSR_ALG2)
        {"name": "spmv_graph_frozen", "path": "spmv", "matrix": "graph", "rows": 6000011, "exponent": 2.0,
         "longest": 200000, "mean": 0.0, "dtype": "f32", "out": "f32", "op": "n", "alg": "frozen", "alpha": 1.0,
         "beta": 0.0},
        # c3 under op(A) = A^T: the adjoint of the same operator
        {"name": "spmv_graph_t", "path": "spmv", "matrix": "graph", "rows": 5000011, "exponent": 2.0,
         "longest": 200000, "mean": 0.0, "dtype": "f32", "out": "f32", "op": "t", "alg": "default", "alpha": 1.0,
         "beta": 0.0},
        # c3 with repeatable sums, through the plan API that promises them
        {"name": "spmvop_graph", "path": "spmvop", "matrix": "graph", "rows": 4000037, "exponent": 2.0,
         "longest": 200000, "mean": 0.0, "dtype": "f32", "out": "f32", "op": "n", "alg": "default", "alpha": 1.0,
         "beta": 0.5},
        # c4: fp32 SpMM, 32 random columns a row, 64 columns of B
        {"name": "spmm_uniform", "path": "spmm", "matrix": "uniform", "rows": 1048576, "per_row": 32, "n": 64,
         "dtype": "f32", "out": "f32", "layout": "row"},
        # c5: a graph layer on fp16 features, forward and backward
        {"name": "train_graph", "path": "train", "matrix": "graph", "rows": 1500007, "exponent": 2.1, "longest": 50000,
         "mean": 16.0, "n": 128, "dtype": "f16", "out": "f32"},
        # the spmm_shapes mode: features on a mesh
        {"name": "spmm_mesh", "path": "spmm", "matrix": "mesh7", "nx": 125, "ny": 131, "nz": 127, "n": 32,
         "dtype": "f32", "out": "f32", "layout": "row"},
        # the few_columns mode: a block method's four right-hand sides
        {"name": "spmm_few_columns", "path": "spmm", "matrix": "mesh5", "nx": 2048, "ny": 2048, "n": 4, "dtype": "f32",
         "out": "f32", "layout": "row"},
        # the convert mode: 33.5 M shuffled triples to sorted CSR and CSC
        {"name": "assemble", "path": "assemble", "start": "triples", "rows": 1048576, "per_row": 32},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _some_mesh(rng, kinds, lo, hi):
    """A mesh of lo .. hi points, its extents unequal and as odd as they come."""
    kind = rng.choice(kinds)
    points = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    dims = 2 if kind in ("mesh5", "mesh9") else 3
    side = points ** (1.0 / dims)
    stretch = math.exp(rng.uniform(-0.5, 0.5))
    c = {"matrix": kind, "nx": max(3, int(side * stretch)), "ny": max(3, int(side / stretch))}
    if dims == 3:
        c["nz"] = max(3, int(side))
    return c


def _some_graph(rng, lo, hi, most_entries):
    """Power-law graphs: either the plain law (its mean follows from it) or one scaled to a mean of 6 - 24."""
    mean = rng.choice([0.0, rng.uniform(6.0, 24.0)])
    exponent, longest = rng.uniform(2.0, 2.5), _log_int(rng, 200, 200000)
    rows = _log_int(rng, lo, hi)
    c = {"matrix": "graph", "rows": rows, "exponent": exponent, "longest": min(longest, rows // 4), "mean": mean}
    per_row = _entries(c) / rows
    c["rows"] = min(rows, int(most_entries / per_row))
    return c


def draw(rng):
    kind = rng.choice(["small", "spmv_mesh", "spmv_mesh", "spmv_graph", "spmv_graph", "spmv_graph_t", "spmvop",
                       "spmm_uniform", "train", "spmm_mesh", "spmm_few", "assemble"])
    scalars = rng.choice([(1.0, 0.0), (1.0, 0.5), (-0.75, 1.0)])
    f16ish = rng.choice(["f32", "f32", "f32", "f16", "bf16"])
    if kind == "small":
        m = rng.choice([_some_mesh(rng, ["mesh5", "mesh7", "mesh9"], 1000, 60000),
                        {"matrix": "uniform", "rows": _log_int(rng, 1000, 60000), "per_row": rng.randint(2, 24)},
                        _some_graph(rng, 2000, 60000, 1 << 20)])
        if rng.random() < 0.3:
            return dict(m, path="spmm", n=rng.choice([3, 8, 16, 33, 64]), dtype="f32", out="f32", layout="row")
        return dict(m, path=rng.choice(["spmv", "spmv", "spmvop"]), dtype="f32", out="f32", op="n", alg="default",
                    alpha=scalars[0], beta=scalars[1])
    if kind == "spmv_mesh":
        if rng.random() < 0.2:
            width = _log_int(rng, 20, 300)
            m = {"matrix": "band", "rows": _log_int(rng, 4000000 // width, 50000000 // width), "per_row": width}
        else:
            m = _some_mesh(rng, ["mesh5", "mesh7", "mesh9", "mesh27"], 100000, 4200000)
            if _entries(m) > 57000000:
                m["nx"] = max(3, int(m["nx"] * 57000000 / _entries(m)))
        out = f16ish if rng.random() < 0.5 else "f32"
        return dict(m, path="spmv", dtype=f16ish, out=out, op="n", alg=rng.choice(["default", "default", "frozen"]),
                    alpha=scalars[0], beta=scalars[1])
    if kind in ("spmv_graph", "spmv_graph_t"):
        m = _some_graph(rng, 200000, 8388608, 60000000)
        if kind == "spmv_graph_t":
            return dict(m, path="spmv", dtype="f32", out="f32", op="t", alg=rng.choice(["default", "frozen"]),
                        alpha=scalars[0], beta=scalars[1])
        return dict(m, path="spmv", dtype=f16ish, out="f32", op="n", alg=rng.choice(["default", "default", "frozen"]),
                    alpha=scalars[0], beta=scalars[1])
    if kind == "spmvop":
        m = rng.choice([_some_graph(rng, 200000, 8388608, 60000000), _some_mesh(rng, ["mesh5", "mesh7"], 100000, 4000000)])
        return dict(m, path="spmvop", dtype="f32", out="f32", op="n", alg=rng.choice(["default", "default", "frozen"]),
                    alpha=scalars[0], beta=scalars[1])
    if kind == "spmm_uniform":
        per_row, n = _log_int(rng, 4, 64), rng.choice([16, 32, 62, 64, 100, 128, 256])
        rows = min(_log_int(rng, 50000, 1500000), int(2.0e9 / (per_row * n)))
        return {"path": "spmm", "matrix": "uniform", "rows": rows, "per_row": per_row, "n": n, "dtype": "f32",
                "out": "f32", "layout": rng.choice(["row", "row", "row", "col"])}
    if kind == "train":
        n, dtype = rng.choice([32, 48, 64, 128, 200, 256]), rng.choice(["f16", "f16", "f32"])
        m = _some_graph(rng, 50000, 1500000, int(2.6e9 / n / (2 if dtype == "f32" else 1)))
        return dict(m, path="train", n=n, dtype=dtype, out="f32")
    if kind == "spmm_mesh":
        n = rng.choice([12, 16, 24, 32, 50, 64, 128])
        if rng.random() < 0.2:
            width = _log_int(rng, 20, 200)
            m = {"matrix": "band", "rows": _log_int(rng, 400000 // width, 400000000 // (n * width)), "per_row": width}
        else:
            m = _some_mesh(rng, ["mesh5", "mesh7", "mesh9", "mesh27"], 50000, 100000000 // n)
        return dict(m, path="spmm", n=n, dtype="f32", out="f32", layout="row")
    if kind == "spmm_few":
        dtype = rng.choice(["f32", "f32", "f32", "f16"])
        n = rng.choice([2, 3, 4, 6, 8]) if dtype == "f32" else rng.choice([8, 16])
        m = rng.choice([_some_mesh(rng, ["mesh5", "mesh7", "mesh27"], 100000, 2500000),
                        _some_graph(rng, 100000, 2000000, 30000000)])
        return dict(m, path="spmm", n=n, dtype=dtype, out="f32", layout=rng.choice(["row", "row", "col"]))
    per_row = _log_int(rng, 4, 48)
    return {"path": "assemble", "start": rng.choice(["triples", "rows"]), "per_row": per_row,
            "rows": _log_int(rng, 50000, min(4000000, 33000000 // per_row))}


# ------------------------------------------------------------------ matrices and vectors

def _law(c):
    """Mean row length of the plain power law on [1, longest]."""
    top = min(c["longest"], c["rows"])
    s0 = s1 = 0.0
    for l in range(1, top + 1):
        w = l ** -c["exponent"]
        s0 += w
        s1 += w * l
    return s1 / s0


def _shape(c):
    return tuple(c[k] for k in ("nx", "ny", "nz") if k in c)


def _rows(c):
    return math.prod(_shape(c)) if c["matrix"].startswith("mesh") else c["rows"]


def _entries(c):
    """Stored entries, as a mean over seeds where the matrix is a random graph."""
    if c["matrix"].startswith("mesh"):
        shape = _shape(c)
        return sum(math.prod(n - abs(s) for n, s in zip(shape, o)) for o in STENCILS[c["matrix"]])
    if c["matrix"] == "graph":
        return int(c["rows"] * (c["mean"] or _law(c)))
    return c["rows"] * c["per_row"]


def _band(rows, width, seed, dev):
    """`width` distinct columns a row inside a window of 4 x width columns round the diagonal."""
    k = torch.arange(width, dtype=torch.int64, device=dev).view(1, width)
    r = torch.arange(rows, dtype=torch.int64, device=dev).view(rows, 1)
    step = wl._lsr(wl.hash64(seed, (r * width + k).reshape(-1)), 11).view(rows, width) % 4
    cols = (r - 2 * width + 4 * k + step).clamp_(0, rows - 1)
    return {"rows": rows, "cols": rows, "colind": cols.reshape(-1).int(),
            "rowptr": (torch.arange(rows + 1, dtype=torch.int64, device=dev) * width).int(),
            "values": wl.uniform(seed + 1, rows * width, -1.0, 1.0, dev)}


def _matrix(c, seed, dev):
    if c["matrix"].startswith("mesh"):
        A = wl.stencil_csr(_shape(c), STENCILS[c["matrix"]], dev)
        # a coefficient that varies over the mesh: every coupling scaled by 0.5 .. 1.5
        A["values"] = A["values"] * wl.uniform(seed + 11, A["values"].numel(), 0.5, 1.5, dev)
        return A
    if c["matrix"] == "graph":
        return wl.power_law_csr(c["rows"], c["rows"], c["exponent"], 1, c["longest"], seed, dev,
                                target_mean=c["mean"] or None)
    if c["matrix"] == "band":
        return _band(c["rows"], c["per_row"], seed, dev)
    return wl.uniform_rows_csr(c["rows"], c["rows"], c["per_row"], seed, dev)


def _row_normalised(A, seed):
    """Edge weights of a mean over neighbours: positive, every row's sum 1 (whole-number sums: the same on every run)."""
    w = (wl._lsr(wl.hash64(seed, torch.arange(A["colind"].numel(), dtype=torch.int64, device=A["colind"].device)), 44)
         + (1 << 10))
    ends = torch.cat([w.new_zeros(1), torch.cumsum(w, 0)])
    at = A["rowptr"].to(torch.int64)
    sums = (ends[at[1:]] - ends[at[:-1]]).to(torch.float32)
    return w.to(torch.float32) / torch.repeat_interleave(sums, at[1:] - at[:-1])


_handles = []


def _handle():
    """One handle for the program, on a stream that is torch's current one too (the library wants a stream of its
    caller's, not the null stream)."""
    if not _handles:
        stream = torch.cuda.Stream()
        torch.cuda.set_stream(stream)
        _handles.append(osa.Handle(stream))
    return _handles[0]


# ------------------------------------------------------------------ one state, one pass

def prepare(case, seed):
    dev, handle = torch.device("cuda:0"), _handle()
    seed = 1000003 * (int(seed) % 1000003) + 17
    gen = torch.Generator(device=dev)
    gen.manual_seed(seed)
    if case["path"] == "assemble":
        return _prepare_assemble(case, dev, gen)
    A = _matrix(case, seed, dev)
    if case["path"] == "train":
        A["values"] = _row_normalised(A, seed + 31)
    dtype = DTYPES[case["dtype"]]
    values = A["values"].to(dtype)
    csr = osa.Csr(A["rows"], A["cols"], A["rowptr"], A["colind"], values)
    s = {"path": case["path"], "csr": csr}
    if case["path"] in ("spmv", "spmvop"):
        t = case["op"] == "t"
        x = wl.uniform(seed + 21, A["rows"] if t else A["cols"], -1.0, 1.0, dev).to(dtype)
        y = wl.uniform(seed + 22, A["cols"] if t else A["rows"], -1.0, 1.0, dev).to(DTYPES[case["out"]])
        s.update(alpha=case["alpha"], beta=case["beta"], x=osa.DnVec(x), y=osa.DnVec(y))
        if case["path"] == "spmv":
            s["out"] = y
            s["op"] = osa.SpmvOp(handle, csr, s["x"], s["y"],
                                 op=osa.ACL_SPARSE_OP_TRANSPOSE if t else osa.ACL_SPARSE_OP_NON_TRANSPOSE,
                                 alg=osa.ACL_SPARSE_SPMV_CSR_ALG2 if case["alg"] == "frozen"
                                 else osa.ACL_SPARSE_SPMV_ALG_DEFAULT)
        else:
            s["out"] = torch.zeros_like(y)
            s["z"] = osa.DnVec(s["out"])
            s["op"] = osa.SpmvOpPlan(handle, csr, s["x"], s["y"], s["z"],
                                     alg=osa.ACL_SPARSE_SPMVOP_ALG2 if case["alg"] == "frozen"
                                     else osa.ACL_SPARSE_SPMVOP_ALG_DEFAULT)
        return s
    n = case["n"]
    if case["path"] == "spmm":
        s["B"] = torch.randn(A["cols"] * n, device=dev, generator=gen).to(dtype)
        s["out"] = torch.zeros(A["rows"] * n, dtype=DTYPES[case["out"]], device=dev)
        col = case["layout"] == "col"
        order = osa.ACL_SPARSE_ORDER_COL if col else osa.ACL_SPARSE_ORDER_ROW
        s["dB"] = osa.DnMat(A["cols"], n, A["cols"] if col else n, s["B"], order)
        s["dC"] = osa.DnMat(A["rows"], n, A["rows"] if col else n, s["out"], order)
        s["op"] = osa.SpmmOp(handle, csr, s["dB"], s["dC"])
        return s
    # train: A^T is made once from A (its CSC arrays are the CSR arrays of A^T), the plans of both are kept
    rows, nnz = A["rows"], csr.nnz
    tptr = torch.empty(A["cols"] + 1, dtype=torch.int32, device=dev)
    tind = torch.empty(nnz, dtype=torch.int32, device=dev)
    tval = torch.empty(nnz, dtype=dtype, device=dev)
    _csr2csc(handle, rows, A["cols"], nnz, values, A["rowptr"], A["colind"], tval, tptr, tind,
             osa.ACL_FLOAT if dtype == torch.float32 else osa.ACL_FLOAT16)()
    s["csr_t"] = osa.Csr(A["cols"], rows, tptr, tind, tval)
    for k, (m, name) in enumerate(((csr, "fwd"), (s["csr_t"], "bwd"))):
        dense = torch.randn(m.cols * n, device=dev, generator=gen).to(dtype)
        out = torch.zeros(m.rows, n, dtype=torch.float32, device=dev)
        s[name + "_out"] = out
        s[name] = osa.SpmmOp(handle, m, osa.DnMat(m.cols, n, n, dense), osa.DnMat(m.rows, n, n, out))
    return s


def _p(t):
    return ctypes.c_void_p(t.data_ptr())


def _csr2csc(handle, m, n, nnz, val, rowptr, col, cval, cptr, cind, acl_type):
    """The csr2csc call with its buffer, ready to be made any number of times."""
    args = (handle.h, m, n, nnz, _p(val), _p(rowptr), _p(col), _p(cval), _p(cptr), _p(cind), acl_type,
            osa.ACL_SPARSE_ACTION_NUMERIC, osa.ACL_SPARSE_INDEX_BASE_ZERO, osa.ACL_SPARSE_CSR2CSC_ALG_DEFAULT)
    size = ctypes.c_size_t(0)
    osa.check(osa.lib().aclsparseCsr2cscEx2_bufferSize(*args, ctypes.byref(size)), "aclsparseCsr2cscEx2_bufferSize")
    buf = torch.empty(max(16, size.value), dtype=torch.uint8, device=val.device)

    def call():
        osa.check(osa.lib().aclsparseCsr2cscEx2(*args, _p(buf)), "aclsparseCsr2cscEx2")
    return call


def _prepare_assemble(case, dev, gen):
    """Entries as an assembly loop or a product leaves them: in no order at all (triples), or by row with the columns of
    a row in no order (rows)."""
    L, handle = osa.lib(), _handle()
    m, per_row = case["rows"], case["per_row"]
    nnz = m * per_row
    s = {"path": "assemble", "start": case["start"], "handle": handle, "m": m, "nnz": nnz}
    col = torch.randint(0, m, (nnz,), device=dev, dtype=torch.int32, generator=gen)
    s["val0"] = torch.rand(nnz, device=dev, generator=gen) * 2 - 1
    s["identity"] = torch.arange(nnz, dtype=torch.int32, device=dev)
    size = ctypes.c_size_t(0)
    if case["start"] == "triples":
        s["row0"] = torch.randint(0, m, (nnz,), device=dev, dtype=torch.int32, generator=gen)
        s["row"], s["rowptr"] = torch.empty_like(col), torch.empty(m + 1, dtype=torch.int32, device=dev)
        osa.check(L.aclsparseXcoosort_bufferSizeExt(handle.h, m, m, nnz, _p(s["row0"]), _p(col), ctypes.byref(size)))
    else:
        s["rowptr"] = (torch.arange(m + 1, device=dev, dtype=torch.int64) * per_row).int()
        osa.check(L.aclsparseXcsrsort_bufferSizeExt(handle.h, m, m, nnz, _p(s["rowptr"]), _p(col), ctypes.byref(size)))
        s["descr"] = ctypes.c_void_p(None)
        osa.check(L.aclsparseCreateMatDescr(ctypes.byref(s["descr"])))
    s["buf"] = torch.empty(max(16, size.value), dtype=torch.uint8, device=dev)
    s["col0"], s["col"], s["perm"] = col, torch.empty_like(col), torch.empty_like(col)
    s["val"], s["cval"] = torch.empty_like(s["val0"]), torch.empty_like(s["val0"])
    s["cptr"], s["cind"] = torch.empty(m + 1, dtype=torch.int32, device=dev), torch.empty_like(col)
    s["csc"] = _csr2csc(handle, m, m, nnz, s["val"], s["rowptr"], s["col"], s["cval"], s["cptr"], s["cind"],
                        osa.ACL_FLOAT)
    return s


def _run_assemble(s):
    L, h, m, nnz = osa.lib(), s["handle"].h, s["m"], s["nnz"]
    # the sorts work in place: the program's own entries stay as they are
    s["col"].copy_(s["col0"])
    s["perm"].copy_(s["identity"])
    if s["start"] == "triples":
        s["row"].copy_(s["row0"])
        osa.check(L.aclsparseXcoosortByRow(h, m, m, nnz, _p(s["row"]), _p(s["col"]), _p(s["perm"]), _p(s["buf"])))
        osa.check(L.aclsparseXcoo2csr(h, _p(s["row"]), nnz, m, _p(s["rowptr"]), osa.ACL_SPARSE_INDEX_BASE_ZERO))
    else:
        osa.check(L.aclsparseXcsrsort(h, m, m, nnz, s["descr"], _p(s["rowptr"]), _p(s["col"]), _p(s["perm"]),
                                      _p(s["buf"])))
    torch.index_select(s["val0"], 0, s["perm"], out=s["val"])
    s["csc"]()
    return [s["rowptr"], s["col"], s["val"], s["cptr"], s["cind"], s["cval"]]


def run(state):
    if state["path"] in ("spmv", "spmvop"):
        state["op"](state["alpha"], state["beta"])
        return state["out"]
    if state["path"] == "spmm":
        state["op"](1.0, 0.0)
        return state["out"]
    if state["path"] == "train":
        state["fwd"](1.0, 0.0)
        state["bwd"](1.0, 0.0)
        return [state["fwd_out"], state["bwd_out"]]
    return _run_assemble(state)


# ------------------------------------------------------------------ what a pass cannot do without

def work(case):
    if case["path"] == "assemble":
        m, nnz = case["rows"], case["rows"] * case["per_row"]
        # triples (or rows, columns) and values in; CSR and CSC out
        read = 12 * nnz if case["start"] == "triples" else 8 * nnz + 4 * m
        return {"bytes": read + 2 * (8 * nnz + 4 * (m + 1)), "flops": 0}
    m, nnz, vb, ob = _rows(case), _entries(case), BYTES[case["dtype"]], BYTES[case["out"]]
    if case["path"] in ("spmv", "spmvop"):
        return {"bytes": wl.spmv_bytes_alg(m, m, nnz, vb, vb, ob, case["beta"] != 0.0), "flops": 2 * nnz}
    n = case["n"]
    bytes_, flops = wl.spmm_bytes_alg(m, m, n, nnz, vb, vb, ob), 2 * nnz * n
    return {"bytes": 2 * bytes_, "flops": 2 * flops} if case["path"] == "train" else {"bytes": bytes_, "flops": flops}


def tolerance(case):
    if case["path"] == "assemble":
        return "exact"
    # Sums are kept in fp64 and rounded once to the output's type: against the same product in 64 bits the relative
    # error is that rounding, 2.5e-8 (fp32), 2.1e-4 (fp16), 1.7e-3 (bf16); four times that.
    rel = {"f32": 1e-7, "f16": 8e-4, "bf16": 7e-3}[case["out"]]
    if case.get("op") == "t":
        rel = 1e-6  # the transposed product of a narrow matrix adds into y in fp32, in any order: 2.4e-7 seen
    return {"rel": rel}
