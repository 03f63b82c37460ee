"""Which matrices of 2 to 7 M entries the default algorithm re-stores: op(A) = A^T over more than 2^18 columns, uneven rows from
2^19 rows and columns on, even rows over an x of 6 MiB and more.  Either side of every bound, by the buffer that
GetBufferSize asks for, and the product against the fp64 oracle (bars as for the layouts at any size)."""
import math

import numpy as np
import pytest
import torch

import oracle
from helpers import to_dev

pytestmark = pytest.mark.gpu


def _matrix(rows, cols, nnz, uneven, seed):
    rng = np.random.default_rng(seed)
    per = nnz // rows
    lengths = np.full(rows, per, np.int64)
    if uneven:
        long_rows = rng.choice(rows, rows // 200, replace=False)
        lengths[long_rows] = 10 * per + 30
    lengths[: nnz - int(lengths.sum())] += 1 if lengths.sum() < nnz else 0
    rowptr = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)
    return rowptr, rng.integers(0, cols, int(rowptr[-1])).astype(np.int32)


@pytest.mark.parametrize("rows,cols,nnz,uneven,transpose,dtype,layout", [
    (1 << 19, 1 << 19, 2_100_000, True, False, "f32", True),
    ((1 << 19) - 1, 1 << 20, 2_100_000, True, False, "f32", False),
    (1 << 20, (1 << 19) - 1, 2_100_000, True, False, "f32", False),
    (1 << 20, 1_572_864, 2_100_000, False, False, "f32", True),
    (1 << 20, 1_572_863, 2_100_000, False, False, "f32", False),
    (1 << 20, 1_572_864, 2_100_000, False, False, "f16", False),
    (1 << 20, 3_145_728, 2_100_000, False, False, "bf16", True),
    (1 << 20, 3_000_000, 1_990_000, False, False, "f32", False),
    (400_000, (1 << 18) + 1, 2_100_000, False, True, "f32", True),
    (400_000, 1 << 18, 2_100_000, False, True, "f32", False),
    (600_000, 600_000, 2_100_000, True, True, "f16", True),
    (600_000, 600_000, 1_990_000, True, True, "f32", False),
    (600_000, 600_000, 2_100_000, False, True, "i32", False),
])
def test_bounds_of_the_layout_below_seven_million_entries(osa, gpu_ctx, monkeypatch, rows, cols, nnz, uneven, transpose, dtype,
                                                          layout):
    for name in ("OPS_SPARSE_DEFAULT_BLOCKED_MIN_NNZ", "OPS_SPARSE_ORDERED_LIVE_MIN_COLS", "OPS_SPARSE_SPMV_REPEATABLE"):
        monkeypatch.delenv(name, raising=False)
    dev, stream, handle = gpu_ctx
    rowptr, colind = _matrix(rows, cols, nnz, uneven, rows + cols)
    nnz = colind.size
    rng = np.random.default_rng(3)
    n_x, n_y = (rows, cols) if transpose else (cols, rows)
    kind = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16, "i32": torch.int32}[dtype]
    if dtype == "i32":
        val, x, y0 = (rng.integers(-5, 6, n).astype(np.int32) for n in (nnz, n_x, n_y))
    else:
        val, x = (torch.from_numpy(rng.uniform(-1, 1, n).astype(np.float32)).to(kind).float().numpy() for n in (nnz, n_x))
        y0 = rng.uniform(-1, 1, n_y).astype(np.float32)
    y = to_dev(y0.astype(np.float32), dev)
    A = osa.Csr(rows, cols, to_dev(rowptr, dev), to_dev(colind, dev), to_dev(val, dev, kind))
    op = osa.SpmvOp(handle, A, osa.DnVec(to_dev(x, dev, kind)), osa.DnVec(y),
                    op=osa.ACL_SPARSE_OP_TRANSPOSE if transpose else osa.ACL_SPARSE_OP_NON_TRANSPOSE)
    assert (op.buffer.numel() > osa.lib().opsparse_spmv_csr_workspace_bytes(rows, nnz)) == layout
    op(1.5, -0.5)
    stream.synchronize()
    fn = oracle.spmv_trans_f64 if transpose else oracle.spmv_f64
    gold = fn(rows, cols, rowptr, colind, val.astype(np.float32), x.astype(np.float32), y0.astype(np.float32), 1.5, -0.5)
    if transpose and not layout:                   # fp32 atomics on y: the bar of test_every_kernel_gpu.py for them
        assert np.abs(y.cpu().numpy() - gold).max() <= (1e-2 if dtype != "i32" else 1e-3 * np.abs(gold).max())
    else:
        assert oracle.max_rel_err(y.cpu().numpy(), gold) <= 1e-5


def test_a_matrix_that_the_ordered_layout_refuses_repeats_below_seven_million_entries(osa, gpu_ctx, monkeypatch):
    """op(A) = A of fewer than 7 M entries with the default algorithm gives the same bits from every call, also where a row of
    more than 65 534 entries whose columns do not ascend keeps the ordered layout away: the buffer has no room for the layout
    that adds with atomics.  Products exact in fp64 whose large ones cancel, so that another order gives other bits."""
    for name in ("OPS_SPARSE_DEFAULT_BLOCKED_MIN_NNZ", "OPS_SPARSE_ORDERED_LIVE_MIN_COLS", "OPS_SPARSE_SPMV_REPEATABLE"):
        monkeypatch.delenv(name, raising=False)
    dev, stream, handle = gpu_ctx
    rows = cols = 1 << 19
    rng = np.random.default_rng(11)
    lengths = np.full(rows, 4, np.int64)
    lengths[rng.choice(rows, 2000, replace=False)] = 60
    lengths[777] = 70_000
    rowptr = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)
    nnz = int(rowptr[-1])
    colind = rng.integers(0, cols, nnz).astype(np.int32)
    a, b = rowptr[777], rowptr[778]
    colind[a:b] = np.sort(rng.choice(cols, b - a, replace=False))[::-1]
    val = np.ldexp(1.0, rng.integers(-30, 1, nnz)).astype(np.float32) * rng.choice([-1.0, 1.0], nnz).astype(np.float32)
    for r in np.nonzero(lengths >= 60)[0]:          # pairs of +-2^40 .. 2^60 at random places of the longer rows
        at = rowptr[r] + rng.choice(lengths[r], 2 * (lengths[r] // 6), replace=False)
        val[at[::2]] = np.ldexp(1.0, rng.integers(40, 61, at.size // 2)).astype(np.float32)
        val[at[1::2]] = -val[at[::2]]
    A = osa.Csr(rows, cols, to_dev(rowptr, dev), to_dev(colind, dev), to_dev(val, dev))
    y = torch.zeros(rows, device=dev)
    op = osa.SpmvOp(handle, A, osa.DnVec(torch.ones(cols, device=dev)), osa.DnVec(y))
    L = osa.lib()
    assert op.buffer.numel() == L.opsparse_spmv_csr_blocked_workspace_bytes(rows, cols, nnz, osa.OPSPARSE_BLOCKED_LIVE_VALUES)
    assert op.buffer.numel() != L.opsparse_spmv_csr_live_workspace_bytes(rows, cols, nnz)
    outs = []
    for _ in range(6):
        op(1.0, 0.0)
        stream.synchronize()
        outs.append(y.clone())
    assert all(torch.equal(o, outs[0]) for o in outs[1:])
    # (whatever the order: fp64 partial sums of n terms stay within n * 2^-53 * sum |terms| of the exact one)
    got = outs[0].cpu().numpy().astype(np.float64)
    for r in [777, *np.nonzero(lengths == 60)[0][:50], *range(64)]:
        terms = val[rowptr[r]:rowptr[r + 1]].astype(np.float64)
        slack = (terms.size + 2) * 2.0 ** -52 * np.abs(terms).sum() + abs(math.fsum(terms)) * 2.0 ** -23
        assert abs(got[r] - math.fsum(terms)) <= slack, r
