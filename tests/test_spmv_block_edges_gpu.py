"""Windowed row blocks at their edges: the four values at the end of the value array, which a lane loads from further in front,
and rows whose pieces lie in several wavefronts and several windows of a block, with an old y to be scaled."""
import numpy as np
import pytest
import torch

import oracle
from helpers import to_dev

pytestmark = pytest.mark.gpu

COLS = 1_400_000


def _matrix(rows, tail, spans, seed):
    """Short rows; `spans`: rows of many entries, their columns in no order, so that they stay in the blocks; the last rows hold
    `tail` entries each."""
    rng = np.random.default_rng(seed)
    lengths = rng.integers(0, 16, rows)
    for row, n in spans.items():
        lengths[row] = n
    lengths[-2:] = tail
    rowptr = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)
    nnz = int(rowptr[-1])
    return rowptr, rng.integers(0, COLS, nnz).astype(np.int32), rng


@pytest.mark.parametrize("tail", [1, 2, 3, 4, 7, 16, 17, 0])
@pytest.mark.parametrize("dtype,alg", [("f32", "default"), ("f16", "default"), ("f32", "frozen")])
def test_last_values_of_the_array_and_rows_across_windows(osa, gpu_ctx, monkeypatch, tail, dtype, alg):
    for name in ("OPS_SPARSE_DEFAULT_BLOCKED_MIN_NNZ", "OPS_SPARSE_ORDERED_LIVE_MIN_COLS"):
        monkeypatch.setenv(name, "0")
    monkeypatch.setenv("OPS_SPARSE_BLOCKED_NO_STREAM", "1")
    dev, stream, handle = gpu_ctx
    rows = 300_001
    spans = {5: 300, 1000: 4096, 1001: 4097, 40_000: 9000, 80_000: 20_000, 80_001: 3, rows - 4: 6000}
    rowptr, colind, rng = _matrix(rows, tail, spans, 100 + tail)
    nnz = colind.size
    kind = {"f32": torch.float32, "f16": torch.float16}[dtype]
    val, x = (torch.from_numpy(rng.uniform(-1, 1, n).astype(np.float32)).to(kind).float().numpy() for n in (nnz, COLS))
    y0 = rng.uniform(-1, 1, rows).astype(np.float32)
    y = to_dev(y0, dev)
    A = osa.Csr(rows, COLS, to_dev(rowptr, dev), to_dev(colind, dev), to_dev(val, dev, kind))
    op = osa.SpmvOp(handle, A, osa.DnVec(to_dev(x, dev, kind)), osa.DnVec(y),
                    alg=osa.ACL_SPARSE_SPMV_CSR_ALG2 if alg == "frozen" else osa.ACL_SPARSE_SPMV_ALG_DEFAULT)
    assert op.buffer.numel() > osa.lib().opsparse_spmv_csr_workspace_bytes(rows, nnz)
    op(1.5, -0.5)
    stream.synchronize()
    gold = oracle.spmv_f64(rows, COLS, rowptr, colind, val, x, y0, 1.5, -0.5)
    assert oracle.max_rel_err(y.cpu().numpy(), gold) <= 1e-5


@pytest.mark.parametrize("rows,longest,ends", [(65_536, 76, False), (65_537, 76, True), (131_071, 40, False), (400_000, 12, True)])
def test_where_the_blocks_are_cut(osa, gpu_ctx, monkeypatch, rows, longest, ends):
    """Blocks end behind their most rows (65 536 are 32 times as many; a stretch of rows of one entry and none) and behind long
    rows (one beside another, the first and the last row of the matrix)."""
    for name in ("OPS_SPARSE_DEFAULT_BLOCKED_MIN_NNZ", "OPS_SPARSE_ORDERED_LIVE_MIN_COLS"):
        monkeypatch.setenv(name, "0")
    dev, stream, handle = gpu_ctx
    rng = np.random.default_rng(rows)
    lengths = rng.integers(0, longest + 1, rows)
    lengths[20_000:26_500] = rng.integers(0, 2, 6500)
    long_rows = [0, 30_000, 30_001, 65_535, rows - 1] if ends else [40_000]
    lengths[long_rows] = 64 * (COLS // 32768 + 1) + 4096
    if rows > 131_072:
        lengths[131_071:131_074] = [7167, 7168, 7169]  # (their columns in no order: they stay in the blocks)
    rowptr = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)
    nnz = int(rowptr[-1])
    colind = rng.integers(0, COLS, nnz).astype(np.int32)
    for r in long_rows:
        colind[rowptr[r]:rowptr[r + 1]].sort()
    val, x = rng.uniform(-1, 1, nnz).astype(np.float32), rng.uniform(-1, 1, COLS).astype(np.float32)
    y = torch.full((rows,), float("nan"), device=dev)
    A = osa.Csr(rows, COLS, to_dev(rowptr, dev), to_dev(colind, dev), to_dev(val, dev))
    op = osa.SpmvOp(handle, A, osa.DnVec(to_dev(x, dev)), osa.DnVec(y))
    assert op.buffer.numel() > osa.lib().opsparse_spmv_csr_workspace_bytes(rows, nnz)
    op(1.0, 0.0)
    stream.synchronize()
    gold = oracle.spmv_f64(rows, COLS, rowptr, colind, val, x, np.zeros(rows, np.float32), 1.0, 0.0)
    assert oracle.max_rel_err(y.cpu().numpy(), gold) <= 1e-5


@pytest.mark.parametrize("rows,least,longest,hubs", [
    (30_000, 380, 420, 0), (131_072, 0, 36, 0), (131_073, 0, 36, 0), (262_145, 0, 16, 0), (70_000, 60, 80, 223), (70_000, 30, 40, 600),
    (200_000, 10, 14, 900)])
def test_where_a_stretch_of_blocks_ends(osa, gpu_ctx, monkeypatch, rows, least, longest, hubs):
    """The blocks are cut by workgroups that take 65 536 rows, or 256 blocks' worth of entries (7168 a block), rows (2048) and long
    rows: several such stretches in the same 65 536 rows, by entries and by long rows, and one."""
    for name in ("OPS_SPARSE_DEFAULT_BLOCKED_MIN_NNZ", "OPS_SPARSE_ORDERED_LIVE_MIN_COLS"):
        monkeypatch.setenv(name, "0")
    dev, stream, handle = gpu_ctx
    rng = np.random.default_rng(rows + hubs)
    lengths = rng.integers(least, longest + 1, rows)
    hub_rows = 1000 + np.arange(hubs) * 3
    lengths[hub_rows] = 64 * (COLS // 32768 + 1) + 4096
    rowptr = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)
    nnz = int(rowptr[-1])
    colind = rng.integers(0, COLS, nnz).astype(np.int32)
    for r in hub_rows:
        colind[rowptr[r]:rowptr[r + 1]].sort()
    val, x = rng.uniform(0.5, 1, nnz).astype(np.float32), rng.uniform(0.5, 1, COLS).astype(np.float32)
    y = torch.full((rows,), float("nan"), device=dev)
    A = osa.Csr(rows, COLS, to_dev(rowptr, dev), to_dev(colind, dev), to_dev(val, dev))
    op = osa.SpmvOp(handle, A, osa.DnVec(to_dev(x, dev)), osa.DnVec(y))
    assert op.buffer.numel() > osa.lib().opsparse_spmv_csr_workspace_bytes(rows, nnz)
    op(1.0, 0.0)
    stream.synchronize()
    gold = oracle.spmv_f64(rows, COLS, rowptr, colind, val, x, np.zeros(rows, np.float32), 1.0, 0.0)
    assert oracle.max_rel_err(y.cpu().numpy(), gold) <= 2 ** -23  # (sums in 64 bits, rounded once)


@pytest.mark.parametrize("streamed", [False, True])
@pytest.mark.parametrize("dtype,alg", [("f16", "default"), ("bf16", "default"), ("f16", "frozen"), ("bf16", "frozen")])
def test_gathered_x_of_16_bits(osa, gpu_ctx, monkeypatch, dtype, alg, streamed):
    """x of every bit pattern, from an odd 16-bit place on.  Eight entries of a row name one column and hold 1/8 each: y is that
    element of x, bit for bit.  A long row over positive elements keeps its values behind the gathered x (frozen)."""
    for name in ("OPS_SPARSE_DEFAULT_BLOCKED_MIN_NNZ", "OPS_SPARSE_ORDERED_LIVE_MIN_COLS"):
        monkeypatch.setenv(name, "0")
    if not streamed:
        monkeypatch.setenv("OPS_SPARSE_BLOCKED_NO_STREAM", "1")
    dev, stream, handle = gpu_ctx
    kind = {"f16": torch.float16, "bf16": torch.bfloat16}[dtype]
    rng = np.random.default_rng(17)
    rows, long_row, long_len = 300_001, 170_000, 20_000
    bits = torch.from_numpy(((np.arange(COLS + 1) * 40503) % 65536).astype(np.uint16).view(np.int16))
    x = bits.view(kind).to(dev)[1:]
    x64 = bits.view(kind)[1:].double().numpy()
    lengths = np.full(rows, 8)
    lengths[long_row] = long_len
    rowptr = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)
    of_row = rng.integers(0, COLS, rows)
    colind = np.repeat(of_row, lengths).astype(np.int32)
    tame = np.flatnonzero((x64 > 0.01) & (x64 < 100.0))
    colind[rowptr[long_row]:rowptr[long_row + 1]] = np.sort(rng.choice(tame, long_len, replace=False))
    val = torch.full((colind.size,), 0.125, dtype=kind, device=dev)
    y = torch.full((rows,), 7.0, device=dev)
    A = osa.Csr(rows, COLS, to_dev(rowptr, dev), to_dev(colind, dev), val)
    op = osa.SpmvOp(handle, A, osa.DnVec(x), osa.DnVec(y),
                    alg=osa.ACL_SPARSE_SPMV_CSR_ALG2 if alg == "frozen" else osa.ACL_SPARSE_SPMV_ALG_DEFAULT)
    assert op.buffer.numel() > osa.lib().opsparse_spmv_csr_workspace_bytes(rows, colind.size)
    op(1.0, 0.0)
    stream.synchronize()
    got, want = y.cpu().numpy(), x64[of_row].astype(np.float32)
    want[long_row] = got[long_row]
    assert np.array_equal(got, want, equal_nan=True)
    total = 0.125 * x64[colind[rowptr[long_row]:rowptr[long_row + 1]]].sum()
    assert abs(got[long_row] - total) <= 2 ** -23 * total  # (a sum in 64 bits, rounded once)


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_pieces_of_long_rows_of_every_length(osa, gpu_ctx, monkeypatch, dtype):
    """Live values: what a long row has in one panel is summed by 16 lanes, 64 entries a request and four requests at a time where
    there are as many; the remainders on either side, and the end of the arrays."""
    monkeypatch.setenv("OPS_SPARSE_DEFAULT_BLOCKED_MIN_NNZ", "0")
    dev, stream, handle = gpu_ctx
    kind = {"f32": torch.float32, "bf16": torch.bfloat16}[dtype]
    rng = np.random.default_rng(23)
    rows, cols, panel = 300_000, 1_000_000, 32768
    pieces = [0, 1, 3, 63, 64, 65, 191, 192, 193, 195, 196, 197, 255, 256, 257, 447, 448, 449, 511, 512, 513, 1024, 1999, 2047]
    lengths = rng.integers(6, 11, rows)
    lengths[-1] = 0
    own = {}
    for k, n in enumerate(pieces):
        row = rows - 1 if k == len(pieces) - 1 else 1000 + 7 * k  # (one of them ends where the arrays do)
        other = np.sort(rng.choice(panel, 4096 - n, replace=False)) if k % 2 else np.sort(rng.choice(cols - 4 * panel, 4096 - n, replace=False) + 4 * panel)
        own[row] = np.sort(np.concatenate([other, 2 * panel + rng.choice(panel, n, replace=False)]))
        lengths[row] = 4096
    rowptr = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)
    colind = rng.integers(0, cols, int(rowptr[-1])).astype(np.int32)
    for row, c in own.items():
        colind[rowptr[row]:rowptr[row + 1]] = c
    val, x = (torch.from_numpy(rng.uniform(0.5, 1, n).astype(np.float32)).to(kind).float().numpy() for n in (colind.size, cols))
    y = torch.full((rows,), float("nan"), device=dev)
    A = osa.Csr(rows, cols, to_dev(rowptr, dev), to_dev(colind, dev), to_dev(val, dev, kind))
    op = osa.SpmvOp(handle, A, osa.DnVec(to_dev(x, dev, kind)), osa.DnVec(y))
    assert op.buffer.numel() > osa.lib().opsparse_spmv_csr_workspace_bytes(rows, colind.size)
    op(1.0, 0.0)
    stream.synchronize()
    gold = oracle.spmv_f64(rows, cols, rowptr, colind, val, x, np.zeros(rows, np.float32), 1.0, 0.0)
    assert oracle.max_rel_err(y.cpu().numpy(), gold) <= 2 ** -23  # (sums in 64 bits, rounded once)
