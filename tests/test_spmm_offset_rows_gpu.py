"""SpMM of a matrix whose rows repeat: the columns of row r are r plus one of a few lists of distances, and Preprocess leaves
a byte a row that the product reads instead of the column indices.  Through aclsparseSpMM, against the fp64 oracle.

Bars as in test_spmm_gpu.py: sums in fp64, rounded once: fp32 C within 1e-5 of the oracle element by element, fp16 C within
one unit in the last place of the oracle rounded to fp16."""
import ctypes

import numpy as np
import pytest
import torch

import oracle
from helpers import run_spmm, to_dev
from test_spmv_offset_rows_gpu import _matrix, _spread, follows_lists, repeating_rows

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _lists_at_any_size(monkeypatch):
    """Preprocess takes the lists where they are the faster plan, which small matrices' seldom are."""
    monkeypatch.setenv("OPS_SPARSE_OFFSETS_ANY_SIZE", "1")


DTYPES = {"f32": (torch.float32, torch.float32), "f16": (torch.float16, torch.float16), "f16_f32": (torch.float16, torch.float32)}


def _seen(a, dtype):
    return torch.from_numpy(np.asarray(a, np.float32)).to(dtype).float().numpy()


def _run(osa, gpu_ctx, rowptr, colind, k, n, types, beta, ldb=None, ldc=None, seed=0, **layout):
    val_dtype, c_dtype = DTYPES[types]
    m, rng = rowptr.size - 1, np.random.default_rng(seed + n)
    b_rm, c_rm = layout.get("b_row_major", True), layout.get("c_row_major", True)
    trans = layout.get("trans_b", False)
    b_rows, b_cols = (n, k) if trans else (k, n)
    ldb = ldb or (b_cols if b_rm else b_rows)
    ldc = ldc or (n if c_rm else m)
    val = _seen(rng.uniform(-1, 1, colind.size), val_dtype)
    B = _seen(rng.uniform(-1, 1, (b_rows if b_rm else b_cols) * ldb), val_dtype)
    C0 = _seen(rng.uniform(-1, 1, (m if c_rm else n) * ldc), c_dtype)
    got = run_spmm(osa, gpu_ctx, m, k, n, rowptr, colind, val, B, ldb, C0, ldc, 1.25, beta,
                   order_b=osa.ACL_SPARSE_ORDER_ROW if b_rm else osa.ACL_SPARSE_ORDER_COL,
                   order_c=osa.ACL_SPARSE_ORDER_ROW if c_rm else osa.ACL_SPARSE_ORDER_COL,
                   op_b=osa.ACL_SPARSE_OP_TRANSPOSE if trans else osa.ACL_SPARSE_OP_NON_TRANSPOSE,
                   val_dtype=val_dtype, c_dtype=c_dtype)
    gold = oracle.spmm_f64(m, n, rowptr, colind, val, B, ldb, C0, ldc, 1.25, beta, **layout)
    idx = (np.arange(m)[:, None] * ldc + np.arange(n)[None, :]) if c_rm else (np.arange(n)[None, :] * ldc + np.arange(m)[:, None])
    if c_dtype == torch.float32:
        assert oracle.max_rel_err(got[idx], gold[idx]) <= 1e-5
    else:
        want = _seen(gold[idx], c_dtype)
        assert np.all(np.abs(got[idx] - want) <= 2.0 ** -10 * np.maximum(np.abs(want), 2.0 ** -14))
    mask = np.ones(got.size, bool)
    mask[idx.ravel()] = False
    assert np.array_equal(got[mask], C0[mask])         # between rows (columns) nothing is written


@pytest.mark.parametrize("n", [4, 8, 16, 32, 64, 128, 256])
@pytest.mark.parametrize("distances", [5, 7, 9, 14, 32])
@pytest.mark.parametrize("types", sorted(DTYPES))
def test_every_width_of_b_and_of_the_list(osa, gpu_ctx, types, distances, n):
    """Every compiled pair of pieces a row and chunk of distances (14: a chunk that is not full), rows that end inside a tile,
    first and last rows cut by the matrix's edges."""
    n = n * 2 if types != "f32" and n < 256 else n
    rowptr, colind = _matrix(1151, 1151, [_spread(distances, 20, distances)], np.zeros(1151, int))
    _run(osa, gpu_ctx, rowptr, colind, 1151, n, types, 0.0 if distances % 2 else -0.5)


STAR2, STAR3 = [-40, -1, 0, 1, 40], [-300, -40, -1, 0, 1, 40, 300]
BOX2 = [40 * i + j for i in (-1, 0, 1) for j in (-1, 0, 1)]
BOX3 = [300 * h + d for h in (-1, 0, 1) for d in BOX2]


@pytest.mark.parametrize("stencil", [STAR2, STAR3, BOX2, BOX3], ids=["star2", "star3", "box2", "box3"])
@pytest.mark.parametrize("types,n", [("f32", 68), ("f32", 128), ("f32", 250), ("f32", 256), ("f16", 136), ("f16", 256), ("f16_f32", 256)])
@pytest.mark.parametrize("rows", [1500, 40_007])
def test_two_rows_a_lane_under_stencils(osa, gpu_ctx, stencil, types, n, rows):
    """Distances in runs of the kinds with a kernel of their own, wide B; rows with gaps inside a run and between runs, alone
    and in pairs, beside whole ones; one to four passes a tile."""
    lists = [stencil, stencil[1:], stencil[:-1], stencil[::2], [d for d in stencil if d not in (0, 40)]]
    choose = np.where(np.arange(rows) % 67 < 60, 0, np.arange(rows) % 5)
    rowptr, colind = _matrix(rows, rows, lists, choose)
    _run(osa, gpu_ctx, rowptr, colind, rows, n, types, 0.5 if n % 8 else 0.0)


@pytest.mark.parametrize("n,ldb,ldc", [(1, 5, 4), (2, 2, 2), (3, 3, 3), (5, 6, 5), (7, 7, 9), (12, 12, 12), (33, 33, 40), (50, 51, 50), (62, 64, 62),
                                       (100, 100, 101), (255, 256, 257)])
def test_ragged_widths_and_leading_dimensions_where_they_are(osa, gpu_ctx, n, ldb, ldc):
    rowptr, colind = _matrix(1283, 1400, [_spread(7, 50, 7), [-50, 0]], (np.arange(1283) % 97 == 96).astype(int))
    for beta in (0.0, 0.5):
        _run(osa, gpu_ctx, rowptr, colind, 1400, n, "f32", beta, ldb, ldc)


@pytest.mark.parametrize("rows,n,reach", [(4096 * 4 * 64 + 130, 4, 1000), (4096 * 4 * 16 + 70, 64, 300), (12_007, 64, 3700),
                                          (70_001, 64, 16_000), (5000, 256, 1030)])
def test_bands_and_more_tiles_than_wavefronts(osa, gpu_ctx, rows, n, reach):
    """Past 16 384 tiles a wavefront takes a second one; a far distance under a wide B makes the XCDs take bands (of the last
    three), with lines that end inside a band and a last line that is not whole."""
    d = np.array([-reach, -1, 0, 1, reach])
    cols = np.arange(rows)[:, None] + d
    ok = (cols >= 0) & (cols < rows)
    rowptr = np.concatenate([[0], np.cumsum(ok.sum(1))]).astype(np.int32)
    _run(osa, gpu_ctx, rowptr, cols[ok].astype(np.int32), rows, n, "f32", 0.5)


@pytest.mark.parametrize("layout", [dict(b_row_major=False), dict(c_row_major=False), dict(b_row_major=False, c_row_major=False),
                                    dict(trans_b=True)])
@pytest.mark.parametrize("n", [1, 2, 6, 16, 33])
def test_column_major_and_transposed_operands(osa, gpu_ctx, layout, n):
    """Through row-major copies, or (one or two columns that are vectors) as SpMV calls."""
    rowptr, colind = _matrix(2100, 2100, [_spread(9, 33, 2)], np.zeros(2100, int))
    _run(osa, gpu_ctx, rowptr, colind, 2100, n, "f32", 0.5, **layout)


def test_one_buffer_for_several_widths_and_live_values(osa, gpu_ctx):
    """Preprocess for the widest B; narrower ones, other values in place, and a transposed B (which takes the kernels for any
    columns and their tables) with the same buffer; a matrix that is none keeps what it had."""
    dev, stream, handle = gpu_ctx
    rng = np.random.default_rng(5)
    for rows_repeat in (True, False):
        rowptr, colind = _matrix(3000, 3000, [_spread(6, 40, 1)], np.zeros(3000, int))
        if not rows_repeat:
            colind = rng.integers(0, 3000, colind.size).astype(np.int32)
        val = rng.uniform(-1, 1, colind.size).astype(np.float32)
        d_val = to_dev(val, dev)
        A = osa.Csr(3000, 3000, to_dev(rowptr, dev), to_dev(colind, dev), d_val)
        wide, size = 64, ctypes.c_size_t(0)

        def operands(n, trans):
            B, C = rng.uniform(-1, 1, 3000 * n).astype(np.float32), rng.uniform(-1, 1, 3000 * n).astype(np.float32)
            dB, dC = to_dev(B, dev), to_dev(C, dev)
            return B, C, dC, osa.DnMat(3000, n, 3000 if trans else n, dB), osa.DnMat(3000, n, n, dC)

        one, half = ctypes.c_float(1.0), ctypes.c_float(0.5)
        buf = None
        for n, trans in ((wide, False), (12, False), (wide, False), (8, True), (wide, False), (5, False)):
            B, C, dC, Bd, Cd = operands(n, trans)
            op = osa.ACL_SPARSE_OP_TRANSPOSE if trans else osa.ACL_SPARSE_OP_NON_TRANSPOSE
            common = (handle.h, osa.ACL_SPARSE_OP_NON_TRANSPOSE, op, ctypes.byref(one), A.d, Bd.d, ctypes.byref(half), Cd.d,
                      osa.ACL_FLOAT, osa.ACL_SPARSE_SPMM_ALG_DEFAULT)
            if buf is None:
                assert osa.lib().aclsparseSpMMGetBufferSize(*common, ctypes.byref(size)) == 0
                guard = 4096
                buf = torch.full((size.value + guard,), 0x77, dtype=torch.uint8, device=dev)
                assert osa.lib().aclsparseSpMMPreprocess(*common, buf.data_ptr()) == 0
            assert osa.lib().aclsparseSpMM(*common, buf.data_ptr()) == 0
            stream.synchronize()
            gold = oracle.spmm_f64(3000, n, rowptr, colind, val, B, 3000 if trans else n, C, n, 1.0, 0.5, trans_b=trans)
            assert oracle.max_rel_err(dC.cpu().numpy(), gold) <= 1e-5
            d_val.mul_(-0.5)
            val = val * np.float32(-0.5)
        assert bool((buf[size.value:] == 0x77).all())


@pytest.mark.parametrize("sized_for,then", [(512, 64), (260, 256), (512, 1), (64, 1), (1, 64)])
def test_buffer_sized_for_another_width_holds_the_lists(osa, gpu_ctx, sized_for, then):
    """GetBufferSize for one width, Preprocess and SpMM for another (one column: SpMV calls), in exactly that many bytes."""
    dev, stream, handle = gpu_ctx
    rng, rows = np.random.default_rng(3), 40_000
    d = np.array([-200, -1, 0, 1, 200])
    cols = np.arange(rows)[:, None] + d
    ok = (cols >= 0) & (cols < rows)
    rowptr, colind = np.concatenate([[0], np.cumsum(ok.sum(1))]).astype(np.int32), cols[ok].astype(np.int32)
    val = rng.uniform(-1, 1, colind.size).astype(np.float32)
    A = osa.Csr(rows, rows, to_dev(rowptr, dev), to_dev(colind, dev), to_dev(val, dev))
    one, none, size = ctypes.c_float(1.0), ctypes.c_float(0.0), ctypes.c_size_t(0)

    def call(n):
        B, C = rng.uniform(-1, 1, rows * n).astype(np.float32), to_dev(np.zeros(rows * n, np.float32), dev)
        Bd, Cd = osa.DnMat(rows, n, n, to_dev(B, dev)), osa.DnMat(rows, n, n, C)
        return B, C, (Bd, Cd), (handle.h, osa.ACL_SPARSE_OP_NON_TRANSPOSE, osa.ACL_SPARSE_OP_NON_TRANSPOSE, ctypes.byref(one), A.d,
                                Bd.d, ctypes.byref(none), Cd.d, osa.ACL_FLOAT, osa.ACL_SPARSE_SPMM_ALG_DEFAULT)

    _, _, keep, common = call(sized_for)
    assert osa.lib().aclsparseSpMMGetBufferSize(*common, ctypes.byref(size)) == 0
    buf = torch.full((size.value + (1 << 20),), 0x77, dtype=torch.uint8, device=dev)
    for n in (then, sized_for):
        B, C, keep, common = call(n)
        if n == then:
            assert osa.lib().aclsparseSpMMPreprocess(*common, buf.data_ptr()) == 0
        assert osa.lib().aclsparseSpMM(*common, buf.data_ptr()) == 0
        stream.synchronize()
        gold = oracle.spmm_f64(rows, n, rowptr, colind, val, B, n, np.zeros(rows * n, np.float32), n, 1.0, 0.0)
        assert oracle.max_rel_err(C.cpu().numpy(), gold) <= 1e-5
    assert bool((buf[size.value:] == 0x77).all())


@pytest.mark.parametrize("types,n", [("f32", 128), ("f32", 256), ("f16", 256), ("f16_f32", 256)])
def test_five_scattered_distances_under_wide_b(osa, gpu_ctx, types, n):
    """Few distances that are no star's: one row a lane under 32 and 64 pieces as well."""
    rowptr, colind = _matrix(1500, 1500, [[-30, -7, 0, 9, 40]], np.zeros(1500, int))
    _run(osa, gpu_ctx, rowptr, colind, 1500, n, types, 0.5)


STAR9 = [-40, -39, -38, -1, 0, 1, 38, 39, 40]                 # a 9-point box
TEN, TWENTY, TWENTY_SEVEN = [*STAR9, 80], [7 * i for i in range(-10, 10)], [7 * i for i in range(-13, 14)]


@pytest.mark.parametrize("distances,types,n,rows,lists", [
    # one piece of B a row, two pieces
    (STAR2, "f32", 4, 147_456, True), (STAR2, "f32", 3, 147_455, False), ([-1, 0, 1], "f32", 4, 200_000, False),
    (TWENTY, "f32", 4, 98_304, True), (STAR9, "f16", 8, 98_303, False), ([-1, 0, 1], "f32", 8, 1 << 17, True),
    (STAR2, "f32", 8, (1 << 17) - 1, False), (STAR2, "f16", 16, 1 << 16, True), (STAR3, "f32", 8, (1 << 16) - 1, False),
    # ragged rows, which the other kernels work on copies of
    (STAR2, "f32", 33, 1024, True), (TWENTY, "f32", 50, 1024, True),
    # whole rows, by the list and the width
    (STAR2, "f32", 12, (1 << 17) - 1, False), (STAR2, "f32", 16, 81_920, True), (STAR2, "f32", 24, 163_839, False),
    (STAR2, "f32", 64, 98_304, True), (STAR2, "f32", 64, 98_303, False), ([-1, 0, 1], "f32", 16, (1 << 19) - 1, False),
    ([-1, 0, 1], "f32", 16, 1 << 19, True), (STAR9, "f32", 32, 81_920, True), (STAR9, "f32", 64, 98_303, False),
    (STAR3, "f32", 12, 163_840, True), (STAR3, "f32", 16, (1 << 19) - 1, False), (STAR3, "f32", 32, 393_215, False),
    (STAR3, "f32", 32, 393_216, True), (STAR3, "f32", 64, 196_607, False), (STAR3, "f32", 64, 196_608, True),
    (TWENTY, "f32", 16, 1 << 16, True), (TWENTY, "f32", 16, (1 << 16) - 1, False), (TEN, "f32", 16, (1 << 20) - 1, False),
    (TEN, "f32", 16, 1 << 20, True), (TEN, "f32", 32, 393_215, False), (TEN, "f32", 64, 1 << 18, True),
    (TWENTY_SEVEN, "f32", 32, 1 << 18, True), (TWENTY_SEVEN, "f32", 32, (1 << 18) - 1, False),
    # wider: slabs give way at every size, whole rows only to two rows a lane
    (STAR2, "f32", 128, 1024, True), (STAR9, "f32", 128, 98_304, True), (STAR9, "f32", 128, 98_303, False),
    (TEN, "f32", 128, 1 << 18, False), (STAR9, "f32", 256, 2000, True),
    # fp16: where the plan is slabs
    (STAR2, "f16", 64, 2000, True), (TEN, "f16", 128, (1 << 17) - 1, True), (TEN, "f16", 128, 1 << 17, False), (STAR9, "f16", 64, 1 << 18, False), (TWENTY, "f16_f32", 64, 1 << 18, False)])
def test_either_side_of_every_bound(osa, gpu_ctx, monkeypatch, distances, types, n, rows, lists):
    """Which matrices Preprocess takes lists of, seen from outside: once it has run, other column indices in place are not
    looked at by the kernel that has lists."""
    monkeypatch.delenv("OPS_SPARSE_OFFSETS_ANY_SIZE")
    dev, stream, handle = gpu_ctx
    val_dtype, c_dtype = DTYPES[types]
    rowptr, colind = repeating_rows(rows, distances, dev)
    B, C = torch.ones(rows, n, dtype=val_dtype, device=dev), torch.zeros(rows, n, dtype=c_dtype, device=dev)
    B[0] = 0
    A = osa.Csr(rows, rows, rowptr, colind, torch.ones(colind.numel(), dtype=val_dtype, device=dev))
    op = osa.SpmmOp(handle, A, osa.DnMat(rows, n, n, B.view(-1)), osa.DnMat(rows, n, n, C.view(-1)))
    assert follows_lists(lambda: op(1.0, 0.0), C, rowptr, colind, stream) == lists


@pytest.mark.parametrize("where", ["a", "b", "beyond_a_list"])
@pytest.mark.parametrize("types,n,stencil", [("f32", 4, STAR2), ("f32", 33, STAR3), ("f32", 128, STAR2), ("f32", 256, BOX3), ("f16", 16, STAR3),
                                             ("f16_f32", 128, BOX2)])
def test_infinities_and_nan(osa, gpu_ctx, types, n, stencil, where):
    """NaN and infinities in A, in B, and in rows of B that a row's list leaves out although its neighbours' lists name them:
    where the plain product has them and nowhere else.  (fp16 C is clamped: infinities become 65504.)"""
    val_dtype, c_dtype = DTYPES[types]
    rows, rng = 3001, np.random.default_rng(n)
    lists = [stencil, [d for d in stencil if d != 1], [d for d in stencil if d != stencil[0]]]
    choose = np.where(np.arange(rows) % 5 == 3, 1 + np.arange(rows) // 5 % 2, 0)
    if where == "beyond_a_list":
        choose[:] = np.where(np.arange(rows) % 2 == 0, 1, choose)      # no even row has distance 1 ...
        lists[0] = lists[2] = [0]                                      # ... and the odd ones only their own column
        lists[1] = [d for d in stencil if d % 2 == 0]
    rowptr, colind = _matrix(rows, rows, lists, choose)
    val = _seen(rng.uniform(-1, 1, colind.size), val_dtype)
    B = _seen(rng.uniform(-1, 1, (rows, n)), val_dtype)
    bad = np.array([np.nan, np.inf, -np.inf], np.float32)
    if where == "a":
        val[rng.choice(val.size, 40, replace=False)] = bad[np.arange(40) % 3]
    else:
        at = 2 * rng.choice(rows // 2, 30, replace=False) + 1          # odd rows of B
        B[at] = bad[np.arange(30) % 3][:, None]
    dev, stream, handle = gpu_ctx
    d = [to_dev(rowptr, dev), to_dev(colind, dev), to_dev(val, dev, val_dtype)]
    A, C = osa.Csr(rows, rows, *d), torch.zeros(rows * n, dtype=c_dtype, device=dev)
    op = osa.SpmmOp(handle, A, osa.DnMat(rows, n, n, to_dev(B.ravel(), dev, val_dtype)), osa.DnMat(rows, n, n, C))
    op(1.0, 0.0)
    stream.synchronize()
    got = C.float().cpu().numpy().reshape(rows, n)
    gold = np.zeros((rows, n))
    with np.errstate(invalid="ignore"):
        entry_row = np.repeat(np.arange(rows), np.diff(rowptr))
        np.add.at(gold, entry_row, val[:, None].astype(np.float64) * B[colind].astype(np.float64))
    if c_dtype == torch.float16:
        gold = np.clip(gold, -65504.0, 65504.0)                        # (NaN stays NaN)
    assert np.array_equal(np.isnan(got), np.isnan(gold)) and np.array_equal(np.isinf(got), np.isinf(gold))
    fine = np.isfinite(gold)
    assert fine.any() and not (fine.all() and c_dtype != torch.float16)
    assert np.allclose(got[fine], gold[fine], rtol=2.0 ** -10 if c_dtype == torch.float16 else 1e-5, atol=1e-5)
    assert np.array_equal(np.sign(got[np.isinf(gold)]), np.sign(gold[np.isinf(gold)]))
