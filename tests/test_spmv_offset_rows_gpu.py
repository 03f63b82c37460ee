"""The plan of a matrix whose rows repeat (plan kernel OPSPARSE_SPMV_OFFSET_ROWS): the columns of row r are r plus one of a
few lists of distances, and the product reads a byte a row instead of the column indices.  Against the fp64 oracle, and
against the row-wise plan of the same matrix.

Bars as for every kernel that sums in fp64 and rounds once: fp32 y within 1e-5 of the oracle element by element, 16-bit y
within one unit in the last place, int32 exactly."""
import ctypes

import numpy as np
import pytest
import torch

import oracle
from helpers import to_dev
from test_every_kernel_gpu import SPMV_TYPES, RawSpmv, _type_code

pytestmark = pytest.mark.gpu


def _matrix(rows, cols, lists, choose, order=None):
    """Row r takes the distances of lists[choose[r]] that stay inside [0, cols)."""
    parts, lengths = [], np.zeros(rows, np.int64)
    for r in range(rows):
        c = r + np.asarray(lists[choose[r]], np.int64)
        c = c[(c >= 0) & (c < cols)]
        if order is not None:
            c = order(r, c)
        parts.append(c)
        lengths[r] = c.size
    rowptr = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)
    return rowptr, (np.concatenate(parts) if rowptr[-1] else np.zeros(0)).astype(np.int32)


def _spread(n, reach, seed):
    """n distances in ascending order, neighbours among them, the furthest `reach` away."""
    rng = np.random.default_rng(seed)
    d = set([-reach, reach, 0, 1, -1][:n])
    while len(d) < n:
        d.add(int(rng.integers(-reach, reach + 1)))
    return sorted(d)


def repeating_rows(rows, distances, dev, others=None):
    """Row offsets and columns, on the device, of the matrix whose row r has the distances that stay inside; stretches of 64
    rows in turns have `others` instead."""
    r = torch.arange(rows, device=dev)[:, None]
    every = sorted(set(distances) | set(others or []))
    cols = r + torch.tensor(every, device=dev)
    has = torch.tensor([[d in l for d in every] for l in (distances, others or distances)], device=dev)
    ok = (cols >= 0) & (cols < rows) & has[r[:, 0] // 64 % 2]
    ends = torch.cumsum(ok.sum(1), 0)
    return torch.cat([ends.new_zeros(1), ends]).int(), cols[ok].int()


def follows_lists(call, out, rowptr, colind, stream):
    """Does `call` multiply by what Preprocess saw (True) or by the column indices as they are?  All ones, but the first
    element (row) of x (B): with every index set to 0 in place, the sums over the indices are 0.  Row sums either way."""
    call()
    stream.synchronize()
    counts = (rowptr[1:] - rowptr[:-1]).float()
    touched = torch.zeros_like(counts).index_add_(0, torch.repeat_interleave(torch.arange(counts.numel(), device=colind.device),
                                                                             rowptr.diff().long()), (colind == 0).float())
    want = (counts - touched).view(-1, *[1] * (out.dim() - 1))
    assert bool((out.float() == want).all())
    kept = colind.clone()
    colind.zero_()
    call()
    stream.synchronize()
    colind.copy_(kept)
    lists = bool((out.float() == want).all())
    assert lists or not bool(out.any())
    return lists


def _offsets_plan(m, want=True):
    osa = m.osa
    plan = m.analyse(osa.OPSPARSE_SPMV_STREAM_ROWS)
    before = bytes(plan)
    rc = m.L.opsparse_spmv_csr_offsets_analyse(m.d_rp.data_ptr(), m.d_ci.data_ptr(), m.rows, m.cols, m.nnz, m.ws.data_ptr(),
                                               m.ws.numel(), ctypes.byref(plan), m.sp)
    if want:
        assert rc == osa.OPSPARSE_OK and plan.kernel == osa.OPSPARSE_SPMV_OFFSET_ROWS
    else:
        assert rc == osa.OPSPARSE_E_UNSUPPORTED and bytes(plan) == before
    return plan


@pytest.mark.parametrize("distances", [1, 5, 6, 7, 8, 9, 10, 18, 19, 27, 28, 32])
@pytest.mark.parametrize("types", sorted(SPMV_TYPES))
def test_every_width_and_type(osa, gpu_ctx, types, distances):
    """Every compiled width at its largest and one more, rows that end inside a tile (1024, and 128 k + 1 or - 1), first
    and last rows cut by the matrix's edges."""
    for rows in (1024, 1281, 1407):
        rowptr, colind = _matrix(rows, rows, [_spread(distances, 20, distances)], np.zeros(rows, int))
        m = RawSpmv(osa, gpu_ctx, rowptr, colind, rows, types, seed=rows)
        plan = _offsets_plan(m)
        assert plan.numDistances == distances
        for alpha, beta in ((1, 0), (2, -1)):
            m.launch_and_check(plan, alpha, beta)


@pytest.mark.parametrize("rows,cols", [(5000, 5000), (5000, 7300), (7300, 5000)])
def test_lists_in_any_order_of_the_rows(osa, gpu_ctx, rows, cols):
    """Several lists mixed at random, one of them empty; more or fewer columns than rows (rows past the last column keep
    the distances that reach back, or none)."""
    rng = np.random.default_rng(rows + cols)
    lists = [_spread(9, 40, 1), _spread(9, 40, 1)[::2], _spread(9, 40, 1)[1:], [], [0]]
    choose = rng.choice(5, rows, p=[0.8, 0.08, 0.08, 0.02, 0.02])
    reach = [-d for d in range(2300, 2303)]
    lists = [sorted(l + reach) if len(l) > 3 else l for l in lists] if rows > cols else lists
    rowptr, colind = _matrix(rows, cols, lists, choose)
    m = RawSpmv(osa, gpu_ctx, rowptr, colind, cols, "f32", seed=4)
    plan = _offsets_plan(m)
    assert plan.numPatterns >= 5
    m.launch_and_check(plan, 1.5, 0.5)


def test_what_is_no_such_matrix_keeps_its_plan(osa, gpu_ctx):
    """Columns that do not ascend, a repeated column, more than 128 lists, more than 32 distances, a column outside, one row
    off by one in the middle of thousands of equal ones counts as a list of its own, mostly empty steps, random columns."""
    rows = 3000
    base = _spread(7, 30, 3)
    same = np.zeros(rows, int)

    def case(rowptr, colind, want, cols=rows):
        m = RawSpmv(osa, gpu_ctx, rowptr, np.clip(colind, 0, cols - 1).astype(np.int32), cols, "f32", seed=1)
        m.d_ci.copy_(to_dev(colind, m.dev))
        plan = _offsets_plan(m, want)
        if want:
            m.launch_and_check(plan, 1.0, 0.5)

    rowptr, colind = _matrix(rows, rows, [base], same)
    case(rowptr, colind, True)
    case(*_matrix(rows, rows, [base], same, lambda r, c: c[::-1]), False)
    twice = colind.copy()
    k = rowptr[1500]
    twice[k + 1] = twice[k]
    case(rowptr, twice, False)
    moved = colind.copy()
    moved[rowptr[1500] + 6] += 1                      # (still ascending: an eighth distance and one more list)
    case(rowptr, moved, True)
    outside = colind.copy()
    outside[rowptr[rows - 1]:] += 40                  # (read by the analysis only: nothing is launched)
    case(rowptr, outside, False)
    many = [sorted(set([0, 1 + i % 16, 17 + i // 16])) for i in range(160)]
    case(*_matrix(rows, rows, many, np.arange(rows) // 18 % 160), False)
    case(*_matrix(rows, rows, [_spread(33, 40, 2)], same), False)
    halves = [[-3, -2, -1, 0], [10, 20, 30], [40, 50, 60, 70]]
    case(*_matrix(rows, rows, halves, np.arange(rows) // 100 % 3), False)
    rng = np.random.default_rng(9)
    case((np.arange(rows + 1) * 6).astype(np.int32), np.sort(rng.integers(0, rows, (rows, 6)), 1).reshape(-1).astype(np.int32),
         False)


def test_more_tiles_than_wavefronts(osa, gpu_ctx):
    """A launch has at most 4096 workgroups of four wavefronts: past 2.1 M rows (two a lane) a wavefront takes a second
    tile, whose bounds and lists were asked for during the first."""
    rows = 4096 * 4 * 128 + 64 * 3 + 1
    d = np.array([-1500, -1, 0, 1, 1500])
    cols = np.arange(rows)[:, None] + d
    ok = (cols >= 0) & (cols < rows)
    rowptr = np.concatenate([[0], np.cumsum(ok.sum(1))]).astype(np.int32)
    m = RawSpmv(osa, gpu_ctx, rowptr, cols[ok].astype(np.int32), rows, "f32", seed=2)
    m.launch_and_check(_offsets_plan(m), 1.0, 0.5)


@pytest.mark.parametrize("shift", [0, 1, 3])
@pytest.mark.parametrize("entry", ["spmv", "alg2", "spmvop_alg2"])
def test_public_calls_follow_the_values_and_agree_with_the_row_wise_plan(osa, gpu_ctx, workloads, monkeypatch, entry, shift):
    """Preprocess / createDescr takes the plan by itself.  Operands that begin `shift` elements behind an aligned address,
    values that change in place, and the same bits as the row-wise plan, which sums short rows in the same order."""
    dev, stream, handle = gpu_ctx
    A = workloads.stencil_csr((37, 41, 29), [(-1, 0, 0), (0, -1, 0), (0, 0, -1), (0, 0, 0), (0, 0, 1), (0, 1, 0), (1, 0, 0)], dev)
    rows, nnz = A["rows"], int(A["colind"].numel())

    def behind(t):
        room = torch.zeros(t.numel() + 8, dtype=t.dtype, device=dev)
        room[shift:shift + t.numel()] = t
        return room[shift:shift + t.numel()]

    values, x = behind(workloads.uniform(1, nnz, -1.0, 1.0, dev)), behind(workloads.uniform(2, rows, -1.0, 1.0, dev))
    y0 = workloads.uniform(3, rows, -1.0, 1.0, dev)
    csr = osa.Csr(rows, rows, behind(A["rowptr"]), behind(A["colind"]), values)
    got = {}
    monkeypatch.setenv("OPS_SPARSE_OFFSETS_ANY_SIZE", "1")   # (at this size the row-wise plan is the faster one)
    for switch in (False, True):
        if switch:
            monkeypatch.setenv("OPS_SPARSE_SPMV_NO_OFFSETS", "1")
        y = behind(y0)
        if entry == "spmvop_alg2":
            z = behind(torch.zeros_like(y0))
            op = osa.SpmvOpPlan(handle, csr, osa.DnVec(x), osa.DnVec(y), osa.DnVec(z), alg=osa.ACL_SPARSE_SPMVOP_ALG2)
        else:
            z = y
            op = osa.SpmvOp(handle, csr, osa.DnVec(x), osa.DnVec(y),
                            alg=osa.ACL_SPARSE_SPMV_CSR_ALG2 if entry == "alg2" else osa.ACL_SPARSE_SPMV_ALG_DEFAULT)
        outs = []
        for round_ in range(2):
            if round_ == 1 and entry == "spmv":
                values.mul_(-0.5)
            y.copy_(y0)
            op(1.5, -0.5)
            stream.synchronize()
            outs.append(z.cpu().numpy().copy())
            gold = oracle.spmv_f64(rows, rows, A["rowptr"].cpu().numpy(), A["colind"].cpu().numpy(), values.cpu().numpy(),
                                   x.cpu().numpy(), y0.cpu().numpy(), 1.5, -0.5)
            assert oracle.max_rel_err(outs[-1], gold) <= 1e-5
        if entry == "spmv":
            values.mul_(-2.0)
        got[switch] = outs
    for a, b in zip(got[False], got[True]):
        assert np.array_equal(a, b)


def test_launch_wants_the_buffer_of_the_plan(osa, gpu_ctx):
    """A workspace that is missing or too small, or a transposed product (which takes the row lengths only)."""
    rows = 2000
    rowptr, colind = _matrix(rows, rows, [_spread(5, 9, 5)], np.zeros(rows, int))
    m = RawSpmv(osa, gpu_ctx, rowptr, colind, rows, "f32", seed=3)
    plan = _offsets_plan(m)
    S = lambda v: osa.OpsparseScalar(float(v), None, 0, 0)
    args = (ctypes.byref(plan), 0, m.d_rp.data_ptr(), m.d_ci.data_ptr(), m.d_val.data_ptr(), m.d_x.data_ptr(),
            m.d_y.data_ptr(), rows, rows, m.nnz, S(1), S(0), osa.OPSPARSE_F32, osa.OPSPARSE_F32, 0)
    assert m.L.opsparse_spmv_csr_launch(*args, None, 0, m.sp) == osa.OPSPARSE_E_WORKSPACE
    assert m.L.opsparse_spmv_csr_launch(*args, m.ws.data_ptr(), plan.bytes - 1, m.sp) == osa.OPSPARSE_E_WORKSPACE


FIVE, NINE, TEN = [-40, -1, 0, 1, 40], [-40, -39, -38, -1, 0, 1, 38, 39, 40], list(range(-5, 5))
TWENTY = list(range(-10, 10))


@pytest.mark.parametrize("entry", ["spmv", "alg2", "spmvop_alg2", "spmm"])
@pytest.mark.parametrize("distances,rows,lists", [
    (FIVE, 1 << 18, True), (FIVE, (1 << 18) - 1, False), (NINE, (1 << 18) - 1, False), (TEN, 98_304, True),
    (TEN, 98_303, False), (TWENTY, (1 << 17) - 1, False), (TWENTY, 1 << 17, True), ("in turns", (1 << 19) - 64, False), ("in turns", 1 << 19, True)])
def test_either_side_of_every_bound(osa, gpu_ctx, monkeypatch, entry, distances, rows, lists):
    """Which matrices Preprocess / createDescr take lists of, seen from outside: column indices that change in place
    afterwards are not looked at where there are lists.  "in turns": stretches of rows with three and four of six distances."""
    monkeypatch.delenv("OPS_SPARSE_OFFSETS_ANY_SIZE", raising=False)
    dev, stream, handle = gpu_ctx
    if distances == "in turns":
        rowptr, colind = repeating_rows(rows, [-3, 2, 9], dev, [-2, 5, 9, 11])
    else:
        rowptr, colind = repeating_rows(rows, distances, dev)
    A = osa.Csr(rows, rows, rowptr, colind, torch.ones(colind.numel(), device=dev))
    x, y = torch.ones(rows, device=dev), torch.zeros(rows, device=dev)
    x[0] = 0
    X, Y = osa.DnVec(x), osa.DnVec(y)
    if entry == "spmvop_alg2":
        op = osa.SpmvOpPlan(handle, A, X, Y, Y, alg=osa.ACL_SPARSE_SPMVOP_ALG2)
    elif entry == "spmm":
        op = osa.SpmmOp(handle, A, osa.DnMat(rows, 1, 1, x), osa.DnMat(rows, 1, 1, y))
    else:
        op = osa.SpmvOp(handle, A, X, Y, alg=osa.ACL_SPARSE_SPMV_CSR_ALG2 if entry == "alg2" else osa.ACL_SPARSE_SPMV_ALG_DEFAULT)
    assert follows_lists(lambda: op(1.0, 0.0), y, rowptr, colind, stream) == lists


@pytest.mark.parametrize("where", ["a", "x", "beyond_a_list"])
@pytest.mark.parametrize("types", ["f32", "bf16_bf16", "f16_f32"])
@pytest.mark.parametrize("distances", [5, 9, 27])
def test_infinities_and_nan(osa, gpu_ctx, distances, types, where):
    """NaN and infinities in A, in x, and in elements of x that a row's list leaves out although its neighbours' lists name
    them: in y where the plain product has them and nowhere else."""
    rows, rng = 3001, np.random.default_rng(distances)
    every = _spread(distances, 40, 1)
    lists = [every, [d for d in every if d != every[1]], every[1:]]
    choose = np.where(np.arange(rows) % 5 == 3, 1 + np.arange(rows) // 5 % 2, 0)
    if where == "beyond_a_list":
        lists = [[0], [d for d in every if d % 2 == 0], every[:1] + [0]]   # even rows: even distances
        choose = np.where(np.arange(rows) % 2 == 0, 1, 0)
    rowptr, colind = _matrix(rows, rows, lists, choose)
    m = RawSpmv(osa, gpu_ctx, rowptr, colind, rows, types, seed=distances)
    row_wise = m.analyse(osa.OPSPARSE_SPMV_STREAM_ROWS)      # (keeps nothing in the workspace)
    plan = _offsets_plan(m)
    bad = torch.tensor([float("nan"), float("inf"), -float("inf")], device=m.dev)
    if where == "a":
        at = torch.from_numpy(rng.choice(m.nnz, 40, replace=False)).to(m.dev)
        m.d_val[at] = bad[torch.arange(40, device=m.dev) % 3].to(m.d_val.dtype)
    else:
        at = torch.from_numpy(2 * rng.choice(rows // 2, 30, replace=False) + 1).to(m.dev)
        m.d_x[at] = bad[torch.arange(30, device=m.dev) % 3].to(m.d_x.dtype)
    S = lambda v: osa.OpsparseScalar(float(v), None, 0, 0)
    got = []
    for p in (plan, row_wise):
        assert m.L.opsparse_spmv_csr_launch(ctypes.byref(p), 0, m.d_rp.data_ptr(), m.d_ci.data_ptr(), m.d_val.data_ptr(),
                                            m.d_x.data_ptr(), m.d_y.data_ptr(), rows, rows, m.nnz, S(1), S(0),
                                            _type_code(osa, m.val_dtype), _type_code(osa, m.out_dtype), 0, m.ws.data_ptr(),
                                            m.ws.numel(), m.sp) == osa.OPSPARSE_OK
        m.stream.synchronize()
        got.append(m.d_y.float().clone())
    assert bool(got[1].isfinite().any()) and not bool(got[1].isfinite().all())
    assert torch.equal(got[0].isnan(), got[1].isnan()) and torch.equal(got[0].isinf(), got[1].isinf())
    # (fp64 sums in another order, rounded once: two units in the last place, or what 32 terms below 1 leave behind)
    ulp = 2.0 ** -7 if m.out_dtype == torch.bfloat16 else 2.0 ** -22
    fine = got[1].isfinite()
    assert bool(((got[0] - got[1])[fine].abs() <= 2 * ulp * got[1][fine].abs() + 1e-12).all())
    assert torch.equal(got[0][got[1].isinf()], got[1][got[1].isinf()])
