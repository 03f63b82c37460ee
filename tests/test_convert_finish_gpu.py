"""csr2csc and coosort where the low bits of the keys are ordered bucket by bucket in LDS: one and two passes over the upper
bits in each workgroup size, buckets up to and beyond the 6 144 entries that one workgroup orders, every entry in a few
buckets, empty buckets, a last bucket cut short by the number of columns.  Bit for bit against the oracle."""
import numpy as np
import pytest

import test_convert_gpu as convert
from test_convert_gpu import NP_TYPE, _typed, run_coosort, run_csr2csc

pytestmark = pytest.mark.gpu

MOST = 6144  # entries of a bucket that one workgroup orders


def columns(what, n, nnz, rng):
    c = rng.integers(0, n, nnz)
    if what == "hubs":
        # the bucket of column 5000 holds nothing else than this column's entries (the widest bucket has 1024 columns)
        c = np.where((c >= 4096) & (c < 10240), c % 4096, c)
        at = rng.permutation(nnz)
        for hub, count in ((5000, MOST), (7000, MOST + 1), (9000, 2 * MOST), (9500, 2 * MOST + 1), (6000, 5 * MOST), (n - 1, 50_000)):
            c[at[:count]] = hub
            at = at[count:]
    elif what == "few":
        c = n // 2 + c % 100
    elif what == "ends":
        c = np.where(c % 2 == 0, 0, n - 1)
    return c.astype(np.int32)


@pytest.mark.parametrize("what", ["uniform", "hubs", "few", "ends"])
@pytest.mark.parametrize("n,nnz,val_type,numeric", [
    (262_143, 400_001, "FP32", True), ((1 << 20) - 77, 3_000_001, "FP16", True), (3_000_001, 6_000_000, "INT8", True),
    ((1 << 20) - 1023, (1 << 23) + 8193, "FP32", True), (700_000, (1 << 23) + 1, "FP32", False)])
def test_csr2csc_buckets(osa, gpu_ctx, n, nnz, val_type, numeric, what):
    rng = np.random.default_rng(nnz + n)
    rowptr = np.concatenate([[0], np.sort(rng.integers(0, nnz + 1, 999)), [nnz]]).astype(np.int32)
    val = _typed(rng.uniform(-1, 1, nnz).astype(np.float32), val_type)
    run_csr2csc(osa, gpu_ctx, 1000, n, rowptr + 1, columns(what, n, nnz, rng) + 1, val, NP_TYPE[val_type], numeric, 1)


@pytest.mark.parametrize("val_type,numeric", [("FP16", True), ("INT8", True), ("FP32", False)])
def test_csr2csc_packed_passes_that_save_none(osa, gpu_ctx, val_type, numeric):
    """17 column bits: two passes either way, over records and with buckets in LDS from 5 M entries on."""
    n, nnz = 100_000, (1 << 23) + 5
    rng = np.random.default_rng(3)
    rowptr = np.array([0, nnz // 3, nnz], np.int32)
    val = _typed(rng.uniform(-1, 1, nnz).astype(np.float32), val_type)
    run_csr2csc(osa, gpu_ctx, 2, n, rowptr, columns("uniform", n, nnz, rng), val, NP_TYPE[val_type], numeric, 0)


@pytest.mark.parametrize("count", [65_537, 2048 * 2048 - 1, 2048 * 2048, 2048 * 2048 + 1])
def test_scan_either_side_of_its_kernels(osa, gpu_ctx, count):
    """Offsets of `count` - 1 rows: from 65 537 on in tiles of 2048, up to 2048 of which add up the sums before their own."""
    convert.test_coo2csr_large_and_unsorted(osa, gpu_ctx, count - 1, 300_000, 1)


@pytest.mark.parametrize("nnz", [1 << 14, (1 << 14) + 1, 61_441])
def test_csr2csc_fewest_entries(osa, gpu_ctx, nnz):
    rng = np.random.default_rng(nnz)
    rowptr = np.array([0, nnz // 3, nnz // 3, nnz], np.int32)
    for n in (3_000, 30_000, 2_000_000):
        run_csr2csc(osa, gpu_ctx, 3, n, rowptr, rng.integers(0, n, nnz).astype(np.int32),
                    rng.uniform(-1, 1, nnz).astype(np.float32), np.float32, True, 0)


@pytest.mark.parametrize("nnz,m,dense,hub,wide", [
    (1_500_000, 60_001, 900, 0, False), ((1 << 23) + 5, 600_001, 3000, 0, False), (1_500_000, 60_001, 0, 0, True),
    (6_000_000, 2_500_000, 0, 0, False), (1_500_000, 200_001, 0, 0, False), (2_000_000, 100_003, 300, 0, True),
    ((1 << 23) + 5, 600_001, 0, 40_000, False), (1_500_000, 60_001, 40, 2500, False), (3_000_000, 400_000, 30_000, 63, False)])
@pytest.mark.parametrize("by_row", [True, False])
def test_coosort_buckets(osa, gpu_ctx, nnz, m, dense, hub, wide, by_row):
    """Short rows, sorted where their bucket is: of 2 - 25 entries on average (every number of lanes to a row); a tenth of the
    entries in `dense` neighbouring rows, which are longer than 64 or lie in buckets that a workgroup cannot order; a row of
    `hub` entries and the next of 64, 65 and 66; rows below zero; column numbers beyond 32-bit keys (`wide`)."""
    rng = np.random.default_rng(nnz + m + dense)
    primary, secondary = rng.integers(0, m, nnz), rng.integers(0, 1 << (30 if wide else 20), nnz)
    at = rng.permutation(nnz)
    if dense:
        primary[at[:nnz // 10]] = rng.integers(1000, 1000 + dense, nnz // 10)
    if hub:
        primary[(primary >= 500) & (primary < 505)] = 7
        for row, count in enumerate((hub, 64, 65, 66)):
            primary[at[-count:]] = 500 + row
            at = at[:-count]
    rows, cols = (primary - 3, secondary) if by_row else (secondary, primary - 3)
    run_coosort(osa, gpu_ctx, 1 << 30, 1 << 30, rows, cols, by_row, perm=rng.permutation(nnz).astype(np.int32))


@pytest.mark.parametrize("m,n,nnz,base", [
    ((1 << 22) - 1, 262_143, 400_001, 1),    # the payload takes 22 bits, the low bits of a key ten
    ((1 << 22) - 1, (1 << 20) - 77, 5_300_003, 0), (1 << 22, (1 << 20) - 77, 5_300_003, 1),  # 22 and 23 bits; one pass fewer or none
    (1 << 24, 300_000, 5_242_880, 1), (3, 300_000, 5_242_879, 0)])
def test_csr2csc_rows_of_many_bits(osa, gpu_ctx, m, n, nnz, base):
    rng = np.random.default_rng(m + n)
    rowptr = np.concatenate([[0], np.sort(rng.integers(0, nnz + 1, m - 1)), [nnz]]).astype(np.int32)
    run_csr2csc(osa, gpu_ctx, m, n, rowptr + base, columns("uniform", n, nnz, rng) + base,
                rng.uniform(-1, 1, nnz).astype(np.float32), np.float32, True, base)


@pytest.mark.parametrize("span,cols,nnz", [(400_000, 1 << 22, 2_000_000), (700_000, (1 << 26) - 2, 5_300_000),
                                           (500_000, 1 << 27, 9_000_000), (700_000, (1 << 31) - 2, 5_300_000),
                                           (147_000, 1 << 26, 5_300_000)])  # (the bits of a column fit beside six of a row's)
def test_coosort_columns_of_many_bits(osa, gpu_ctx, span, cols, nnz):
    rng = np.random.default_rng(span + nnz)
    rows, c = rng.integers(0, span, nnz).astype(np.int32), rng.integers(0, cols, nnz).astype(np.int32)
    c[:2] = [0, cols - 1]
    run_coosort(osa, gpu_ctx, span, cols, rows, c, True, perm=rng.permutation(nnz).astype(np.int32))


VALUES = [("FP32", True), ("FP16", True), ("INT8", True), ("FP32", False)]


@pytest.mark.parametrize("val_type,numeric", VALUES)
def test_csr2csc_two_packed_passes_of_the_smallest_workgroups(osa, gpu_ctx, val_type, numeric):
    """21 column bits, ten of them in LDS, under 2^20 entries."""
    n, nnz = (1 << 20) + 3, 700_001
    rng = np.random.default_rng(5)
    rowptr = np.array([0, nnz // 3, nnz // 3, nnz], np.int32)
    val = _typed(rng.uniform(-1, 1, nnz).astype(np.float32), val_type)
    run_csr2csc(osa, gpu_ctx, 3, n, rowptr + 1, columns("uniform", n, nnz, rng) + 1, val, NP_TYPE[val_type], numeric, 1)


@pytest.mark.parametrize("val_type,numeric", VALUES)
def test_csr2csc_plain_passes_of_the_largest_workgroups(osa, gpu_ctx, val_type, numeric):
    """25 column bits, buckets of 429 entries on average: three passes over keys, rows and values, the last one writes the outputs."""
    n, nnz = 20_000_003, (1 << 23) + 5
    rng = np.random.default_rng(4)
    rowptr = np.array([0, nnz // 3, nnz], np.int32)
    val = _typed(rng.uniform(-1, 1, nnz).astype(np.float32), val_type)
    run_csr2csc(osa, gpu_ctx, 2, n, rowptr, columns("uniform", n, nnz, rng), val, NP_TYPE[val_type], numeric, 0)


def test_csr2csc_fullest_packed_passes(osa, gpu_ctx):
    """Whole tiles and two digits of eight bits: the tables of both passes fill their room to the last number."""
    m, n, nnz = 3_000_000, (1 << 25) + 3, 3 << 23
    rng = np.random.default_rng(9)
    rowptr = np.concatenate([[0], np.sort(rng.integers(0, nnz + 1, m - 1)), [nnz]]).astype(np.int32)
    c = columns("uniform", n, nnz, rng)
    c[:2] = [n - 1, 0]
    run_csr2csc(osa, gpu_ctx, m, n, rowptr, c, rng.uniform(-1, 1, nnz).astype(np.float32), np.float32, True, 0)


@pytest.mark.parametrize("val_type,numeric", VALUES)
def test_csr2csc_of_few_entries_a_column_and_many_rows(osa, gpu_ctx, val_type, numeric):
    """24 row bits leave eight in a record, whose buckets would hold 128 entries: the rows' top bits travel beside it."""
    m, n, nnz = (1 << 23) + 7, (1 << 24) - 3, (1 << 23) + 5
    rng = np.random.default_rng(6)
    rowptr = np.concatenate([[0], np.sort(rng.integers(0, nnz + 1, m - 1)), [nnz]]).astype(np.int32)
    val = _typed(rng.uniform(-1, 1, nnz).astype(np.float32), val_type)
    run_csr2csc(osa, gpu_ctx, m, n, rowptr, columns("uniform", n, nnz, rng), val, NP_TYPE[val_type], numeric, 0)


MANY = (1 << 23) + 9  # rows: 24 bits, of which 22 stand beside ten low bits of a key


@pytest.mark.parametrize("val_type,numeric", VALUES)
@pytest.mark.parametrize("n,nnz", [(400_003, 800_001), ((1 << 20) + 3, 700_001), (500_001, 1_200_003), ((1 << 21) + 3, 2_000_001),
                                   ((1 << 25) + 3, 5 * (1 << 23) + 8195)])
def test_csr2csc_top_bits_of_rows_beside_the_records(osa, gpu_ctx, n, nnz, val_type, numeric):
    """One pass and two of every size of workgroup; the last one's two passes take eight bits each."""
    rng = np.random.default_rng(nnz)
    rowptr = np.concatenate([[0], np.sort(rng.integers(0, nnz + 1, MANY - 1)), [nnz]]).astype(np.int32)
    val = _typed(rng.uniform(-1, 1, nnz).astype(np.float32), val_type)
    run_csr2csc(osa, gpu_ctx, MANY, n, rowptr + 1, columns("uniform", n, nnz, rng) + 1, val, NP_TYPE[val_type], numeric, 1)


@pytest.mark.parametrize("what", ["hubs", "few", "ends"])
def test_csr2csc_top_bits_in_buckets_that_do_not_fit(osa, gpu_ctx, what):
    n, nnz = (1 << 20) - 77, 3_000_001
    rng = np.random.default_rng(8)
    rowptr = np.concatenate([[0], np.sort(rng.integers(0, nnz + 1, MANY - 1)), [nnz]]).astype(np.int32)
    run_csr2csc(osa, gpu_ctx, MANY, n, rowptr, columns(what, n, nnz, rng), rng.uniform(-1, 1, nnz).astype(np.float32),
                np.float32, True, 0)


@pytest.mark.parametrize("span,cols,nnz", [(700_001, 1 << 25, 2_500_000), (300_001, 1 << 25, 2_000_000),
                                           (200_001, (1 << 26) - 2, 2_000_000), (100_001, (1 << 26) - 2, 1_850_000),
                                           (2_000_000, (1 << 31) - 2, 5_300_000)])
@pytest.mark.parametrize("hub", [0, 40_000])
def test_coosort_top_bits_of_columns_beside_the_records(osa, gpu_ctx, span, cols, nnz, hub):
    """Rows of every number of lanes, sorted where their bucket is, and rows whose columns do not fit their 32-bit keys; with
    `hub`, a row that no workgroup orders and rows of 64, 65 and 66 entries."""
    rng = np.random.default_rng(span)
    rows, c = rng.integers(0, span, nnz).astype(np.int32), rng.integers(0, cols, nnz).astype(np.int32)
    c[:2] = [0, cols - 1]
    if hub:
        at = rng.permutation(nnz)
        for row, count in enumerate((hub, 64, 65, 66)):
            rows[at[:count]] = 500 + row
            at = at[count:]
    run_coosort(osa, gpu_ctx, span, cols, rows, c, True, perm=rng.permutation(nnz).astype(np.int32))
