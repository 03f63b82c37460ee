// aclsparseSpMMGetBufferSize / aclsparseSpMMPreprocess / aclsparseSpMM.
//
// Validation order and status codes follow the reference's arch35 host code
// (sparse/spmm/arch35/spmm_host.cpp:152-191 for the shared checks, :213-234,
// :335-362, :364-394 for the three entry points).  Not carried over: the
// synchronous device<->host round trip of the tiling struct on every SpMM call
// (:281-308); alpha / beta travel as kernel arguments instead.
#include <climits>

#include <cstdint>
#include <cstdlib>

#include "internal.h"
#include "offset_rows.h"

namespace {

struct SpmmTypes {
    int32_t valType;
    int32_t cType;
};

// (A, B, C, compute) combinations with a kernel.  The first three rows are the
// reference's table (spmm_host.cpp:103-120); the fourth is the fp16-in /
// fp32-out case.
bool ResolveTypes(const aclsparseSpMatDescr *A, const aclsparseDnMatDescr *B, const aclsparseDnMatDescr *C,
                  aclDataType computeType, SpmmTypes *t)
{
    const aclDataType a = A->valueType, b = B->valueType, c = C->valueType;
    if (a == ACL_FLOAT && b == ACL_FLOAT && c == ACL_FLOAT && computeType == ACL_FLOAT) {
        *t = {OPSPARSE_F32, OPSPARSE_F32};
        return true;
    }
    if (a == ACL_FLOAT16 && b == ACL_FLOAT16 && c == ACL_FLOAT16 && computeType == ACL_FLOAT) {
        *t = {OPSPARSE_F16, OPSPARSE_F16};
        return true;
    }
    if (a == ACL_INT8 && b == ACL_INT8 && c == ACL_INT32 && computeType == ACL_INT32) {
        *t = {OPSPARSE_I8, OPSPARSE_I32};
        return true;
    }
    if (a == ACL_FLOAT16 && b == ACL_FLOAT16 && c == ACL_FLOAT && computeType == ACL_FLOAT) {
        *t = {OPSPARSE_F16, OPSPARSE_F32};
        return true;
    }
    return false;
}

aclsparseStatus_t Validate(const aclsparseSpMatDescr *A, const aclsparseDnMatDescr *B, const aclsparseDnMatDescr *C,
                           aclsparseOperation_t opA, aclsparseOperation_t opB, aclDataType computeType,
                           aclsparseSpMMAlg_t alg, SpmmTypes *types)
{
    if (A == nullptr || B == nullptr || C == nullptr) {
        return ACL_SPARSE_STATUS_HANDLE_IS_NULLPTR;
    }
    if (opA != ACL_SPARSE_OP_NON_TRANSPOSE) {
        return ACL_SPARSE_STATUS_NOT_SUPPORTED;
    }
    if (opB != ACL_SPARSE_OP_NON_TRANSPOSE && opB != ACL_SPARSE_OP_TRANSPOSE) {
        return ACL_SPARSE_STATUS_NOT_SUPPORTED;
    }
    if (A->format != ACL_SPARSE_FORMAT_CSR) {
        return ACL_SPARSE_STATUS_MATRIX_TYPE_NOT_SUPPORTED;
    }
    if (A->rowOffsetsType != ACL_SPARSE_INDEX_32I || A->colIndType != ACL_SPARSE_INDEX_32I) {
        return ACL_SPARSE_STATUS_NOT_SUPPORTED;
    }
    if (A->idxBase != ACL_SPARSE_INDEX_BASE_ZERO) {
        return ACL_SPARSE_STATUS_NOT_SUPPORTED;
    }
    if (!ResolveTypes(A, B, C, computeType, types)) {
        return ACL_SPARSE_STATUS_NOT_SUPPORTED;
    }
    // The reference compares the descriptors' own rows / cols, not those of
    // op(B) (spmm_host.cpp:122-131); kept, so the same descriptors are accepted.
    if (A->cols != B->rows || A->rows != C->rows || B->cols != C->cols) {
        return ACL_SPARSE_STATUS_INVALID_VALUE;
    }
    if (alg != ACL_SPARSE_SPMM_ALG_DEFAULT && alg != ACL_SPARSE_SPMM_CSR_ALG1 &&
        alg != ACL_SPARSE_SPMM_CSR_FP32_HIGH_PRECISION_ALG) {
        return ACL_SPARSE_STATUS_NOT_SUPPORTED;
    }
    if (A->rows > INT32_MAX || C->cols > INT32_MAX) {
        return ACL_SPARSE_STATUS_NOT_SUPPORTED;
    }
    return ACL_SPARSE_STATUS_SUCCESS;
}

aclsparseStatus_t FromLaunch(int rc)
{
    switch (rc) {
        case OPSPARSE_OK: return ACL_SPARSE_STATUS_SUCCESS;
        case OPSPARSE_E_INVALID: return ACL_SPARSE_STATUS_INVALID_VALUE;
        case OPSPARSE_E_UNSUPPORTED: return ACL_SPARSE_STATUS_NOT_SUPPORTED;
        case OPSPARSE_E_WORKSPACE: return ACL_SPARSE_STATUS_INSUFFICIENT_RESOURCES;
        default: return ACL_SPARSE_STATUS_EXECUTION_FAILED;
    }
}

int64_t ElementBytes(int32_t type)
{
    return type == OPSPARSE_F32 || type == OPSPARSE_I32 ? 4 : (type == OPSPARSE_I8 ? 1 : 2);
}

// Column-major or transposed B, column-major C: the reference kernel reads them in place through its index
// formulas (spmm_kernel.cpp:155-168, :215-219), which here would mean one cache line per element (32/row, n = 64,
// column-major B: 37.8 ms against 1.2 ms row-major).  Instead the SpMM buffer carries, behind the plan's tables,
// room for compact row-major copies of such operands: B is copied in, the row-major kernels run, C is copied
// in (unless beta is known to be 0) and out.  n is padded to whole 16-byte vectors in the copies, so row-major
// operands of a width or leading dimension the vector kernels do not take go the same way (n = 62: 3.2 ms in
// place, n = 64: 1.2 ms).
struct Staging {
    bool b = false, c = false;
    int64_t nPadded = 0, bOff = 0, cOff = 0;
    int64_t bytes = 0;  // beyond the plan's own bytes, 0: the operands are used where they are
};

Staging MakeStaging(const aclsparseSpMatDescr *A, const aclsparseDnMatDescr *B, const aclsparseDnMatDescr *C,
                    aclsparseOperation_t opB, const SpmmTypes &t, int64_t planBytes)
{
    Staging g{};
    const bool bColMajor = (B->order == ACL_SPARSE_ORDER_COL) != (opB == ACL_SPARSE_OP_TRANSPOSE);
    const bool cColMajor = C->order == ACL_SPARSE_ORDER_COL;
    if (A->rows <= 0 || A->cols <= 0 || C->cols <= 0) {
        return g;
    }
    const int64_t vec = 16 / ElementBytes(t.valType);
    g.nPadded = (C->cols + vec - 1) / vec * vec;
    // a width that is not whole vectors needs both copies: the kernels then run on the padded width; a row-major
    // operand whose leading dimension is not whole vectors needs its own
    g.b = bColMajor || g.nPadded != C->cols || B->ld % vec != 0;
    g.c = cColMajor || g.nPadded != C->cols || C->ld % vec != 0;
    if (!g.b && !g.c) {
        return g;
    }
    auto align = [](int64_t v) { return (v + 255) / 256 * 256; };
    int64_t off = align(planBytes);
    g.bOff = off;
    off += g.b ? align(A->cols * g.nPadded * ElementBytes(t.valType)) : 0;
    g.cOff = off;
    off += g.c ? align(A->rows * g.nPadded * ElementBytes(t.cType)) : 0;
    g.bytes = off - planBytes;
    return g;
}

// The width the plan is made for: the padded one when the product runs on staged copies.
int64_t PlanWidth(const aclsparseSpMatDescr *A, const aclsparseDnMatDescr *B, const aclsparseDnMatDescr *C,
                  aclsparseOperation_t opB, const SpmmTypes &t)
{
    const Staging g = MakeStaging(A, B, C, opB, t, 0);
    return g.bytes > 0 ? g.nPadded : C->cols;
}

// One or two columns that lie in memory as vectors (column-major operands; a single column with a leading dimension
// of 1): the product is then n SpMV calls, which read the matrix n times and still beat the SpMM kernels, whose
// rows of B would be padded to 16 bytes in the staging area (5-point mesh of 4 M rows, n = 1: 37 us against 98 us;
// n = 2: 75 against 103; from n = 3 on the padded product wins, and for n = 2 already under rows of 27 entries:
// 244 us against 206, so two columns go this way up to 16 entries a row on average).  fp32, and fp16 with fp32 C:
// the fp16 C of SpMM is clamped to the finite range before rounding, which the SpMV kernels do not do.
bool ColumnsAreVectors(const aclsparseSpMatDescr *A, const aclsparseDnMatDescr *B, const aclsparseDnMatDescr *C,
                       aclsparseOperation_t opB, const SpmmTypes &t)
{
    const int64_t n = C->cols;
    if (n < 1 || n > 2 || opB != ACL_SPARSE_OP_NON_TRANSPOSE || A->rows <= 0 || A->cols <= 0 || A->nnz <= 0 ||
        A->nnz > INT32_MAX || t.cType != OPSPARSE_F32 || (t.valType != OPSPARSE_F32 && t.valType != OPSPARSE_F16)) {
        return false;
    }
    if (n == 2 && A->nnz > 16 * A->rows) {
        return false;
    }
    const bool bVectors = B->order == ACL_SPARSE_ORDER_COL ? B->ld >= A->cols : (n == 1 && B->ld == 1);
    const bool cVectors = C->order == ACL_SPARSE_ORDER_COL ? C->ld >= A->rows : (n == 1 && C->ld == 1);
    return bVectors && cVectors;
}

// Whether a matrix without long rows, under a B of n elements of elemBytes, is better served by the kernel that
// gives every row whole to one lane group straight from memory than by the slabs staged through LDS.  Measured on
// fp32 (us, slabs / rows; 1 - 2 M rows of meshes, bands, and uniformly random columns):
//   n = 16: 5-point mesh 224 / 104, 27-point 439 / 280, band of 50 245 / 153, 32 random columns a row 494 / 415
//   n = 32: 5-point 255 / 182, 27-point 558 / 263, band of 200 190 / 103, 8 random 191 / 181, 32 random 315 / 375
//   n = 64: 5-point 392 / 365, 7-point 521 / 425, 27-point 772 / 423, band of 50 340 / 193, 32 random 592 / 631
//   n = 128: 5-point 694 / 730, 7-point 905 / 888, 27-point 1135 / 748, band of 200 458 / 299, 32 random 1198 / 1215
// The slabs win where the gathers of B are what the product waits for (random columns, wide rows of B) and on
// the shortest rows under the widest B; rows of even length whose columns stay near the diagonal, and any narrow
// B, run faster row by row.  Uneven rows stay with the slabs, which share them out by work.
bool PrefersWholeRows(const aclsparseSpMatDescr *A, const OpsparseSpmmPlan &plan, int64_t n, int64_t elemBytes,
                      void *buffer, hipStream_t stream)
{
    if (std::getenv("OPS_SPARSE_SPMM_NO_ROWS_RULE") != nullptr || stream == nullptr || elemBytes < 2 ||
        plan.kernel == OPSPARSE_SPMM_BINNED || plan.numLongRows != 0 || plan.maxRowNnz <= 0 || A->rows <= 0 ||
        A->colInd == nullptr) {
        return false;
    }
    const int64_t rowBytes = n * elemBytes;
    const double mean = static_cast<double>(A->nnz) / static_cast<double>(A->rows);
    if ((rowBytes == 16 || rowBytes == 32) && plan.maxRowNnz <= 200) {
        return false;  // the kernel for a B of one or two 16-byte pieces a row takes these
    }
    // (fp32, n = 256, local columns: 27-point mesh of 614 K rows 2142 / 936, band of 12 675 / 492, of 20 485 / 388; but
    // 9-point 1229 / 1329)
    const int64_t widest = elemBytes == 4 && mean >= 12.0 ? 1024 : 512;
    if (rowBytes > widest || static_cast<double>(plan.maxRowNnz) > 4.0 * mean + 8.0) {
        return false;
    }
    if (elemBytes == 2) {
        // fp16 keeps the slabs, tuned on c5, except under local rows of 12 entries or more (us, slabs / rows, pipelined:
        // band of 12 n = 64 45 / 35, n = 128 71 / 63, n = 256 144 / 143; 27-point mesh n = 64 203 / 145, n = 256 612 /
        // 508; 32 random columns a row n = 32 292 / 412) and shorter ones where the table had the rows ahead.  Up to 128
        // bytes of B a row, from 6 entries: 7-point mesh of 1 M rows n = 32 110 / 84, n = 64 160 / 143, 9-point n = 64
        // 121 / 119.  Up to 256, from 10 entries (band of 10 n = 96 46 / 43) or with rows enough for several turns of
        // the pipeline (7-point, 1 M rows, n = 128 298 / 280; 9-point of 2.3 M rows n = 112 712 / 645, of 720 K rows
        // n = 96 196 / 209; band of 7, 300 K rows, n = 128 72 / 77).  Above 384, not 9-point meshes: 7-point n = 224
        // 565 / 516, band of 10 94 / 85, 9-point 1248 / 1299.  In between, from 12: 9-point n = 160 966 / 1154, band of
        // 10 74 / 78, 7-point 919 / 963.
        const bool ninePoint = mean >= 8.0 && mean < 10.0;
        const bool ahead = rowBytes <= 128 || (rowBytes <= 256 && (mean >= 10.0 || A->rows >= 786432)) ||
                           (rowBytes > 384 && !ninePoint);
        if (mean < 6.0 || (mean < 12.0 && !ahead)) {
            return false;
        }
    } else {
        if (rowBytes <= 64 || (rowBytes <= 128 && mean < 24.0)) {
            return true;
        }
        if (rowBytes > 256 && mean < 6.0) {
            return false;
        }
    }
    // what is left depends on whether the rows of B a row needs lie near each other: the sample of the SpMV plans
    // (the first 256 bytes of the buffer are the analyses' scratch: no launch reads them)
    int32_t scattered = 1000;
    if (opsparse_spmv_csr_gathers_scattered(static_cast<const int32_t *>(A->rowOffsets),
                                            static_cast<const int32_t *>(A->colInd), A->rows, A->cols, A->nnz, buffer,
                                            256, &scattered, stream) != OPSPARSE_OK) {
        return false;
    }
    return scattered < 250;
}

int64_t Align256(int64_t v)
{
    return (v + 255) / 256 * 256;
}

// Bytes at the start of the buffer for the lists of a matrix whose rows repeat, or for the SpMV plan that one or two columns
// run under.  By the sizes of A alone, not by the operands: a buffer sized for a wide B serves a narrower one, and nothing
// tells Preprocess which operands the buffer it is given was sized for.  (0: no such matrix by its sizes; the SpMV plan
// then lies behind everything else, in buffers sized for such columns.)
int64_t FrontBytes(const aclsparseSpMatDescr *A)
{
    return (A->valueType == ACL_FLOAT || A->valueType == ACL_FLOAT16) &&
                   opsparse_spmv_csr_offsets_workspace_bytes(A->rows, A->cols, A->nnz) > 0
               ? Align256(static_cast<int64_t>(opsparse_spmv_csr_workspace_bytes(A->rows, A->nnz)))
               : 0;
}

// Where the plan's tables, and the staging area behind them, begin.
void *Tables(const aclsparseSpMatDescr *A, void *buffer)
{
    return static_cast<unsigned char *>(buffer) + FrontBytes(A);
}

// Row statistics and long-row tables for width n into `buffer`; binds the buffer to A.
aclsparseStatus_t BuildPlan(const aclsparseSpMatDescr *A, int64_t n, int64_t elemBytes, void *buffer,
                            hipStream_t stream)
{
    // An empty matrix has nothing to preprocess (spmm_csr_mat.cpp:148-150).
    if (A->rows <= 0) {
        return ACL_SPARSE_STATUS_INVALID_VALUE;
    }
    if (A->rowOffsets == nullptr) {
        return ACL_SPARSE_STATUS_INVALID_VALUE;
    }
    OpsparseSpmmPlan plan{};
    // Nothing says how large the caller's buffer is: it was sized by GetBufferSize for this matrix and width, and the
    // analysis lays out exactly what GetBufferSize counted (one reduction over the row offsets, no allocation).
    const size_t bytes = static_cast<size_t>(INT64_MAX);
    void *const tables = Tables(A, buffer);
    const int rc = opsparse_spmm_csr_analyse(static_cast<const int32_t *>(A->rowOffsets), A->rows, A->nnz, n, tables,
                                             bytes, OPSPARSE_SPMM_AUTO, &plan, stream);
    if (rc != OPSPARSE_OK) {
        opsparse::LogError("aclsparseSpMM: analysis failed (%d)", rc);
        return FromLaunch(rc);
    }
    const int32_t maxRow = plan.maxRowNnz;
    const bool wholeRows = PrefersWholeRows(A, plan, n, elemBytes, tables, stream);
    if (wholeRows) {
        // a plan without tables: the launch layer then takes a lane group a row
        const int again = opsparse_spmm_csr_analyse(static_cast<const int32_t *>(A->rowOffsets), A->rows, A->nnz, n,
                                                    tables, bytes, OPSPARSE_SPMM_ROW_SPLIT, &plan, stream);
        if (again != OPSPARSE_OK) {
            return FromLaunch(again);
        }
    }
    if (A->spmm.buffer != buffer) {
        A->spmm.widestN = 0;
        A->spmm.offsetPatterns = 0;
    }
    A->spmm.widestN = A->spmm.widestN > n ? A->spmm.widestN : n;
    A->spmm.buffer = buffer;
    A->spmm.plan = plan;
    A->spmm.stagingBytes = 0;
    A->spmm.vectorOff = 0;
    A->spmm.vectorBytes = 0;
    A->spmm.maxRowNnz = maxRow;
    A->spmm.wholeRows = wholeRows;
    return ACL_SPARSE_STATUS_SUCCESS;
}

// Where the lists of a matrix whose rows repeat are ahead of the plan that was just made for a C of n columns.  us a launch,
// plan / lists:
//   - one 16-byte piece of B a row: n = 4 of 80 K rows 5-point mesh 4.2 / 4.5, 7-point 4.6 / 6.2, 9-point 5.6 / 5.6, 27-point 11.1 / 12.4,
//     of 160 K 5.4 / 5.2, 6.2 / 6.1, 9.1 / 6.5, 18.6 / 12.0; 3 distances of 320 K 5.9 / 6.3, of 2.5 M 28.1 / 29.8; fp16 n = 8 of 80 K
//     7-point 7.8 / 9.1, 9-point 9.9 / 7.6, of 160 K 10.9 / 8.7, 16.5 / 9.4;
//   - two: n = 8 of 80 K rows 4.5 / 5.0, 5.9 / 5.6, 7.0 / 6.2, 14.7 / 10.7, 5-point of 160 K 7.7 / 6.4; fp16 n = 16 5-point of 80 K 10.2 / 7.4;
//   - row-major fp32 rows that are not whole 16-byte pieces, which the plan copies: ahead at every size, n = 33 of 5000 rows 5-point
//     11.1 / 4.6, 27-point 15.8 / 9.2, of 290 K 120 / 33, 188 / 114;
//   - slabs staged through LDS: ahead at every size, 5-point n = 128 of 2000 rows 27 / 6, of 320 K 127 / 80; 7-point n = 256 75 / 7,
//     312 / 198; fp16 5-point n = 64 25 / 7, 69 / 48, 9-point n = 128 35 / 8, 137 / 108; only fp16 under lists with many empty
//     steps is behind (10 distances, which are 18 steps, n = 128 of 40 K rows 23 / 21, of 150 K 57 / 60, of 500 K 166 / 180);
//   - whole rows, fp16: behind nearly everywhere (7-point of 320 K rows n = 32 24 / 36, 27-point n = 64 102 / 141);
//   - whole rows, fp32, by the list and the width (a lane group has a power of two of lanes, so that n = 24 idles as many as 32 uses):
//     5-point mesh of 100 K rows n = 12 7.0 / 7.7, n = 24 9.9 / 10.7, n = 48 17.4 / 17.2, of 150 K 8.8 / 8.1, 13.7 / 14.2, 23.9 / 21.4, of
//     250 K 14.6 / 12.3, 20.3 / 18.5, 44 / 33, of 80 K n = 16 6.8 / 6.1, n = 64 15.0 / 13.8;
//     7-point of 150 K 10.4 / 10.4, 15.0 / 16.4, 25.7 / 27.3, of 250 K 16.5 / 14.7, 21.8 / 23.0, 45 / 39, of 400 K 24 / 22, 34 / 32, 73 / 50,
//     n = 16 of 320 K 20.1 / 21.1, of 640 K 37.5 / 32.9;
//     9-point of 70 K 7.5 / 8.0, 13.4 / 11.7, 17.4 / 22.4, of 100 K 10.8 / 9.2, 15.6 / 13.4, 23.0 / 23.3, n = 96 41 / 36, of 250 K 21 / 16,
//     32 / 26, 57 / 45, 111 / 76;
//     27-point of 70 K 18.5 / 14.2, 19.4 / 21.8, 31 / 44, 45 / 83, of 250 K 56 / 36, 59 / 57, 102 / 97, 166 / 173, of 400 K 91 / 56, 94 / 76,
//     161 / 125, 250 / 214; 19 distances, which are 27 steps, n = 16 of 40 K 7.0 / 9.0, of 80 K 14.7 / 14.0, n = 32 of 320 K 61 / 66, of
//     640 K 125 / 107, n = 64 of 160 K 59 / 64, of 320 K 116 / 100; 15, 18 steps, n = 16 of 320 K 37 / 36, of 640 K 76 / 57; 10, 18 steps,
//     n = 16 of 640 K 49 / 51, of 1.25 M 102 / 84;
//   - beyond 64 columns only where there is a kernel for two rows a lane (of 320 K rows, n = 128, 27-point 224 / 188, but 19-point
//     190 / 210, 15 distances n = 256 351 / 553).
// `copied`: the plan copies rows that the kernel for lists takes where they are.  `mayHaveRuns`: two rows a lane.
bool ListsAhead(const aclsparseSpMatDescr *A, int64_t n, int64_t elemBytes, int32_t distances, bool copied, bool mayHaveRuns)
{
    const int64_t pieces = (n * elemBytes + 15) / 16;
    const int64_t chunk = distances <= 5 ? 5 : distances <= 7 ? 7 : 9, steps = (distances + chunk - 1) / chunk * chunk;
    const bool emptySteps = 2 * steps * A->rows > 3 * A->nnz;
    if (opsparse::OffsetsAtAnySize()) {
        return true;
    }
    const int64_t k16 = int64_t{1} << 14;
    if (pieces == 1) {
        return distances >= 4 && A->rows >= (distances < 8 ? 9 * k16 : 6 * k16);
    }
    if (pieces == 2) {
        return distances >= 3 && A->rows >= (distances <= 5 && elemBytes == 4 ? 8 * k16 : 4 * k16);
    }
    if (copied) {
        return true;
    }
    if (!A->spmm.wholeRows) {
        return elemBytes == 4 || !emptySteps || A->rows < int64_t{1} << 17;
    }
    if (elemBytes == 2) {
        return false;
    }
    int64_t least;
    if (distances <= 5) {
        least = emptySteps ? (pieces <= 4 ? 32 : 8) : pieces == 3 ? 8 : pieces == 4 ? 5 : pieces <= 8 ? 10 : 6;
    } else if (distances <= 7) {
        least = pieces == 3 ? 10 : pieces == 4 ? 32 : pieces <= 8 ? 24 : pieces <= 16 ? 12 : 9;
    } else if (distances <= 9) {
        least = pieces <= 8 ? 5 : 6;
    } else if (pieces <= 4) {
        least = emptySteps ? 64 : distances >= 18 ? 4 : 32;
    } else {
        least = pieces <= 8 ? (steps == distances ? 16 : 24) : pieces <= 32 ? 16 : 8;
    }
    return A->rows >= least * k16 && (pieces <= 16 || mayHaveRuns);
}

bool ScalarIsZero(const void *host, aclDataType computeType)
{
    return computeType == ACL_INT32 ? *static_cast<const int32_t *>(host) == 0
                                    : *static_cast<const float *>(host) == 0.0f;
}

// The product of a matrix whose rows repeat, row-major operands; false: not with these operands.
bool OffsetsTake(const aclsparseSpMatDescr *A, int64_t n, int64_t ldb, int64_t ldc, const void *B, const void *C,
                 const SpmmTypes &t)
{
    return A->spmm.offsetPatterns > 0 && A->nnz > 0 && opsparse::OffsetSpmmTakes(n, ldb, ldc, B, C, t.valType, t.cType);
}
int RunOffsets(const aclsparseSpMatDescr *A, int64_t n, int64_t ldb, int64_t ldc, const void *B, void *C,
               OpsparseScalar alpha, OpsparseScalar beta, const SpmmTypes &t, const void *buffer, hipStream_t stream)
{
    const opsparse::OffsetSpmmArgs a{static_cast<const int32_t *>(A->rowOffsets), A->values, B, C, A->rows, A->cols, n,
                                     A->nnz, ldb, ldc, alpha, beta,
                                     static_cast<const unsigned char *>(buffer), A->spmm.offsetPatterns, A->spmm.offsetDistances, A->spmm.offsetReach, A->spmm.offsetRuns, stream};
    return opsparse::LaunchOffsetSpmm(a, t.valType, t.cType);
}

// The product through the staging area: B copied to compact row-major (padded width), the row-major kernels,
// C copied in (unless beta is 0 for certain) and out.  Kernels only, all on `stream`.
int RunStaged(const Staging &g, const aclsparseSpMatDescr *A, const aclsparseDnMatDescr *B,
              const aclsparseDnMatDescr *C, aclsparseOperation_t opB, OpsparseScalar alpha, OpsparseScalar beta,
              const SpmmTypes &t, bool betaIsZero, void *buffer, hipStream_t stream)
{
    auto *base = static_cast<unsigned char *>(Tables(A, buffer));
    const int64_t k = A->cols, m = A->rows, n = C->cols;
    const bool bColMajor = (B->order == ACL_SPARSE_ORDER_COL) != (opB == ACL_SPARSE_OP_TRANSPOSE);
    const bool cColMajor = C->order == ACL_SPARSE_ORDER_COL;
    const void *bUse = B->values;
    void *cUse = C->values;
    int64_t ldb = B->ld, ldc = C->ld;
    int rc = OPSPARSE_OK;
    if (g.b) {
        rc = opsparse_dense_restage(B->values, base + g.bOff, k, n, g.nPadded, B->ld, bColMajor ? 1 : 0, g.nPadded, 0,
                                    static_cast<int32_t>(ElementBytes(t.valType)), stream);
        bUse = base + g.bOff;
        ldb = g.nPadded;
    }
    if (rc == OPSPARSE_OK && g.c) {
        cUse = base + g.cOff;
        ldc = g.nPadded;
        if (!betaIsZero) {
            rc = opsparse_dense_restage(C->values, cUse, m, n, g.nPadded, C->ld, cColMajor ? 1 : 0, g.nPadded, 0,
                                        static_cast<int32_t>(ElementBytes(t.cType)), stream);
        }
    }
    if (rc != OPSPARSE_OK) {
        return rc;
    }
    // both copies exist whenever the width was padded, so the kernels may take the padded width as theirs
    const int64_t nRun = A->spmm.plan.n;  // the padded width, which the plan was made for
    if ((g.c || !cColMajor) && OffsetsTake(A, nRun, ldb, ldc, bUse, cUse, t)) {
        rc = RunOffsets(A, nRun, ldb, ldc, bUse, cUse, alpha, beta, t, buffer, stream);
    } else {
        rc = opsparse_spmm_csr_launch(&A->spmm.plan, static_cast<const int32_t *>(A->rowOffsets),
                                      static_cast<const int32_t *>(A->colInd), A->values, bUse, cUse, m, k, nRun, A->nnz,
                                      ldb, ldc, 0, g.c ? 0 : (cColMajor ? 1 : 0), 0, alpha, beta, t.valType, t.cType,
                                      base, static_cast<size_t>(A->spmm.plan.bytes), stream);
    }
    if (rc == OPSPARSE_OK && g.c) {
        rc = opsparse_dense_restage(cUse, C->values, m, n, n, g.nPadded, 0, C->ld, cColMajor ? 1 : 0,
                                    static_cast<int32_t>(ElementBytes(t.cType)), stream);
    }
    return rc;
}

}  // namespace

extern "C" {

aclsparseStatus_t aclsparseSpMMGetBufferSize(aclsparseHandle_t handle, aclsparseOperation_t opA,
                                             aclsparseOperation_t opB, const void * /*alpha*/,
                                             aclsparseConstSpMatDescr_t matA, aclsparseConstDnMatDescr_t matB,
                                             const void * /*beta*/, aclsparseDnMatDescr_t matC,
                                             aclDataType computeType, aclsparseSpMMAlg_t alg, size_t *size)
{
    if (size == nullptr) {
        return ACL_SPARSE_STATUS_INVALID_VALUE;
    }
    SpmmTypes t{};
    const aclsparseStatus_t st = Validate(matA, matB, matC, opA, opB, computeType, alg, &t);
    if (st != ACL_SPARSE_STATUS_SUCCESS) {
        return st;
    }
    // Matrices in which no row can be long need the 256-byte header only (no
    // device access); otherwise the long rows are counted on the device.
    if (matA->rows > 0 && matA->rowOffsets == nullptr) {
        return ACL_SPARSE_STATUS_INVALID_VALUE;
    }
    const int rc = opsparse_spmm_csr_workspace_bytes(static_cast<const int32_t *>(matA->rowOffsets), matA->rows,
                                                     matA->nnz, PlanWidth(matA, matB, matC, opB, t),
                                                     handle != nullptr ? handle->stream : nullptr, size);
    if (rc == OPSPARSE_OK) {
        *size += static_cast<size_t>(MakeStaging(matA, matB, matC, opB, t, static_cast<int64_t>(*size)).bytes);
        if (const int64_t front = FrontBytes(matA)) {
            *size += static_cast<size_t>(front);
        } else if (ColumnsAreVectors(matA, matB, matC, opB, t)) {
            // behind everything else: the workspace of the SpMV plan the columns run under
            *size = static_cast<size_t>(Align256(static_cast<int64_t>(*size))) +
                    opsparse_spmv_csr_workspace_bytes(matA->rows, matA->nnz);
        }
    }
    return FromLaunch(rc);
}

aclsparseStatus_t aclsparseSpMMPreprocess(aclsparseHandle_t handle, aclsparseOperation_t opA,
                                          aclsparseOperation_t opB, const void * /*alpha*/,
                                          aclsparseConstSpMatDescr_t matA, aclsparseConstDnMatDescr_t matB,
                                          const void * /*beta*/, aclsparseDnMatDescr_t matC, aclDataType computeType,
                                          aclsparseSpMMAlg_t alg, void *buffer)
{
    SpmmTypes t{};
    const aclsparseStatus_t st = Validate(matA, matB, matC, opA, opB, computeType, alg, &t);
    if (st != ACL_SPARSE_STATUS_SUCCESS) {
        return st;
    }
    if (buffer == nullptr) {
        return ACL_SPARSE_STATUS_INSUFFICIENT_RESOURCES;
    }
    // The reference ignores the handle here; its stream is used when there is one.
    hipStream_t stream = handle != nullptr ? handle->stream : nullptr;
    const aclsparseStatus_t built =
        BuildPlan(matA, PlanWidth(matA, matB, matC, opB, t), ElementBytes(t.valType), buffer, stream);
    if (built == ACL_SPARSE_STATUS_SUCCESS) {
        // the buffer was sized by GetBufferSize for these operands: their staging area exists
        matA->spmm.stagingBytes = MakeStaging(matA, matB, matC, opB, t, matA->spmm.plan.bytes).bytes;
        matA->spmm.offsetPatterns = 0;
        const int64_t front = FrontBytes(matA);
        const bool copied = matA->spmm.stagingBytes > 0 && t.valType == OPSPARSE_F32 && opB == ACL_SPARSE_OP_NON_TRANSPOSE &&
                            matB->order == ACL_SPARSE_ORDER_ROW && matC->order == ACL_SPARSE_ORDER_ROW;
        if (ColumnsAreVectors(matA, matB, matC, opB, t)) {
            // (GetBufferSize counted this region: at the start for every operand, or at the end for these)
            const int64_t off = front > 0 ? 0 : Align256(matA->spmm.plan.bytes + matA->spmm.stagingBytes);
            const size_t bytes = opsparse_spmv_csr_workspace_bytes(matA->rows, matA->nnz);
            OpsparseSpmvPlan vectorPlan{};
            const int rc = opsparse_spmv_csr_analyse(static_cast<const int32_t *>(matA->rowOffsets), matA->rows,
                                                     matA->cols, matA->nnz, static_cast<unsigned char *>(buffer) + off,
                                                     bytes, OPSPARSE_SPMV_AUTO, &vectorPlan, stream);
            if (rc == OPSPARSE_OK &&
                (stream == nullptr ||
                 opsparse::LookForOffsets(static_cast<const int32_t *>(matA->rowOffsets),
                                          static_cast<const int32_t *>(matA->colInd), matA->rows, matA->cols, matA->nnz,
                                          static_cast<unsigned char *>(buffer) + off, &vectorPlan,
                                          stream) == OPSPARSE_OK)) {
                matA->spmm.vectorPlan = vectorPlan;
                matA->spmm.vectorOff = off;
                matA->spmm.vectorBytes = static_cast<int64_t>(bytes);
            }
        } else if (front > 0 && matC->cols >= 1 && matC->cols <= opsparse::kOffsetMaxColumns && stream != nullptr &&
                   matA->colInd != nullptr && std::getenv("OPS_SPARSE_SPMM_NO_OFFSETS") == nullptr &&
                   ListsAhead(matA, matA->spmm.plan.n, ElementBytes(t.valType), matA->spmm.maxRowNnz, copied, true)) {
            opsparse::OffsetFound found;
            const int rc = opsparse::AnalyseOffsetRows(static_cast<const int32_t *>(matA->rowOffsets),
                                                       static_cast<const int32_t *>(matA->colInd), matA->rows, matA->cols,
                                                       matA->nnz, matA->spmm.maxRowNnz,
                                                       static_cast<unsigned char *>(buffer), &found, stream);
            if (rc != OPSPARSE_OK) {
                return FromLaunch(rc);
            }
            const int32_t runs = opsparse::OffsetRuns(found);
            if (found.patterns > 0 && ListsAhead(matA, matA->spmm.plan.n, ElementBytes(t.valType), found.distances, copied,
                                                 runs != opsparse::kOffsetRunsAny)) {
                matA->spmm.offsetPatterns = found.patterns;
                matA->spmm.offsetDistances = found.distances;
                matA->spmm.offsetRuns = runs;
                const int64_t back = -static_cast<int64_t>(found.distance[0]), on = found.distance[found.distances - 1];
                matA->spmm.offsetReach = back > on ? back : on;
            }
        }
    }
    return built;
}

aclsparseStatus_t aclsparseSpMM(aclsparseHandle_t handle, aclsparseOperation_t opA, aclsparseOperation_t opB,
                                const void *alpha, aclsparseConstSpMatDescr_t matA,
                                aclsparseConstDnMatDescr_t matB, const void *beta, aclsparseDnMatDescr_t matC,
                                aclDataType computeType, aclsparseSpMMAlg_t alg, void *buffer)
{
    SpmmTypes t{};
    aclsparseStatus_t st = Validate(matA, matB, matC, opA, opB, computeType, alg, &t);
    if (st != ACL_SPARSE_STATUS_SUCCESS) {
        return st;
    }
    if (buffer == nullptr) {
        return ACL_SPARSE_STATUS_INSUFFICIENT_RESOURCES;
    }
    if (handle == nullptr) {
        return ACL_SPARSE_STATUS_HANDLE_IS_NULLPTR;
    }
    // Staged copies of B / C only in a buffer that Preprocess was given for operands needing at least as much:
    // nothing else says how large the buffer is.  A buffer that is not the one bound to matA is preprocessed first
    // (spmm_host.cpp:310-321), without a staging area.
    const Staging g = MakeStaging(matA, matB, matC, opB, t, matA->spmm.plan.bytes);
    const bool bound = matA->spmm.buffer == buffer && matA->spmm.plan.rows == matA->rows &&
                       matA->spmm.plan.nnz == matA->nnz;
    bool staged = bound && g.bytes > 0 && g.bytes <= matA->spmm.stagingBytes && matA->spmm.plan.n == g.nPadded &&
                  matA->nnz > 0;
    const OpsparseSpmmPlan *plan = &matA->spmm.plan;
    void *const tables = Tables(matA, buffer);
    // A few row-major fp32 columns under a plan cut for the kernel for narrow B: that kernel reads and writes rows of
    // any width up to 8, leading dimension and 4-byte alignment where they are, and the copies through the staging
    // area are saved.
    const bool direct = staged && opB == ACL_SPARSE_OP_NON_TRANSPOSE && matB->order == ACL_SPARSE_ORDER_ROW &&
                        matC->order == ACL_SPARSE_ORDER_ROW &&
                        opsparse_spmm_csr_narrow_rows(plan, tables, matC->cols, matA->nnz, t.valType, t.cType) != 0;
    // Rows that repeat: the kernel for them takes row-major operands of any width where they are.
    const bool vectors = bound && matA->spmm.vectorBytes > 0 && matA->spmm.vectorPlan.rows == matA->rows &&
                         matA->spmm.vectorPlan.nnz == matA->nnz && ColumnsAreVectors(matA, matB, matC, opB, t);
    const bool offsets = bound && !vectors && opB == ACL_SPARSE_OP_NON_TRANSPOSE && matB->order == ACL_SPARSE_ORDER_ROW &&
                         matC->order == ACL_SPARSE_ORDER_ROW &&
                         OffsetsTake(matA, matC->cols, matB->ld, matC->ld, matB->values, matC->values, t);
    if (direct || offsets) {
        staged = false;
    }
    if (!direct && !offsets && !staged && (!bound || matA->spmm.plan.n != matC->cols)) {
        // The analysis reads two numbers back and synchronises, which a stream under capture must not: such a call
        // runs without a plan (a lane group per row, no tables), like the raw launch layer with plan == NULL.
        hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
        if (hipStreamIsCapturing(handle->stream, &capturing) != hipSuccess ||
            capturing != hipStreamCaptureStatusNone) {
            (void)hipGetLastError();
            plan = nullptr;
        } else if (bound && matC->cols > matA->spmm.widestN) {
            // The bound buffer was sized for a narrower C: the tables of a wider one (8 bytes per long-row segment
            // and column) need not fit it, and nothing says how large it is.  Without tables, then.
            plan = nullptr;
        } else {
            st = BuildPlan(matA, matC->cols, ElementBytes(t.valType), buffer, handle->stream);
            if (st != ACL_SPARSE_STATUS_SUCCESS) {
                return st;
            }
        }
    }
    // NULL scalars read as 0 (spmm_host.cpp:62-74).
    const OpsparseScalar a = opsparse::MakeScalar(alpha, computeType, handle->pointerMode, 0.0);
    const OpsparseScalar b = opsparse::MakeScalar(beta, computeType, handle->pointerMode, 0.0);
    int rc;
    const OpsparseSpmmBinding &bind = matA->spmm;
    if (offsets) {
        rc = RunOffsets(matA, matC->cols, matB->ld, matC->ld, matB->values, matC->values, a, b, t, buffer, handle->stream);
    } else if (vectors && bind.vectorBytes > 0) {
        const int64_t bStep = matB->order == ACL_SPARSE_ORDER_COL ? matB->ld : 0;
        const int64_t cStep = matC->order == ACL_SPARSE_ORDER_COL ? matC->ld : 0;
        rc = OPSPARSE_OK;
        for (int64_t j = 0; j < matC->cols && rc == OPSPARSE_OK; ++j) {
            const auto *x = static_cast<const unsigned char *>(matB->values) + j * bStep * ElementBytes(t.valType);
            auto *y = static_cast<unsigned char *>(matC->values) + j * cStep * ElementBytes(t.cType);
            rc = opsparse_spmv_csr_launch_zy(&bind.vectorPlan, 0, static_cast<const int32_t *>(matA->rowOffsets),
                                             static_cast<const int32_t *>(matA->colInd), matA->values, x, y, y,
                                             matA->rows, matA->cols, matA->nnz, a, b, t.valType, t.cType, 0,
                                             static_cast<unsigned char *>(buffer) + bind.vectorOff,
                                             static_cast<size_t>(bind.vectorBytes), handle->stream);
        }
    } else if (staged) {
        rc = RunStaged(g, matA, matB, matC, opB, a, b, t, handle->pointerMode == ACL_SPARSE_POINTER_MODE_HOST &&
                                                              beta != nullptr && ScalarIsZero(beta, computeType),
                       buffer, handle->stream);
    } else {
        rc = opsparse_spmm_csr_launch(
            plan, static_cast<const int32_t *>(matA->rowOffsets),
            static_cast<const int32_t *>(matA->colInd), matA->values, matB->values, matC->values, matA->rows,
            matA->cols, matC->cols, matA->nnz, matB->ld, matC->ld, matB->order == ACL_SPARSE_ORDER_COL ? 1 : 0,
            matC->order == ACL_SPARSE_ORDER_COL ? 1 : 0, opB == ACL_SPARSE_OP_TRANSPOSE ? 1 : 0, a, b, t.valType,
            t.cType, tables, plan != nullptr ? static_cast<size_t>(plan->bytes) : 0, handle->stream);
    }
    if (rc != OPSPARSE_OK) {
        opsparse::LogError("aclsparseSpMM: launch failed (%d)", rc);
    }
    return FromLaunch(rc);
}

}  // extern "C"
