// CSR producers for gfx950: COO rows -> CSR row offsets, CSR row offsets -> COO
// rows, per-row stable sort of CSR column indices with a permutation, and CSR ->
// CSC.  All of it is integer / byte work whose results must be bit-exact, and
// all of it is bound by memory traffic, so the kernels stream their operands
// with coalesced accesses and keep the shuffling in LDS.
//
// They replace the device side of
//   aclsparseXcoo2csr     sparse/coo2csr/arch35/coo2csr_kernel.cpp   (count + prefix sum)
//   aclsparseXcsr2coo     sparse/csr2coo/arch35/csr2coo_kernel.cpp   (row expansion)
//   aclsparseXcsrsort     sparse/csrsort/arch35/csrsort_kernel.cpp   (runs + serial merge)
//   aclsparseCsr2cscEx2   sparse/csr2csc_ex2/arch35/csr2csc_ex2_kernel.cpp (striped counting sort)
// and produce what the reference's CPU goldens produce
// (test/coo2csr/coo2csr_golden.h:44-77, test/csr2coo/csr2coo_golden.h:37-61,
// test/csrsort/arch35/csrsort_golden.h:38-70, test/csr2csc_ex2/csr2csc_ex2_golden.h:50-110).
//
// Building blocks:
//   * an inclusive scan of int32 (tile sums, then a tile rescan; many tiles: a
//     one-workgroup scan of the sums in between), in place if wanted;
//   * least-significant-digit radix sorts of (key, payload) pairs: one of up to ten
//     bits a pass, whose tiles are ordered in LDS and leave as runs of whole lines
//     (csr2csc, coosort; the last bits bucket by bucket in LDS), and one of four bits a pass (the SpMV layouts, csrsort of
//     very long rows).  In the latter a thread owns consecutive items of its tile,
//     counts them per digit, the workgroup scans the 16 x 256 counters digit-major,
//     and every item goes to digit base + number of earlier items with its digit:
//     stable by construction;
//   * bitonic sorts of 64-bit (column, position) keys in registers (a wavefront per
//     row of up to 64 entries) and in LDS (a workgroup per row of up to 2048); the
//     position in the low half makes every key distinct, so any correct sort is
//     the stable sort.
#include <climits>
#include <type_traits>
#include <cstdlib>

#include "convert_internal.h"
#include "device_utils.h"

namespace opsparse {

constexpr int kScanItems = 8;                             // consecutive elements a thread scans
constexpr int kScanTile = kBlockThreads * kScanItems;     // elements per workgroup
constexpr int kRadixBits = 4;
constexpr int kRadixDigits = 1 << kRadixBits;
constexpr int kRadixItems = 4;                            // consecutive items a thread ranks
constexpr int kRadixTile = kBlockThreads * kRadixItems;
constexpr int kSortWaveRow = 64;                          // rows up to this length: one wavefront, registers
constexpr int kSortLdsRow = 2048;                         // rows up to this length: one workgroup, LDS
constexpr int kSortListBlocks = 2048;                     // workgroups walking the list of longer rows
constexpr int kSortWideRow = 16384;                       // listed rows longer than this get 1024 lanes instead of 256

// ------------------------------------------------------------------- fill

__global__ __launch_bounds__(kBlockThreads) void FillI32Kernel(int32_t *__restrict__ p, int64_t n, int32_t v)
{
    const int64_t stride = static_cast<int64_t>(gridDim.x) * kBlockThreads;
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * kBlockThreads + threadIdx.x; i < n; i += stride) {
        p[i] = v;
    }
}

// ------------------------------------------------------------------- scan

// Exclusive scan of one value per thread over the workgroup; *total gets the sum.  Its barriers order LDS only.
__device__ __forceinline__ int32_t BlockExclusiveScan(int32_t v, int32_t *waveSums /* [4] in LDS */, int32_t *total)
{
    const int32_t lane = threadIdx.x % kWave;
    const int32_t wave = threadIdx.x / kWave;
    int32_t incl = v;
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
        const int32_t up = __shfl_up(incl, off, kWave);
        if (lane >= off) {
            incl += up;
        }
    }
    if (lane == kWave - 1) {
        waveSums[wave] = incl;
    }
    LdsBarrier();
    int32_t base = 0, all = 0;
#pragma unroll
    for (int w = 0; w < kBlockThreads / kWave; ++w) {
        const int32_t s = waveSums[w];
        base += (w < wave) ? s : 0;
        all += s;
    }
    LdsBarrier();  // waveSums may be reused by the caller's next call
    *total = all;
    return base + incl - v;
}

__global__ __launch_bounds__(kBlockThreads) void ScanTileSumsKernel(const int32_t *__restrict__ in, int64_t n,
                                                                   int32_t *__restrict__ tileSums)
{
    __shared__ int32_t waveSums[kBlockThreads / kWave];
    const int64_t base = static_cast<int64_t>(blockIdx.x) * kScanTile;
    int32_t sum = 0;
#pragma unroll
    for (int i = 0; i < kScanItems; ++i) {
        const int64_t p = base + i * kBlockThreads + threadIdx.x;
        sum += p < n ? in[p] : 0;
    }
    int32_t total;
    (void)BlockExclusiveScan(sum, waveSums, &total);
    if (threadIdx.x == 0) {
        tileSums[blockIdx.x] = total;
    }
}

// One workgroup: tileSums[i] <- sum of tileSums[0..i).
__global__ __launch_bounds__(kBlockThreads) void ScanTileOffsetsKernel(int32_t *__restrict__ tileSums, int64_t numTiles)
{
    __shared__ int32_t waveSums[kBlockThreads / kWave];
    int32_t carry = 0;
    for (int64_t c0 = 0; c0 < numTiles; c0 += kBlockThreads) {
        const int64_t p = c0 + threadIdx.x;
        const int32_t v = p < numTiles ? tileSums[p] : 0;
        int32_t total;
        const int32_t excl = BlockExclusiveScan(v, waveSums, &total);
        if (p < numTiles) {
            tileSums[p] = carry + excl;
        }
        carry += total;
    }
}

// out[i] = add + in[0] + ... + in[i]; out may be in.  tiles: offsets of the tiles, or (Sums) their sums, of which a workgroup
// then adds up those before its own: up to kScanSumsMost tiles that is eight loads a thread at most and takes less than the
// launch of the kernel above between the other two (csr2csc, three scans: 6 M entries over 300 K columns 197 -> 191 us, 5 M over
// 500 K 189 -> 184).
constexpr int64_t kScanSumsMost = 8 * kBlockThreads;

template <bool Sums>
__global__ __launch_bounds__(kBlockThreads) void ScanApplyKernel(const int32_t *in, int32_t *out, int64_t n,
                                                                const int32_t *__restrict__ tiles, int32_t add)
{
    __shared__ int32_t waveSums[kBlockThreads / kWave];
    int32_t offset = 0;
    if (Sums) {
        int32_t part = 0;
#pragma unroll
        for (int i = 0; i < kScanSumsMost / kBlockThreads; ++i) {
            const uint32_t t = i * kBlockThreads + threadIdx.x;
            part += t < blockIdx.x ? tiles[t] : 0;
        }
        (void)BlockExclusiveScan(part, waveSums, &offset);
    } else {
        offset = tiles[blockIdx.x];
    }
    const int64_t first = static_cast<int64_t>(blockIdx.x) * kScanTile + static_cast<int64_t>(threadIdx.x) * kScanItems;
    int32_t v[kScanItems];
    int32_t sum = 0;
#pragma unroll
    for (int i = 0; i < kScanItems; ++i) {
        v[i] = first + i < n ? in[first + i] : 0;
        sum += v[i];
        v[i] = sum;  // inclusive within the thread
    }
    int32_t total;
    const int32_t before = BlockExclusiveScan(sum, waveSums, &total) + offset + add;
#pragma unroll
    for (int i = 0; i < kScanItems; ++i) {
        if (first + i < n) {
            out[first + i] = before + v[i];
        }
    }
}

// The same in one launch: one workgroup, a thread takes kScanOneItems consecutive elements of a chunk.  For arrays of up
// to kScanOneMost elements, where the three launches above are three times the 4 us between two dependent kernels.
constexpr int kScanOneThreads = 1024;
constexpr int kScanOneItems = 16;
constexpr int64_t kScanOneMost = int64_t{4} * kScanOneThreads * kScanOneItems;

__global__ __launch_bounds__(kScanOneThreads) void ScanOneKernel(const int32_t *in, int32_t *out, int64_t n, int32_t add)
{
    // A chunk passes through LDS: memory is read and written a line a wavefront, the threads take consecutive elements.
    // (one word of padding after every kScanOneItems: the threads' strides fall on all banks)
    __shared__ int32_t chunk[kScanOneThreads * (kScanOneItems + 1)];
    __shared__ int32_t waveSums[kScanOneThreads / kWave];
    const int32_t tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
    int32_t carry = add;
    for (int64_t c0 = 0; c0 < n; c0 += kScanOneThreads * kScanOneItems) {
        int32_t v[kScanOneItems];
#pragma unroll
        for (int i = 0; i < kScanOneItems; ++i) {
            const int64_t p = c0 + i * kScanOneThreads + tid;
            v[i] = in[p < n ? p : n - 1];
        }
#pragma unroll
        for (int i = 0; i < kScanOneItems; ++i) {
            const int32_t p = i * kScanOneThreads + tid;
            chunk[p + p / kScanOneItems] = c0 + p < n ? v[i] : 0;
        }
        __syncthreads();
        int32_t sum = 0;
#pragma unroll
        for (int i = 0; i < kScanOneItems; ++i) {
            sum += chunk[tid * (kScanOneItems + 1) + i];
            v[i] = sum;
        }
        int32_t incl = sum;
#pragma unroll
        for (int off = 1; off < kWave; off <<= 1) {
            const int32_t up = __shfl_up(incl, off, kWave);
            incl += lane >= off ? up : 0;
        }
        if (lane == kWave - 1) {
            waveSums[wave] = incl;
        }
        __syncthreads();
        int32_t base = carry + incl - sum;
#pragma unroll
        for (int w = 0; w < kScanOneThreads / kWave; ++w) {
            base += w < wave ? waveSums[w] : 0;
            carry += waveSums[w];
        }
#pragma unroll
        for (int i = 0; i < kScanOneItems; ++i) {
            chunk[tid * (kScanOneItems + 1) + i] = base + v[i];
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < kScanOneItems; ++i) {
            const int32_t p = i * kScanOneThreads + tid;
            if (c0 + p < n) {
                out[c0 + p] = chunk[p + p / kScanOneItems];
            }
        }
        __syncthreads();
    }
}

// ---------------------------------------------------------------- coo2csr

// counts[r + 1] += number of entries with row r (rows outside [0, m) are
// skipped, as the golden does).  A wavefront reads 64 consecutive entries at a
// time; the first lane of every run of equal rows adds the run's length with
// one atomic, so sorted input costs about one atomic per distinct row and
// unsorted input still counts correctly.
__global__ __launch_bounds__(kBlockThreads) void CountRunsKernel(const int32_t *__restrict__ ind, int64_t nnz,
                                                                int64_t m, int32_t base, int32_t *counts)
{
    constexpr int kRounds = 8;
    const int32_t lane = threadIdx.x % kWave;
    const int64_t wave = static_cast<int64_t>(blockIdx.x) * (kBlockThreads / kWave) + threadIdx.x / kWave;
    const int64_t first = wave * (kWave * kRounds);
    // all loads first, unconditionally (a position past the end re-reads the last entry and is not counted): behind
    // the branch around the atomic the compiler would wait for each load before issuing the next
    int32_t raw[kRounds];
#pragma unroll
    for (int r = 0; r < kRounds; ++r) {
        const int64_t p = first + r * kWave + lane;
        raw[r] = LoadStream(ind + (p < nnz ? p : nnz - 1));
    }
#pragma unroll
    for (int r = 0; r < kRounds; ++r) {
        const int64_t p = first + r * kWave + lane;
        const bool valid = p < nnz;
        // unsigned subtraction, like the reference kernel: no signed overflow on hostile input
        const int32_t row = valid ? static_cast<int32_t>(static_cast<uint32_t>(raw[r]) - static_cast<uint32_t>(base))
                                  : -1;
        const int32_t prev = __shfl_up(row, 1, kWave);
        const bool head = valid && (lane == 0 || prev != row);
        const uint64_t heads = __ballot(head);
        const uint64_t valids = __ballot(valid);
        if (head && row >= 0 && row < m) {
            // the run ends in front of the next head, or with the last valid lane
            const uint64_t later = lane == kWave - 1 ? 0 : (heads >> (lane + 1)) << (lane + 1);
            const int32_t end = later != 0 ? __ffsll(static_cast<long long>(later)) - 1 : __popcll(valids);
            atomicAdd(counts + row + 1, end - lane);
        }
    }
}

// ---------------------------------------------------------------- csr2coo

// A wavefront takes 64 consecutive rows.  Where their bounds chain (every row ends where the next begins, as in
// any well-formed CSR matrix) the 64 rows are one contiguous piece of the output: lane l writes positions
// first + l, first + l + 64, ..., a whole 256-byte line per store instruction, and finds the row of a position
// by walking the wavefront's 65 offsets, kept in LDS, forwards.  Otherwise (a row whose bounds do not describe
// a range inside [0, nnz) is skipped, csr2coo_golden.h:51-53, and rows may overlap or leave gaps) rows of up to
// 16 entries are written by their own lane and a longer row by the whole wavefront, 64 entries per store.
__global__ __launch_bounds__(kBlockThreads) void ExpandRowsKernel(const int32_t *__restrict__ rowPtr, int64_t m,
                                                                 int64_t nnz, int32_t base,
                                                                 int32_t *__restrict__ rowInd)
{
    __shared__ int32_t offs[kBlockThreads / kWave][kWave + 1];
    const int32_t lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
    const int64_t row = (static_cast<int64_t>(blockIdx.x) * kBlockThreads + threadIdx.x);
    int64_t lo = 0, hi = 0;
    bool bad = false;
    if (row < m) {
        lo = static_cast<int64_t>(rowPtr[row]) - base;
        hi = static_cast<int64_t>(rowPtr[row + 1]) - base;
        if (lo < 0 || hi > nnz || lo > hi) {
            lo = hi = 0;
            bad = true;
        }
    }
    const int32_t value = static_cast<int32_t>(row) + base;
    const int32_t live = __popcll(__ballot(row < m));  // rows of this wavefront: the first `live` lanes
    if (live == 0) {
        return;
    }
    const int64_t nextLo = __shfl_down(lo, 1, kWave);
    const bool chained = !bad && (lane + 1 >= live || hi == nextLo);
    if (__all(chained || lane >= live)) {
        int32_t *mine = offs[wave];
        if (lane < live) {
            mine[lane] = static_cast<int32_t>(lo);
        }
        if (lane == live - 1) {
            mine[live] = static_cast<int32_t>(hi);
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        const int32_t first = mine[0], last = mine[live];
        const int32_t row0 = static_cast<int32_t>(row) - lane + base;
        if (static_cast<int64_t>(last - first) >= 11 * static_cast<int64_t>(live)) {
            // rows of 11 entries and more on average: from one position of a lane to its next (64 further) at most
            // six row ends are passed, and walking past them is cheaper than searching
            int32_t cur = 0;
            for (int32_t p = first + lane; p < last; p += kWave) {
                while (mine[cur + 1] <= p) {  // ends at the latest at cur + 1 == live, whose offset is `last` > p
                    ++cur;
                }
                rowInd[p] = row0 + cur;
            }
        } else {
            for (int32_t p = first + lane; p < last; p += kWave) {
                int32_t a = 0, b = live - 1;  // the last row with mine[row] <= p (mine[0] <= p < mine[live]): 64 candidates
#pragma unroll
                for (int step = 0; step < 6; ++step) {
                    const int32_t mid = (a + b + 1) >> 1;
                    const bool right = mine[mid] <= p;
                    a = right ? mid : a;
                    b = right ? b : mid - 1;
                }
                rowInd[p] = row0 + a;
            }
        }
        return;
    }
    const int64_t len = hi - lo;
    if (len <= 16) {
        for (int64_t j = 0; j < len; ++j) {
            rowInd[lo + j] = value;
        }
    }
    uint64_t longRows = __ballot(len > 16);
    while (longRows != 0) {
        const int32_t src = __ffsll(static_cast<long long>(longRows)) - 1;
        longRows &= longRows - 1;
        const int64_t l = __shfl(lo, src, kWave);
        const int64_t h = __shfl(hi, src, kWave);
        const int32_t v = __shfl(value, src, kWave);
        for (int64_t p = l + lane; p < h; p += kWave) {
            rowInd[p] = v;
        }
    }
}

// ------------------------------------------------------------- radix sort

// Digit of a key for the pass at `shift`.
__device__ __forceinline__ int32_t RadixDigit(int32_t key, int32_t shift)
{
    return static_cast<int32_t>((static_cast<uint32_t>(key) >> shift) & (kRadixDigits - 1));
}

// table[1 + digit * numTiles + tile] = items of that digit in the tile
// (table[0] stays 0: an inclusive scan of the table then leaves, at the same
// place shifted down by one, the first output position of every (digit, tile)).
__global__ __launch_bounds__(kBlockThreads) void RadixCountKernel(const int32_t *__restrict__ keys, int64_t n,
                                                                 int32_t keyBase, int32_t shift,
                                                                 int32_t *__restrict__ table, int64_t numTiles)
{
    __shared__ int32_t hist[kRadixDigits];
    if (threadIdx.x < kRadixDigits) {
        hist[threadIdx.x] = 0;
    }
    __syncthreads();
    const int64_t first = static_cast<int64_t>(blockIdx.x) * kRadixTile + static_cast<int64_t>(threadIdx.x) * kRadixItems;
#pragma unroll
    for (int i = 0; i < kRadixItems; ++i) {
        if (first + i < n) {
            atomicAdd(&hist[RadixDigit(keys[first + i] - keyBase, shift)], 1);
        }
    }
    __syncthreads();
    if (threadIdx.x < kRadixDigits) {
        table[1 + static_cast<int64_t>(threadIdx.x) * numTiles + blockIdx.x] = hist[threadIdx.x];
    }
}

// LDS arrays that one phase reads with lane t at t * 16 + i and another with lane t at d * 256 + t: one unused
// word after every 32 keeps both patterns free of bank conflicts (unpadded, the first puts all lanes on two banks).
__device__ __forceinline__ int32_t Padded(int32_t i)
{
    return i + (i >> 5);
}
constexpr int kCounterSlots = kRadixDigits * kBlockThreads + kRadixDigits * kBlockThreads / 32;

// Exclusive scan, digit-major, of the 16 x 256 per-thread digit counters of a
// workgroup.  counters[d * 256 + t] holds thread t's count of digit d on entry
// and the number of items that sort before thread t's first item of digit d on
// exit.
__device__ __forceinline__ void ScanDigitCounters(int32_t *counters, int32_t *waveSums)
{
    constexpr int kPer = kRadixDigits;  // 4096 counters / 256 threads
    int32_t v[kPer];
    int32_t sum = 0;
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
        v[i] = counters[Padded(threadIdx.x * kPer + i)];
        sum += v[i];
    }
    int32_t total;
    int32_t run = BlockExclusiveScan(sum, waveSums, &total);
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
        counters[Padded(threadIdx.x * kPer + i)] = run;
        run += v[i];
    }
    LdsBarrier();
}

// What travels with the keys through a pass.  kPayIndex: one int32 per item (a source position; payloadIn ==
// NULL means "the payload of item i is i").  The pair modes carry csr2csc's (row, value) itself, 8 bytes, so that
// no gather by source position is left at the end: kPayPairFirst builds the pair from the row-of-position and
// value arrays (read in order), kPayPair moves it, kPayPairLast writes its two halves to the output arrays.
enum RadixPayload { kPayIndex = 0, kPayPairFirst = 1, kPayPair = 2, kPayPairLast = 3 };

struct RadixPairIo {
    const int32_t *rowSrc;  // kPayPairFirst: row (with the output's index base) of every source position
    const void *valSrc;     //                the values, valueBytes each (0: none)
    int32_t *rowOut;        // kPayPairLast: the sorted rows
    void *valOut;           //               the sorted values
    int32_t valueBytes;
};

struct RadixPair {
    int32_t row;
    uint32_t val;
};

// One pass: items of tile `blockIdx.x` go to prefix[digit][tile] + their rank
// among the tile's items of the same digit.  keyBase is subtracted from the keys
// read (first pass: the index base of the column indices) and the keys are
// written without it.
template <int Mode>
__global__ __launch_bounds__(kBlockThreads) void RadixScatterKernel(
    const int32_t *__restrict__ keysIn, const void *__restrict__ payloadIn, int32_t *__restrict__ keysOut,
    void *__restrict__ payloadOut, int64_t n, int32_t keyBase, int32_t shift, const int32_t *__restrict__ prefix,
    int64_t numTiles, RadixPairIo io)
{
    __shared__ int32_t counters[kCounterSlots];
    __shared__ int32_t waveSums[kBlockThreads / kWave];
    const int64_t first = static_cast<int64_t>(blockIdx.x) * kRadixTile + static_cast<int64_t>(threadIdx.x) * kRadixItems;
    int32_t key[kRadixItems], dig[kRadixItems];
    RadixPair pay[kRadixItems];  // kPayIndex uses .row only
    int32_t cnt[kRadixDigits];
#pragma unroll
    for (int d = 0; d < kRadixDigits; ++d) {
        cnt[d] = 0;
    }
#pragma unroll
    for (int i = 0; i < kRadixItems; ++i) {
        dig[i] = -1;
        pay[i] = RadixPair{0, 0u};
        if (first + i < n) {
            key[i] = keysIn[first + i] - keyBase;
            if (Mode == kPayIndex) {
                pay[i].row = payloadIn != nullptr ? static_cast<const int32_t *>(payloadIn)[first + i]
                                                  : static_cast<int32_t>(first + i);
            } else if (Mode == kPayPairFirst) {
                pay[i].row = io.rowSrc[first + i];
                if (io.valueBytes == 4) {
                    pay[i].val = static_cast<const uint32_t *>(io.valSrc)[first + i];
                } else if (io.valueBytes == 2) {
                    pay[i].val = static_cast<const uint16_t *>(io.valSrc)[first + i];
                } else if (io.valueBytes == 1) {
                    pay[i].val = static_cast<const uint8_t *>(io.valSrc)[first + i];
                }
            } else {
                pay[i] = static_cast<const RadixPair *>(payloadIn)[first + i];
            }
            dig[i] = RadixDigit(key[i], shift);
#pragma unroll
            for (int d = 0; d < kRadixDigits; ++d) {
                cnt[d] += (dig[i] == d) ? 1 : 0;
            }
        }
    }
#pragma unroll
    for (int d = 0; d < kRadixDigits; ++d) {
        counters[Padded(d * kBlockThreads + threadIdx.x)] = cnt[d];
    }
    __syncthreads();
    ScanDigitCounters(counters, waveSums);
#pragma unroll
    for (int i = 0; i < kRadixItems; ++i) {
        if (dig[i] >= 0) {
            // rank inside the tile among items of this digit: the thread's base for the digit, less the
            // digit's own start, plus the thread's earlier items of the digit
            int32_t earlier = 0;
#pragma unroll
            for (int j = 0; j < kRadixItems; ++j) {
                earlier += (j < i && dig[j] == dig[i]) ? 1 : 0;
            }
            const int32_t inTile = counters[Padded(dig[i] * kBlockThreads + threadIdx.x)] -
                                   counters[Padded(dig[i] * kBlockThreads)] + earlier;
            const int64_t dst = static_cast<int64_t>(prefix[static_cast<int64_t>(dig[i]) * numTiles + blockIdx.x]) + inTile;
            keysOut[dst] = key[i];
            if (Mode == kPayPairLast) {
                io.rowOut[dst] = pay[i].row;
                if (io.valueBytes == 4) {
                    static_cast<uint32_t *>(io.valOut)[dst] = pay[i].val;
                } else if (io.valueBytes == 2) {
                    static_cast<uint16_t *>(io.valOut)[dst] = static_cast<uint16_t>(pay[i].val);
                } else if (io.valueBytes == 1) {
                    static_cast<uint8_t *>(io.valOut)[dst] = static_cast<uint8_t>(pay[i].val);
                }
            } else if (Mode == kPayIndex) {
                static_cast<int32_t *>(payloadOut)[dst] = pay[i].row;
            } else {
                static_cast<RadixPair *>(payloadOut)[dst] = pay[i];
            }
        }
    }
}

// ----------------------------------------- radix sort, up to 10 bits a pass
// The passes of csr2csc and coosort over (key, row, value) triples.  A pass reads 12 bytes an entry and writes 12, so
// the number of passes is what counts, and with it the number of buckets a pass may have: with 1024 of them a tile's
// run in a bucket is eight entries.  Such runs reach memory as whole lines all the same, because the workgroups of an
// XCD work on neighbouring tiles at the same time: their runs of a bucket follow one another, and the lines between
// them are completed in the L2 that the workgroups share.
//
// Inside a workgroup: a wavefront takes 512 consecutive entries of the tile, 64 at a time, and finds every lane's peers
// (the lanes with its digit) from one ballot a digit bit; a counter a digit and wavefront in LDS carries the count from
// one 64 to the next.  The running sums of those counters over (digit, wavefront) are where a wavefront's entries of a
// digit start in the ordered tile; the entries are put there in LDS and leave in that order, neighbouring lanes writing
// neighbouring addresses.
//
// Measured on 33.5 M entries: 190 us a pass over 128 buckets, 4.5 TB/s (448 MB written for 402 of entries), 275 us over
// 1024; 285 us over 128 while tiles of 3840 were ordered by two 4-bit splits and every workgroup walked a range of its
// own.  What is left is the length of a turn: one workgroup of 1024 a compute unit, six barriers a tile.

constexpr int kWideItems = 8;      // entries of a thread
constexpr int kWideMaxBits = 10;   // ... of a digit

template <int T>
struct WideShape {
    static constexpr int kTile = T * kWideItems;
    static constexpr int kWaves = T / kWave;
    static constexpr int kPer = (1 << kWideMaxBits) > T ? (1 << kWideMaxBits) / T : 1;  // digits of a thread
};

// key - keyBase in wrap-around arithmetic (the keys of a COO sort may span the whole int32 range).
__device__ __forceinline__ int32_t Rebased(int32_t key, int32_t keyBase)
{
    return static_cast<int32_t>(static_cast<uint32_t>(key) - static_cast<uint32_t>(keyBase));
}

// A pass's digit: `mask` = 2^bits - 1 with bits <= kWideMaxBits (the passes of a sort share its key bits evenly).
__device__ __forceinline__ uint32_t WideDigit(int32_t key, int32_t shift, int32_t mask)
{
    return (static_cast<uint32_t>(key) >> shift) & static_cast<uint32_t>(mask);
}

// Exclusive scan of one value a thread over a workgroup of T threads; its barriers order LDS only.
template <int T>
__device__ __forceinline__ int32_t WideBlockScan(int32_t v, int32_t *waveSums)
{
    const int32_t lane = threadIdx.x % kWave;
    const int32_t wave = threadIdx.x / kWave;
    int32_t incl = v;
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
        const int32_t up = __shfl_up(incl, off, kWave);
        incl += lane >= off ? up : 0;
    }
    if (lane == kWave - 1) {
        waveSums[wave] = incl;
    }
    LdsBarrier();
    int32_t base = 0;
#pragma unroll
    for (int w = 0; w < T / kWave; ++w) {
        base += w < wave ? waveSums[w] : 0;
    }
    return base + incl - v;
}

// table[1 + digit * numTiles + tile] = entries of that digit in the tile (table[0] = 0: an inclusive scan of the table
// then leaves, at the same place shifted down by one, the first output position of every (digit, tile)).  A workgroup
// counts kWideCountTiles consecutive tiles and writes their counts of one digit side by side.
constexpr int kWideCountTiles = 4;

template <int T>
__global__ __launch_bounds__(T) void WideCountKernel(const int32_t *__restrict__ keys, int64_t n, int32_t keyBase,
                                                     int32_t shift, int32_t mask, int32_t *__restrict__ table,
                                                     int64_t numTiles)
{
    constexpr int kTile = WideShape<T>::kTile;
    __shared__ int32_t hist[kWideCountTiles << kWideMaxBits];
    const int32_t digits = mask + 1;
    for (int32_t i = threadIdx.x; i < kWideCountTiles * digits; i += T) {
        hist[i] = 0;
    }
    const int64_t firstTile = static_cast<int64_t>(XcdContiguousTile(blockIdx.x, gridDim.x)) * kWideCountTiles;
    // The keys of a tile are loaded, all of them, a tile ahead of their counting: the compiler keeps a load and the
    // LDS atomic after it in program order, and an atomic straight behind its load is a round trip to memory for
    // every entry.  No branch around a load: an entry past the end reads the last key and counts for nothing.
    int32_t key[2][kWideItems];
    auto fetch = [&](int j) {
#pragma unroll
        for (int i = 0; i < kWideItems; ++i) {
            const int64_t at = (firstTile + j) * kTile + i * T + threadIdx.x;
            key[j & 1][i] = keys[at < n ? at : n - 1];
        }
    };
    fetch(0);
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kWideCountTiles; ++j) {
        if (j + 1 < kWideCountTiles) {
            fetch(j + 1);
        }
#pragma unroll
        for (int i = 0; i < kWideItems; ++i) {
            const int64_t at = (firstTile + j) * kTile + i * T + threadIdx.x;
            atomicAdd(&hist[j * digits + WideDigit(Rebased(key[j & 1][i], keyBase), shift, mask)], at < n ? 1 : 0);
        }
    }
    __syncthreads();
    // the lanes of a group of kWideCountTiles write neighbouring tiles of one digit
    for (int32_t i = threadIdx.x; i < kWideCountTiles * digits; i += T) {
        const int64_t tile = firstTile + i % kWideCountTiles;
        if (tile < numTiles) {
            const int32_t d = i / kWideCountTiles;
            table[1 + static_cast<int64_t>(d) * numTiles + tile] = hist[i % kWideCountTiles * digits + d];
        }
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        table[0] = 0;
    }
}

// Between two passes the n (row, value) pairs lie as n rows followed by n values in the 8 n bytes of their buffer:
// 4-byte stores to a bucket's run, as for the keys.
template <typename P>
__device__ __forceinline__ auto WideRows(P *pairs)
{
    return reinterpret_cast<std::conditional_t<std::is_const<P>::value, const int32_t, int32_t> *>(pairs);
}
template <typename P>
__device__ __forceinline__ auto WideVals(P *pairs, int64_t n)
{
    return reinterpret_cast<std::conditional_t<std::is_const<P>::value, const uint32_t, uint32_t> *>(pairs) + n;
}

typedef uint32_t Uint2U __attribute__((ext_vector_type(2), aligned(4)));
typedef uint64_t Record __attribute__((aligned(4)));  // (a caller's buffer may begin at any 4-byte-aligned address)

// A tile's entries as the loads deliver them: lane l of wavefront w holds entries 512 w + l, 512 w + 64 + l, ...
template <int T>
struct WideTileRegs {
    int32_t key[kWideItems];
    RadixPair pay[kWideItems];
    int32_t first[WideShape<T>::kPer];  // first output position of the thread's digits
};

template <int T, int Mode, int VB, bool Full>
__device__ __forceinline__ void WideFetch(WideTileRegs<T> &r, int64_t tile, const int32_t *__restrict__ keysIn,
                                          const RadixPair *__restrict__ pairsIn, int64_t n, int32_t keyBase,
                                          int32_t shift, int32_t mask, const int32_t *__restrict__ prefix,
                                          int64_t numTiles, const RadixPairIo &io)
{
    constexpr int kPer = WideShape<T>::kPer;
    const int tid = threadIdx.x;
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
        const int32_t d = tid * kPer + j;
        r.first[j] = prefix[static_cast<int64_t>(d <= mask ? d : mask) * numTiles + tile];
    }
    const int64_t wave0 = tile * WideShape<T>::kTile + tid / kWave * (kWave * kWideItems) + tid % kWave;
#pragma unroll
    for (int i = 0; i < kWideItems; ++i) {
        const int64_t at = wave0 + i * kWave;
        // a slot past the end gets the largest digit, so that it sorts behind every real entry
        r.key[i] = static_cast<int32_t>(static_cast<uint32_t>(mask) << shift);
        r.pay[i] = RadixPair{0, 0u};
        if (Full || at < n) {
            r.key[i] = Rebased(LoadStream(keysIn + at), keyBase);
            if (Mode == kPayPairFirst) {
                r.pay[i].row = LoadStream(io.rowSrc + at);
                if (VB == 4) {
                    r.pay[i].val = LoadStream(static_cast<const uint32_t *>(io.valSrc) + at);
                } else if (VB == 2) {
                    r.pay[i].val = static_cast<const uint16_t *>(io.valSrc)[at];
                } else if (VB == 1) {
                    r.pay[i].val = static_cast<const uint8_t *>(io.valSrc)[at];
                }
            } else {
                r.pay[i] = RadixPair{LoadStream(WideRows(pairsIn) + at), LoadStream(WideVals(pairsIn, n) + at)};
            }
        }
    }
}

template <int T>
struct WideLds {
    union {
        int32_t counters[WideShape<T>::kWaves << kWideMaxBits];  // [wavefront][digit]
        struct {
            int32_t key[WideShape<T>::kTile];
            int32_t row[WideShape<T>::kTile];
            uint32_t val[WideShape<T>::kTile];
        };
    };
    int32_t outOf[1 << kWideMaxBits];  // output position less slot in the ordered tile, for the entries of a digit
    int32_t waveSums[WideShape<T>::kWaves];
};

// rank[i]: the place in the order of the tile's digits of the thread's entry i, whose digit is dig[i]; lds.outOf: where the
// entries of a digit go, less their places there.  Ends with a barrier, behind which lds.counters is free.
template <int T, typename Lds>
__device__ __forceinline__ void WideRank(Lds &lds, const uint32_t (&dig)[kWideItems],
                                         const int32_t (&first)[WideShape<T>::kPer], int32_t mask, int32_t bits,
                                         uint32_t (&rank)[kWideItems])
{
    constexpr int kPer = WideShape<T>::kPer, kWaves = WideShape<T>::kWaves;
    const int tid = threadIdx.x, lane = tid % kWave;
    const int32_t digits = mask + 1;
    int32_t *mine = lds.counters + tid / kWave * digits;
    for (int32_t d = lane; d < digits; d += kWave) {
        mine[d] = 0;
    }
    uint64_t peers[kWideItems];
#pragma unroll
    for (int i = 0; i < kWideItems; ++i) {
        peers[i] = ~uint64_t{0};
    }
    for (int32_t b = 0; b < bits; ++b) {
#pragma unroll
        for (int i = 0; i < kWideItems; ++i) {
            const uint32_t ones = static_cast<uint32_t>(__builtin_amdgcn_sbfe(dig[i], b, 1));  // the bit in every place
            const uint64_t m = __ballot(ones != 0);
            // peers & ~(m ^ ones)
            const uint32_t lo = __builtin_amdgcn_bitop3_b32(static_cast<uint32_t>(peers[i]), static_cast<uint32_t>(m), ones, 0x90);
            const uint32_t hi = __builtin_amdgcn_bitop3_b32(static_cast<uint32_t>(peers[i] >> 32), static_cast<uint32_t>(m >> 32), ones, 0x90);
            peers[i] = (static_cast<uint64_t>(hi) << 32) | lo;
        }
    }
    // (a wavefront's own counters: LDS serves a wavefront's instructions in their order)
#pragma unroll
    for (int i = 0; i < kWideItems; ++i) {
        const uint32_t below = __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(peers[i] >> 32),
                                                         __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(peers[i]), 0));
        const uint32_t before = static_cast<uint32_t>(mine[dig[i]]);
        rank[i] = before + below;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
        __builtin_amdgcn_wave_barrier();
        if (below == 0) {
            mine[dig[i]] = static_cast<int32_t>(before + __popcll(peers[i]));
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
        __builtin_amdgcn_wave_barrier();
    }
    LdsBarrier();
    {
        // digits of this thread: the counters become the start of every (digit, wavefront) in the ordered tile (read
        // twice rather than kept: the registers hold two tiles)
        int32_t sum = 0;
#pragma unroll
        for (int j = 0; j < kPer; ++j) {
            const int32_t d = tid * kPer + j;
            if (d < digits) {
#pragma unroll
                for (int w = 0; w < kWaves; ++w) {
                    sum += lds.counters[w * digits + d];
                }
            }
        }
        int32_t run = WideBlockScan<T>(sum, lds.waveSums);
#pragma unroll
        for (int j = 0; j < kPer; ++j) {
            const int32_t d = tid * kPer + j;
            if (d < digits) {
                lds.outOf[d] = first[j] - run;
                constexpr int kAtOnce = 4;
#pragma unroll
                for (int w0 = 0; w0 < kWaves; w0 += kAtOnce) {
                    int32_t count[kAtOnce];
#pragma unroll
                    for (int w = 0; w < kAtOnce; ++w) {
                        count[w] = lds.counters[(w0 + w) * digits + d];
                    }
#pragma unroll
                    for (int w = 0; w < kAtOnce; ++w) {
                        lds.counters[(w0 + w) * digits + d] = run;
                        run += count[w];
                    }
                }
            }
        }
    }
    LdsBarrier();
#pragma unroll
    for (int i = 0; i < kWideItems; ++i) {
        rank[i] += static_cast<uint32_t>(mine[dig[i]]);
    }
    LdsBarrier();  // the counters make room for the entries
}

// Puts the tile held in registers into the LDS arrays in the order of its digits.  Ends with a barrier.
template <int T>
__device__ __forceinline__ void WideOrder(WideLds<T> &lds, const WideTileRegs<T> &r, int32_t shift, int32_t mask,
                                          int32_t bits)
{
    uint32_t dig[kWideItems], rank[kWideItems];
#pragma unroll
    for (int i = 0; i < kWideItems; ++i) {
        dig[i] = WideDigit(r.key[i], shift, mask);
    }
    WideRank<T>(lds, dig, r.first, mask, bits, rank);
#pragma unroll
    for (int i = 0; i < kWideItems; ++i) {
        lds.key[rank[i]] = r.key[i];
        lds.row[rank[i]] = r.pay[i].row;
        lds.val[rank[i]] = r.pay[i].val;
    }
    LdsBarrier();
}

// Writes the ordered tile out.  Ends with the stores issued and no barrier behind them.
template <int T, int Mode, int VB, bool Full>
__device__ __forceinline__ void WideWrite(const WideLds<T> &lds, int64_t tile, int64_t n, int32_t shift, int32_t mask,
                                          int32_t *__restrict__ keysOut, RadixPair *__restrict__ pairsOut,
                                          const RadixPairIo &io)
{
    const int tid = threadIdx.x;
    const int32_t valid = Full ? WideShape<T>::kTile : static_cast<int32_t>(n - tile * WideShape<T>::kTile);
#pragma unroll
    for (int i = 0; i < kWideItems; ++i) {
        const int32_t p = i * T + tid;
        if (Full || p < valid) {  // the real entries are the first `valid` slots of the ordered tile
            const int32_t key = lds.key[p];
            const int64_t dst = static_cast<int64_t>(lds.outOf[WideDigit(key, shift, mask)] + p);
            keysOut[dst] = key;
            if (Mode == kPayPairLast) {
                io.rowOut[dst] = lds.row[p];
                if (VB == 4) {
                    static_cast<uint32_t *>(io.valOut)[dst] = lds.val[p];
                } else if (VB == 2) {
                    static_cast<uint16_t *>(io.valOut)[dst] = static_cast<uint16_t>(lds.val[p]);
                } else if (VB == 1) {
                    static_cast<uint8_t *>(io.valOut)[dst] = static_cast<uint8_t>(lds.val[p]);
                }
            } else {
                WideRows(pairsOut)[dst] = lds.row[p];
                WideVals(pairsOut, n)[dst] = lds.val[p];
            }
        }
    }
}

// The tiles of a pass.  Every XCD has a range of tiles, its workgroups take neighbouring tiles of it in the same turn, and a
// workgroup has the loads of its next tile in flight while it writes the current one: two sets of registers used in turn.  The
// tile that the end of the array cuts short is done last, by workgroup 0, with bounds checks.
template <int T, typename Regs, typename Fetch, typename Order, typename Write>
__device__ __forceinline__ void WideTurns(int64_t n, int64_t numTiles, Fetch &&fetch, Order &&order, Write &&write)
{
    const int64_t fullTiles = n / WideShape<T>::kTile;
    Regs r;
    const uint32_t xcds = gridDim.x < kNumXcd ? gridDim.x : kNumXcd;
    const uint32_t xcd = blockIdx.x % xcds;
    const int64_t step = (gridDim.x - xcd + xcds - 1) / xcds;
    const int64_t tileEnd = fullTiles * (xcd + 1) / xcds;
    int64_t tile = fullTiles * xcd / xcds + blockIdx.x / xcds;
    // (The last turn fetches its own tile again rather than branch around the loads: a wait for "all but what was issued
    // since" needs one straight path.)
    auto turn = [&](Regs &now, Regs &next) {
        const int64_t ahead = tile + step < tileEnd ? tile + step : tile;
        fetch(next, ahead, std::true_type{});
        __builtin_amdgcn_sched_barrier(0);  // the loads are issued here, not where the scheduler finds room later
        order(now, tile, std::true_type{});
        write(tile, std::true_type{});
        LdsBarrier();  // the tile's LDS is free again
        tile += step;
    };
    if (tile < tileEnd) {
        fetch(r, tile, std::true_type{});
        Regs other;
        // the first turn stands outside the loop: entered from here, with no stores behind the loads, the loop's
        // wait for the loads would be a wait for everything, the stores of the turn before included
        turn(r, other);
        while (tile < tileEnd) {
            turn(other, r);
            if (tile >= tileEnd) {
                break;
            }
            turn(r, other);
        }
    }
    if (blockIdx.x == 0 && fullTiles < numTiles) {
        fetch(r, fullTiles, std::false_type{});
        order(r, fullTiles, std::false_type{});
        write(fullTiles, std::false_type{});
    }
}

// One pass; the payload modes are those of RadixScatterKernel (pairs only), VB the bytes of a value in the arrays
// that the first pass reads and the last one writes (a template parameter: a branch on it among the loads would
// leave the compiler unable to count what is in flight).  prefix is the scanned table of WideCountKernel:
// prefix[digit * numTiles + tile] is the first output position of the tile's entries of that digit.
template <int T, int Mode, int VB>
__global__ __launch_bounds__(T) void WideScatterKernel(
    const int32_t *__restrict__ keysIn, const RadixPair *__restrict__ pairsIn, int32_t *__restrict__ keysOut,
    RadixPair *__restrict__ pairsOut, int64_t n, int32_t keyBase, int32_t shift, int32_t mask, int32_t bits,
    const int32_t *__restrict__ prefix, int64_t numTiles, RadixPairIo io)
{
    __shared__ WideLds<T> lds;
    WideTurns<T, WideTileRegs<T>>(
        n, numTiles,
        [&](WideTileRegs<T> &r, int64_t tile, auto full) {
            WideFetch<T, Mode, VB, decltype(full)::value>(r, tile, keysIn, pairsIn, n, keyBase, shift, mask, prefix, numTiles,
                                                          io);
        },
        [&](const WideTileRegs<T> &r, int64_t, auto) { WideOrder<T>(lds, r, shift, mask, bits); },
        [&](int64_t tile, auto full) {
            WideWrite<T, Mode, VB, decltype(full)::value>(lds, tile, n, shift, mask, keysOut, pairsOut, io);
        });
}

// ------------------------------- passes in front of buckets that are ordered in LDS
// Where the last bits of a key are ordered bucket by bucket (below), a pass need not carry the bits that the passes before have
// ordered by: an entry's bucket is where it stands.  What travels is a record of 8 bytes, the low bits of the key above the
// payload in one word and the value in the other, and between two passes a byte beside it, the second pass's digit, which is
// also all that its count has to read.  Bound by memory: 12 bytes an entry in and 9 out, 9 and 8, where key, row and value were
// 12 in and 12 out in either pass; a tile's run in a bucket is a piece of one array instead of three.
// Where the low bits and the payload take more than a word (more than 2^22 rows under ten low bits) the payload's top bits travel
// in 16 bits of their own (Tops): 2 bytes an entry more into and out of every step behind the first.
struct PackIo {
    const int32_t *keys;  // first pass: keyBase + key, payload and value of every entry
    int32_t keyBase;
    const int32_t *pays;
    const void *vals;
    const uint8_t *digitsIn;  // second pass
    const Record *recsIn;
    uint8_t *digitsOut;  // first pass of two
    Record *recsOut;
    const uint16_t *topsIn;  // Tops: what is above payBits of a payload, beside the records
    uint16_t *topsOut;
    int64_t n;
    int32_t low, payBits;  // bits of a key below its bucket; of a payload in the record (together 32 at most)
    int32_t nextShift;     // first pass of two: the second one's digit is what is above this bit of a key
};

enum PackMode { kPackOnly = 0, kPackFirst = 1, kPackSecond = 2 };

template <int T, int Mode, bool Tops>
struct PackRegs {
    uint32_t key[kWideItems], pay[kWideItems], val[kWideItems];
    int32_t first[WideShape<T>::kPer];
};
template <int T, bool Tops>
struct PackRegs<T, kPackSecond, Tops> {
    uint64_t rec[kWideItems];
    uint32_t digit[kWideItems];
    uint32_t top[Tops ? kWideItems : 1];
    int32_t first[WideShape<T>::kPer];
};

// Low bits of a key above its payload, and the value.
__device__ __forceinline__ uint64_t PackedRecord(uint32_t word, uint32_t val)
{
    return (static_cast<uint64_t>(val) << 32) | word;
}

template <int T, bool Tops>
struct PackLds {
    union {
        int32_t counters[WideShape<T>::kWaves << kWideMaxBits];
        struct {
            uint64_t rec[WideShape<T>::kTile];
            uint16_t digit[WideShape<T>::kTile * (Tops ? 2 : 1)];  // kPackFirst: the next pass's above the lower eight
                                                                   // bits; behind the tile's digits its tops
        };
    };
    int32_t outOf[1 << kWideMaxBits];
    int32_t waveSums[WideShape<T>::kWaves];
};

// prefix, shift, mask, bits: as WideScatterKernel; the first digit of two has eight bits at most.
template <int T, int Mode, int VB, bool Tops>
__global__ __launch_bounds__(T, 4) void PackScatterKernel(PackIo io, int32_t shift, int32_t mask, int32_t bits,
                                                          const int32_t *__restrict__ prefix, int64_t numTiles)
{
    __shared__ PackLds<T, Tops> lds;
    constexpr int kTile = WideShape<T>::kTile, kPer = WideShape<T>::kPer;
    const uint32_t lowMask = (1u << io.low) - 1u;
    auto fetch = [&](PackRegs<T, Mode, Tops> &r, int64_t tile, auto full) {
        const int tid = MadeAnew(threadIdx.x);
#pragma unroll
        for (int j = 0; j < kPer; ++j) {
            const int32_t d = tid * kPer + j;
            r.first[j] = prefix[static_cast<int64_t>(d <= mask ? d : mask) * numTiles + tile];
        }
        const int64_t wave0 = tile * kTile + tid / kWave * (kWave * kWideItems) + tid % kWave;
#pragma unroll
        for (int i = 0; i < kWideItems; ++i) {
            // (a slot past the end reads the last entry)
            const int64_t at = decltype(full)::value || wave0 + i * kWave < io.n ? wave0 + i * kWave : io.n - 1;
            if constexpr (Mode == kPackSecond) {
                r.rec[i] = __builtin_nontemporal_load(io.recsIn + at);
                r.digit[i] = LoadStream(io.digitsIn + at);
                if constexpr (Tops) {
                    r.top[i] = LoadStream(io.topsIn + at);
                }
            } else {
                r.key[i] = static_cast<uint32_t>(LoadStream(io.keys + at));
                r.pay[i] = static_cast<uint32_t>(LoadStream(io.pays + at));
                r.val[i] = 0;
                if constexpr (VB == 4) {
                    r.val[i] = LoadStream(static_cast<const uint32_t *>(io.vals) + at);
                } else if constexpr (VB == 2) {
                    r.val[i] = static_cast<const uint16_t *>(io.vals)[at];
                } else if constexpr (VB == 1) {
                    r.val[i] = static_cast<const uint8_t *>(io.vals)[at];
                }
            }
        }
    };
    auto order = [&](const PackRegs<T, Mode, Tops> &r, int64_t tile, auto full) {
        const int tid = MadeAnew(threadIdx.x);
        uint32_t dig[kWideItems], rank[kWideItems];
        const int64_t wave0 = tile * kTile + tid / kWave * (kWave * kWideItems) + tid % kWave;
#pragma unroll
        for (int i = 0; i < kWideItems; ++i) {
            if constexpr (Mode == kPackSecond) {
                dig[i] = r.digit[i] & static_cast<uint32_t>(mask);
            } else {
                dig[i] = WideDigit(Rebased(static_cast<int32_t>(r.key[i]), io.keyBase), shift, mask);
            }
            // a slot past the end gets the largest digit, so that it sorts behind every real entry
            dig[i] = decltype(full)::value || wave0 + i * kWave < io.n ? dig[i] : static_cast<uint32_t>(mask);
        }
        WideRank<T>(lds, dig, r.first, mask, bits, rank);
#pragma unroll
        for (int i = 0; i < kWideItems; ++i) {
            if constexpr (Mode == kPackSecond) {
                lds.rec[rank[i]] = r.rec[i];
                lds.digit[rank[i]] = static_cast<uint16_t>(dig[i]);
                if constexpr (Tops) {
                    lds.digit[kTile + rank[i]] = static_cast<uint16_t>(r.top[i]);
                }
            } else {
                const uint32_t key = static_cast<uint32_t>(Rebased(static_cast<int32_t>(r.key[i]), io.keyBase));
                const uint32_t pay = Tops ? r.pay[i] & ((1u << io.payBits) - 1u) : r.pay[i];
                lds.rec[rank[i]] = PackedRecord(((key & lowMask) << io.payBits) | pay, r.val[i]);
                if constexpr (Tops) {
                    lds.digit[kTile + rank[i]] = static_cast<uint16_t>(r.pay[i] >> io.payBits);
                }
                lds.digit[rank[i]] = static_cast<uint16_t>(Mode == kPackFirst ? dig[i] | (key >> io.nextShift << 8) : dig[i]);
            }
        }
        LdsBarrier();
    };
    auto write = [&](int64_t tile, auto full) {
        const int tid = MadeAnew(threadIdx.x);
        const int32_t valid = decltype(full)::value ? kTile : static_cast<int32_t>(io.n - tile * kTile);
#pragma unroll
        for (int i = 0; i < kWideItems; ++i) {
            const int32_t p = i * T + tid;
            if (decltype(full)::value || p < valid) {  // the real entries are the first `valid` slots of the ordered tile
                const uint32_t digit = lds.digit[p];
                const int64_t dst = static_cast<int64_t>(lds.outOf[Mode == kPackFirst ? digit & 0xffu : digit] + p);
                io.recsOut[dst] = lds.rec[p];
                if constexpr (Tops) {
                    io.topsOut[dst] = lds.digit[kTile + p];
                }
                if constexpr (Mode == kPackFirst) {
                    io.digitsOut[dst] = static_cast<uint8_t>(digit >> 8);
                }
            }
        }
    };
    WideTurns<T, PackRegs<T, Mode, Tops>>(io.n, numTiles, fetch, order, write);
}

// WideCountKernel's table from the digits that the first pass left: a thread takes eight of a tile's together.
template <int T>
__global__ __launch_bounds__(T) void DigitCountKernel(const uint8_t *__restrict__ digits, int64_t n, int32_t mask,
                                                      int32_t *__restrict__ table, int64_t numTiles)
{
    constexpr int kTile = WideShape<T>::kTile;
    static_assert(kWideItems == 8, "eight digits a load");
    __shared__ int32_t hist[kWideCountTiles << 8];
    const int32_t count = mask + 1;
    for (int32_t i = threadIdx.x; i < kWideCountTiles * count; i += T) {
        hist[i] = 0;
    }
    const int64_t firstTile = static_cast<int64_t>(XcdContiguousTile(blockIdx.x, gridDim.x)) * kWideCountTiles;
    Uint2U eight[kWideCountTiles];
#pragma unroll
    for (int j = 0; j < kWideCountTiles; ++j) {
        const int64_t at = (firstTile + j) * kTile + 8 * threadIdx.x;
        eight[j] = *reinterpret_cast<const Uint2U *>(digits + (at < n ? at : 0));  // (the array's room ends on such a piece)
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kWideCountTiles; ++j) {
        const int64_t at = (firstTile + j) * kTile + 8 * threadIdx.x;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const uint32_t d = ((i < 4 ? eight[j].x : eight[j].y) >> (8 * (i % 4))) & static_cast<uint32_t>(mask);
            atomicAdd(&hist[j * count + d], at + i < n ? 1 : 0);
        }
    }
    __syncthreads();
    for (int32_t i = threadIdx.x; i < kWideCountTiles * count; i += T) {
        const int64_t tile = firstTile + i % kWideCountTiles;
        if (tile < numTiles) {
            const int32_t d = i / kWideCountTiles;
            table[1 + static_cast<int64_t>(d) * numTiles + tile] = hist[i % kWideCountTiles * count + d];
        }
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        table[0] = 0;
    }
}

// csrsort of a matrix of long rows, between its two sorts: the entries are sorted by column and carry (row,
// permutation value); the second sort is by row and carries (column, permutation value).
__global__ __launch_bounds__(kBlockThreads) void RegroupByRowKernel(const int32_t *__restrict__ colKeys,
                                                                   const RadixPair *__restrict__ rowAndPerm, int64_t n,
                                                                   int32_t colBase, int32_t *__restrict__ rowKeys,
                                                                   RadixPair *__restrict__ colAndPerm)
{
    const int64_t i = static_cast<int64_t>(blockIdx.x) * kBlockThreads + threadIdx.x;
    if (i < n) {
        const RadixPair in = rowAndPerm[i];
        rowKeys[i] = in.row;
        colAndPerm[i] = RadixPair{colKeys[i] + colBase, in.val};
    }
}

// ---------------------------------------------------------------- csr2csc

// cscRowInd[d] = row of source position pos[d] (+ base); cscVal[d] = csrVal[pos[d]].
template <typename T>
__global__ __launch_bounds__(kBlockThreads) void GatherByPositionKernel(const int32_t *__restrict__ pos,
                                                                       const int32_t *__restrict__ rowOfPos,
                                                                       const T *__restrict__ srcVal, int64_t nnz,
                                                                       int32_t *__restrict__ rowOut,
                                                                       T *__restrict__ valOut)
{
    const int64_t d = static_cast<int64_t>(blockIdx.x) * kBlockThreads + threadIdx.x;
    if (d >= nnz) {
        return;
    }
    const int32_t p = LoadStream(pos + d);
    rowOut[d] = rowOfPos[p];
    if (valOut != nullptr) {
        valOut[d] = srcVal[p];
    }
}

// ---------------------------------------------------------------- csrsort

// Orders by signed column first, position in the row second.
__device__ __forceinline__ uint64_t SortKey(int32_t col, uint32_t idx)
{
    return (static_cast<uint64_t>(static_cast<uint32_t>(col) ^ 0x80000000u) << 32) | idx;
}
__device__ __forceinline__ int32_t SortKeyColumn(uint64_t key)
{
    return static_cast<int32_t>(static_cast<uint32_t>(key >> 32) ^ 0x80000000u);
}

// The value of lane (l ^ J) for every lane l of a wavefront, all of whose lanes are active.  Distances 1, 2, 4
// and 8 stay inside a row of 16 lanes and are data-parallel-primitive moves in the vector ALU (quad permutes,
// rotations of a row); only 16 and 32 go through the LDS crossbar, where every distance went before (the sort of
// a 64-lane group issued 42 such operations and spent its time waiting for them).  `ror4` says whether the
// rotation by 4 or the one by 12 brings lane l the value of lane l ^ 4: found once per thread by sending the
// lane numbers through both, which leaves the direction of the rotation out of the argument.
__device__ __forceinline__ uint32_t DppMove(uint32_t v, int ctrl)
{
    switch (ctrl) {  // the control word is an immediate of the instruction
        case 0xB1: return static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0xB1, 0xF, 0xF, false));
        case 0x4E: return static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x4E, 0xF, 0xF, false));
        case 0x124: return static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x124, 0xF, 0xF, false));
        case 0x128: return static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x128, 0xF, 0xF, false));
        default: return static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x12C, 0xF, 0xF, false));
    }
}

__device__ __forceinline__ bool Ror4IsXor4()
{
    const uint32_t lane = threadIdx.x % kWave;
    return DppMove(lane, 0x124) == (lane ^ 4u);
}

template <int J>
__device__ __forceinline__ uint32_t XorLanes(uint32_t v, bool ror4)
{
    if (J == 1) {
        return DppMove(v, 0xB1);  // quad_perm [1, 0, 3, 2]
    } else if (J == 2) {
        return DppMove(v, 0x4E);  // quad_perm [2, 3, 0, 1]
    } else if (J == 4) {
        const uint32_t a = DppMove(v, 0x124), b = DppMove(v, 0x12C);  // row_ror 4 and 12
        return ror4 ? a : b;
    } else if (J == 8) {
        return DppMove(v, 0x128);  // row_ror 8: the same in either direction
    } else {
        return static_cast<uint32_t>(__shfl_xor(static_cast<int>(v), J, kWave));
    }
}

template <int J>
__device__ __forceinline__ uint64_t XorLanes(uint64_t v, bool ror4)
{
    const uint32_t lo = XorLanes<J>(static_cast<uint32_t>(v), ror4);
    const uint32_t hi = XorLanes<J>(static_cast<uint32_t>(v >> 32), ror4);
    return (static_cast<uint64_t>(hi) << 32) | lo;
}

template <int K, int J, typename KeyT>
__device__ __forceinline__ void BitonicStep(KeyT &key, int32_t g, bool ror4)
{
    const KeyT other = XorLanes<J>(key, ror4);
    const bool ascending = (g & K) == 0;
    const bool lower = (g & J) == 0;
    const KeyT mn = key < other ? key : other;
    const KeyT mx = key < other ? other : key;
    key = (ascending == lower) ? mn : mx;
}

template <int K, int J, typename KeyT>
__device__ __forceinline__ void BitonicMerge(KeyT &key, int32_t g, bool ror4)
{
    BitonicStep<K, J>(key, g, ror4);
    if constexpr (J > 1) {
        BitonicMerge<K, J / 2>(key, g, ror4);
    }
}

template <int G, int K, typename KeyT>
__device__ __forceinline__ void BitonicStages(KeyT &key, int32_t g, bool ror4)
{
    BitonicMerge<K, K / 2>(key, g, ror4);
    if constexpr (K < G) {
        BitonicStages<G, K * 2>(key, g, ror4);
    }
}

// Bitonic sort of one key per lane over the G lanes of a group (all 64 lanes of the wavefront take part); `g` is
// the lane's index in its group.  The low bits of a key hold the group lane its entry came from, so all keys
// differ and the sort is the stable one.  Returns the sorted key.
template <int G, typename KeyT>
__device__ __forceinline__ KeyT GroupBitonicSort(KeyT key, int32_t g)
{
    const bool ror4 = Ror4IsXor4();
    BitonicStages<G, 2>(key, g, ror4);
    return key;
}

// The middle one of three: with c = 0 the smaller of a and b, with c = ~0 the larger.
__device__ __forceinline__ uint32_t Median(uint32_t a, uint32_t b, uint32_t c)
{
    const uint32_t mn = a < b ? a : b, mx = a < b ? b : a;
    const uint32_t up = mx < c ? mx : c;
    return mn > up ? mn : up;
}

// The sort of 32-bit keys over groups of G lanes, two vector instructions for most steps: the other lane's key by a move inside
// the vector unit, and the median of both keys and 0 or ~0, by the lane's place in its pair.  Up to 16 lanes the first step of a
// merge exchanges the lanes from the outside in (lane i with lane K - 1 - i), so that all of them sort upwards; the exchanges at
// 16 and 32 are swaps of rows and of halves, which leave both keys of a pair in both its lanes, and there the upper block of a
// merge has been sorted downwards, which is upwards in its complements.  33.5 M entries in rows of 32: csrsort 213 -> 169 us,
// coosort by row 731 -> 676 against steps of a minimum, a maximum and a choice with the moves at 16 and 32 through the LDS
// crossbar.
template <int kCtrl>
__device__ __forceinline__ uint32_t DppOf(uint32_t v)
{
    return static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), kCtrl, 0xF, 0xF, false));
}
template <int G>
__device__ __forceinline__ uint32_t GroupSort(uint32_t key, int32_t lane)
{
    constexpr int kQuad1 = 0xB1, kQuad2 = 0x4E, kQuad3 = 0x1B, kMirror8 = 0x141, kMirror16 = 0x140, kTurn8 = 0x128;
    auto upper = [&](int bit) { return static_cast<uint32_t>(__builtin_amdgcn_sbfe(lane, bit, 1)); };  // ~0 where the bit is set
    const uint32_t up0 = upper(0), up1 = upper(1), up2 = upper(2), up3 = upper(3), up4 = upper(4), up5 = upper(5);
    auto by1 = [&] { key = Median(key, DppOf<kQuad1>(key), up0); };
    auto by2 = [&] { key = Median(key, DppOf<kQuad2>(key), up1); };
    auto by4 = [&] { key = Median(key, DppOf<kQuad3>(DppOf<kMirror8>(key)), up2); };
    auto by8 = [&] { key = Median(key, DppOf<kTurn8>(key), up3); };
    auto by16 = [&] {
        const auto pair = __builtin_amdgcn_permlane16_swap(key, key, false, false);
        key = Median(pair[0], pair[1], up4);
    };
    auto by32 = [&] {
        const auto pair = __builtin_amdgcn_permlane32_swap(key, key, false, false);
        key = Median(pair[0], pair[1], up5);
    };
    if constexpr (G >= 32) {
        key ^= G == 64 ? up4 ^ up5 : up4;
    }
    by1();
    key = Median(key, DppOf<kQuad3>(key), up1);
    by1();
    key = Median(key, DppOf<kMirror8>(key), up2);
    by2();
    by1();
    if constexpr (G >= 16) {
        key = Median(key, DppOf<kMirror16>(key), up3);
        by4();
        by2();
        by1();
    }
    if constexpr (G >= 32) {
        key ^= up4;
        by16();
        by8();
        by4();
        by2();
        by1();
    }
    if constexpr (G >= 64) {
        key ^= up5;
        by32();
        by16();
        by8();
        by4();
        by2();
        by1();
    }
    return key;
}

// Packed: the key is (column << log2 G | lane) in 32 bits, half the moves of the 64-bit key; the launcher takes
// it when every column index of a valid matrix fits (columns outside [0, n) then only lose their order: the
// entries themselves travel by source lane, not inside the key).
// The entry a lane holds of its group's row, sorted within the group: (col, pay) of lane g become those of the
// g-th entry of the sorted row.
template <int G, bool Packed>
__device__ __forceinline__ void SortHeldRow(bool valid, int32_t g, int32_t *col, int32_t *pay)
{
    constexpr int kLog = G == 64 ? 6 : G == 32 ? 5 : G == 16 ? 4 : 3;
    static_assert((1 << kLog) == G, "8, 16, 32 or 64 lanes a row");
    const int32_t lane = threadIdx.x % kWave;
    int32_t from;
    if (Packed) {
        uint32_t key = valid ? (static_cast<uint32_t>(*col) << kLog) | static_cast<uint32_t>(g) : ~0u;  // padding last
        key = GroupSort<G>(key, lane);
        from = (lane - g) + static_cast<int32_t>(key & (G - 1));
    } else {
        uint64_t key = valid ? SortKey(*col, static_cast<uint32_t>(g)) : ~0ull;
        key = GroupBitonicSort<G>(key, g);
        from = (lane - g) + (static_cast<int32_t>(key & 0xffffffffu) & (G - 1));
    }
    *col = __shfl(*col, from, kWave);
    *pay = __shfl(*pay, from, kWave);
}

template <int G, bool Packed>
__device__ __forceinline__ void SortRowInGroup(int64_t begin, int64_t len, int32_t g, int32_t *colInd, int32_t *perm)
{
    const bool valid = g < len;
    int32_t col = 0, pay = 0;
    if (valid) {
        col = colInd[begin + g];
        pay = perm[begin + g];
    }
    SortHeldRow<G, Packed>(valid, g, &col, &pay);
    if (valid) {
        colInd[begin + g] = col;
        perm[begin + g] = pay;
    }
}

// ------------------------------------- the last bits of a key, in LDS
// Stable passes over the upper bits of the keys (csr2csc, coosort) leave the entries in buckets of 2^low neighbouring
// keys, and a bucket of a few thousand entries is ordered in LDS by one workgroup.  It leaves as one piece, whole lines,
// where a pass writes a run of tens of entries for each of its buckets; the starts of its keys are the offsets that
// another two passes over the sorted keys found by counting, and the sorted keys themselves need not be written where
// nobody asks for them.  Bound by memory: 8 bytes an entry in, 8 (csr2csc) or 12 (coosort) out, three or two workgroups a
// compute unit, one of which loads while another orders; coosort's by its vector instructions, which sort the rows.
//
// Buckets that do not fit go on lists.  Of up to kFinishLarge entries: a workgroup twice as large orders them.  Beyond (hubs):
// three kernels count, scan and scatter pieces of kFinishMost entries as a pass does its tiles.  With nothing on the lists
// these kernels end at once, 14 us for the three.
//
// 33.5 M entries over 2^20 keys: csr2csc 797 -> 651 us (the last pass with its count and scan, 213 us, and the counting of the
// sorted columns, 70, became 133 us and 19 for the buckets' starts), and 498 with packed records in front of the buckets (114 us);
// 400 K entries over 50 000 columns 95 -> 64 us.  Before the records were packed: where half of the keys are met, so that every
// bucket is twice as full as planned, the larger workgroups made it 772 -> 742 us (925 while such buckets went in pieces, 1139
// with each entry of theirs written straight to its place); with a tenth of the entries in one column 1487 -> 762.
//
// coosort's rows lie side by side in LDS then, and those of up to 64 entries are sorted in registers on their way out; the
// rest go on csrsort's lists.  A kernel over the sorted entries that did this read and wrote 8 bytes an entry once more: 33.5 M
// entries, 32 a row, 897 -> 779 us, 8 a row over 4 M rows 904 -> 747 (without the digits in LDS there is room for three
// workgroups a compute unit instead of two, too).  With packed records in front and the faster networks 676 us, the buckets 225.

constexpr int kFinishThreads = 512;
constexpr int kFinishItems = 12;  // entries of a thread
constexpr int kFinishMost = kFinishThreads * kFinishItems;  // entries of a bucket that fits
constexpr int kFinishLargeThreads = 1024;
constexpr int kFinishLarge = kFinishLargeThreads * kFinishItems;  // ... the larger workgroup
constexpr int kFinishMaxBits = 10;                          // bits of a key that are ordered here
constexpr int kFinishScanThreads = 1 << kFinishMaxBits;

// The buckets that do not fit; the first three are the lengths of the lists.
struct FinishList {
    int32_t *large, *pieces, *buckets;
    int32_t *largeOf;                 // buckets of up to kFinishLarge entries
    int32_t *pieceBucket, *pieceNo;   // of a piece: its bucket, its number in there
    int32_t *bucketOf, *bucketFirst;  // of a bucket in pieces: which, its first piece (they follow one another)
    int32_t *table;                   // [piece][digit]: how many, then where they go
};

constexpr int kFinishLengths = 32;  // ints from `large` on that are zero at the start: the lists' lengths, csrsort's counters

struct FinishIo {
    const Record *recs;  // in the order of the keys' upper bits: low bits of the key above the payload, and the value
    const uint16_t *tops;  // Tops: what is above payBits of the payloads
    int32_t payBits;
    int64_t n;
    const int32_t *starts;  // bucket b begins at starts[b * startStride]; there is one more than buckets
    int64_t startStride;
    int32_t low;            // bits of a key below its bucket
    int64_t numKeys;
    int32_t base;
    int32_t *ptr;     // [numKeys + 1]: base + the position of every key's first entry
    int32_t *keyOut;  // coosort
    int32_t *rowOut;
    void *valOut;
    FinishList list;
    // rows that csrsort's kernels have to sort: counters[0] in midList (up to 64 entries), counters[1] in longList
    int32_t *rowCounters, *midList, *longList;
};

// Lanes: 0, or coosort's rows (the entries of a key) are sorted by column as well, Lanes of a wavefront to a row.
template <int T, bool Digits, int Lanes>
struct FinishLds {
    union {
        int32_t counters[T / kWave << kFinishMaxBits];  // [wavefront][digit]
        struct {
            int32_t row[T * kFinishItems];
            uint32_t val[T * kFinishItems];
        };
    };
    uint16_t digit[Digits ? T * kFinishItems : 1];
    int32_t outOf[Digits || Lanes != 0 ? (1 << kFinishMaxBits) + 1 : 1];  // with rows to sort: where each begins
    int32_t longRows, longRow[Lanes != 0 ? T * kFinishItems / kSortWaveRow : 1];
    int32_t waveSums[T / kWave];
};

// A wavefront sorts the rows of the ordered entries that fall to it and writes them: as many at a time as it has groups of
// Lanes, those that a group cannot hold by itself, and those of more than 64 entries unsorted (they are on a list).
template <int T, int Lanes, typename Lds>
__device__ __forceinline__ void FinishRows(const Lds &lds, const FinishIo &io, int32_t first, int32_t key0)
{
    const int32_t lane = threadIdx.x % kWave, wave = threadIdx.x / kWave, g = lane % Lanes;
    const int32_t digits = 1 << io.low;
    auto write = [&](int64_t dst, int32_t key, int32_t col, int32_t pay) {
        io.keyOut[dst] = key;
        io.rowOut[dst] = col;
        static_cast<int32_t *>(io.valOut)[dst] = pay;
    };
    constexpr int32_t kRows = kWave / Lanes;
    for (int32_t d0 = wave * kRows; d0 < digits; d0 += T / kWave * kRows) {
        const int32_t d = d0 + lane / Lanes;
        const int32_t begin = d < digits ? lds.outOf[d] : 0;
        const int32_t len = d < digits ? lds.outOf[d + 1] - begin : 0;
        const bool valid = len <= Lanes && g < len;
        int32_t col = 0, pay = 0;
        if (valid) {
            col = lds.row[begin + g];
            pay = static_cast<int32_t>(lds.val[begin + g]);
        }
        SortHeldRow<Lanes, true>(valid, g, &col, &pay);
        if (valid) {
            write(static_cast<int64_t>(first) + begin + g, key0 + d, col, pay);
        }
        uint64_t left = __ballot(g == 0 && len > Lanes);
        while (left != 0) {
            const int32_t src = __ffsll(static_cast<long long>(left)) - 1;
            left &= left - 1;
            const int32_t at = __shfl(begin, src, kWave), n = __shfl(len, src, kWave), key = key0 + d0 + src / Lanes;
            if (n <= kSortWaveRow) {
                col = lane < n ? lds.row[at + lane] : 0;
                pay = lane < n ? static_cast<int32_t>(lds.val[at + lane]) : 0;
                SortHeldRow<kWave, true>(lane < n, lane, &col, &pay);
                if (lane < n) {
                    write(static_cast<int64_t>(first) + at + lane, key, col, pay);
                }
            } else {
                for (int32_t i = lane; i < n; i += kWave) {
                    write(static_cast<int64_t>(first) + at + i, key, lds.row[at + i], static_cast<int32_t>(lds.val[at + i]));
                }
            }
        }
    }
}

// The low bits of the key that a record holds.
__device__ __forceinline__ int32_t FinishDigit(uint64_t rec, int32_t payBits, int32_t mask)
{
    return static_cast<int32_t>(static_cast<uint32_t>(rec) >> payBits) & mask;
}

// Orders the `len` entries at `first` by the low bits of their keys and writes them: a whole bucket (Big = false) where it
// stands, a piece of one where the scanned table says.
template <int T, bool Keys, int VB, bool Big, bool Tops, bool Digits, int Lanes>
__device__ __forceinline__ void FinishPiece(FinishLds<T, Digits, Lanes> &lds, const FinishIo &io, int32_t first, int32_t len,
                                            uint32_t bucket, const int32_t *__restrict__ places)
{
    const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
    const int32_t digits = 1 << io.low, mask = digits - 1;
    // lane l of wavefront w holds the entries l, l + 64, ... of the w-th stretch of `rounds` x 64; the slots past the end
    // have the largest digit and so come behind every entry
    const int32_t rounds = (len + T - 1) / T;
    const int32_t at0 = wave * rounds * kWave + lane;
    // (no branch around a load: a slot past the end reads the last entry)
    uint64_t rec[kFinishItems];
    uint32_t top[Tops ? kFinishItems : 1];
    const int32_t lastSlot = len > 0 ? len - 1 : 0;
#pragma unroll
    for (int i = 0; i < kFinishItems; ++i) {
        const int32_t slot = at0 + i * kWave;
        const int64_t at = static_cast<int64_t>(first) + (slot < lastSlot ? slot : lastSlot);
        rec[i] = __builtin_nontemporal_load(io.recs + (at < io.n ? at : io.n - 1));
        if constexpr (Tops) {
            top[i] = LoadStream(io.tops + (at < io.n ? at : io.n - 1));
        }
    }
    int32_t *mine = lds.counters + wave * digits;
    for (int32_t d = lane; d < digits; d += kWave) {
        mine[d] = 0;
    }
    if (tid == 0) {
        lds.longRows = 0;
    }
    // (a wavefront's own counters: LDS serves a wavefront's instructions in their order)
    uint32_t rank[kFinishItems];
#pragma unroll
    for (int i = 0; i < kFinishItems; ++i) {
        rank[i] = 0;
        rec[i] = at0 + i * kWave < len ? rec[i] : ~uint64_t{0};
        if (i < rounds) {
            const int32_t key = FinishDigit(rec[i], io.payBits, mask);
            uint64_t peers = ~uint64_t{0};
            for (int32_t b = 0; b < io.low; ++b) {
                const uint32_t ones = static_cast<uint32_t>(__builtin_amdgcn_sbfe(key, b, 1));
                const uint64_t m = __ballot(ones != 0);
                // peers & ~(m ^ ones)
                const uint32_t lo = __builtin_amdgcn_bitop3_b32(static_cast<uint32_t>(peers), static_cast<uint32_t>(m), ones, 0x90);
                const uint32_t hi = __builtin_amdgcn_bitop3_b32(static_cast<uint32_t>(peers >> 32), static_cast<uint32_t>(m >> 32), ones, 0x90);
                peers = (static_cast<uint64_t>(hi) << 32) | lo;
            }
            const uint32_t below = __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(peers >> 32),
                                                             __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(peers), 0));
            const uint32_t before = static_cast<uint32_t>(mine[key]);
            rank[i] = before + below;
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
            __builtin_amdgcn_wave_barrier();
            if (below == 0) {
                mine[key] = static_cast<int32_t>(before + __popcll(peers));
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
            __builtin_amdgcn_wave_barrier();
        }
    }
    LdsBarrier();
    {
        // the counters become the start of every (digit, wavefront) among the ordered entries
        const int32_t per = digits > T ? (1 << kFinishMaxBits) / T : 1;
        int32_t sum = 0;
        for (int32_t j = 0; j < per; ++j) {
            const int32_t d = tid * per + j;
            if (d < digits) {
#pragma unroll
                for (int w = 0; w < (T / kWave); ++w) {
                    sum += lds.counters[w * digits + d];
                }
            }
        }
        int32_t run = WideBlockScan<T>(sum, lds.waveSums);
        for (int32_t j = 0; j < per; ++j) {
            const int32_t d = tid * per + j;
            if (d < digits) {
                if constexpr (Big) {
                    lds.outOf[d] = places[d] - run;
                } else {
                    const int64_t k = (static_cast<int64_t>(bucket) << io.low) + d;
                    if (k <= io.numKeys) {
                        io.ptr[k] = io.base + first + run;
                    }
                    if constexpr (Lanes != 0) {
                        lds.outOf[d] = run;
                        if (d == mask) {
                            lds.outOf[digits] = len;
                        }
                    }
                }
                const int32_t begin = run;
                int32_t count[(T / kWave)];
#pragma unroll
                for (int w = 0; w < (T / kWave); ++w) {
                    count[w] = lds.counters[w * digits + d];
                }
#pragma unroll
                for (int w = 0; w < (T / kWave); ++w) {
                    lds.counters[w * digits + d] = run;
                    run += count[w];
                }
                if constexpr (Lanes != 0 && !Big) {
                    if ((d == mask ? len : run) - begin > kSortWaveRow) {
                        lds.longRow[atomicAdd(&lds.longRows, 1)] = static_cast<int32_t>(bucket << io.low) + d;
                    }
                }
            }
        }
    }
    LdsBarrier();
#pragma unroll
    for (int i = 0; i < kFinishItems; ++i) {
        if (i < rounds) {
            // (Tops: the digit is worked out again: kept beside the record it would make the compiler spill)
            const uint64_t again = Tops ? static_cast<uint32_t>(MadeAnew(static_cast<int>(rec[i]))) : rec[i];
            rank[i] += static_cast<uint32_t>(mine[FinishDigit(again, io.payBits, mask)]);
        }
    }
    LdsBarrier();  // the counters make room for the entries
#pragma unroll
    for (int i = 0; i < kFinishItems; ++i) {
        if (i < rounds) {
            uint32_t pay = static_cast<uint32_t>(rec[i]) & ((1u << io.payBits) - 1u);
            if constexpr (Tops) {
                pay |= top[i] << io.payBits;
            }
            lds.row[rank[i]] = static_cast<int32_t>(pay);
            lds.val[rank[i]] = static_cast<uint32_t>(rec[i] >> 32);
            if constexpr ((Keys && Lanes == 0) || Big) {
                lds.digit[rank[i]] = static_cast<uint16_t>(FinishDigit(rec[i], io.payBits, mask));
            }
        }
    }
    LdsBarrier();
    if constexpr (Lanes != 0 && !Big) {
        const int32_t longRows = lds.longRows;
        if (wave == 0 && longRows > 0) {
            // (one addition a bucket to the list's length: additions to one word are served one after the other)
            int32_t at = lane == 0 ? atomicAdd(io.rowCounters + 1, longRows) : 0;
            at = __shfl(at, 0, kWave);
            for (int32_t i = lane; i < longRows; i += kWave) {
                io.longList[at + i] = lds.longRow[i];
            }
        }
        FinishRows<T, Lanes>(lds, io, first, static_cast<int32_t>(bucket << io.low));
        return;
    }
    for (int32_t p = tid; p < len; p += T) {
        int64_t dst = static_cast<int64_t>(first) + p;
        if constexpr (Big) {
            dst = lds.outOf[lds.digit[p]] + p;
        }
        if constexpr (Keys) {
            io.keyOut[dst] = static_cast<int32_t>((bucket << io.low) | lds.digit[p]);
        }
        io.rowOut[dst] = lds.row[p];
        if (VB == 4) {
            static_cast<uint32_t *>(io.valOut)[dst] = lds.val[p];
        } else if (VB == 2) {
            static_cast<uint16_t *>(io.valOut)[dst] = static_cast<uint16_t>(lds.val[p]);
        } else if (VB == 1) {
            static_cast<uint8_t *>(io.valOut)[dst] = static_cast<uint8_t>(lds.val[p]);
        }
    }
}

// A workgroup a bucket (neighbouring buckets on one XCD).
template <bool Keys, int VB, int Lanes, bool Tops>
__global__ __launch_bounds__(kFinishThreads, Keys && Lanes == 0 ? 4 : 6) void FinishBucketsKernel(FinishIo io)
{
    __shared__ FinishLds<kFinishThreads, Keys && Lanes == 0, Lanes> lds;
    const uint32_t bucket = XcdContiguousTile(blockIdx.x, gridDim.x);
    const int32_t first = io.starts[bucket * io.startStride];
    const int32_t len = io.starts[(bucket + 1) * io.startStride] - first;
    if (blockIdx.x == 0 && threadIdx.x == 0 && io.numKeys == static_cast<int64_t>(gridDim.x) << io.low) {
        io.ptr[io.numKeys] = io.base + static_cast<int32_t>(io.n);  // (otherwise the first key past the last one's)
    }
    if (len > kFinishMost && len <= kFinishLarge) {
        if (threadIdx.x == 0) {
            io.list.largeOf[atomicAdd(io.list.large, 1)] = static_cast<int32_t>(bucket);
        }
        return;
    }
    if (len > kFinishLarge) {
        __shared__ int32_t at;
        const int32_t pieces = (len - 1) / kFinishMost + 1;  // (len may be all of 2^31 - 1)
        if (threadIdx.x == 0) {
            at = atomicAdd(io.list.pieces, pieces);
            const int32_t b = atomicAdd(io.list.buckets, 1);
            io.list.bucketOf[b] = static_cast<int32_t>(bucket);
            io.list.bucketFirst[b] = at;
        }
        __syncthreads();
        for (int32_t i = threadIdx.x; i < pieces; i += kFinishThreads) {
            io.list.pieceBucket[at + i] = static_cast<int32_t>(bucket);
            io.list.pieceNo[at + i] = i;
        }
        return;
    }
    FinishPiece<kFinishThreads, Keys, VB, false, Tops>(lds, io, first, len, bucket, nullptr);
}

// The first position and the length of piece `i` of the list.
__device__ __forceinline__ int32_t FinishPieceAt(const FinishIo &io, int32_t i, uint32_t *bucket, int32_t *len)
{
    *bucket = static_cast<uint32_t>(io.list.pieceBucket[i]);
    const int32_t first = io.starts[*bucket * io.startStride];
    const int64_t all = io.starts[(*bucket + 1) * io.startStride] - first;
    const int64_t pieces = (all + kFinishMost - 1) / kFinishMost, no = io.list.pieceNo[i];
    const int32_t from = static_cast<int32_t>(all * no / pieces);  // (pieces of about the same length)
    *len = static_cast<int32_t>(all * (no + 1) / pieces) - from;
    return first + from;
}

__global__ __launch_bounds__(kFinishThreads) void FinishCountKernel(FinishIo io)
{
    __shared__ int32_t hist[1 << kFinishMaxBits];
    const int32_t digits = 1 << io.low, pieces = *io.list.pieces;
    for (int32_t piece = blockIdx.x; piece < pieces; piece += gridDim.x) {
        for (int32_t d = threadIdx.x; d < digits; d += kFinishThreads) {
            hist[d] = 0;
        }
        uint32_t bucket;
        int32_t len;
        const int32_t first = FinishPieceAt(io, piece, &bucket, &len);
        // all loads ahead of the LDS atomics; an entry past the end reads the last one and counts for nothing
        uint64_t rec[kFinishItems];
#pragma unroll
        for (int i = 0; i < kFinishItems; ++i) {
            const int32_t at = i * kFinishThreads + threadIdx.x;
            rec[i] = io.recs[static_cast<int64_t>(first) + (at < len ? at : len - 1)];
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < kFinishItems; ++i) {
            const int32_t at = i * kFinishThreads + threadIdx.x;
            atomicAdd(&hist[FinishDigit(rec[i], io.payBits, digits - 1)], at < len ? 1 : 0);
        }
        __syncthreads();
        for (int32_t d = threadIdx.x; d < digits; d += kFinishThreads) {
            io.list.table[(static_cast<int64_t>(piece) << io.low) + d] = hist[d];
        }
        __syncthreads();
    }
}

// The table's counts become positions, and the offsets of the bucket's keys are known.  A workgroup a bucket; its threads
// share the pieces of a digit out among them.
__global__ __launch_bounds__(kFinishScanThreads) void FinishScanKernel(FinishIo io)
{
    __shared__ int32_t sums[kFinishScanThreads];   // [part][digit]
    __shared__ int32_t begins[1 << kFinishMaxBits];
    __shared__ int32_t waveSums[kFinishScanThreads / kWave];
    const int32_t digits = 1 << io.low, buckets = *io.list.buckets, tid = threadIdx.x;
    const int32_t parts = kFinishScanThreads >> io.low, d = tid & (digits - 1), part = tid >> io.low;
    for (int32_t b = blockIdx.x; b < buckets; b += gridDim.x) {
        const uint32_t bucket = static_cast<uint32_t>(io.list.bucketOf[b]);
        const int32_t first = io.starts[bucket * io.startStride];
        const int32_t len = io.starts[(bucket + 1) * io.startStride] - first;
        const int64_t pieces = (len - 1) / kFinishMost + 1;
        const int64_t from = pieces * part / parts, to = pieces * (part + 1) / parts;
        int32_t *mine = io.list.table + (static_cast<int64_t>(io.list.bucketFirst[b]) << io.low) + d;
        int32_t sum = 0;
#pragma unroll 8
        for (int64_t p = from; p < to; ++p) {
            sum += mine[p << io.low];
        }
        sums[tid] = sum;
        __syncthreads();
        int32_t total = 0;
        if (tid < digits) {
            for (int32_t q = 0; q < parts; ++q) {
                total += sums[(q << io.low) + d];
            }
        }
        const int32_t begin = first + WideBlockScan<kFinishScanThreads>(total, waveSums);
        if (tid < digits) {
            begins[d] = begin;
            const int64_t k = (static_cast<int64_t>(bucket) << io.low) + d;
            if (k <= io.numKeys) {
                io.ptr[k] = io.base + begin;
            }
        }
        if (io.rowCounters != nullptr) {
            // the rows of a bucket in pieces are left to csrsort's kernels
            const bool isMid = tid < digits && total > 1 && total <= kSortWaveRow, isLong = tid < digits && total > kSortWaveRow;
            const int32_t lane = tid % kWave;
#pragma unroll
            for (int list = 0; list < 2; ++list) {
                const uint64_t in = __ballot(list == 0 ? isMid : isLong);
                if (in != 0) {
                    int32_t at = lane == 0 ? atomicAdd(io.rowCounters + list, __popcll(in)) : 0;
                    at = __shfl(at, 0, kWave);
                    if ((in >> lane & 1) != 0) {
                        (list == 0 ? io.midList : io.longList)[at + __popcll(in & ((uint64_t{1} << lane) - 1))] =
                            static_cast<int32_t>(bucket << io.low) + d;
                    }
                }
            }
        }
        __syncthreads();
        int32_t run = begins[d];
        for (int32_t q = 0; q < part; ++q) {
            run += sums[(q << io.low) + d];
        }
#pragma unroll 8
        for (int64_t p = from; p < to; ++p) {
            const int32_t count = mine[p << io.low];
            mine[p << io.low] = run;
            run += count;
        }
        __syncthreads();
    }
}

template <bool Keys, int VB, int Lanes, bool Tops>
__global__ __launch_bounds__(kFinishLargeThreads) void FinishListsKernel(FinishIo io)
{
    __shared__ FinishLds<kFinishLargeThreads, true, Lanes> lds;
    const int32_t large = *io.list.large, pieces = *io.list.pieces;
    for (int32_t i = blockIdx.x; i < large; i += gridDim.x) {
        const int32_t bucket = io.list.largeOf[i];
        const int32_t first = io.starts[bucket * io.startStride];
        FinishPiece<kFinishLargeThreads, Keys, VB, false, Tops>(lds, io, first,
                                                                io.starts[(bucket + 1) * io.startStride] - first,
                                                                static_cast<uint32_t>(bucket), nullptr);
        LdsBarrier();
    }
    for (int32_t piece = blockIdx.x; piece < pieces; piece += gridDim.x) {
        uint32_t bucket;
        int32_t len;
        const int32_t first = FinishPieceAt(io, piece, &bucket, &len);
        FinishPiece<kFinishLargeThreads, Keys, VB, true, Tops>(lds, io, first, len, bucket,
                                                               io.list.table + (static_cast<int64_t>(piece) << io.low));
        LdsBarrier();
    }
}

// Where the buckets of two passes begin, without a look at every key: between the passes the entries with lower digit dl are
// one stretch, and of those with upper digit dh the second pass puts as many in front of (dh, dl) as its table has for the
// tiles in front of the stretch, and as lie in the stretch's first tile in front of it.  A workgroup a lower digit.
// `upper`: the digits that the second pass read; starts[buckets] = n and the lists' lengths = 0 come from here, too.
__global__ __launch_bounds__(kFinishScanThreads) void FinishStartsKernel(const uint8_t *__restrict__ upper, int64_t n,
                                                                    int64_t tile, int64_t numTiles,
                                                                    int32_t lowerBits, int32_t upperBits,
                                                                    const int32_t *__restrict__ lowerPrefix,
                                                                    const int32_t *__restrict__ upperPrefix,
                                                                    int32_t *__restrict__ starts, FinishList list)
{
    __shared__ int32_t hist[1 << kWideMaxBits];
    const int32_t digits = 1 << upperBits;
    for (int32_t d = threadIdx.x; d < digits; d += kFinishScanThreads) {
        hist[d] = 0;
    }
    __syncthreads();
    const int64_t stretch = lowerPrefix[static_cast<int64_t>(blockIdx.x) * numTiles];
    const int64_t t = stretch / tile;
    // (all loads of a turn ahead of the LDS atomics)
    for (int64_t i0 = t * tile; i0 < stretch; i0 += kWideItems * kFinishScanThreads) {
        uint32_t digit[kWideItems];
#pragma unroll
        for (int j = 0; j < kWideItems; ++j) {
            const int64_t i = i0 + j * kFinishScanThreads + threadIdx.x;
            digit[j] = upper[i < stretch ? i : stretch - 1];
        }
#pragma unroll
        for (int j = 0; j < kWideItems; ++j) {
            const int64_t i = i0 + j * kFinishScanThreads + threadIdx.x;
            atomicAdd(&hist[digit[j] & static_cast<uint32_t>(digits - 1)], i < stretch ? 1 : 0);
        }
    }
    __syncthreads();
    for (int32_t d = threadIdx.x; d < digits; d += kFinishScanThreads) {
        // (t may be numTiles, behind the last entry: that is where the next digit's first tile stands in the table)
        starts[(static_cast<int64_t>(d) << lowerBits) + blockIdx.x] =
            upperPrefix[static_cast<int64_t>(d) * numTiles + t] + hist[d];
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        starts[int64_t{1} << (lowerBits + upperBits)] = static_cast<int32_t>(n);
    }
    if (blockIdx.x == 0 && threadIdx.x < kFinishLengths) {
        list.large[threadIdx.x] = 0;
    }
}

// A group of G lanes per row: rows of 2..G entries are sorted in registers (bitonic
// network over the group's lanes); rows of up to 64 entries that do not fit the
// group go to midList (one wavefront each, next kernel), longer rows to longList.
// counters[0] / counters[1] are the two list lengths.  A group takes kSortRowsPerGroup consecutive rows and loads
// all of them before it sorts the first: with a row a group, a wavefront's life was one round trip to memory for
// the offsets, one for the entries and a store, and a million such wavefronts waited more than they moved.
constexpr int kSortRowsPerGroup = 8;

template <int G, bool Packed>
__global__ __launch_bounds__(kBlockThreads, 8) void SortShortRowsKernel(const int32_t *__restrict__ rowPtr, int64_t m,
                                                                       int64_t nnz, int32_t base, int32_t *colInd,
                                                                       int32_t *perm, int32_t *counters,
                                                                       int32_t *__restrict__ midList,
                                                                       int32_t *__restrict__ longList)
{
    constexpr int R = kSortRowsPerGroup;
    constexpr int kWaveRows = kWave / G * R;  // rows of a wavefront
    const int32_t g = threadIdx.x % G;
    const int64_t row0 = (static_cast<int64_t>(blockIdx.x) * (kBlockThreads / G) + threadIdx.x / G) * R;
    int32_t off[R + 1];
#pragma unroll
    for (int r = 0; r <= R; ++r) {
        off[r] = rowPtr[row0 + r <= m ? row0 + r : m];  // (rowPtr has m + 1 entries)
    }
    int64_t begin[R], len[R];
    int32_t col[R], pay[R];
    // The wavefront's rows for midList from the front, for longList from the back; how many.
    __shared__ int32_t listed[kBlockThreads / kWave][kWaveRows];
    __shared__ int32_t counts[kBlockThreads / kWave][2];
    const int32_t lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
    int32_t nMid = 0, nLong = 0;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int64_t row = row0 + r;
        begin[r] = 0;
        len[r] = 0;
        if (row < m) {
            begin[r] = static_cast<int64_t>(off[r]) - base;
            len[r] = static_cast<int64_t>(off[r + 1]) - base - begin[r];
            if (len[r] <= 1 || begin[r] < 0 || begin[r] + len[r] > nnz) {
                len[r] = 0;  // nothing to sort, or bounds that do not describe a range of the arrays
            }
        }
        if (__ballot(len[r] > G) != 0) {
            const bool mid = g == 0 && len[r] > G && len[r] <= kSortWaveRow, isLong = g == 0 && len[r] > kSortWaveRow;
            const uint64_t inMid = __ballot(mid), inLong = __ballot(isLong), below = (uint64_t{1} << lane) - 1;
            if (mid) {
                listed[wave][nMid + __popcll(inMid & below)] = static_cast<int32_t>(row);
            } else if (isLong) {
                listed[wave][kWaveRows - 1 - nLong - __popcll(inLong & below)] = static_cast<int32_t>(row);
            }
            nMid += __popcll(inMid);
            nLong += __popcll(inLong);
            len[r] = len[r] > G ? 0 : len[r];
        }
        col[r] = 0;
        pay[r] = 0;
        if (g < len[r]) {
            col[r] = colInd[begin[r] + g];
            pay[r] = perm[begin[r] + g];
        }
    }
    // The workgroup's rows take their places in the lists with one addition a list, while the entries are on their way.
    // An addition a row, to the same two words, was served one after the other, 10 ns each (33 M entries, 4.4 random ones a
    // row, of which 4 % of the rows do not fit eight lanes: 3116 us, 422 now).  Behind the sort, with barriers that wait for
    // its stores, this cost equal rows up to 8 % (2 M rows of 13: 156 us without any lists, 167, 158 now; 4 M of 5: 135,
    // 145, 136); with counters in LDS and the work left to the wavefront that arrives last, half as much.  So a wavefront has a
    // piece of LDS and counts of its own, and one barrier, of LDS alone, is all they share.  Eight wavefronts a SIMD, as
    // without lists.
    if (lane < 2) {
        counts[wave][lane] = lane == 0 ? nMid : nLong;
    }
    LdsBarrier();
    if (wave < 2) {
        // wavefront 0 writes midList, wavefront 1 longList
        int32_t all = 0;
#pragma unroll 1
        for (int w = 0; w < kBlockThreads / kWave; ++w) {
            all += counts[w][wave];
        }
        if (all > 0) {
            int32_t at = 0;
            if (lane == 0) {
                at = atomicAdd(counters + wave, all);
            }
            at = __shfl(at, 0);
#pragma unroll 1
            for (int w = 0; w < kBlockThreads / kWave; ++w) {
                const int32_t n = counts[w][wave];
                for (int32_t i = lane; i < n; i += kWave) {
                    (wave == 0 ? midList : longList)[at + i] = listed[w][wave == 0 ? i : kWaveRows - 1 - i];
                }
                at += n;
            }
        }
    }
    // every lane takes part in the shuffles; groups without a row sort padding
#pragma unroll
    for (int r = 0; r < R; ++r) {
        SortHeldRow<G, Packed>(g < len[r], g, &col[r], &pay[r]);
        if (g < len[r]) {
            colInd[begin[r] + g] = col[r];
            perm[begin[r] + g] = pay[r];
        }
    }
}

// Wavefronts walk midList: rows of up to 64 entries, one wavefront each.
template <bool Packed>
__global__ __launch_bounds__(kBlockThreads) void SortMidRowsKernel(const int32_t *__restrict__ rowPtr, int32_t base,
                                                                  int32_t *colInd, int32_t *perm,
                                                                  const int32_t *__restrict__ counters,
                                                                  const int32_t *__restrict__ midList)
{
    const int32_t lane = threadIdx.x % kWave;
    const int32_t count = counters[0];
    const int32_t wavesInGrid = gridDim.x * (kBlockThreads / kWave);
    for (int32_t item = blockIdx.x * (kBlockThreads / kWave) + threadIdx.x / kWave; item < count; item += wavesInGrid) {
        const int32_t row = midList[item];
        const int64_t begin = static_cast<int64_t>(rowPtr[row]) - base;
        const int64_t len = static_cast<int64_t>(rowPtr[row + 1]) - base - begin;
        SortRowInGroup<kWave, Packed>(begin, len, lane, colInd, perm);
    }
}

// Workgroups walk the list of rows longer than 64 entries.  Up to 2048 entries:
// bitonic sort of the keys in LDS.  Longer: a workgroup-local radix sort, four
// bits a pass, between the row and its place in the scratch arrays; thread t
// owns the t-th contiguous part of the row, so the same counter scan as in
// RadixScatterKernel keeps it stable.
template <int kThreads>
__global__ __launch_bounds__(kThreads) void SortListedRowsKernel(const int32_t *__restrict__ rowPtr, int32_t base,
                                                                     int32_t keyBits, int32_t *colInd, int32_t *perm,
                                                                     int32_t *tmpCol, int32_t *tmpPerm,
                                                                     int32_t *listCounts, const int32_t *__restrict__ list,
                                                                     int32_t countSlot, int64_t lenTo,
                                                                     int32_t *__restrict__ longerList)
{
    __shared__ uint64_t keys[kSortLdsRow];                          // 16 KB, doubles as the radix counters
    __shared__ int32_t pays[kSortLdsRow];
    static_assert(sizeof(uint64_t) * kSortLdsRow >= sizeof(int32_t) * 2 * (kThreads / kWave) * kRadixDigits, "counter space");
    int32_t *counters = reinterpret_cast<int32_t *>(keys);

    const int32_t count = listCounts[countSlot];
    for (int32_t item = blockIdx.x; item < count; item += gridDim.x) {
        const int32_t row = list[item];
        const int64_t begin = static_cast<int64_t>(rowPtr[row]) - base;
        const int64_t len = static_cast<int64_t>(rowPtr[row + 1]) - base - begin;
        if (len > lenTo) {
            // too long for this launch: listed for the next one, which runs with more lanes per row
            if (threadIdx.x == 0) {
                longerList[atomicAdd(&listCounts[2], 1)] = row;
            }
            continue;
        }
        if (len <= kSortLdsRow) {
            int32_t npad = 128;
            while (npad < len) {
                npad <<= 1;
            }
            for (int32_t i = threadIdx.x; i < npad; i += kThreads) {
                keys[i] = i < len ? SortKey(colInd[begin + i], static_cast<uint32_t>(i)) : ~0ull;
                pays[i] = i < len ? perm[begin + i] : 0;
            }
            __syncthreads();
            for (int32_t k = 2; k <= npad; k <<= 1) {
                for (int32_t j = k >> 1; j > 0; j >>= 1) {
                    for (int32_t i = threadIdx.x; i < npad; i += kThreads) {
                        const int32_t partner = i ^ j;
                        if (partner > i) {
                            const uint64_t a = keys[i], b = keys[partner];
                            const bool ascending = (i & k) == 0;
                            if ((a > b) == ascending) {
                                keys[i] = b;
                                keys[partner] = a;
                            }
                        }
                    }
                    __syncthreads();
                }
            }
            for (int32_t i = threadIdx.x; i < len; i += kThreads) {
                const uint64_t key = keys[i];
                colInd[begin + i] = SortKeyColumn(key);
                perm[begin + i] = pays[static_cast<uint32_t>(key & 0xffffffffu)];
            }
            __syncthreads();
            continue;
        }
        // Stable 4-bit radix passes over [begin, begin + len) between the row and the scratch arrays.  Wavefront w
        // owns the w-th quarter of the row and walks it 64 consecutive entries at a time, so every load is
        // coalesced.  Counting pass: per-lane digit counts, added up over the wavefront.  Then the first output
        // slot of every (digit, wavefront), digit-major, so that equal digits keep their order.  Scatter pass: the
        // lanes of a round that hold the same digit are found with four ballots, the rank among them is a population
        // count, and a running count per digit carries on from round to round.
        constexpr int kWaves = kThreads / kWave;
        constexpr int kRounds = 8;  // rounds whose loads are issued together
        int32_t *waveDigit = counters;                        // [kWaves][kRadixDigits] counts, then first slots
        int32_t *running = counters + kWaves * kRadixDigits;  // [kWaves][kRadixDigits] entries placed so far
        const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
        const uint64_t below = (uint64_t{1} << lane) - 1;
        const int64_t quarter = (len + kWaves - 1) / kWaves;
        const int64_t lo = begin + wave * quarter < begin + len ? begin + wave * quarter : begin + len;
        const int64_t hi = lo + quarter < begin + len ? lo + quarter : begin + len;
        int32_t *srcCol = colInd, *srcPerm = perm, *dstCol = tmpCol, *dstPerm = tmpPerm;
        for (int32_t shift = 0; shift < keyBits; shift += kRadixBits) {
            int32_t cnt[kRadixDigits];
#pragma unroll
            for (int d = 0; d < kRadixDigits; ++d) {
                cnt[d] = 0;
            }
            for (int64_t p0 = lo + lane; p0 < hi; p0 += kRounds * kWave) {
                int32_t c[kRounds];
#pragma unroll
                for (int u = 0; u < kRounds; ++u) {  // the loads of kRounds rounds issued together
                    const int64_t p = p0 + u * kWave;
                    c[u] = p < hi ? srcCol[p] : -1;
                }
#pragma unroll
                for (int u = 0; u < kRounds; ++u) {
                    const int32_t dg = p0 + u * kWave < hi ? RadixDigit(c[u] - base, shift) : -1;
#pragma unroll
                    for (int d = 0; d < kRadixDigits; ++d) {
                        cnt[d] += (dg == d) ? 1 : 0;
                    }
                }
            }
#pragma unroll
            for (int d = 0; d < kRadixDigits; ++d) {
                int32_t c = cnt[d];
#pragma unroll
                for (int off = kWave / 2; off > 0; off >>= 1) {
                    c += __shfl_xor(c, off, kWave);
                }
                if (lane == 0) {
                    waveDigit[wave * kRadixDigits + d] = c;
                    running[wave * kRadixDigits + d] = 0;
                }
            }
            __syncthreads();
            if (threadIdx.x == 0) {  // 64 numbers: first slot of (digit, wavefront), digit-major
                int32_t run = 0;
                for (int d = 0; d < kRadixDigits; ++d) {
                    for (int w = 0; w < kWaves; ++w) {
                        const int32_t c = waveDigit[w * kRadixDigits + d];
                        waveDigit[w * kRadixDigits + d] = run;
                        run += c;
                    }
                }
            }
            __syncthreads();
            for (int64_t p0 = lo; p0 < hi; p0 += kRounds * kWave) {
                int32_t c[kRounds], pv[kRounds];
                bool valid[kRounds];
#pragma unroll
                for (int u = 0; u < kRounds; ++u) {
                    const int64_t p = p0 + u * kWave + lane;
                    valid[u] = p < hi;
                    c[u] = valid[u] ? srcCol[p] : 0;
                    pv[u] = valid[u] ? srcPerm[p] : 0;
                }
#pragma unroll
                for (int u = 0; u < kRounds; ++u) {
                    const int32_t dg = RadixDigit(c[u] - base, shift);
                    uint64_t same = __ballot(valid[u]);
#pragma unroll
                    for (int b = 0; b < kRadixBits; ++b) {
                        const bool bit = (dg >> b) & 1;
                        const uint64_t votes = __ballot(valid[u] && bit);
                        same &= bit ? votes : ~votes;
                    }
                    const int32_t before = running[wave * kRadixDigits + dg];
                    if (valid[u]) {
                        const int64_t slot = begin + waveDigit[wave * kRadixDigits + dg] + before + __popcll(same & below);
                        dstCol[slot] = c[u];
                        dstPerm[slot] = pv[u];
                        if ((same & below) == 0) {  // the lowest lane of every digit present in this round
                            running[wave * kRadixDigits + dg] = before + __popcll(same);
                        }
                    }
                }
            }
            __threadfence_block();
            __syncthreads();
            int32_t *t = srcCol;
            srcCol = dstCol;
            dstCol = t;
            t = srcPerm;
            srcPerm = dstPerm;
            dstPerm = t;
        }
        if (srcCol != colInd) {  // an odd number of passes left the result in the scratch arrays
            for (int64_t p = begin + threadIdx.x; p < begin + len; p += kThreads) {
                colInd[p] = srcCol[p];
                perm[p] = srcPerm[p];
            }
        }
        __syncthreads();
    }
}

// =============================================================== host side

namespace {

inline int CheckLaunch()
{
    return hipGetLastError() == hipSuccess ? OPSPARSE_OK : OPSPARSE_E_LAUNCH;
}

inline int64_t Align256(int64_t v) { return (v + 255) / 256 * 256; }

inline uint32_t GridFor(int64_t items, int64_t perBlock, int64_t cap = INT32_MAX)
{
    int64_t g = (items + perBlock - 1) / perBlock;
    g = g < 1 ? 1 : g;
    return static_cast<uint32_t>(g > cap ? cap : g);
}

inline int64_t ScanTiles(int64_t count) { return (count + kScanTile - 1) / kScanTile; }

// out[i] = add + in[0..i]; `tiles` holds ScanTiles(count) ints.
void LaunchInclusiveScan(const int32_t *in, int32_t *out, int64_t count, int32_t add, int32_t *tiles, hipStream_t s)
{
    if (count <= 0) {
        return;
    }
    if (count <= kScanOneMost) {
        hipLaunchKernelGGL(ScanOneKernel, dim3(1), dim3(kScanOneThreads), 0, s, in, out, count, add);
        return;
    }
    const int64_t numTiles = ScanTiles(count);
    hipLaunchKernelGGL(ScanTileSumsKernel, dim3(static_cast<uint32_t>(numTiles)), dim3(kBlockThreads), 0, s, in, count,
                       tiles);
    const auto grid = dim3(static_cast<uint32_t>(numTiles));
    if (numTiles <= kScanSumsMost) {
        hipLaunchKernelGGL(ScanApplyKernel<true>, grid, dim3(kBlockThreads), 0, s, in, out, count, tiles, add);
        return;
    }
    hipLaunchKernelGGL(ScanTileOffsetsKernel, dim3(1), dim3(kBlockThreads), 0, s, tiles, numTiles);
    hipLaunchKernelGGL(ScanApplyKernel<false>, grid, dim3(kBlockThreads), 0, s, in, out, count, tiles, add);
}

void LaunchFill(int32_t *p, int64_t n, int32_t v, hipStream_t s)
{
    if (n > 0) {
        hipLaunchKernelGGL(FillI32Kernel, dim3(GridFor(n, kBlockThreads, 8192)), dim3(kBlockThreads), 0, s, p, n, v);
    }
}

}  // namespace

int64_t ScanScratchInts(int64_t count) { return count <= 0 ? 0 : ScanTiles(count); }

void LaunchInclusiveScanI32(const int32_t *in, int32_t *out, int64_t count, int32_t add, int32_t *scratch, hipStream_t s)
{
    LaunchInclusiveScan(in, out, count, add, scratch, s);
}

void LaunchFillI32(int32_t *p, int64_t n, int32_t v, hipStream_t s)
{
    LaunchFill(p, n, v, s);
}

void LaunchExpandRows(const int32_t *rowPtr, int64_t m, int64_t nnz, int32_t base, int32_t *rowInd, hipStream_t s)
{
    if (m > 0 && nnz > 0) {
        hipLaunchKernelGGL(ExpandRowsKernel, dim3(GridFor(m, kBlockThreads)), dim3(kBlockThreads), 0, s, rowPtr, m, nnz,
                           base, rowInd);
    }
}

int64_t RadixTiles(int64_t n) { return (n + kRadixTile - 1) / kRadixTile; }
int64_t RadixTableInts(int64_t n) { return static_cast<int64_t>(kRadixDigits) * RadixTiles(n) + 1; }

void LaunchRadixPass(const int32_t *keysIn, const int32_t *payIn, int32_t *keysOut, int32_t *payOut, int64_t n,
                     int32_t keyBase, int32_t shift, int32_t *table, int32_t *scratch, hipStream_t s)
{
    if (n <= 0) {
        return;
    }
    const int64_t numTiles = RadixTiles(n);
    const auto grid = dim3(static_cast<uint32_t>(numTiles));
    LaunchFill(table, 1, 0, s);
    hipLaunchKernelGGL(RadixCountKernel, grid, dim3(kBlockThreads), 0, s, keysIn, n, keyBase, shift, table, numTiles);
    LaunchInclusiveScan(table, table, RadixTableInts(n), 0, scratch, s);
    hipLaunchKernelGGL(RadixScatterKernel<kPayIndex>, grid, dim3(kBlockThreads), 0, s, keysIn,
                       static_cast<const void *>(payIn), keysOut, static_cast<void *>(payOut), n, keyBase, shift, table,
                       numTiles, RadixPairIo{});
}

// The same pass carrying csr2csc's (row, value) pairs: mode is one of the pair modes of RadixPayload.
void LaunchRadixPairPass(int mode, const int32_t *keysIn, const void *pairsIn, int32_t *keysOut, void *pairsOut,
                         int64_t n, int32_t keyBase, int32_t shift, int32_t *table, int32_t *scratch,
                         const RadixPairIo &io, hipStream_t s)
{
    if (n <= 0) {
        return;
    }
    const int64_t numTiles = RadixTiles(n);
    const auto grid = dim3(static_cast<uint32_t>(numTiles));
    LaunchFill(table, 1, 0, s);
    hipLaunchKernelGGL(RadixCountKernel, grid, dim3(kBlockThreads), 0, s, keysIn, n, keyBase, shift, table, numTiles);
    LaunchInclusiveScan(table, table, RadixTableInts(n), 0, scratch, s);
    switch (mode) {
        case kPayPairFirst:
            hipLaunchKernelGGL(RadixScatterKernel<kPayPairFirst>, grid, dim3(kBlockThreads), 0, s, keysIn, pairsIn,
                               keysOut, pairsOut, n, keyBase, shift, table, numTiles, io);
            break;
        case kPayPairLast:
            hipLaunchKernelGGL(RadixScatterKernel<kPayPairLast>, grid, dim3(kBlockThreads), 0, s, keysIn, pairsIn,
                               keysOut, pairsOut, n, keyBase, shift, table, numTiles, io);
            break;
        default:
            hipLaunchKernelGGL(RadixScatterKernel<kPayPair>, grid, dim3(kBlockThreads), 0, s, keysIn, pairsIn, keysOut,
                               pairsOut, n, keyBase, shift, table, numTiles, io);
            break;
    }
}

// Threads of the wide pass' workgroups.  Large ones write long runs, small ones occupy the chip with few entries (csr2csc
// of 2.7 M entries: 171 us with 1024 threads, 125 with 512, 134 with 256; of 250 K: 99, 86 and 68; of 33.5 M: 790, 870
// and 980).
int WideThreads(int64_t n)
{
    return n >= (int64_t{1} << 23) ? 1024 : n >= (int64_t{1} << 20) ? 512 : 256;
}
int64_t WideTiles(int64_t n)
{
    const int64_t tile = static_cast<int64_t>(WideThreads(n)) * kWideItems;
    return (n + tile - 1) / tile;
}
// Room for the table of a pass of ten bits, and for the two of the passes that leave records (PackTiles), a total behind each.
int64_t WideTableInts(int64_t n) { return (WideTiles(n) << kWideMaxBits) + 2; }

// ... of the passes that leave records.  Half as many as the other passes of many entries have: two workgroups a compute unit,
// one of which loads while the other orders, and runs that are as long, in bytes, as theirs of three arrays (17 M triples over 1 M
// rows 865 us with 1024, 777 with 512; 33.5 M 2032 and 2029; 3.3 M over 300 000 with 256 707, with 512 626).  With tops, whose keys
// have many buckets, the run of a tile in one of them is a line with 1024 and half of one with 512: csr2csc of 12 M entries over
// 8.4 M columns 426 us with 1024, 377 with 512, 33.6 M over 8.4 M 781 and 771, 48 M over 12 M 959 and 1023, 80 M over 20 M 1711 and
// 1910.  Their tables have as many counts as one of ten bits of the others' at most: from 2^23 entries on twice the tiles, but nine
// bits in one pass, and eight in each of two.
int PackThreads(int64_t n, bool tops)
{
    return tops && n >= int64_t{5} << 23 ? 1024 : n >= (int64_t{1} << 20) ? 512 : 256;
}
int64_t PackTiles(int64_t n, bool tops)
{
    const int64_t tile = static_cast<int64_t>(PackThreads(n, tops)) * kWideItems;
    return (n + tile - 1) / tile;
}

// Passes of a sort of n entries over `keyBits` bits of key, and the bits each takes.  At least two: a first pass that
// reads the sources and a last one that writes the outputs.  The passes share the key's bits evenly: the fewer buckets
// a pass has, the longer the runs its tiles write.  (Nine bits at most where the workgroups are large: 20 bits of 33.5 M
// keys in three passes of 7, 775 us, against two of 10, 784; in ten bits the counts and their table cost more, too.)
struct WidePasses {
    int32_t passes, bits;
};
WidePasses WidePassesOf(int32_t keyBits, int64_t n)
{
    const int32_t most = WideThreads(n) == 1024 ? 9 : kWideMaxBits;
    const int32_t passes = keyBits <= 2 * most ? 2 : (keyBits + most - 1) / most;
    return {passes, (keyBits + passes - 1) / passes};
}

// Workgroups of the scatter pass: as many as are resident (LDS and registers).
uint32_t WideScatterBlocks(int64_t n, int threads)
{
    static const int64_t cus = [] {
        int dev = 0, count = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&count, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || count <= 0) {
            (void)hipGetLastError();
            return int64_t{256};
        }
        return static_cast<int64_t>(count);
    }();
    const int64_t resident = cus * (1024 / threads);
    const int64_t fullTiles = n / (static_cast<int64_t>(threads) * kWideItems);
    return static_cast<uint32_t>(fullTiles < 1 ? 1 : (fullTiles < resident ? fullTiles : resident));
}

// One pass carrying (row, value) pairs; table: WideTableInts(n) ints.
template <int T>
void LaunchWidePairPassOf(int mode, const int32_t *keysIn, const void *pairsIn, int32_t *keysOut, void *pairsOut,
                          int64_t n, int32_t keyBase, int32_t shift, int32_t bits, int32_t *table, int32_t *scratch,
                          const RadixPairIo &io, hipStream_t s)
{
    const int32_t mask = (1 << bits) - 1;
    const int64_t numTiles = WideTiles(n);
    const auto *pin = static_cast<const RadixPair *>(pairsIn);
    auto *pout = static_cast<RadixPair *>(pairsOut);
    hipLaunchKernelGGL(WideCountKernel<T>, dim3(static_cast<uint32_t>((numTiles + kWideCountTiles - 1) / kWideCountTiles)),
                       dim3(T), 0, s, keysIn, n, keyBase, shift, mask, table, numTiles);
    LaunchInclusiveScan(table, table, (numTiles << bits) + 1, 0, scratch, s);
    const auto grid = dim3(WideScatterBlocks(n, T));
#define OPSPARSE_WIDE_SCATTER(MODE, VB)                                                                               \
    hipLaunchKernelGGL((WideScatterKernel<T, MODE, VB>), grid, dim3(T), 0, s, keysIn, pin, keysOut, pout, n, keyBase, \
                       shift, mask, bits, table, numTiles, io)
#define OPSPARSE_WIDE_SCATTER_BY_VALUE(MODE)                                                                          \
    switch (io.valueBytes) {                                                                                          \
        case 4: OPSPARSE_WIDE_SCATTER(MODE, 4); break;                                                                \
        case 2: OPSPARSE_WIDE_SCATTER(MODE, 2); break;                                                                \
        case 1: OPSPARSE_WIDE_SCATTER(MODE, 1); break;                                                                \
        default: OPSPARSE_WIDE_SCATTER(MODE, 0); break;                                                               \
    }
    switch (mode) {
        case kPayPairFirst:
            OPSPARSE_WIDE_SCATTER_BY_VALUE(kPayPairFirst);
            break;
        case kPayPairLast:
            OPSPARSE_WIDE_SCATTER_BY_VALUE(kPayPairLast);
            break;
        default:
            OPSPARSE_WIDE_SCATTER(kPayPair, 4);
            break;
    }
#undef OPSPARSE_WIDE_SCATTER_BY_VALUE
#undef OPSPARSE_WIDE_SCATTER
}

void LaunchWidePairPass(int mode, const int32_t *keysIn, const void *pairsIn, int32_t *keysOut, void *pairsOut,
                        int64_t n, int32_t keyBase, int32_t shift, int32_t bits, int32_t *table, int32_t *scratch,
                        const RadixPairIo &io, hipStream_t s)
{
    if (n <= 0) {
        return;
    }
    const int threads = WideThreads(n);
    const auto launch = threads == 1024  ? LaunchWidePairPassOf<1024>
                        : threads == 512 ? LaunchWidePairPassOf<512>
                                         : LaunchWidePairPassOf<256>;
    launch(mode, keysIn, pairsIn, keysOut, pairsOut, n, keyBase, shift, bits, table, scratch, io, s);
}

void LaunchGatherByPosition(const int32_t *pos, const int32_t *rowOfPos, const uint32_t *srcVal, int64_t nnz,
                            int32_t *rowOut, uint32_t *valOut, hipStream_t s)
{
    if (nnz > 0) {
        hipLaunchKernelGGL(GatherByPositionKernel<uint32_t>, dim3(GridFor(nnz, kBlockThreads)), dim3(kBlockThreads), 0,
                           s, pos, rowOfPos, srcVal, nnz, rowOut, valOut);
    }
}

// ptr[0..m] from sorted (or unsorted) indices: zero, count runs, scan.
void LaunchIndicesToOffsets(const int32_t *ind, int64_t nnz, int64_t m, int32_t base, int32_t *ptr, int32_t *tiles,
                            hipStream_t s)
{
    LaunchFill(ptr, m + 1, 0, s);
    if (nnz > 0 && m > 0) {
        hipLaunchKernelGGL(CountRunsKernel, dim3(GridFor(nnz, kBlockThreads * 8)), dim3(kBlockThreads), 0, s, ind, nnz,
                           m, base, ptr);
    }
    LaunchInclusiveScan(ptr, ptr, m + 1, base, tiles, s);
}

namespace {

int32_t KeyBits(int64_t n)
{
    int32_t bits = 1;
    while (bits < 31 && (int64_t{1} << bits) < n) {
        ++bits;
    }
    return bits;
}

// How a stable sort by keys in [0, numKeys) ends in LDS: `high` upper bits in one or two passes, `low` bits at the end.
// Taken where that saves a pass, and where it saves none from 5 M entries on: the passes in front of buckets move less (triples,
// the same number of passes, plain / with buckets: 4 M over 100 000 rows 433 / 451 us, 6 M over 300 000 630 / 601, 6 M over 600 000
// 642 / 596, 9.6 M over 200 000 795 / 714).  kFinishMean leaves a fifth of the room for buckets fuller than the average (with three
// fifths, and one more bit in the passes: 33.5 M entries 683 us, 651 so); below kFinishLeast the workgroups' start and end
// outweigh their work.
struct FinishPlan {
    bool use, tops;
    int32_t passes, low, lowerBits, upperBits;
    int32_t payBits;  // of a payload in the record; `tops`: the others travel beside it
    int64_t buckets;
};
constexpr int64_t kFinishMean = kFinishMost * 4 / 5;
constexpr int64_t kFinishLeast = 512;
constexpr int64_t kFinishSamePasses = 5 << 20;
constexpr int64_t kFinishMin = 1 << 14;  // entries (the lists' room in the second pair buffer is counted from here)

FinishPlan FinishPlanWith(int64_t numKeys, int64_t n, int32_t payBits, int32_t mostLow)
{
    FinishPlan f{};
    const int32_t keyBits = KeyBits(numKeys);
    int32_t low = keyBits - 1 < mostLow ? keyBits - 1 : mostLow;
    auto mean = [&](int32_t bits) {  // entries of a bucket
        return static_cast<double>(n) * static_cast<double>(int64_t{1} << bits) / static_cast<double>(numKeys);
    };
    while (low > 0 && mean(low) > static_cast<double>(kFinishMean)) {
        --low;
    }
    const int32_t high = keyBits - low, most = WideThreads(n) == 1024 ? 9 : kWideMaxBits;
    if (n < kFinishMin || low < 1 || mean(low) < static_cast<double>(kFinishLeast) || high > 16) {
        return f;
    }
    f.tops = payBits > 32 - low;
    f.payBits = f.tops ? 32 - low : payBits;
    f.passes = high <= most ? 1 : 2;
    f.low = low;
    f.lowerBits = f.passes == 1 ? high : (high + 1) / 2;
    f.upperBits = high - f.lowerBits;
    f.buckets = int64_t{1} << high;
    const int32_t plain = WidePassesOf(keyBits, n).passes;
    f.use = f.passes < plain || (f.passes == plain && n >= kFinishSamePasses);
    return f;
}

// With tops where a word leaves a key two low bits fewer than it might have, or a pass more.  Without them, and the plain passes where those buckets are too small, csr2csc of 33.6 M entries, 8.4 M x 8.4 M, takes 909 us
// (765 with), of 80 M, 20 M x 20 M, 2440 (1680), of 1 M over 1 M columns and 5 M rows 116 (77), coosort by row of 80 M, 20 M x 20 M,
// 3450 (2120).  One bit fewer costs less than the tops: 20 M entries, 5 M x 5 M, 415 us without and 423 with.
FinishPlan FinishPlanOf(int64_t numKeys, int64_t n, int32_t payBits)
{
    const int32_t room = 32 - payBits < kFinishMaxBits ? 32 - payBits : kFinishMaxBits;
    const FinishPlan inWord = FinishPlanWith(numKeys, n, payBits, room);
    const FinishPlan most = FinishPlanWith(numKeys, n, payBits, kFinishMaxBits);
    return inWord.use && inWord.passes <= most.passes && inWord.low + 1 >= most.low ? inWord : most;
}

// Lanes per row from the mean row length: twice the mean, a power of two in [8, 64].
int SortLanes(int64_t nnz, int64_t m)
{
    const int64_t mean2 = 2 * nnz / m;
    return mean2 <= 8 ? 8 : mean2 <= 16 ? 16 : mean2 <= 32 ? 32 : 64;
}

// Are columns below n, and a lane of so many, one 32-bit key?
bool SortPacked(int64_t n, int64_t indexBase, int lanes)
{
    int log = 0;
    while ((1 << log) < lanes) {
        ++log;
    }
    return n + indexBase < (int64_t{1} << (32 - log)) - 1;
}

// The rows of longList.  Of up to kSortWideRow entries: 256 lanes each, many rows at a time.  The few beyond: 1024 lanes
// each, because the longest of them is what the call waits for (a row of 1 M entries 12.5 -> 6 ms).
// (the list of the mid rows has been used up by then: its space takes the rows handed on)
void LaunchSortListedRows(const int32_t *rowPtr, int32_t base, int64_t n, int32_t *colInd, int32_t *perm, int32_t *tmpCol,
                          int32_t *tmpPerm, int32_t *counters, int32_t *midList, const int32_t *longList, hipStream_t s)
{
    hipLaunchKernelGGL(SortListedRowsKernel<kBlockThreads>, dim3(kSortListBlocks), dim3(kBlockThreads), 0, s, rowPtr, base,
                       KeyBits(n), colInd, perm, tmpCol, tmpPerm, counters, longList, 1, int64_t{kSortWideRow}, midList);
    hipLaunchKernelGGL(SortListedRowsKernel<1024>, dim3(kSortListBlocks / 4), dim3(1024), 0, s, rowPtr, base, KeyBits(n),
                       colInd, perm, tmpCol, tmpPerm, counters, midList, 2, int64_t{INT32_MAX},
                       static_cast<int32_t *>(nullptr));
}

template <int T, int Mode, bool Tops>
void LaunchPackPassOf(const PackIo &io, int32_t valueBytes, int32_t shift, int32_t bits, int32_t *table, int32_t *scratch,
                      hipStream_t s)
{
    const int32_t mask = (1 << bits) - 1;
    const int64_t numTiles = PackTiles(io.n, Tops);
    const auto counts = dim3(static_cast<uint32_t>((numTiles + kWideCountTiles - 1) / kWideCountTiles));
    if (Mode == kPackSecond) {
        hipLaunchKernelGGL(DigitCountKernel<T>, counts, dim3(T), 0, s, io.digitsIn, io.n, mask, table, numTiles);
    } else {
        hipLaunchKernelGGL(WideCountKernel<T>, counts, dim3(T), 0, s, io.keys, io.n, io.keyBase, shift, mask, table, numTiles);
    }
    LaunchInclusiveScan(table, table, (numTiles << bits) + 1, 0, scratch, s);
    auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(WideScatterBlocks(io.n, T)), dim3(T), 0, s, io, shift, mask, bits, table, numTiles);
    };
    if constexpr (Mode == kPackSecond) {
        launch(PackScatterKernel<T, Mode, 4, Tops>);
    } else {
        switch (valueBytes) {
            case 4: launch(PackScatterKernel<T, Mode, 4, Tops>); break;
            case 2: launch(PackScatterKernel<T, Mode, 2, Tops>); break;
            case 1: launch(PackScatterKernel<T, Mode, 1, Tops>); break;
            default: launch(PackScatterKernel<T, Mode, 0, Tops>); break;
        }
    }
}

// One pass of a sort that ends in LDS; table: WideTableInts(n) ints.
template <int Mode>
void LaunchPackPass(const PackIo &io, int32_t valueBytes, int32_t shift, int32_t bits, int32_t *table, int32_t *scratch,
                    hipStream_t s)
{
    const bool tops = io.topsOut != nullptr;
    const int threads = PackThreads(io.n, tops);
    auto launch = tops ? (threads == 256 ? LaunchPackPassOf<256, Mode, true> : LaunchPackPassOf<512, Mode, true>)
                       : (threads == 256 ? LaunchPackPassOf<256, Mode, false> : LaunchPackPassOf<512, Mode, false>);
    if constexpr (Mode != kPackOnly) {  // (so many entries take two passes)
        launch = threads == 1024 ? LaunchPackPassOf<1024, Mode, true> : launch;
    }
    launch(io, valueBytes, shift, bits, table, scratch, s);
}

struct FinishSort {
    const int32_t *keysIn;  // keyBase + key
    int32_t keyBase;
    RadixPairIo io;         // the first pass's sources and the outputs
    int32_t *keyOut;        // coosort's sorted keys (zero-based), or NULL
    int64_t rowBound;       // coosort: sort the entries of a key by their rows as well, which are below this; or 0
    int32_t *ptr;           // base + the first position of every key, numKeys + 1 of them
    int32_t base;
    int64_t n, numKeys;
};

// keys[], pairs[]: 4 n and 8 n bytes each; table: WideTableInts(n).  The entries pass through the first of the buffers and
// lie in the second when the last kernels start, whose lists then use the first pair buffer; `ptr` may be keys[0].
void LaunchFinishSort(const FinishSort &sort, const FinishPlan &plan, int32_t *const *keys, void *const *pairs,
                      int32_t *table, int32_t *scratch, hipStream_t s)
{
    const int64_t n = sort.n, numTiles = PackTiles(n, plan.tops), most = n / kFinishMost + 1;  // (buckets on a list: fewer)
    FinishIo io{};
    auto *at = static_cast<int32_t *>(pairs[0]);
    auto take = [&](int64_t ints) {
        int32_t *p = at;
        at += ints;
        return p;
    };
    io.list.large = take(kFinishLengths);
    io.list.pieces = io.list.large + 1;
    io.list.buckets = io.list.large + 2;
    io.list.largeOf = take(most);
    io.list.pieceBucket = take(2 * most);  // a bucket in pieces has fewer than twice its entries / kFinishMost of them
    io.list.pieceNo = take(2 * most);
    io.list.bucketOf = take(most);
    io.list.bucketFirst = take(most);
    int32_t *starts = take(plan.buckets + 1);
    io.list.table = take(2 * most << plan.low);
    // Rows of two entries and more out of pieces, and rows of more than 64: fewer than n / 2 and n / 64.  (With the table,
    // a third of n, and the lists above that is less than the 2 n ints of the buffer.)
    if (sort.rowBound > 0) {
        io.rowCounters = io.list.large + 8;
        io.midList = take(n / 2);
        io.longList = take(n / kSortWaveRow);
    }
    PackIo pack{};
    pack.keys = sort.keysIn;
    pack.keyBase = sort.keyBase;
    pack.pays = sort.io.rowSrc;
    pack.vals = sort.io.valSrc;
    pack.n = n;
    pack.low = plan.low;
    pack.payBits = plan.payBits;
    pack.nextShift = plan.low + plan.lowerBits;
    auto *last = static_cast<Record *>(pairs[1]);
    // (between two passes the digits are the first n bytes of a key buffer, the tops the last 2 n)
    auto *lastTops = plan.tops ? reinterpret_cast<uint16_t *>(keys[1]) : nullptr;
    if (plan.passes == 1) {
        pack.recsOut = last;
        pack.topsOut = lastTops;
        LaunchPackPass<kPackOnly>(pack, sort.io.valueBytes, plan.low, plan.lowerBits, table, scratch, s);
        LaunchFill(io.list.large, kFinishLengths, 0, s);
        io.starts = table;
        io.startStride = numTiles;
    } else {
        // (up to eight bits each: WideTableInts has room for both tables)
        int32_t *upper = table + (numTiles << plan.lowerBits) + 1;
        auto *digits = reinterpret_cast<uint8_t *>(keys[0]);
        pack.recsOut = static_cast<Record *>(pairs[0]);
        pack.digitsOut = digits;
        pack.topsOut = plan.tops ? reinterpret_cast<uint16_t *>(digits + 2 * n) : nullptr;
        LaunchPackPass<kPackFirst>(pack, sort.io.valueBytes, plan.low, plan.lowerBits, table, scratch, s);
        pack.recsIn = pack.recsOut;
        pack.digitsIn = digits;
        pack.topsIn = pack.topsOut;
        pack.recsOut = last;
        pack.topsOut = lastTops;
        LaunchPackPass<kPackSecond>(pack, 4, 0, plan.upperBits, upper, scratch, s);
        hipLaunchKernelGGL(FinishStartsKernel, dim3(1u << plan.lowerBits), dim3(kFinishScanThreads), 0, s, digits, n,
                           static_cast<int64_t>(PackThreads(n, plan.tops)) * kWideItems, numTiles, plan.lowerBits, plan.upperBits, table,
                           upper, starts, io.list);
        io.starts = starts;
        io.startStride = 1;
    }
    io.recs = last;
    io.tops = lastTops;
    io.payBits = plan.payBits;
    io.n = n;
    io.low = plan.low;
    io.numKeys = sort.numKeys;
    io.base = sort.base;
    io.ptr = sort.ptr;
    io.keyOut = sort.keyOut;
    io.rowOut = sort.io.rowOut;
    io.valOut = sort.io.valOut;
    // a workgroup a compute unit for the lists, no more than there may be buckets on them
    auto launch = [&](auto buckets, auto lists) {
        hipLaunchKernelGGL(buckets, dim3(static_cast<uint32_t>(plan.buckets)), dim3(kFinishThreads), 0, s, io);
        hipLaunchKernelGGL(FinishCountKernel, dim3(GridFor(2 * most, 1, 512)), dim3(kFinishThreads), 0, s, io);
        hipLaunchKernelGGL(FinishScanKernel, dim3(GridFor(most, 1, 512)), dim3(kFinishScanThreads), 0, s, io);
        hipLaunchKernelGGL(lists, dim3(GridFor(2 * most, 1, 256)), dim3(kFinishLargeThreads), 0, s, io);
    };
    auto finish = [&](auto withTops) {
        constexpr bool Tops = decltype(withTops)::value;
        if (sort.rowBound > 0) {
            switch (SortLanes(n, sort.numKeys)) {
                case 8: launch(FinishBucketsKernel<true, 4, 8, Tops>, FinishListsKernel<true, 4, 8, Tops>); break;
                case 16: launch(FinishBucketsKernel<true, 4, 16, Tops>, FinishListsKernel<true, 4, 16, Tops>); break;
                case 32: launch(FinishBucketsKernel<true, 4, 32, Tops>, FinishListsKernel<true, 4, 32, Tops>); break;
                default: launch(FinishBucketsKernel<true, 4, 64, Tops>, FinishListsKernel<true, 4, 64, Tops>); break;
            }
        } else if (sort.keyOut != nullptr) {
            launch(FinishBucketsKernel<true, 4, 0, Tops>, FinishListsKernel<true, 4, 0, Tops>);
        } else {
            switch (sort.io.valueBytes) {
                case 4: launch(FinishBucketsKernel<false, 4, 0, Tops>, FinishListsKernel<false, 4, 0, Tops>); break;
                case 2: launch(FinishBucketsKernel<false, 2, 0, Tops>, FinishListsKernel<false, 2, 0, Tops>); break;
                case 1: launch(FinishBucketsKernel<false, 1, 0, Tops>, FinishListsKernel<false, 1, 0, Tops>); break;
                default: launch(FinishBucketsKernel<false, 0, 0, Tops>, FinishListsKernel<false, 0, 0, Tops>); break;
            }
        }
    };
    plan.tops ? finish(std::true_type{}) : finish(std::false_type{});
    if (sort.rowBound > 0) {
        // the buffers that the entries lay in are csrsort's scratch now
        hipLaunchKernelGGL(SortMidRowsKernel<true>, dim3(kSortListBlocks), dim3(kBlockThreads), 0, s, sort.ptr, sort.base,
                           sort.io.rowOut, static_cast<int32_t *>(sort.io.valOut), io.rowCounters, io.midList);
        LaunchSortListedRows(sort.ptr, sort.base, sort.rowBound, sort.io.rowOut, static_cast<int32_t *>(sort.io.valOut),
                             keys[1], static_cast<int32_t *>(pairs[1]), io.rowCounters, io.midList, io.longList, s);
    }
}

struct Csr2CscLayout {
    int64_t keysA, keysB, payA, payB, rowOfPos, table, tiles, bytes;
    int64_t tableCount;
};

Csr2CscLayout LayoutCsr2Csc(int64_t n, int64_t nnz)
{
    Csr2CscLayout l{};
    l.tableCount = WideTableInts(nnz);
    int64_t off = 0;
    const int64_t arr = Align256(4 * nnz);
    l.keysA = off; off += arr;
    l.keysB = off; off += arr;
    l.payA = off; off += Align256(8 * nnz);  // (row, value) pairs
    l.payB = off; off += Align256(8 * nnz);
    l.rowOfPos = off; off += arr;
    l.table = off; off += Align256(4 * l.tableCount);
    const int64_t scanCount = l.tableCount > n + 1 ? l.tableCount : n + 1;
    l.tiles = off; off += Align256(4 * ScanTiles(scanCount));
    l.bytes = off;
    return l;
}

}  // namespace
}  // namespace opsparse

using namespace opsparse;

extern "C" {

size_t opsparse_scan_workspace_bytes(int64_t count)
{
    return count <= 0 ? 0 : static_cast<size_t>(Align256(4 * ScanTiles(count)));
}

int opsparse_coo2csr_launch(const int32_t *cooRowInd, int64_t nnz, int64_t m, int32_t *csrRowPtr, int32_t indexBase,
                            void *workspace, size_t workspaceBytes, void *stream)
{
    if (nnz < 0 || m < 0 || nnz > INT32_MAX || m >= INT32_MAX || (indexBase != 0 && indexBase != 1) ||
        csrRowPtr == nullptr || (nnz > 0 && (cooRowInd == nullptr || m == 0))) {
        return OPSPARSE_E_INVALID;
    }
    if (workspace == nullptr || workspaceBytes < opsparse_scan_workspace_bytes(m + 1)) {
        return OPSPARSE_E_WORKSPACE;
    }
    LaunchIndicesToOffsets(cooRowInd, nnz, m, indexBase, csrRowPtr, static_cast<int32_t *>(workspace),
                           static_cast<hipStream_t>(stream));
    return CheckLaunch();
}

int opsparse_csr2coo_launch(const int32_t *csrRowPtr, int64_t nnz, int64_t m, int32_t *cooRowInd, int32_t indexBase,
                            void *stream)
{
    if (nnz < 0 || m < 0 || nnz > INT32_MAX || m > INT32_MAX || (indexBase != 0 && indexBase != 1) ||
        (m == 0 && nnz != 0) || (m > 0 && csrRowPtr == nullptr) || (nnz > 0 && cooRowInd == nullptr)) {
        return OPSPARSE_E_INVALID;
    }
    if (nnz == 0 || m == 0) {
        return OPSPARSE_OK;
    }
    hipLaunchKernelGGL(ExpandRowsKernel, dim3(GridFor(m, kBlockThreads)), dim3(kBlockThreads), 0,
                       static_cast<hipStream_t>(stream), csrRowPtr, m, nnz, indexBase, cooRowInd);
    return CheckLaunch();
}

// Rows of thousands of entries on average: too few rows to occupy the GPU with a workgroup each (one row of 4 M
// entries: 128 ms that way).  The whole matrix is then sorted with the device-wide radix passes, by column and
// after that, stably, by row, 0.1 - 0.2 ms a pass for such sizes.  The mean is known on the host; a matrix of short
// rows with single very long ones among them still takes the per-row kernels.
constexpr int64_t kSortWholeMeanRow = 4096;

static bool SortWhole(int64_t m, int64_t nnz) { return nnz / m >= kSortWholeMeanRow; }

struct SortWholeLayout {
    int64_t keysA, keysB, pairsA, pairsB, rowOfPos, table, tiles, bytes;
};

static SortWholeLayout LayoutSortWhole(int64_t nnz)
{
    SortWholeLayout l{};
    int64_t off = 0;
    l.keysA = off; off += Align256(4 * nnz);
    l.keysB = off; off += Align256(4 * nnz);
    l.pairsA = off; off += Align256(8 * nnz);
    l.pairsB = off; off += Align256(8 * nnz);
    l.rowOfPos = off; off += Align256(4 * nnz);
    l.table = off; off += Align256(4 * RadixTableInts(nnz));
    l.tiles = off; off += Align256(4 * ScanTiles(RadixTableInts(nnz)));
    l.bytes = off;
    return l;
}

size_t opsparse_csrsort_workspace_bytes(int64_t m, int64_t nnz)
{
    if (m <= 0 || nnz <= 0) {
        return 0;
    }
    if (SortWhole(m, nnz)) {
        return static_cast<size_t>(LayoutSortWhole(nnz).bytes);
    }
    return static_cast<size_t>(2 * Align256(4 * nnz) + 256 + 2 * Align256(4 * m));
}

int opsparse_csrsort_launch(int64_t m, int64_t n, int64_t nnz, int32_t indexBase, const int32_t *csrRowPtr,
                            int32_t *csrColInd, int32_t *perm, void *workspace, size_t workspaceBytes, void *stream)
{
    if (m < 0 || n < 0 || nnz < 0 || m > INT32_MAX || nnz > INT32_MAX || (indexBase != 0 && indexBase != 1) ||
        ((m == 0 || n == 0) && nnz != 0)) {
        return OPSPARSE_E_INVALID;
    }
    if (nnz == 0) {
        return OPSPARSE_OK;
    }
    if (csrRowPtr == nullptr || csrColInd == nullptr || perm == nullptr) {
        return OPSPARSE_E_INVALID;
    }
    if (workspace == nullptr || workspaceBytes < opsparse_csrsort_workspace_bytes(m, nnz)) {
        return OPSPARSE_E_WORKSPACE;
    }
    auto s = static_cast<hipStream_t>(stream);
    auto *base = static_cast<unsigned char *>(workspace);
    if (SortWhole(m, nnz)) {
        const SortWholeLayout l = LayoutSortWhole(nnz);
        auto at = [&](int64_t off) { return reinterpret_cast<int32_t *>(base + off); };
        int32_t *keys[2] = {at(l.keysA), at(l.keysB)};
        void *pairs[2] = {base + l.pairsA, base + l.pairsB};
        int32_t *rowOfPos = at(l.rowOfPos), *table = at(l.table), *tiles = at(l.tiles);
        hipLaunchKernelGGL(ExpandRowsKernel, dim3(GridFor(m, kBlockThreads)), dim3(kBlockThreads), 0, s, csrRowPtr, m,
                           nnz, indexBase, rowOfPos);  // rows numbered from indexBase: the order is what matters
        // by column, carrying (row, permutation value) ...
        const RadixPairIo in{rowOfPos, perm, nullptr, nullptr, 4};
        const int32_t colPasses = (KeyBits(n) + kRadixBits - 1) / kRadixBits;
        const int32_t *keysIn = csrColInd;
        const void *pairsIn = nullptr;
        int cur = 0;
        for (int32_t pass = 0; pass < colPasses; ++pass) {
            LaunchRadixPairPass(pass == 0 ? kPayPairFirst : kPayPair, keysIn, pairsIn, keys[cur], pairs[cur], nnz,
                                pass == 0 ? indexBase : 0, pass * kRadixBits, table, tiles, in, s);
            keysIn = keys[cur];
            pairsIn = pairs[cur];
            cur ^= 1;
        }
        // ... then, stably, by row, carrying (column, permutation value); the last pass writes both in place
        hipLaunchKernelGGL(RegroupByRowKernel, dim3(GridFor(nnz, kBlockThreads)), dim3(kBlockThreads), 0, s, keysIn,
                           static_cast<const RadixPair *>(pairsIn), nnz, indexBase, keys[cur],
                           static_cast<RadixPair *>(pairs[cur]));
        keysIn = keys[cur];
        pairsIn = pairs[cur];
        cur ^= 1;
        const RadixPairIo out{nullptr, nullptr, csrColInd, perm, 4};
        const int32_t rowPasses = (KeyBits(m + indexBase) + kRadixBits - 1) / kRadixBits;
        for (int32_t pass = 0; pass < rowPasses; ++pass) {
            LaunchRadixPairPass(pass == rowPasses - 1 ? kPayPairLast : kPayPair, keysIn, pairsIn, keys[cur], pairs[cur],
                                nnz, 0, pass * kRadixBits, table, tiles, out, s);
            keysIn = keys[cur];
            pairsIn = pairs[cur];
            cur ^= 1;
        }
        return CheckLaunch();
    }
    const int64_t arr = Align256(4 * nnz);
    auto *tmpCol = reinterpret_cast<int32_t *>(base);
    auto *tmpPerm = reinterpret_cast<int32_t *>(base + arr);
    auto *counters = reinterpret_cast<int32_t *>(base + 2 * arr);
    auto *midList = reinterpret_cast<int32_t *>(base + 2 * arr + 256);
    auto *longList = reinterpret_cast<int32_t *>(base + 2 * arr + 256 + Align256(4 * m));
    LaunchFill(counters, 3, 0, s);
    const int g = SortLanes(nnz, m);
    const auto shortGrid = dim3(GridFor(m, static_cast<int64_t>(kBlockThreads / g) * kSortRowsPerGroup));
    // 32-bit keys (column and lane packed) where the columns of a valid matrix leave room for the lane number
    auto packedFor = [&](int lanes) { return SortPacked(n, indexBase, lanes); };
#define OPSPARSE_SORT_SHORT(G, PACKED)                                                                              \
    hipLaunchKernelGGL((SortShortRowsKernel<G, PACKED>), shortGrid, dim3(kBlockThreads), 0, s, csrRowPtr, m, nnz,    \
                       indexBase, csrColInd, perm, counters, midList, longList)
#define OPSPARSE_SORT_SHORT_G(G)            \
    if (packedFor(G)) {                     \
        OPSPARSE_SORT_SHORT(G, true);       \
    } else {                                \
        OPSPARSE_SORT_SHORT(G, false);      \
    }
    switch (g) {
        case 8: OPSPARSE_SORT_SHORT_G(8); break;
        case 16: OPSPARSE_SORT_SHORT_G(16); break;
        case 32: OPSPARSE_SORT_SHORT_G(32); break;
        default: OPSPARSE_SORT_SHORT_G(64); break;
    }
#undef OPSPARSE_SORT_SHORT_G
#undef OPSPARSE_SORT_SHORT
    if (g < kSortWaveRow) {
        if (packedFor(kWave)) {
            hipLaunchKernelGGL(SortMidRowsKernel<true>, dim3(kSortListBlocks), dim3(kBlockThreads), 0, s, csrRowPtr,
                               indexBase, csrColInd, perm, counters, midList);
        } else {
            hipLaunchKernelGGL(SortMidRowsKernel<false>, dim3(kSortListBlocks), dim3(kBlockThreads), 0, s, csrRowPtr,
                               indexBase, csrColInd, perm, counters, midList);
        }
    }
    LaunchSortListedRows(csrRowPtr, indexBase, n, csrColInd, perm, tmpCol, tmpPerm, counters, midList, longList, s);
    return CheckLaunch();
}

size_t opsparse_csr2csc_workspace_bytes(int64_t m, int64_t n, int64_t nnz)
{
    if (m <= 0 || n <= 0 || nnz <= 0) {
        return 0;
    }
    return static_cast<size_t>(LayoutCsr2Csc(n, nnz).bytes);
}

int opsparse_csr2csc_launch(int64_t m, int64_t n, int64_t nnz, const void *csrVal, const int32_t *csrRowPtr,
                            const int32_t *csrColInd, void *cscVal, int32_t *cscColPtr, int32_t *cscRowInd,
                            int32_t valueBytes, int32_t indexBase, void *workspace, size_t workspaceBytes,
                            void *stream)
{
    if (m < 0 || n < 0 || nnz < 0 || m > INT32_MAX || n >= INT32_MAX || nnz > INT32_MAX - indexBase ||
        (indexBase != 0 && indexBase != 1) || ((m == 0 || n == 0) && nnz != 0) || cscColPtr == nullptr ||
        (valueBytes != 0 && valueBytes != 1 && valueBytes != 2 && valueBytes != 4)) {
        return OPSPARSE_E_INVALID;
    }
    auto s = static_cast<hipStream_t>(stream);
    if (nnz == 0) {
        LaunchFill(cscColPtr, n + 1, indexBase, s);
        return CheckLaunch();
    }
    if (csrRowPtr == nullptr || csrColInd == nullptr || cscRowInd == nullptr ||
        (valueBytes != 0 && (csrVal == nullptr || cscVal == nullptr))) {
        return OPSPARSE_E_INVALID;
    }
    const Csr2CscLayout l = LayoutCsr2Csc(n, nnz);
    if (workspace == nullptr || static_cast<int64_t>(workspaceBytes) < l.bytes) {
        return OPSPARSE_E_WORKSPACE;
    }
    auto *base = static_cast<unsigned char *>(workspace);
    auto at = [&](int64_t off) { return reinterpret_cast<int32_t *>(base + off); };
    int32_t *keys[2] = {at(l.keysA), at(l.keysB)};
    void *pairs[2] = {base + l.payA, base + l.payB};
    int32_t *rowOfPos = at(l.rowOfPos), *table = at(l.table), *tiles = at(l.tiles);

    // Row index of every source position, with the output's index base.
    hipLaunchKernelGGL(ExpandRowsKernel, dim3(GridFor(m, kBlockThreads)), dim3(kBlockThreads), 0, s, csrRowPtr, m, nnz,
                       indexBase, rowOfPos);

    // Stable sort by column of (column; row, value): the pair travels with its key, 8 bytes a pass and entry more
    // than a source position would, and the last pass writes rows and values where they belong — no gather by
    // position at the end, which cost two cache-line fills per entry (33.5 M entries: 2.9 -> 1.9 ms).
    // Up to ten bits a pass (WidePassesOf), the tile ordered through LDS before it leaves, and the last bits in LDS where
    // that saves a pass or there are many entries (33.5 M over 2^20 columns: three passes of seven bits 0.80 ms, two over packed
    // records and the last bits 0.50).
    const RadixPairIo io{rowOfPos, csrVal, cscRowInd, cscVal, valueBytes};
    const FinishPlan plan = FinishPlanOf(n, nnz, KeyBits(m + indexBase));
    if (plan.use) {
        const FinishSort sort{csrColInd, indexBase, io, nullptr, 0, cscColPtr, indexBase, nnz, n};
        LaunchFinishSort(sort, plan, keys, pairs, table, tiles, s);
        return CheckLaunch();
    }
    const auto [passes, perPass] = WidePassesOf(KeyBits(n), nnz);
    const int32_t *keysIn = csrColInd;
    const void *pairsIn = nullptr;
    int cur = 0;
    for (int32_t pass = 0; pass < passes; ++pass) {
        const int mode = pass == 0 ? kPayPairFirst : (pass == passes - 1 ? kPayPairLast : kPayPair);
        LaunchWidePairPass(mode, keysIn, pairsIn, keys[cur], pairs[cur], nnz, pass == 0 ? indexBase : 0,
                           pass * perPass, perPass, table, tiles, io, s);
        keysIn = keys[cur];
        pairsIn = pairs[cur];
        cur ^= 1;
    }

    // Column offsets from the sorted (zero-based) columns.
    LaunchFill(cscColPtr, n + 1, 0, s);
    hipLaunchKernelGGL(CountRunsKernel, dim3(GridFor(nnz, kBlockThreads * 8)), dim3(kBlockThreads), 0, s, keysIn, nnz,
                       n, 0, cscColPtr);
    LaunchInclusiveScan(cscColPtr, cscColPtr, n + 1, indexBase, tiles, s);
    return CheckLaunch();
}


// ------------------------------------------------------------------ coosort
//
// aclsparseXcoosortByRow / ByColumn (sparse/coosort/arch35/coosort_host.cpp:309-371; the order is the one of
// test/coosort/arch35/coosort_golden.h:52-85): a stable sort of (primary, secondary, P) triples, signed keys,
// ascending in the primary key and, among equal ones, in the secondary.  Least-significant-key first: the wide
// passes of csr2csc over the secondary key, the primary key and P travelling as the pair, then over the primary
// key with the secondary key and P as the pair; the last pass writes the caller's three arrays.  Where there are
// 2^20 entries or more and a sample says that they lie in short rows, the passes run over the primary key only and
// csrsort's kernels order each row in place (kRowsFirstLongest).  The keys are taken relative to their minimum,
// found on the device first, so that a pass count follows from the range the indices really span (one read-back of
// five integers, the ranges and the sample's count: the call synchronises its stream once).

}  // extern "C"

namespace opsparse {
namespace {

// range[0..3] = min / max of a[], min / max of b[] (pre-filled with INT32_MAX / INT32_MIN alternately).
__global__ __launch_bounds__(kBlockThreads) void CooRangeKernel(const int32_t *__restrict__ a,
                                                                const int32_t *__restrict__ b, int64_t n,
                                                                int32_t *__restrict__ range)
{
    int32_t lo[2] = {INT32_MAX, INT32_MAX}, hi[2] = {INT32_MIN, INT32_MIN};
    auto take = [&](int k, int32_t v) {
        lo[k] = v < lo[k] ? v : lo[k];
        hi[k] = v > hi[k] ? v : hi[k];
    };
    // four groups of four entries of each array asked for together; a group past the end re-reads the last whole one
    constexpr int kAtOnce = 4;
    const int64_t groups = n / 4, stride = static_cast<int64_t>(gridDim.x) * kBlockThreads;
    const int64_t me = static_cast<int64_t>(blockIdx.x) * kBlockThreads + threadIdx.x;
    for (int64_t i = me; i < groups; i += stride * kAtOnce) {
        Int4U v[2][kAtOnce];
#pragma unroll
        for (int j = 0; j < kAtOnce; ++j) {
            const int64_t at = i + j * stride < groups ? i + j * stride : groups - 1;
            v[0][j] = *reinterpret_cast<const Int4U *>(a + 4 * at);
            v[1][j] = *reinterpret_cast<const Int4U *>(b + 4 * at);
        }
#pragma unroll
        for (int j = 0; j < kAtOnce; ++j) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                take(0, v[0][j][e]);
                take(1, v[1][j][e]);
            }
        }
    }
    if (me < n - 4 * groups) {
        take(0, a[4 * groups + me]);
        take(1, b[4 * groups + me]);
    }
#pragma unroll
    for (int k = 0; k < 2; ++k) {
#pragma unroll
        for (int off = kWave / 2; off > 0; off >>= 1) {
            const int32_t l = __shfl_xor(lo[k], off), h = __shfl_xor(hi[k], off);
            lo[k] = l < lo[k] ? l : lo[k];
            hi[k] = h > hi[k] ? h : hi[k];
        }
    }
    // one set of atomics a workgroup (a set a wavefront of 8192 workgroups took 1.2 ms on four addresses)
    __shared__ int32_t part[kBlockThreads / kWave][4];
    if (threadIdx.x % kWave == 0) {
        int32_t *mine = part[threadIdx.x / kWave];
        mine[0] = lo[0];
        mine[1] = hi[0];
        mine[2] = lo[1];
        mine[3] = hi[1];
    }
    __syncthreads();
    if (threadIdx.x < 4) {
        int32_t v = part[0][threadIdx.x];
        for (int w = 1; w < kBlockThreads / kWave; ++w) {
            const int32_t o = part[w][threadIdx.x];
            v = (threadIdx.x & 1) ? (o > v ? o : v) : (o < v ? o : v);
        }
        if (threadIdx.x & 1) {
            atomicMax(range + threadIdx.x, v);
        } else {
            atomicMin(range + threadIdx.x, v);
        }
    }
}

// ... and range[4] = 0, counters[0 .. count) = 0 for the kernel below.
__global__ __launch_bounds__(kBlockThreads) void CooRangeInitKernel(int32_t *range, int32_t *counters, int32_t count)
{
    if (blockIdx.x == 0 && threadIdx.x < 5) {
        range[threadIdx.x] = threadIdx.x == 4 ? 0 : (threadIdx.x & 1) ? INT32_MIN : INT32_MAX;
    }
    for (int32_t i = blockIdx.x * kBlockThreads + threadIdx.x; i < count; i += gridDim.x * kBlockThreads) {
        counters[i] = 0;
    }
}

// How long are the rows that the entries lie in?  Of `samples` evenly spaced entries, range[4] = the pairs that share a
// row (a counter: the rows are hashed onto 2^bits of them): samples^2 / (2 n) x (mean row length over the entries).
__global__ __launch_bounds__(kBlockThreads) void CooSampleKernel(const int32_t *__restrict__ primary, int64_t n,
                                                                 int32_t samples, int32_t *__restrict__ counters,
                                                                 int32_t bits, int32_t *__restrict__ range)
{
    const int32_t i = blockIdx.x * kBlockThreads + threadIdx.x;
    int32_t pairs = 0;
    if (i < samples) {
        // one entry of every stretch, from a place of its own in each: entries in a periodic order (a long row at every
        // other position, triples column by column) are seen as often as they are there
        const int64_t first = static_cast<int64_t>(i) * n / samples, next = static_cast<int64_t>(i + 1) * n / samples;
        uint32_t mix = static_cast<uint32_t>(i) * 0x85EBCA6Bu;
        mix = (mix ^ (mix >> 15)) * 0xC2B2AE35u;
        const int64_t place = static_cast<int64_t>(static_cast<uint64_t>(mix) * static_cast<uint64_t>(next - first) >> 32);
        const uint32_t row = static_cast<uint32_t>(primary[first + place]);
        pairs = atomicAdd(counters + ((row * 0x9E3779B1u) >> (32 - bits)), 1);
    }
    __shared__ int32_t part[kBlockThreads / kWave];
    pairs = GroupSum<kWave>(pairs);
    if (threadIdx.x % kWave == 0) {
        part[threadIdx.x / kWave] = pairs;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        pairs = 0;
        for (int w = 0; w < kBlockThreads / kWave; ++w) {
            pairs += part[w];
        }
        atomicAdd(range + 4, pairs);
    }
}

// a[i] += addA, b[i] += addB (wrap-around: the sorted keys come back relative to their minimum).
__global__ __launch_bounds__(kBlockThreads) void CooRebaseKernel(int32_t *__restrict__ a, int32_t *__restrict__ b,
                                                                 int64_t n, int32_t addA, int32_t addB)
{
    const int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += stride) {
        a[i] = static_cast<int32_t>(static_cast<uint32_t>(a[i]) + static_cast<uint32_t>(addA));
        b[i] = static_cast<int32_t>(static_cast<uint32_t>(b[i]) + static_cast<uint32_t>(addB));
    }
}

// From this many entries on a sample of the rows is taken, and rows of up to this mean length over the entries are
// sorted by csrsort after one sort by row.
constexpr int64_t kRowsFirstMin = int64_t{1} << 20;
constexpr int32_t kRowSamples = 65536;
constexpr double kRowsFirstLongest = 50.0;

struct CoosortLayout {
    int64_t range, keysA, keysB, pairsA, pairsB, table, tiles, bytes;
};

CoosortLayout LayoutCoosort(int64_t nnz)
{
    CoosortLayout l{};
    int64_t off = 0;
    l.range = off; off += 256;
    l.keysA = off; off += Align256(4 * nnz);
    l.keysB = off; off += Align256(4 * nnz);
    l.pairsA = off; off += Align256(8 * nnz);
    l.pairsB = off; off += Align256(8 * nnz);
    const int64_t tableCount = WideTableInts(nnz);
    l.table = off; off += Align256(4 * tableCount);
    // (scanned are the table and, where the rows come first, the offsets of fewer than nnz rows: span + 1 <= nnz)
    l.tiles = off; off += Align256(4 * ScanTiles(tableCount > nnz ? tableCount : nnz));
    l.bytes = off;
    return l;
}

// Bits that hold hi - lo (both int32, hi >= lo), at least 1.
int32_t RangeBits(int32_t lo, int32_t hi)
{
    const uint32_t span = static_cast<uint32_t>(hi) - static_cast<uint32_t>(lo);
    int32_t bits = 1;
    while (bits < 32 && (span >> bits) != 0) {
        ++bits;
    }
    return bits;
}

}  // namespace
}  // namespace opsparse

extern "C" {

size_t opsparse_coosort_workspace_bytes(int64_t nnz)
{
    return nnz <= 0 ? 0 : static_cast<size_t>(LayoutCoosort(nnz).bytes);
}

int opsparse_coosort_launch(int64_t nnz, int32_t byRow, int32_t *cooRows, int32_t *cooCols, int32_t *perm,
                            void *workspace, size_t workspaceBytes, void *stream)
{
    if (nnz < 0 || nnz > INT32_MAX) {
        return OPSPARSE_E_INVALID;
    }
    if (nnz == 0) {
        return OPSPARSE_OK;
    }
    if (cooRows == nullptr || cooCols == nullptr || perm == nullptr) {
        return OPSPARSE_E_INVALID;
    }
    const CoosortLayout l = LayoutCoosort(nnz);
    if (workspace == nullptr || static_cast<int64_t>(workspaceBytes) < l.bytes) {
        return OPSPARSE_E_WORKSPACE;
    }
    auto s = static_cast<hipStream_t>(stream);
    auto *base = static_cast<unsigned char *>(workspace);
    auto at = [&](int64_t off) { return reinterpret_cast<int32_t *>(base + off); };
    int32_t *keys[2] = {at(l.keysA), at(l.keysB)};
    void *pairs[2] = {base + l.pairsA, base + l.pairsB};
    int32_t *table = at(l.table), *tiles = at(l.tiles), *range = at(l.range);
    int32_t *primary = byRow != 0 ? cooRows : cooCols, *secondary = byRow != 0 ? cooCols : cooRows;

    // (the counters of the sample: in the first key buffer, a power of two of them that fits)
    int32_t sampleBits = 1;
    while (sampleBits < 20 && (int64_t{2} << sampleBits) <= nnz) {
        ++sampleBits;
    }
    const bool ask = nnz >= kRowsFirstMin;
    hipLaunchKernelGGL(CooRangeInitKernel, dim3(ask ? 1024 : 1), dim3(kBlockThreads), 0, s, range, keys[0],
                       ask ? 1 << sampleBits : 0);
    // (two workgroups a compute unit keep memory busy, 5.8 TB/s; more of them cost their ends: 33.5 M entries 46 us with
    // 512, 65 with 2048)
    hipLaunchKernelGGL(CooRangeKernel, dim3(GridFor(nnz, kBlockThreads * 16, 512)), dim3(kBlockThreads), 0, s, primary,
                       secondary, nnz, range);
    if (ask) {
        hipLaunchKernelGGL(CooSampleKernel, dim3(kRowSamples / kBlockThreads), dim3(kBlockThreads), 0, s, primary, nnz,
                           kRowSamples, keys[0], sampleBits, range);
    }
    int32_t r[5] = {0, 0, 0, 0, 0};  // min / max of the primary key, of the secondary key; pairs of the sample
    if (hipMemcpyAsync(r, range, sizeof(r), hipMemcpyDeviceToHost, s) != hipSuccess ||
        hipStreamSynchronize(s) != hipSuccess) {
        (void)hipGetLastError();
        return OPSPARSE_E_LAUNCH;
    }

    int cur = 0;
    // One key's passes: the first reads (key, pair) from three arrays, the last writes three arrays.
    auto sortBy = [&](const int32_t *keySrc, int32_t keyBase, int32_t bits, const int32_t *pairRowSrc,
                      const void *pairValSrc, int32_t *keyDst, int32_t *pairRowDst, void *pairValDst) {
        const auto [passes, perPass] = WidePassesOf(bits, nnz);
        const RadixPairIo io{pairRowSrc, pairValSrc, pairRowDst, pairValDst, 4};
        const int32_t *keysIn = keySrc;
        const void *pairsIn = nullptr;
        for (int32_t pass = 0; pass < passes; ++pass) {
            const bool last = pass == passes - 1;
            const int mode = pass == 0 ? kPayPairFirst : (last ? kPayPairLast : kPayPair);
            int32_t *keysOut = last ? keyDst : keys[cur];
            LaunchWidePairPass(mode, keysIn, pairsIn, keysOut, pairs[cur], nnz, pass == 0 ? keyBase : 0, pass * perPass,
                               perPass, table, tiles, io, s);
            keysIn = keysOut;
            pairsIn = pairs[cur];
            cur ^= 1;
        }
    };
    const int32_t bitsS = RangeBits(r[2], r[3]), bitsP = RangeBits(r[0], r[1]);
    const int64_t span = static_cast<int64_t>(r[1]) - r[0] + 1;
    // (two rows that share a counter look like one: as many pairs of theirs as the counters would give anyway come off)
    const double rowLength = (2.0 * r[4] / (static_cast<double>(kRowSamples) * kRowSamples) -
                              1.0 / static_cast<double>(int64_t{1} << sampleBits)) * static_cast<double>(nnz);
    // (nor can the rows be shorter than the entries over the rows' range, whatever the sample says: csrsort's scratch for
    // short rows fits the passes' buffers, the one for a matrix of rows of thousands of entries would not)
    const bool mayBeShort = static_cast<double>(nnz) <= kRowsFirstLongest * static_cast<double>(span);
    if (ask && mayBeShort && rowLength <= kRowsFirstLongest && span < nnz && r[2] >= 0 && r[3] < INT32_MAX) {
        // Rows short enough for csrsort's registers: by row only, then every row by its secondary key in one pass over
        // the entries instead of one a digit.
        int32_t *rowPtr = keys[0];  // (the passes' buffers are free when it is written)
        const int64_t bound = static_cast<int64_t>(r[3]) + 1;
        const FinishPlan plan = FinishPlanOf(span, nnz, KeyBits(bound));
        const bool rowsToo = plan.use && SortPacked(bound, 0, kWave);
        if (plan.use) {
            const FinishSort sort{primary, r[0], RadixPairIo{secondary, perm, secondary, perm, 4}, primary,
                                  rowsToo ? bound : 0, rowPtr, 0, nnz, span};
            LaunchFinishSort(sort, plan, keys, pairs, table, tiles, s);
        } else {
            sortBy(primary, r[0], bitsP, secondary, perm, primary, secondary, perm);
            LaunchIndicesToOffsets(primary, nnz, span, 0, rowPtr, tiles, s);
        }
        if (!rowsToo) {
            const int rc = opsparse_csrsort_launch(span, bound, nnz, 0, rowPtr, secondary, perm, keys[1],
                                                   static_cast<size_t>(l.table - l.keysB), stream);
            if (rc != OPSPARSE_OK) {
                return rc;
            }
        }
        if (r[0] != 0) {
            hipLaunchKernelGGL(CooRebaseKernel, dim3(GridFor(nnz, kBlockThreads * 8)), dim3(kBlockThreads), 0, s, primary,
                               secondary, nnz, r[0], 0);
        }
        return CheckLaunch();
    }
    // by the secondary key, (primary key, P) as the pair: the result stays in the workspace ...
    int32_t *midKeys = keys[1];                                   // (two or four passes: the last one writes buffer 1
    auto *midRows = static_cast<int32_t *>(pairs[1]);             //  only when their number is even)
    const int lastBuf = (WidePassesOf(bitsS, nnz).passes - 1) & 1;                        // buffer the last pass of that stage writes
    midKeys = keys[lastBuf];
    midRows = static_cast<int32_t *>(pairs[lastBuf]);
    uint32_t *midVals = reinterpret_cast<uint32_t *>(pairs[lastBuf]) + nnz;
    sortBy(secondary, r[2], bitsS, primary, perm, midKeys, midRows, midVals);
    // ... then, stably, by the primary key, (secondary key, P) as the pair, into the caller's arrays
    sortBy(midRows, r[0], bitsP, midKeys, midVals, primary, secondary, perm);
    if (r[0] != 0 || r[2] != 0) {
        hipLaunchKernelGGL(CooRebaseKernel, dim3(GridFor(nnz, kBlockThreads * 8)), dim3(kBlockThreads), 0, s, primary,
                           secondary, nnz, r[0], r[2]);
    }
    return CheckLaunch();
}

}  // extern "C"
