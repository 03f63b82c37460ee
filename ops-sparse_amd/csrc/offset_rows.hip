// Matrices whose rows repeat (OPSPARSE_SPMV_OFFSET_ROWS): analysis and SpMV.
//
// On a mesh the columns of row r are r + d for a list of distances d that a handful of lists serve for every row, the
// faces included.  The analysis finds the lists, checks every entry of the matrix against them and keeps a byte a row;
// the product then never reads the column indices, half of what the row-wise kernels move.  It asks of the
// matrix ascending columns, at most 32 distances in at most 128 lists, and rows that have most of them.
//
// us a call, beta != 0, row-wise kernels / here: 5-point 2048 x 2048 39.6 / 26.4 (5.2 TB/s of the bytes it needs), 9-point
// 1500 x 1501 38.6 / 23.4, 7-point 125 x 131 x 127 31.3 / 20.0, 27-point 131 x 127 x 129 125 / 56 (4.6 TB/s), bf16 118 /
// 47, 83 x 141 x 109 71 / 31; below some 250 000 points (27: 90 000) the row-wise kernels are ahead, and Preprocess keeps them.
// The analysis reads the columns twice: Preprocess of the first takes 0.37 ms instead of 0.18, of the 27-point one 0.60 instead
// of 0.19, of a matrix that is none 0.05 - 0.1 more.
//
// No counterpart in the reference, whose kernels read a column index an entry
// (sparse/spmv/arch22/kernels/spmv_kernel.h:27-310).
#include <type_traits>

#include "convert_internal.h"
#include "device_utils.h"
#include "offset_device.h"
#include "offset_rows.h"
#include "spmv_internal.h"

namespace opsparse {

namespace {

// ------------------------------------------------------------- analysis

constexpr int32_t kKeySlots = 512;  // open addressing, at most a quarter full
constexpr int32_t kMaxProbes = 32;  // slots looked at for a list
// Different lists among 64 neighbouring rows beyond which a matrix is none: without a look at the table (random columns
// would fill it, one atomic after the other: 5 ms)
constexpr int32_t kStretchLists = 32;
// header of the part: [0] lists found, [1] "this is no such matrix", [2] distances in all, and from
// kOffsetHeaderDistances on these
constexpr int kHeaderInts = 64;
static_assert(kOffsetHeaderDistances + kOffsetMaxDistances <= kHeaderInts, "the header holds the distances");

constexpr int kWaves = kBlockThreads / kWave;

// The columns of 64 consecutive rows into the wavefront's LDS, and the lane's row among them (start < 0: no row).
// Offsets that are no offsets of a matrix with `nnz` entries give a row that `bad` reports.
struct LaneRow {
    int32_t start, len;
    bool bad;
};
__device__ __forceinline__ LaneRow StageColumns(const int32_t *__restrict__ rowOffsets,
                                                const int32_t *__restrict__ colInd, int64_t rows, int64_t nnz,
                                                int64_t r0, int32_t maxRow, int32_t *__restrict__ cols)
{
    const int lane = threadIdx.x % kWave;
    const int64_t rEnd = r0 + kWave < rows ? r0 + kWave : rows;
    const int64_t r = r0 + lane;
    LaneRow mine{-1, 0, false};
    if (r0 >= rows) {
        return mine;
    }
    const int64_t base = rowOffsets[r0];
    const int64_t count = rowOffsets[rEnd] - base;
    mine.bad = base < 0 || count < 0 || base + count > nnz || count > static_cast<int64_t>(kWave) * maxRow;
    if (r < rEnd) {
        mine.start = static_cast<int32_t>(rowOffsets[r] - base);
        mine.len = rowOffsets[r + 1] - rowOffsets[r];
        mine.bad = mine.bad || mine.len < 0 || mine.len > maxRow || mine.start < 0 || mine.start + mine.len > count;
    }
    if (__ballot(mine.bad) == 0) {
        for (int32_t k = lane; k < count; k += kWave) {
            cols[k] = LoadStream(colInd + base + k);
        }
    }
    return mine;
}

__device__ __forceinline__ uint64_t HashRow(const int32_t *__restrict__ cols, int32_t start, int32_t len, int32_t row)
{
    uint64_t h = 0x9e3779b97f4a7c15ull * static_cast<uint64_t>(len + 1);
    for (int32_t k = 0; k < len; ++k) {
        h ^= static_cast<uint32_t>(cols[start + k] - row);
        h *= 0xbf58476d1ce4e5b9ull;
        h ^= h >> 29;
    }
    h *= 0x94d049bb133111ebull;
    h ^= h >> 32;
    return h == 0 ? 1 : h;
}

// Enters the hashes of the lists into `keys`, with one row of each list: of every `stretchStride`-th stretch of 64 rows.
__global__ __launch_bounds__(kBlockThreads) void OffsetCollectKernel(
    const int32_t *__restrict__ rowOffsets, const int32_t *__restrict__ colInd, int64_t rows, int64_t nnz,
    int64_t stretchStride, int32_t maxRow, int32_t *header, unsigned long long *keys, int32_t *keyRow)
{
    extern __shared__ int32_t staged[];
    const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
    int32_t *const cols = staged + wave * kWave * maxRow;
    uint64_t known = 0;  // the list that this wavefront entered or found last
    for (int64_t r0 = (static_cast<int64_t>(blockIdx.x) * kWaves + wave) * kWave * stretchStride; r0 < rows;
         r0 += static_cast<int64_t>(gridDim.x) * kWaves * kWave * stretchStride) {
        if (__builtin_amdgcn_readfirstlane(
                __hip_atomic_load(header + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) != 0) {
            return;  // no such matrix: nothing to look for any more
        }
        const LaneRow mine = StageColumns(rowOffsets, colInd, rows, nnz, r0, maxRow, cols);
        if (__ballot(mine.bad) != 0) {
            if (lane == 0) {
                __hip_atomic_store(header + 1, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            return;
        }
        __builtin_amdgcn_wave_barrier();
        const bool have = mine.start >= 0;
        const uint64_t hash = have ? HashRow(cols, mine.start, mine.len, static_cast<int32_t>(r0 + lane)) : known;
        // one lane a list enters it: most wavefronts hold one list, or three
        const uint64_t news = __ballot(have && hash != known);
        uint64_t leaders = 0;
        int32_t lists = 0;
        for (uint64_t todo = news; todo != 0 && lists <= kStretchLists; ++lists) {
            const int leader = __ffsll(static_cast<unsigned long long>(todo)) - 1;
            const uint64_t key = __shfl(hash, leader, kWave);
            todo &= ~__ballot(have && hash == key);
            leaders |= uint64_t{1} << leader;
            known = key;
        }
        bool none = lists > kStretchLists;
        if (!none && ((leaders >> lane) & 1) != 0) {
            none = true;
            uint32_t slot = static_cast<uint32_t>(hash) % kKeySlots;
            for (int32_t probe = 0; probe < kMaxProbes && none; ++probe, slot = (slot + 1) % kKeySlots) {
                unsigned long long there = __hip_atomic_load(keys + slot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if (there == 0) {
                    there = atomicCAS(keys + slot, 0ull, static_cast<unsigned long long>(hash));
                    if (there == 0) {
                        keyRow[slot] = static_cast<int32_t>(r0 + lane);
                        none = atomicAdd(header, 1) >= kOffsetMaxPatterns;
                        break;
                    }
                }
                none = there != hash;
            }
        }
        if (__ballot(none) != 0) {
            if (lane == 0) {
                __hip_atomic_store(header + 1, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            return;
        }
        __builtin_amdgcn_wave_barrier();
    }
}

// One workgroup: numbers the lists (a slot's list in keyRow from here on), writes their distances, and makes one list of
// all distances and the masks of the lists over it.
__global__ __launch_bounds__(kKeySlots) void OffsetNumberKernel(const int32_t *__restrict__ rowOffsets,
                                                                const int32_t *__restrict__ colInd, int32_t maxRow,
                                                                int32_t *header,
                                                                const unsigned long long *__restrict__ keys,
                                                                int32_t *keyRow, int32_t *lens, int32_t *table,
                                                                uint32_t *masks)
{
    constexpr int kSlotWaves = kKeySlots / kWave;
    __shared__ int32_t waveCount[kSlotWaves], waveMin[kSlotWaves];
    __shared__ int32_t distances[kOffsetMaxDistances];
    if (header[1] != 0) {
        return;
    }
    const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
    const bool used = keys[threadIdx.x] != 0;
    const uint64_t votes = __ballot(used);
    if (lane == 0) {
        waveCount[wave] = __popcll(votes);
    }
    __syncthreads();
    int32_t id = __popcll(votes & ((uint64_t{1} << lane) - 1)), lists = 0;
    for (int w = 0; w < kSlotWaves; ++w) {
        id += w < wave ? waveCount[w] : 0;
        lists += waveCount[w];
    }
    bool bad = lists > kOffsetMaxPatterns;
    if (used && !bad) {
        const int32_t row = keyRow[threadIdx.x];
        const int32_t s = rowOffsets[row];
        const int32_t n = rowOffsets[row + 1] - s;
        lens[id] = n;
        for (int32_t k = 0; k < n; ++k) {
            table[id * maxRow + k] = colInd[s + k] - row;
            bad = bad || (k > 0 && colInd[s + k] <= colInd[s + k - 1]);  // (distances in ascending order only)
        }
        keyRow[threadIdx.x] = id;
    }
    if (__syncthreads_or(bad)) {
        header[1] = 1;
        return;
    }
    // the smallest distance above the last one, again and again
    int32_t found = 0;
    int64_t last = INT64_MIN;
    while (true) {
        int32_t best = INT32_MAX;
        for (int32_t k = threadIdx.x; k < lists * maxRow; k += kKeySlots) {
            if (k % maxRow < lens[k / maxRow] && table[k] > last && table[k] < best) {
                best = table[k];
            }
        }
#pragma unroll
        for (int off = kWave / 2; off > 0; off >>= 1) {
            const int32_t other = __shfl_xor(best, off, kWave);
            best = other < best ? other : best;
        }
        if (lane == 0) {
            waveMin[wave] = best;
        }
        __syncthreads();
        for (int w = 0; w < kSlotWaves; ++w) {
            best = waveMin[w] < best ? waveMin[w] : best;
        }
        __syncthreads();
        if (best == INT32_MAX || found == kOffsetMaxDistances) {
            bad = best != INT32_MAX;
            break;
        }
        if (threadIdx.x == 0) {
            distances[found] = best;
        }
        ++found;
        last = best;
    }
    __syncthreads();
    if (bad || found == 0) {
        header[1] = 1;
        return;
    }
    if (static_cast<int32_t>(threadIdx.x) < lists) {
        uint32_t mask = 0;
        int32_t k = 0;
        for (int32_t d = 0; d < found; ++d) {
            if (k < lens[threadIdx.x] && table[threadIdx.x * maxRow + k] == distances[d]) {
                mask |= 1u << d;
                ++k;
            }
        }
        masks[threadIdx.x] = mask;
    }
    if (threadIdx.x < kHeaderInts - kOffsetHeaderDistances) {
        // (behind the last distance the last again: the loads there stay where the others are)
        header[kOffsetHeaderDistances + threadIdx.x] =
            distances[static_cast<int32_t>(threadIdx.x) < found ? threadIdx.x : found - 1];
    }
    if (threadIdx.x == 0) {
        header[2] = found;
    }
}

// Every row's list by its number, checked entry by entry.
__global__ __launch_bounds__(kBlockThreads) void OffsetAssignKernel(
    const int32_t *__restrict__ rowOffsets, const int32_t *__restrict__ colInd, int64_t rows, int64_t cols, int64_t nnz,
    int32_t maxRow, int32_t *header, const unsigned long long *__restrict__ keys, const int32_t *__restrict__ keyRow,
    const int32_t *__restrict__ lens, const int32_t *__restrict__ table, uint8_t *__restrict__ ids)
{
    extern __shared__ int32_t staged[];
    const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
    int32_t *const mineCols = staged + wave * kWave * maxRow;
    for (int64_t r0 = (static_cast<int64_t>(blockIdx.x) * kWaves + wave) * kWave; r0 < rows;
         r0 += static_cast<int64_t>(gridDim.x) * kWaves * kWave) {
        if (__builtin_amdgcn_readfirstlane(
                __hip_atomic_load(header + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) != 0) {
            return;
        }
        const LaneRow mine = StageColumns(rowOffsets, colInd, rows, nnz, r0, maxRow, mineCols);
        __builtin_amdgcn_wave_barrier();
        bool wrong = mine.bad;
        if (__ballot(mine.bad) == 0 && mine.start >= 0) {
            const int32_t row = static_cast<int32_t>(r0 + lane);
            const uint64_t hash = HashRow(mineCols, mine.start, mine.len, row);
            uint32_t slot = static_cast<uint32_t>(hash) % kKeySlots;
            for (int32_t probe = 0; probe < kMaxProbes && keys[slot] != hash && keys[slot] != 0; ++probe) {
                slot = (slot + 1) % kKeySlots;
            }
            wrong = keys[slot] != hash;
            if (!wrong) {
                const int32_t id = keyRow[slot];
                wrong = lens[id] != mine.len;
                for (int32_t k = 0; k < mine.len && !wrong; ++k) {
                    const int32_t c = mineCols[mine.start + k];
                    wrong = table[id * maxRow + k] != c - row || c < 0 || c >= cols;
                }
                ids[r0 + lane] = static_cast<uint8_t>(id);
            }
        }
        if (__ballot(wrong) != 0) {
            if (lane == 0) {
                __hip_atomic_store(header + 1, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            return;
        }
        __builtin_amdgcn_wave_barrier();
    }
}

// ------------------------------------------------------------- SpMV

// Workgroups of a launch at most: two rounds of the eight a compute unit takes (5 distances on 2048 x 2048 points: 26.4 us;
// 28.6, 26.7 and 26.0 with 4, 8 and 64 a compute unit; 9 on 1500 x 1501: 23.4; 28.3, 25.4, 24.6).
constexpr int64_t kOffsetGrid = 16 * 256;

typedef int32_t Int2U __attribute__((ext_vector_type(2), aligned(4)));
typedef uint16_t Short2U __attribute__((ext_vector_type(2), aligned(2)));
// One or two neighbours.
template <typename T, int V>
using Some = typename std::conditional<sizeof(T) == 4, typename std::conditional<V == 2, Int2U, int32_t>::type,
                                       typename std::conditional<V == 2, Short2U, uint16_t>::type>::type;

struct OffsetList {
    // all distances in ascending order, and the last one again behind them: the loads there stay in range, and the bound of
    // a tile's columns is the entry of the compiled width
    int32_t d[kOffsetMaxDistances];
};

// A wavefront walks over tiles of 128 consecutive rows, a lane taking two neighbours.  The distances of all lists, in
// ascending order, are one list and a row's own a mask over it.  So the loop over the distances is the same for the whole
// wavefront: a distance is a scalar, and one load of two neighbours a lane brings x for 128 rows (a load instruction takes
// 16 cycles of a compute unit's address path whatever it brings; a column index an entry needs one for 64 entries).  The
// values, one contiguous range a tile, come in through full-width loads and pass through the wavefront's own LDS to the
// lanes whose rows they are; where a row's begin is a scan of the masks' bits.  No barrier, and no branch around a load:
// a tile that is not whole, or whose loads could leave the arrays, is summed straight from memory instead.
//
// Bytes a row of K fp32 entries: 4 K of values, 1 for the list, 4 of x, 4 or 8 of y; the column indices and the row
// offsets would be another 4 K + 4.  A tile has two round trips to memory and hides the first: where its values begin and
// which lists its rows have is asked for a tile ahead; the second is left to the other wavefronts of the compute unit (20 of them
// with 27 distances): over a call on 131 x 127 x 129 points the data path of the vector memory is 73 % busy, its address path
// 59 %.  K >= the distances there are, in chunks of U whose loads of x are in flight together.
template <typename ValT, typename OutT, typename AccT, int V, int K, int U>
__global__ __launch_bounds__(kBlockThreads) void SpmvOffsetRowsKernel(
    const int32_t *__restrict__ rowOffsets, const ValT *__restrict__ vals, const ValT *__restrict__ x, OutT *y,
    const OutT *yIn, int64_t rows, int64_t cols, int64_t nnz, const uint8_t *__restrict__ ids,
    const uint32_t *__restrict__ masks, OffsetList all, int32_t distances, int32_t patterns, OpsparseScalar alphaS,
    OpsparseScalar betaS)
{
    static_assert(K % U == 0 && (V == 1 || V == 2), "whole chunks");
    constexpr int32_t kTileRows = V * kWave;
    constexpr int Q = (kTileRows * K + 4 * kWave - 1) / (4 * kWave);  // quads of values a lane loads
    // (what the masked reads may touch past the last row's end behind them)
    __shared__ __align__(16) ValT stagedOf[kWaves][Q * 4 * kWave + 8];
    __shared__ uint32_t maskOf[kOffsetMaxPatterns];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
    ValT *const staged = stagedOf[wave];
    if (threadIdx.x < kOffsetMaxPatterns) {
        maskOf[threadIdx.x] = static_cast<int32_t>(threadIdx.x) < patterns ? masks[threadIdx.x] : 0;
    }
    __syncthreads();

    const AccT alpha = ReadScalar<AccT>(alphaS);
    const AccT beta = ReadScalar<AccT>(betaS);
    const bool betaZero = (beta == AccT(0));

    // This XCD's tiles, and this wavefront's stride through them: neighbours share lines of x in that XCD's L2.  (A grid of
    // fewer workgroups than XCDs lives on as many.)
    const uint32_t numTiles = static_cast<uint32_t>((rows + kTileRows - 1) / kTileRows);
    const uint32_t dies = gridDim.x < kNumXcd ? gridDim.x : kNumXcd;
    const uint32_t xcd = blockIdx.x % dies;
    const uint32_t perXcd = numTiles / dies, rem = numTiles % dies;
    const int64_t xcdFirst = xcd * perXcd + (xcd < rem ? xcd : rem);
    const int64_t xcdTiles = perXcd + (xcd < rem ? 1 : 0);
    const int64_t step = (gridDim.x - xcd + dies - 1) / dies * kWaves;  // wavefronts living on this XCD
    int64_t t = static_cast<int64_t>(blockIdx.x / dies) * kWaves + wave;
    if (t >= xcdTiles) {
        return;
    }

    // (bounds by a vector load: a scalar one would have to be waited for with the first LDS read of the tile before)
    int32_t bound;
    uint32_t idPair;
    auto askTile = [&](int64_t tile) {
        const int64_t first = (xcdFirst + tile) * kTileRows;
        const int64_t last = first + kTileRows < rows ? first + kTileRows : rows;
        bound = LoadStream(rowOffsets + ((lane & 1) != 0 ? last : first));
        // (the table is padded to whole tiles)
        if constexpr (V == 2) {
            idPair = LoadStream(reinterpret_cast<const uint16_t *>(ids + first) + lane);
        } else {
            idPair = LoadStream(ids + first + lane);
        }
    };
    askTile(t);
    while (true) {
        const int64_t r0 = (xcdFirst + t) * kTileRows;
        const int64_t tNext = t + step;
        const bool more = tNext < xcdTiles;
        const uint32_t pair = idPair;
        const int32_t first = __builtin_amdgcn_readlane(bound, 0);
        const int32_t count = __builtin_amdgcn_readlane(bound, 1) - first;
        const bool whole = r0 + kTileRows <= rows && r0 + all.d[0] >= 0 && r0 + kTileRows + all.d[K - 1] <= cols &&
                           first >= 0 && count >= 1 && count <= Q * 4 * kWave &&
                           first + static_cast<int64_t>(count) + 3 <= nnz;
        if (whole) {
            FourOf<ValT> q[Q];
#pragma unroll
            for (int u = 0; u < Q; ++u) {
                int32_t k = (u * kWave + lane) * 4;  // (lanes past the end: the last quad again, not used)
                k = k < count ? k : (count - 1) & ~3;
                q[u] = __builtin_nontemporal_load(reinterpret_cast<const FourOf<ValT> *>(vals + first + k));
            }
            Some<ValT, V> xv[2][U];
            auto gather = [&](int chunk) {
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    xv[chunk % 2][u] = reinterpret_cast<const Some<ValT, V> *>(x + (r0 + all.d[chunk * U + u]))[lane];
                }
            };
            gather(0);
            Some<OutT, V> yOld{};
            if (!betaZero) {
                yOld = __builtin_nontemporal_load(reinterpret_cast<const Some<OutT, V> *>(yIn + r0) + lane);
            }
            if (more) {
                askTile(tNext);
            }
            const uint32_t m0 = maskOf[(pair & 0xff) % kOffsetMaxPatterns];
            const uint32_t m1 = V == 2 ? maskOf[(pair >> 8) % kOffsetMaxPatterns] : 0;
            const int32_t n0 = __popc(m0), n1 = __popc(m1);
            int32_t at0 = WaveScan(n0 + n1) - n0 - n1;
            at0 = at0 + n0 + n1 > count ? 0 : at0;  // (never, in the matrix that was analysed)
            int32_t at1 = at0 + n0;
#pragma unroll
            for (int u = 0; u < Q; ++u) {
                __builtin_memcpy(__builtin_assume_aligned(staged + (u * kWave + lane) * 4, 4 * sizeof(ValT)), &q[u],
                                 4 * sizeof(ValT));
            }
            // (a shorter path for tiles whose rows have every distance measured the same, 26.4 / 26.7 us)
            AccT sum0 = AccT(0), sum1 = AccT(0);
#pragma unroll
            for (int chunk = 0; chunk < K / U; ++chunk) {
                if (chunk + 1 < K / U) {
                    gather(chunk + 1);
                }
                ValT v0[U], v1[U];
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    v0[u] = staged[at0];
                    v1[u] = V == 2 ? staged[at1] : ValT{};
                    at0 += (m0 >> (chunk * U + u)) & 1;
                    at1 += (m1 >> (chunk * U + u)) & 1;
                }
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    ValT two[V];
                    __builtin_memcpy(two, &xv[chunk % 2][u], sizeof(two));
                    const bool in0 = ((m0 >> (chunk * U + u)) & 1) != 0, in1 = ((m1 >> (chunk * U + u)) & 1) != 0;
                    sum0 += (in0 ? ToAcc<AccT>(v0[u]) : AccT(0)) * (in0 ? ToAcc<AccT>(two[0]) : AccT(0));
                    if constexpr (V == 2) {
                        sum1 += (in1 ? ToAcc<AccT>(v1[u]) : AccT(0)) * (in1 ? ToAcc<AccT>(two[1]) : AccT(0));
                    }
                }
            }
            AccT res0 = alpha * sum0, res1 = alpha * sum1;
            if (!betaZero) {
                OutT old[V];
                __builtin_memcpy(old, &yOld, sizeof(old));
                res0 += beta * ToAcc<AccT>(old[0]);
                res1 += beta * ToAcc<AccT>(old[V - 1]);
            }
            const OutT out[2] = {FromAcc<OutT>(res0), FromAcc<OutT>(res1)};
            Some<OutT, V> o;
            __builtin_memcpy(&o, out, sizeof(o));
            reinterpret_cast<Some<OutT, V> *>(y + r0)[lane] = o;
        } else {
            for (int i = 0; i < V; ++i) {
                const int64_t r = r0 + V * lane + i;
                if (r < rows) {
                    const uint32_t m = maskOf[(i == 0 ? pair & 0xff : pair >> 8) % kOffsetMaxPatterns];
                    int64_t k = rowOffsets[r];
                    AccT sum = AccT(0);
                    for (int32_t e = 0; e < distances; ++e) {
                        if (((m >> e) & 1) != 0 && k >= 0 && k < nnz) {
                            int64_t c = r + all.d[e];
                            c = c < 0 ? 0 : (c < cols ? c : cols - 1);
                            sum += ToAcc<AccT>(vals[k]) * ToAcc<AccT>(x[c]);
                            ++k;
                        }
                    }
                    AccT res = alpha * sum;
                    if (!betaZero) {
                        res += beta * ToAcc<AccT>(yIn[r]);
                    }
                    y[r] = FromAcc<OutT>(res);
                }
            }
            if (more) {
                askTile(tNext);
            }
        }
        if (!more) {
            break;
        }
        t = tNext;
    }
}

}  // namespace

OffsetLayout MakeOffsetLayout(int64_t rows)
{
    OffsetLayout l{};
    int64_t off = kHeaderInts * 4;
    l.keyOff = off;
    off += 8 * kKeySlots;
    l.rowOff = off;
    off += 4 * kKeySlots;
    l.lenOff = off;
    off += 4 * kOffsetMaxPatterns;
    l.maskOff = off;
    off += 4 * kOffsetMaxPatterns;
    l.tableOff = off;
    off += 4 * kOffsetMaxPatterns * kOffsetMaxRow;
    l.idOff = off;
    off += (rows + 255) / 256 * 256;
    l.bytes = off;
    return l;
}

int32_t OffsetRuns(const OffsetFound &found)
{
    int32_t size[kOffsetMaxDistances] = {}, runs = 0;
    bool threes = true;
    for (int32_t k = 0; k < found.distances; ++runs) {
        size[runs] = 1;
        while (k + size[runs] < found.distances && found.distance[k + size[runs]] == found.distance[k] + size[runs]) {
            ++size[runs];
        }
        k += size[runs];
        threes = threes && size[runs] == 3;
    }
    if (threes && (runs == 3 || runs == 9)) {
        return kOffsetRuns333;
    }
    if (runs == 3 && size[0] == 1 && size[1] == 3 && size[2] == 1) {
        return kOffsetRuns131;
    }
    return runs == 5 && size[0] == 1 && size[1] == 1 && size[2] == 3 && size[3] == 1 && size[4] == 1 ? kOffsetRuns11311
                                                                                                  : kOffsetRunsAny;
}

bool OffsetRowsApply(int64_t rows, int64_t cols, int64_t nnz)
{
    // Rows and columns within 2^30 (32-bit byte offsets into x and a row number plus a distance in 32 bits).
    return rows >= 1024 && cols > 0 && nnz > 0 && rows < (int64_t{1} << 30) && cols <= (int64_t{1} << 30) &&
           nnz <= INT32_MAX && nnz <= rows * kOffsetMaxRow;
}

int AnalyseOffsetRows(const int32_t *rowOffsets, const int32_t *colInd, int64_t rows, int64_t cols, int64_t nnz,
                      int32_t maxRow, unsigned char *part, OffsetFound *found, hipStream_t stream)
{
    *found = OffsetFound{};
    if (maxRow < 1 || maxRow > kOffsetMaxRow || !OffsetRowsApply(rows, cols, nnz)) {
        return OPSPARSE_OK;
    }
    const OffsetLayout l = MakeOffsetLayout(rows);
    auto *header = reinterpret_cast<int32_t *>(part);
    auto *keys = reinterpret_cast<unsigned long long *>(part + l.keyOff);
    auto *keyRow = reinterpret_cast<int32_t *>(part + l.rowOff);
    auto *lens = reinterpret_cast<int32_t *>(part + l.lenOff);
    auto *table = reinterpret_cast<int32_t *>(part + l.tableOff);
    auto *masks = reinterpret_cast<uint32_t *>(part + l.maskOff);
    LaunchFillI32(header, l.tableOff / 4, 0, stream);  // header, keys, rows and lengths
    const size_t lds = static_cast<size_t>(kBlockThreads) * maxRow * sizeof(int32_t);
    // A look at 2048 stretches first: a matrix that is none fills the table there, and the other kernels leave at once.
    const int64_t stretches = (rows + kWave - 1) / kWave;
    constexpr int64_t kSampleStretches = 2048;
    const int64_t sampleStride = stretches / kSampleStretches + 1;
    auto blocks = [](int64_t n) {
        const int64_t b = (n + kWaves - 1) / kWaves;
        return dim3(static_cast<uint32_t>(b < 2048 ? b : 2048));
    };
    if (sampleStride > 1) {
        hipLaunchKernelGGL(OffsetCollectKernel, blocks((stretches + sampleStride - 1) / sampleStride),
                           dim3(kBlockThreads), lds, stream, rowOffsets, colInd, rows, nnz, sampleStride, maxRow, header,
                           keys, keyRow);
    }
    hipLaunchKernelGGL(OffsetCollectKernel, blocks(stretches), dim3(kBlockThreads), lds, stream, rowOffsets, colInd,
                       rows, nnz, int64_t{1}, maxRow, header, keys, keyRow);
    hipLaunchKernelGGL(OffsetNumberKernel, dim3(1), dim3(kKeySlots), 0, stream, rowOffsets, colInd, maxRow, header, keys,
                       keyRow, lens, table, masks);
    hipLaunchKernelGGL(OffsetAssignKernel, blocks(stretches), dim3(kBlockThreads), lds, stream, rowOffsets, colInd,
                       rows, cols, nnz, maxRow, header, keys, keyRow, lens, table, part + l.idOff);
    int32_t seen[kHeaderInts] = {};
    if (CheckLaunch() != OPSPARSE_OK ||
        hipMemcpyAsync(seen, header, sizeof(seen), hipMemcpyDeviceToHost, stream) != hipSuccess ||
        hipStreamSynchronize(stream) != hipSuccess) {
        return OPSPARSE_E_LAUNCH;
    }
    if (seen[1] != 0 || seen[0] < 1 || seen[0] > kOffsetMaxPatterns) {
        return OPSPARSE_OK;
    }
    if (seen[2] < 1 || seen[2] > kOffsetMaxDistances) {
        return OPSPARSE_OK;
    }
    // Every row takes a step a distance, whether it has an entry there or not: not worth it where most steps are empty.
    if (seen[2] * rows > 2 * nnz) {
        return OPSPARSE_OK;
    }
    found->patterns = seen[0];
    found->distances = seen[2];
    for (int32_t k = 0; k < kOffsetMaxDistances; ++k) {
        found->distance[k] = seen[kOffsetHeaderDistances + k];
    }
    return OPSPARSE_OK;
}

template <typename ValT, typename OutT, typename AccT>
static int LaunchOffsetRowsTyped(const SpmvArgs &a, const OpsparseSpmvPlan &plan)
{
    const OffsetLayout l = MakeOffsetLayout(a.rows);
    if (a.ws == nullptr || static_cast<int64_t>(a.wsBytes) < l.bytes || plan.bytes != l.bytes) {
        return OPSPARSE_E_WORKSPACE;
    }
    if (a.cols < 1 || plan.numPatterns < 1 || plan.numPatterns > kOffsetMaxPatterns || plan.numDistances < 1 ||
        plan.numDistances > kOffsetMaxDistances || plan.maxRowNnz < 1 || plan.maxRowNnz > kOffsetMaxRow) {
        return OPSPARSE_E_INVALID;
    }
    const auto *part = static_cast<const unsigned char *>(a.ws);
    OffsetList all{};
    for (int32_t k = 0; k < kOffsetMaxDistances; ++k) {
        all.d[k] = plan.distances[k];  // (behind the last one the last again)
    }
    auto launch = [&](auto rowsTag, auto widthTag, auto chunkTag) {
        constexpr int V = decltype(rowsTag)::value, K = decltype(widthTag)::value, U = decltype(chunkTag)::value;
        int64_t grid = (a.rows + kBlockThreads * V - 1) / (kBlockThreads * V);
        grid = grid > kOffsetGrid ? kOffsetGrid : grid;
        hipLaunchKernelGGL((SpmvOffsetRowsKernel<ValT, OutT, AccT, V, K, U>), dim3(static_cast<uint32_t>(grid)),
                           dim3(kBlockThreads), 0, a.stream, a.rowOffsets, static_cast<const ValT *>(a.vals),
                           static_cast<const ValT *>(a.x), static_cast<OutT *>(a.y), static_cast<const OutT *>(a.yIn),
                           a.rows, a.cols, a.nnz, part + l.idOff, reinterpret_cast<const uint32_t *>(part + l.maskOff), all,
                           plan.numDistances, plan.numPatterns, a.alpha, a.beta);
    };
#define OFFSET_ROWS_CASE(V, K, U)                                                                                      \
    if (plan.numDistances <= K) {                                                                                      \
        launch(std::integral_constant<int, V>{}, std::integral_constant<int, K>{}, std::integral_constant<int, U>{});  \
        return CheckLaunch();                                                                                          \
    }
    // Two rows a lane while the values of a tile leave room in LDS for the wavefronts it takes: 27 distances on 131 x 127 x
    // 129 points 56 us with one row a lane (20 wavefronts a compute unit), 65 us with two (8); 9 on 1500 x 1501 24.2
    // and 23.4; 5 on 2048 x 2048 28 and 26.4.
    OFFSET_ROWS_CASE(2, 5, 5)
    OFFSET_ROWS_CASE(2, 7, 7)
    OFFSET_ROWS_CASE(2, 9, 9)
    OFFSET_ROWS_CASE(1, 18, 9)
    OFFSET_ROWS_CASE(1, 27, 9)
    OFFSET_ROWS_CASE(1, 32, 8)
#undef OFFSET_ROWS_CASE
    return OPSPARSE_E_INVALID;
}

int LaunchOffsetRows(const SpmvArgs &a, const OpsparseSpmvPlan &plan, int32_t valType, int32_t outType,
                     int32_t computeIsInt)
{
    if (computeIsInt) {
        return valType == OPSPARSE_I32 && outType == OPSPARSE_I32
                   ? LaunchOffsetRowsTyped<int32_t, int32_t, int32_t>(a, plan)
                   : OPSPARSE_E_UNSUPPORTED;
    }
    switch (valType) {
        case OPSPARSE_F32:
            if (outType == OPSPARSE_F32) return LaunchOffsetRowsTyped<float, float, double>(a, plan);
            break;
        case OPSPARSE_F16:
            if (outType == OPSPARSE_F32) return LaunchOffsetRowsTyped<Half, float, double>(a, plan);
            if (outType == OPSPARSE_F16) return LaunchOffsetRowsTyped<Half, Half, double>(a, plan);
            break;
        case OPSPARSE_BF16:
            if (outType == OPSPARSE_F32) return LaunchOffsetRowsTyped<Bf16, float, double>(a, plan);
            if (outType == OPSPARSE_BF16) return LaunchOffsetRowsTyped<Bf16, Bf16, double>(a, plan);
            break;
        case OPSPARSE_I32:
            if (outType == OPSPARSE_F32) return LaunchOffsetRowsTyped<int32_t, float, double>(a, plan);
            break;
        default:
            break;
    }
    return OPSPARSE_E_UNSUPPORTED;
}

}  // namespace opsparse

using namespace opsparse;

extern "C" {

size_t opsparse_spmv_csr_offsets_workspace_bytes(int64_t rows, int64_t cols, int64_t nnz)
{
    return OffsetRowsApply(rows, cols, nnz) ? static_cast<size_t>(MakeOffsetLayout(rows).bytes) : 0;
}

int opsparse_spmv_csr_offsets_analyse(const int32_t *rowOffsets, const int32_t *colInd, int64_t rows, int64_t cols,
                                      int64_t nnz, void *workspace, size_t workspaceBytes, OpsparseSpmvPlan *plan,
                                      void *stream)
{
    if (plan == nullptr || rows < 0 || cols < 0 || nnz < 0 || plan->rows != rows || plan->nnz != nnz ||
        (rows > 0 && rowOffsets == nullptr) || (nnz > 0 && colInd == nullptr)) {
        return OPSPARSE_E_INVALID;
    }
    if (plan->kernel != OPSPARSE_SPMV_STREAM_ROWS || !OffsetRowsApply(rows, cols, nnz)) {
        return OPSPARSE_E_UNSUPPORTED;
    }
    const int64_t bytes = MakeOffsetLayout(rows).bytes;
    if (workspace == nullptr || static_cast<int64_t>(workspaceBytes) < bytes) {
        return OPSPARSE_E_WORKSPACE;
    }
    OffsetFound found;
    const int rc = AnalyseOffsetRows(rowOffsets, colInd, rows, cols, nnz, plan->maxRowNnz,
                                     static_cast<unsigned char *>(workspace), &found,
                                     static_cast<hipStream_t>(stream));
    if (rc != OPSPARSE_OK) {
        return rc;
    }
    if (found.patterns == 0) {
        return OPSPARSE_E_UNSUPPORTED;
    }
    plan->kernel = OPSPARSE_SPMV_OFFSET_ROWS;
    plan->numPatterns = found.patterns;
    plan->numDistances = found.distances;
    for (int32_t k = 0; k < kOffsetMaxDistances; ++k) {
        plan->distances[k] = found.distance[k];
    }
    plan->bytes = bytes;
    return OPSPARSE_OK;
}

}  // extern "C"
