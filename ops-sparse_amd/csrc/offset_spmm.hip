// SpMM of a matrix whose rows repeat (offset_rows.hip has the analysis and the SpMV).
//
// No counterpart in the reference, whose kernel reads a column index an entry
// (sparse/spmm/arch35/spmm_kernel.cpp:155-219).
#include <type_traits>

#include "device_utils.h"
#include "offset_device.h"
#include "offset_rows.h"
#include "spmv_internal.h"

namespace opsparse {

namespace {

constexpr int kWaves = kBlockThreads / kWave;
// Passes over a wavefront's tile under P pieces a row and `rowsALane` rows a lane, at most: 64 rows, but no more than four
// times those of one pass.
constexpr int32_t MostPasses(int pieces, int rowsALane)
{
    return pieces / rowsALane < 1 ? 1 : pieces / rowsALane < 4 ? pieces / rowsALane : 4;
}

// How a lane takes the list of distances.  Chunks: one row a lane, U distances with their loads in flight together, at most
// K of them.  Runs: two neighbouring rows a lane, the distances of a chunk in runs of S... consecutive ones; a run of s
// takes s + 1 loads for both rows instead of 2 s, and every element of B loaded is widened once for both.
template <int U, int K>
struct Chunks {
    static constexpr int kRows = 1, kChunk = U, kMost = K, kLoads = U;
};
template <int K, int... S>
struct Runs {
    static constexpr int kRows = 2, kChunk = (S + ... + 0), kMost = K, kLoads = ((S + 1) + ... + 0), kRuns = sizeof...(S);
    static constexpr int kSize[kRuns] = {S...};
};
constexpr int64_t kEnoughTiles = 16 * 256;  // below that many tiles there are fewer passes a tile instead
constexpr int64_t kOffsetGrid = 16 * 256;   // workgroups of a launch at most
constexpr int64_t kBandBytes = 7 << 17;     // of B between a row and the furthest one it meets

// V elements of a row of B or C, a lane's piece.
template <typename T, int V>
struct __align__(sizeof(T)) Piece {
    T e[V];
};
template <typename T, int V>
__device__ __forceinline__ Piece<T, V> LoadPiece(const void *p)
{
    Piece<T, V> r;
    if constexpr (sizeof(T) == 4) {
        for (int i = 0; i < V; i += 4) {
            const Int4U q = *reinterpret_cast<const Int4U *>(static_cast<const T *>(p) + i);
            __builtin_memcpy(r.e + i, &q, 16);
        }
    } else {
        typedef int32_t Int4A __attribute__((ext_vector_type(4)));
        static_assert(V * sizeof(T) == 16, "one 16-byte piece");
        const Int4A q = *static_cast<const Int4A *>(p);
        __builtin_memcpy(r.e, &q, 16);
    }
    return r;
}
template <typename T, int V>
__device__ __forceinline__ void StorePiece(T *p, const Piece<T, V> &v)
{
    if constexpr (sizeof(T) == 4) {
        for (int i = 0; i < V; i += 4) {
            Int4U q;
            __builtin_memcpy(&q, v.e + i, 16);
            __builtin_nontemporal_store(q, reinterpret_cast<Int4U *>(p + i));
        }
    } else {
        typedef int32_t Int4A __attribute__((ext_vector_type(4)));
        Int4A q;
        __builtin_memcpy(&q, v.e, 16);
        __builtin_nontemporal_store(q, reinterpret_cast<Int4A *>(p));
    }
}

// Which tiles an XCD works, in order.  period == 0: a contiguous range of them.  Else a band: the tiles are lines of `period`
// (the rows between a row and the furthest one it meets), and an XCD takes its eighth of every line, line after line, so
// that what neighbouring lines share of B meets in that XCD's L2 an eighth of a line later instead of a whole one.
struct TileWalk {
    int64_t first, tiles, numTiles;
    uint32_t dies, period, from, width;
    __device__ __forceinline__ TileWalk(int64_t rows, int32_t tileRows, int32_t periodTiles)
    {
        numTiles = (rows + tileRows - 1) / tileRows;
        dies = gridDim.x < kNumXcd ? gridDim.x : kNumXcd;
        const uint32_t xcd = blockIdx.x % dies;
        period = periodTiles;
        const uint32_t span = period > 0 ? period : static_cast<uint32_t>(numTiles);
        const uint32_t per = span / dies, rem = span % dies;
        from = xcd * per + (xcd < rem ? xcd : rem);
        width = per + (xcd < rem ? 1 : 0);
        first = from;
        tiles = width;
        if (period > 0) {
            const int64_t whole = numTiles / period, rest = numTiles % period;
            const int64_t last = rest - from;
            tiles = whole * width + (last < 0 ? 0 : last < width ? last : width);
        }
    }
    __device__ __forceinline__ int64_t Tile(int64_t t) const
    {
        if (period == 0) {
            return first + t;
        }
        const uint32_t line = static_cast<uint32_t>(t) / width;
        return static_cast<int64_t>(line) * period + from + (static_cast<uint32_t>(t) - line * width);
    }
};

// A wavefront walks over tiles of 64 consecutive rows: values, lists and row starts as in SpmvOffsetRowsKernel.  P lanes
// take the 16-byte pieces of a row of B and C, so that 64 / P rows are worked at a time; the gathers of one distance are
// then 64 / P neighbouring rows of B, read as one stretch.  C is written past the caches: it would push the rows of B out
// that the next line of the mesh meets again (5-point 2048 x 2048, n = 4, 54 -> 48 us; 7-point 125 x 131 x 127, n = 32, 176 ->
// 169).  K >= the distances there are, U of them with their loads in flight together.
//
// us a call, the kernels for any columns / here: 5-point 2048 x 2048 n = 4 78 / 48 (the 320 MB it cannot do without at
// 6.6 TB/s), n = 8 120 / 88; 7-point 125 x 131 x 127 n = 16 131 / 97, n = 32 213 / 169; 9-point 900 x 901 n = 64 190 / 134;
// 27-point 71 x 77 x 79 n = 8 61 / 37, n = 64 184 / 156.  Wide B is bound by the data path of the vector memory, 86 % busy over a
// call of n = 32 (its address path 80 %): a row of B passes it once a distance, wherever it comes from (with every gather sent
// to the row itself and no C written n = 32 still takes 110 us).  Passes whose rows
// all have every distance, as inside a mesh, go without a branch an entry, one distance's elements widened at a time (9-point 1300 x
// 1200 n = 24 120 -> 105, n = 64 127 -> 114; 27-point 100 x 100 x 101 n = 4 47 -> 43, n = 64 153 -> 142; 7-point n = 12 82 -> 76).
template <typename ValT, typename CT, int P, typename Shape>
__global__ __launch_bounds__(kBlockThreads) void SpmmOffsetRowsKernel(
    const int32_t *__restrict__ rowOffsets, const ValT *__restrict__ vals, const ValT *__restrict__ B, CT *C, int64_t rows,
    int64_t cols, int32_t n, int64_t nnz, int64_t ldb, int64_t ldc, const uint8_t *__restrict__ ids,
    const uint32_t *__restrict__ masks, const int32_t *__restrict__ distance, int32_t distances, int32_t patterns,
    int32_t clampF16, int32_t period, int32_t passes, OpsparseScalar alphaS, OpsparseScalar betaS)
{
    using AccT = double;
    constexpr int V = 16 / sizeof(ValT);
    constexpr int kPassRows = kWave / P * Shape::kRows, U = Shape::kChunk;
    constexpr int Q = (kPassRows * MostPasses(P, Shape::kRows) * Shape::kMost + 4 * kWave - 1) / (4 * kWave);
    const int32_t tileRows = kPassRows * passes;
    struct RowInfo {
        uint32_t mask;
        int32_t at;
    };
    // (what the masked reads may touch past the last row's end behind them)
    __shared__ __align__(16) ValT stagedOf[kWaves][Q * 4 * kWave + 8];
    __shared__ RowInfo infoOf[kWaves][kWave];
    __shared__ uint32_t maskOf[kOffsetMaxPatterns];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
    ValT *const staged = stagedOf[wave];
    RowInfo *const info = infoOf[wave];
    if (threadIdx.x < kOffsetMaxPatterns) {
        maskOf[threadIdx.x] = static_cast<int32_t>(threadIdx.x) < patterns ? masks[threadIdx.x] : 0;
    }
    __syncthreads();

    const AccT alpha = ReadScalar<AccT>(alphaS);
    const AccT beta = ReadScalar<AccT>(betaS);
    const bool betaZero = (beta == AccT(0));

    const TileWalk walk(rows, tileRows, period);
    int64_t t = static_cast<int64_t>(blockIdx.x / walk.dies) * kWaves + wave;
    const int64_t step = (gridDim.x - blockIdx.x % walk.dies + walk.dies - 1) / walk.dies * kWaves;
    if (t >= walk.tiles) {
        return;
    }
    const int32_t piece = lane % P;
    // (lanes past the row's pieces take the last one again and store nothing)
    const int32_t col = piece * V < n ? piece * V : (n - 1) / V * V;
    const int32_t width = piece * V < n ? (n - col < V ? n - col : V) : 0;
    const int32_t dMin = distance[0], dMax = distance[distances - 1];

    int32_t bound;
    uint32_t id;
    auto askTile = [&](int64_t tile) {
        const int64_t first = walk.Tile(tile) * tileRows;
        const int64_t last = first + tileRows < rows ? first + tileRows : rows;
        bound = LoadStream(rowOffsets + ((lane & 1) != 0 ? last : first));
        id = LoadStream(ids + first + (lane < tileRows ? lane : 0));  // (the table is padded to whole tiles)
    };
    // One row's piece out (beta == 0 and != 0 apart: a wait for old C would be one for the stores before it, too).
    auto result = [&](AccT v) {
        if (std::is_same<CT, Half>::value && clampF16 != 0) {
            v = v > AccT(65504.0) ? AccT(65504.0) : v;
            v = v < AccT(-65504.0) ? AccT(-65504.0) : v;
        }
        return FromAcc<CT>(v);
    };
    auto store = [&](CT *out, const Piece<CT, V> &res) {
        if (width == V) {
            StorePiece<CT, V>(out, res);
        } else {
#pragma unroll
            for (int i = 0; i < V; ++i) {
                if (i < width) {
                    out[i] = res.e[i];
                }
            }
        }
    };
    auto finish = [&](AccT (&acc)[V], int64_t r) {
        CT *const out = C + r * ldc + col;
        Piece<CT, V> res;
        if (betaZero) {
#pragma unroll
            for (int i = 0; i < V; ++i) {
                res.e[i] = result(alpha * acc[i]);
            }
            store(out, res);
        } else {
#pragma unroll
            for (int i = 0; i < V; ++i) {
                // (a piece of fewer columns reads its first one again behind them)
                res.e[i] = result(alpha * acc[i] + beta * ToAcc<AccT>(out[i < width ? i : 0]));
            }
            store(out, res);
        }
    };
    askTile(t);
    while (true) {
        const int64_t r0 = walk.Tile(t) * tileRows;
        const int64_t tNext = t + step;
        const bool more = tNext < walk.tiles;
        const uint32_t list = id;
        const int32_t first = __builtin_amdgcn_readlane(bound, 0);
        const int32_t count = __builtin_amdgcn_readlane(bound, 1) - first;
        // (a piece of fewer than V columns reads on into the next rows: up to V - 1 of them where ldb is 1)
        const bool whole = r0 + tileRows <= rows && r0 + dMin >= 0 && r0 + tileRows + dMax + V <= cols && first >= 0 &&
                           count >= 1 && count <= Q * 4 * kWave && first + static_cast<int64_t>(count) + 3 <= nnz;
        if (whole) {
            FourOf<ValT> q[Q];
#pragma unroll
            for (int u = 0; u < Q; ++u) {
                int32_t k = (u * kWave + lane) * 4;  // (lanes past the end: the last quad again, not used)
                k = k < count ? k : (count - 1) & ~3;
                if (u * 4 * kWave < count) {
                    q[u] = __builtin_nontemporal_load(reinterpret_cast<const FourOf<ValT> *>(vals + first + k));
                }
            }
            if (more) {
                askTile(tNext);
            }
            const uint32_t mask = lane < tileRows ? maskOf[list % kOffsetMaxPatterns] : 0;
            const int32_t size = __popc(mask);
            int32_t start = WaveScan(size) - size;
            start = start + size > count ? 0 : start;  // (never, in the matrix that was analysed)
            info[lane] = RowInfo{mask, start};
#pragma unroll
            for (int u = 0; u < Q; ++u) {
                if (u * 4 * kWave < count) {
                    __builtin_memcpy(__builtin_assume_aligned(staged + (u * kWave + lane) * 4, 4 * sizeof(ValT)), &q[u],
                                     4 * sizeof(ValT));
                }
            }
            for (int32_t pass = 0; pass < passes; ++pass) {
                if constexpr (Shape::kRows == 2) {
                    const int32_t l = pass * kPassRows + lane / P * 2;
                    const ValT *const from = B + ((r0 + l) * ldb + col);
                    AccT acc[2][V] = {};
                    const RowInfo mine[2] = {info[l], info[l + 1]};
                    int32_t at[2] = {mine[0].at, mine[1].at};
                    for (int32_t k0 = 0; k0 < distances; k0 += U) {
                        Piece<ValT, V> b[Shape::kLoads];
                        {
                            int load = 0, k = 0;
#pragma unroll
                            for (int g = 0; g < Shape::kRuns; ++g) {
                                const ValT *const run = from + static_cast<int64_t>(distance[k0 + k]) * ldb;
#pragma unroll
                                for (int i = 0; i <= Shape::kSize[g]; ++i) {
                                    b[load++] = LoadPiece<ValT, V>(run + i * ldb);
                                }
                                k += Shape::kSize[g];
                            }
                        }
                        const uint32_t bits[2] = {mine[0].mask >> k0, mine[1].mask >> k0};
                        ValT v[2][U];
#pragma unroll
                        for (int j = 0; j < 2; ++j) {
#pragma unroll
                            for (int u = 0; u < U; ++u) {
                                v[j][u] = staged[at[j]];
                                at[j] += (bits[j] >> u) & 1;
                            }
                        }
                        constexpr uint32_t kAll = (1u << U) - 1;
                        if (__all((bits[0] & bits[1] & kAll) == kAll)) {
                            int load = 0, k = 0;
#pragma unroll
                            for (int g = 0; g < Shape::kRuns; ++g) {
#pragma unroll
                                for (int i = 0; i <= Shape::kSize[g]; ++i, ++load) {
                                    AccT wide[V];
#pragma unroll
                                    for (int c = 0; c < V; ++c) {
                                        wide[c] = ToAcc<AccT>(b[load].e[c]);
                                    }
#pragma unroll
                                    for (int j = 0; j < 2; ++j) {
                                        if (i - j >= 0 && i - j < Shape::kSize[g]) {
                                            const AccT w = ToAcc<AccT>(v[j][k + i - j]);
#pragma unroll
                                            for (int c = 0; c < V; ++c) {
                                                acc[j][c] += w * wide[c];
                                            }
                                        }
                                    }
                                }
                                k += Shape::kSize[g];
                            }
                        } else {
                            int load = 0, k = 0;
#pragma unroll
                            for (int g = 0; g < Shape::kRuns; ++g) {
#pragma unroll
                                for (int i = 0; i <= Shape::kSize[g]; ++i, ++load) {
                                    // (opaque, so that its conversions are not made ahead of the branch for both of its arms:
                                    // that takes twice the registers of b)
                                    Int4U raw;
                                    __builtin_memcpy(&raw, b[load].e, 16);
                                    asm volatile("" : "+v"(raw));
                                    Piece<ValT, V> here;
                                    __builtin_memcpy(here.e, &raw, 16);
#pragma unroll
                                    for (int j = 0; j < 2; ++j) {
                                        if (i - j >= 0 && i - j < Shape::kSize[g] && ((bits[j] >> (k + i - j)) & 1) != 0) {
                                            const AccT w = ToAcc<AccT>(v[j][k + i - j]);
#pragma unroll
                                            for (int c = 0; c < V; ++c) {
                                                acc[j][c] += w * ToAcc<AccT>(here.e[c]);
                                            }
                                        }
                                    }
                                }
                                k += Shape::kSize[g];
                            }
                        }
                    }
                    finish(acc[0], r0 + l);
                    finish(acc[1], r0 + l + 1);
                } else {
                    const int32_t l = pass * kPassRows + lane / P;
                    const ValT *const from = B + ((r0 + l) * ldb + col);
                    AccT acc[V] = {};
                    const RowInfo mine = info[l];
                    int32_t at = mine.at;
                    auto chunk = [&](int32_t k0) {
                        Piece<ValT, V> b[U];
#pragma unroll
                        for (int u = 0; u < U; ++u) {
                            b[u] = LoadPiece<ValT, V>(from + static_cast<int64_t>(distance[k0 + u]) * ldb);
                        }
                        const uint32_t bits = mine.mask >> k0;
                        ValT v[U];
                        constexpr uint32_t kAll = (1u << U) - 1;
                        if (__all((bits & kAll) == kAll)) {
#pragma unroll
                            for (int u = 0; u < U; ++u) {
                                v[u] = staged[at + u];
                            }
                            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                            for (int u = 0; u < U; ++u) {
                                const AccT w = ToAcc<AccT>(v[u]);
#pragma unroll
                                for (int i = 0; i < V; ++i) {
                                    acc[i] += w * ToAcc<AccT>(b[u].e[i]);
                                }
                                __builtin_amdgcn_sched_barrier(0);  // (what a distance widens is not kept beside the next one's)
                            }
                            at += U;
                        } else {
#pragma unroll
                            for (int u = 0; u < U; ++u) {
                                v[u] = staged[at];
                                at += (bits >> u) & 1;
                            }
#pragma unroll
                            for (int u = 0; u < U; ++u) {
                                // (opaque, so that its conversions are not made ahead of the branch for both of its arms)
                                Int4U raw;
                                __builtin_memcpy(&raw, b[u].e, 16);
                                asm volatile("" : "+v"(raw));
                                Piece<ValT, V> here;
                                __builtin_memcpy(here.e, &raw, 16);
                                if (((bits >> u) & 1) != 0) {
                                    const AccT w = ToAcc<AccT>(v[u]);
#pragma unroll
                                    for (int i = 0; i < V; ++i) {
                                        acc[i] += w * ToAcc<AccT>(here.e[i]);
                                    }
                                }
                            }
                        }
                    };
                    if constexpr (Shape::kMost == U) {
                        chunk(0);
                    } else {
                        for (int32_t k0 = 0; k0 < distances; k0 += U) {
                            chunk(k0);
                        }
                    }
                    finish(acc, r0 + l);
                }
            }
        } else {
            for (int32_t l0 = 0; l0 < tileRows; l0 += kWave / P) {
                const int64_t r = r0 + l0 + lane / P;
                const uint32_t mask = maskOf[__shfl(static_cast<int32_t>(list), l0 + lane / P, kWave) %
                                             kOffsetMaxPatterns];
                if (r < rows) {
                    int64_t k = rowOffsets[r];
                    AccT acc[V] = {};
                    for (int32_t e = 0; e < distances; ++e) {
                        if (((mask >> e) & 1) != 0 && k >= 0 && k < nnz) {
                            int64_t c = r + distance[e];
                            c = c < 0 ? 0 : (c < cols ? c : cols - 1);
                            const AccT v = ToAcc<AccT>(vals[k]);
#pragma unroll
                            for (int i = 0; i < V; ++i) {
                                acc[i] += v * ToAcc<AccT>(B[c * ldb + (i < width ? col + i : col)]);
                            }
                            ++k;
                        }
                    }
                    finish(acc, r);
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

template <typename ValT, typename CT>
int LaunchTyped(const OffsetSpmmArgs &a)
{
    const OffsetLayout l = MakeOffsetLayout(a.rows);
    constexpr int V = 16 / sizeof(ValT);
    auto launch = [&](auto piecesTag, auto shapeTag) {
        constexpr int P = decltype(piecesTag)::value;
        using Shape = decltype(shapeTag);
        constexpr int32_t kPassRows = kWave / P * Shape::kRows;
        int32_t passes = MostPasses(P, Shape::kRows);
        while (passes > 1 && a.rows < kEnoughTiles * passes * kPassRows) {
            passes /= 2;  // (9-point mesh of 140 K rows, n = 12: 14.3 us with four passes, 12.6 by the other kernels)
        }
        const int32_t tileRows = passes * kPassRows;
        // Bands where a line is too long for the L2s to keep and wide enough to be cut in eight (us, contiguous / bands:
        // 7-point mesh of 125 x 131 x 127, lines of 16 375 rows, n = 12 85.2 / 87.8, n = 16 105 / 97, n = 32 190 / 169;
        // 101 x 97 x 99, n = 64, 175 / 158; 27-point of 71 x 77 x 79, 5 546 rows, n = 32 93 / 91, n = 64 171 / 156; 9-point
        // mesh with lines of 901 rows, 28 tiles, n = 32 71 / 82).
        const int64_t line = (a.reach + tileRows / 2) / tileRows;
        const bool bands = line >= 16 * kNumXcd && a.reach * a.n * static_cast<int64_t>(sizeof(ValT)) >= kBandBytes;
        const int32_t period = bands ? static_cast<int32_t>(line) : 0;
        int64_t grid = (a.rows + kWaves * tileRows - 1) / (kWaves * tileRows);
        grid = grid > kOffsetGrid ? kOffsetGrid : grid;
        hipLaunchKernelGGL((SpmmOffsetRowsKernel<ValT, CT, P, Shape>), dim3(static_cast<uint32_t>(grid)),
                           dim3(kBlockThreads), 0, a.stream, a.rowOffsets, static_cast<const ValT *>(a.vals),
                           static_cast<const ValT *>(a.B), static_cast<CT *>(a.C), a.rows, a.cols,
                           static_cast<int32_t>(a.n), a.nnz, a.ldb, a.ldc, a.part + l.idOff,
                           reinterpret_cast<const uint32_t *>(a.part + l.maskOff),
                           reinterpret_cast<const int32_t *>(a.part) + kOffsetHeaderDistances, a.distances, a.patterns,
                           std::is_same<CT, Half>::value ? 1 : 0, period, passes, a.alpha, a.beta);
        return CheckLaunch();
    };
    auto chunked = [&](auto piecesTag) {
        // Two rows a lane under the widest B only: it takes 150 - 200 registers, two wavefronts a SIMD (us, one row / two:
        // n = 128 7-point 213 / 192, 9-point 291 / 230, 5-point 174 / 154, 27-point 304 / 267; n = 256 7-point 146 / 125; but
        // n = 64 155 / 159, 140 / 123, 132 / 127, 157 / 179 and n = 32 172 / 190, 72 / 85, -, 93 / 113).
        if constexpr (decltype(piecesTag)::value >= 32) {
            if (a.runs == kOffsetRuns131) return launch(piecesTag, Runs<5, 1, 3, 1>{});
            if (a.runs == kOffsetRuns11311) return launch(piecesTag, Runs<7, 1, 1, 3, 1, 1>{});
            if (a.runs == kOffsetRuns333 && a.distances <= 9) return launch(piecesTag, Runs<9, 3, 3, 3>{});
            if (a.runs == kOffsetRuns333) return launch(piecesTag, Runs<27, 3, 3, 3>{});
        }
        if (a.distances <= 5) return launch(piecesTag, Chunks<5, 5>{});
        if (a.distances <= 7) return launch(piecesTag, Chunks<7, 7>{});
        if (a.distances <= 9) return launch(piecesTag, Chunks<9, 9>{});
        return launch(piecesTag, Chunks<9, 32>{});
    };
    const int64_t pieces = (a.n + V - 1) / V;
    if (pieces <= 1) return chunked(std::integral_constant<int, 1>{});
    if (pieces <= 2) return chunked(std::integral_constant<int, 2>{});
    if (pieces <= 4) return chunked(std::integral_constant<int, 4>{});
    if (pieces <= 8) return chunked(std::integral_constant<int, 8>{});
    if (pieces <= 16) return chunked(std::integral_constant<int, 16>{});
    if (pieces <= 32) return chunked(std::integral_constant<int, 32>{});
    if constexpr (sizeof(ValT) == 4) {
        if (pieces <= 64) return chunked(std::integral_constant<int, 64>{});
    }
    return OPSPARSE_E_UNSUPPORTED;
}

}  // namespace

bool OffsetSpmmTakes(int64_t n, int64_t ldb, int64_t ldc, const void *B, const void *C, int32_t valType, int32_t cType)
{
    if (n < 1 || n > kOffsetMaxColumns || ldb < n || ldc < n) {
        return false;
    }
    if (valType == OPSPARSE_F32 && cType == OPSPARSE_F32) {
        return reinterpret_cast<uintptr_t>(B) % 4 == 0 && reinterpret_cast<uintptr_t>(C) % 4 == 0;
    }
    return valType == OPSPARSE_F16 && (cType == OPSPARSE_F16 || cType == OPSPARSE_F32) && n % 8 == 0 && ldb % 8 == 0 &&
           ldc % 8 == 0 && reinterpret_cast<uintptr_t>(B) % 16 == 0 && reinterpret_cast<uintptr_t>(C) % 16 == 0;
}

int LaunchOffsetSpmm(const OffsetSpmmArgs &a, int32_t valType, int32_t cType)
{
    if (a.part == nullptr || a.cols < 1 || a.rows < 1 || a.patterns < 1 || a.patterns > kOffsetMaxPatterns ||
        a.distances < 1 || a.distances > kOffsetMaxDistances ||
        !OffsetSpmmTakes(a.n, a.ldb, a.ldc, a.B, a.C, valType, cType)) {
        return OPSPARSE_E_INVALID;
    }
    if (valType == OPSPARSE_F32) return LaunchTyped<float, float>(a);
    return cType == OPSPARSE_F16 ? LaunchTyped<Half, Half>(a) : LaunchTyped<Half, float>(a);
}

}  // namespace opsparse
