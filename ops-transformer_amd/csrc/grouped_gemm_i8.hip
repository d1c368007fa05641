// Expert-grouped int8 x int8 -> int32 GEMM for gfx950 (CDNA4) with fused epilogues.
//
// Computes, for every group e and every row r of that group, acc[r, c] = sum_k x[r, k] * w[e, k, c] on
// v_mfma_i32_16x16x64_i8 and applies one of three epilogues in registers:
//   kInt32   raw accumulators                                   (aclnnGroupedMatmulV4, int32 output)
//   kDequant (float(acc) * scale[e, c]) * rowScale[r] -> bf16 / fp16 / fp32
//            (reference order: gmm/grouped_matmul/op_kernel/grouped_matmul_quant_mixcore.h:248-291,293-310)
//   kSwiglu  C = (float(acc) * rowScale[r]) * scale[e, c];  S = swish(C[:, j]) * C[:, j + N/2]
//            (reference order: gmm/grouped_matmul_swiglu_quant/op_kernel/grouped_matmul_swiglu_quant.h:368-399,446-474),
//            S is written as fp32 together with one partial max |S| per (n-tile, row); a second, bandwidth-trivial
//            kernel folds the partials and turns S into int8 with the row scale max/127 (same file :477-513).
//
// Scheduling.  Group sizes live in device memory, so a one-workgroup kernel (here) turns groupList into one table entry
// per m-tile -- big m-tiles first, then those of at most 64 rows -- plus tile counters.  Each run of the table is cut
// into eight contiguous shares, one per XCD, so that the workgroups of an XCD sit on neighbouring tiles (shared
// activation rows and weight columns stay in that XCD's L2); workgroups pull their tiles from the counters, or walk
// fixed shares where tiles are too short to hide a draw.
//
// This file: the scheduling kernel, the requantisation kernel, planning and the launch sequence.  The GEMM kernels
// themselves are in grouped_gemm_i8_kernels.h and are instantiated by one translation unit per epilogue:
//   StreamGemmKernel  the fast path (K a multiple of 16; K-contiguous, blocked or row-major [K, N] weights).  Persistent
//                     workgroups; operands go global -> LDS with global_load_lds_dwordx4 into rings of 2..4 stages of
//                     128 k-bytes (192-row tiles: two activation and three weight stages), so several stages of weights
//                     are in flight per CU with no staging registers, and the rings already hold the next tile's first
//                     steps while the current tile's epilogue runs.
//   MixedGemmKernel   the same body twice, once per run of the table with a stage geometry of its own (pulled tiles of
//                     192 and 256 rows).
//   GenericGemmKernel byte-wise loader for K off the 16-byte grid or below 128 and, with the other two weight layouts,
//                     channel counts off theirs: correct, slow.
// LDS rows are XOR-swizzled in 16-byte chunks so that the 16 lanes the LDS serves per clock (64 banks) never collide,
// for the DMA writes as well as for the MFMA operand reads.
#include "grouped_gemm_i8.h"

#include <cmath>
#include <mutex>
#include <vector>

#include "grouped_gemm_i8_kernels.h"

namespace gemm {
namespace {

// ---------------------------------------------------------------------------------------------- scheduling kernel
struct SchedArgs {
    const void* groupList;
    int32_t* sched;
    int32_t groups;
    int32_t groupListIsInt64;
    int32_t isCount;  // 0 cumsum, 1 counts, 2 sparse (expert id, count) pairs
    int32_t tileM;
    int32_t mayLower;  // 1: m-tiles of kLowTileM rows instead where they leave at most an eighth of the groups a small last one;
                       // 3: for means below those, by how many groups are small or have several m-tiles;
                       // 2: where they fill at most two rounds of the machine, and no more of them than the tall ones
    // with mayLower 3:
    int32_t lowIsWide;   // the tiles of the lower m-tiles are two 256-channel units wide
    int32_t offGrid;     // weights whose rows begin inside cache lines (Plan::offGrid)
    int32_t maySmall;    // or all m-tiles of kSmallRows rows
    int32_t kSteps;
    int32_t cus, tilesN;
    int32_t maxMTiles;
    int64_t M;
    int64_t rowBegin, rowEnd;  // only rows in [rowBegin, rowEnd) get tiles (one band of a launch that runs in row bands)
};

// A group's m-tiles of at most `cut` rows, and the cost of the big ones.
struct Cut {
    int32_t big, small, bigCost;
};
__device__ __forceinline__ Cut CutOf(int32_t rows, int32_t cut, bool allSmall, bool oneList) {
    const int32_t tiles = (rows + cut - 1) / cut, lastRows = tiles > 0 ? rows - (tiles - 1) * cut : 0;
    Cut c{};
    c.small = allSmall ? tiles : (!oneList && tiles > 0 && lastRows <= kSmallRows ? 1 : 0);
    c.big = tiles - c.small;
    if (c.big > 0) {
        const bool lastIsBig = c.small == 0;
        c.bigCost = (c.big - (lastIsBig ? 1 : 0)) * max(cut >> 5, kSmallCost) + (lastIsBig ? max((lastRows + 31) >> 5, kSmallCost) : 0);
    }
    return c;
}

// One workgroup a table: two problems on one group list share a launch (SharedSchedule).
__global__ __launch_bounds__(1024) void ScheduleKernel(SchedArgs first, SchedArgs second) {
    const SchedArgs a = blockIdx.x == 0 ? first : second;
    __shared__ int32_t scan[1024];
    const int t = threadIdx.x;
    auto at = [&](int i) -> int64_t {
        return a.groupListIsInt64 ? static_cast<const int64_t*>(a.groupList)[i]
                                  : static_cast<int64_t>(static_cast<const int32_t*>(a.groupList)[i]);
    };
    // Inclusive prefix sums over the 1024 threads: shuffles inside each wave, then the sixteen wave totals through LDS, all of
    // which every thread reads (one round trip; a loop over the waves before it was fifteen).  Each is called once at most, so that
    // nobody waits for earlier totals to have been read.
    __shared__ int32_t waveTotal[16];
    auto inclusiveScan = [&](int32_t v) -> int32_t {
        const int lane = t & 63, wave = t >> 6;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int32_t below = __shfl_up(v, d, 64);
            if (lane >= d) v += below;
        }
        if (lane == 63) waveTotal[wave] = v;
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 15; ++i) v += i < wave ? waveTotal[i] : 0;
        return v;
    };
    // the same over two values of two 32-bit counts each, packed into 64 bits (neither half may overflow into the other)
    __shared__ uint64_t waveTotal64[2][16];
    auto inclusiveScan64 = [&](uint64_t& v, uint64_t& w) {
        const int lane = t & 63, wave = t >> 6;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const uint64_t belowV = __shfl_up(v, d, 64), belowW = __shfl_up(w, d, 64);
            if (lane >= d) {
                v += belowV;
                w += belowW;
            }
        }
        if (lane == 63) {
            waveTotal64[0][wave] = v;
            waveTotal64[1][wave] = w;
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 15; ++i) {
            v += i < wave ? waveTotal64[0][i] : 0;
            w += i < wave ? waveTotal64[1][i] : 0;
        }
    };
    // group boundaries, clamped into [0, M], no end before its begin, so that a malformed list cannot push rows out of range
    int64_t begin = 0, end = 0;
    if (a.isCount == 2) {
        // Sparse list [groups, 2]: pair p = (expert id, rows); pairs take consecutive row ranges in list order and the
        // list ends at the first pair without rows.  The table stays indexed by expert: an expert named by a pair gets
        // that pair's row range, every other expert none (an expert named twice keeps the later range only).
        __shared__ int32_t firstEmpty;
        __shared__ int32_t expertBegin[kMaxGroups], expertEnd[kMaxGroups];
        if (t == 0) firstEmpty = a.groups;
        expertBegin[t] = 0;
        expertEnd[t] = 0;
        __syncthreads();
        int64_t key = -1, val = 0;
        if (t < a.groups) {
            key = at(2 * t);
            val = at(2 * t + 1);
            if (val <= 0) atomicMin(&firstEmpty, t);
        }
        __syncthreads();
        if (t >= firstEmpty) val = 0;
        val = val > a.M ? a.M : val;
        const int32_t inc = inclusiveScan(static_cast<int32_t>(val));
        int64_t pairEnd = inc, pairBegin = inc - val;
        pairBegin = pairBegin > a.M ? a.M : pairBegin;
        pairEnd = pairEnd > a.M ? a.M : pairEnd;
        if (val > 0 && key >= 0 && key < a.groups) {
            expertBegin[key] = static_cast<int32_t>(pairBegin);
            expertEnd[key] = static_cast<int32_t>(pairEnd);
        }
        __syncthreads();
        begin = expertBegin[t];
        end = expertEnd[t];
    } else if (t < a.groups) {
        if (a.isCount) {
            int64_t c = at(t);
            c = c < 0 ? 0 : (c > a.M ? a.M : c);
            end = c;  // turned into a cumsum below
        } else {
            end = at(t);
            begin = t > 0 ? at(t - 1) : 0;
        }
    }
    if (a.isCount == 1) {
        const int32_t inc = inclusiveScan(static_cast<int32_t>(end));
        begin = static_cast<int64_t>(inc) - end;
        end = inc;
    }
    begin = begin < 0 ? 0 : (begin > a.M ? a.M : begin);
    end = end < begin ? begin : (end > a.M ? a.M : end);
    // the band of rows this launch covers: a group keeps the part of its rows that lies inside
    begin = begin < a.rowBegin ? a.rowBegin : (begin > a.rowEnd ? a.rowEnd : begin);
    end = end < a.rowBegin ? a.rowBegin : (end > a.rowEnd ? a.rowEnd : end);
    const int32_t rows = t < a.groups ? static_cast<int32_t>(end - begin) : 0;
    int32_t tileM = a.tileM, cut = tileM;  // cut: rows per m-tile of this group
    int32_t wide = 0;
    bool oneList = false;  // small m-tiles among the big ones
    bool dealt = false;    // every tile belongs to a workgroup from the start
    if (a.mayLower == 2) {
        // Whole rounds of the machine, one of low tiles costing 0.7 to 0.85 of one of tall ones: their ring is a stage deeper, and
        // the launch ends with its tallest tile.  Low tiles where they are one round; where they are two, only if the tall ones
        // are two as well, not counting what runs as small tiles.  us, planned height -> this, K-contiguous / row-major:
        //   8 experts, K 14336 x N 4096: 180 rows each 157 -> 134 / 164 -> 141, 250 rows 176 -> 143 / 176 -> 154, 600 rows 326 -> 274 / 330 -> 293
        //   8 experts, 1024 x 1024 and gate/up 1024 x 2 x 1024: 250 rows 31 -> 27 and 34 -> 30
        //   two rounds for one and a few small tiles, left alone: 16 experts, K 8192 x N 1024, 1000 rows 149 (154 low)
        const uint32_t low = (rows + kLowTileM - 1) / kLowTileM, tall = (rows + tileM - 1 - kSmallRows) / tileM;
        __shared__ uint32_t sLow, sTall;
        if (t == 0) sLow = sTall = 0;
        __syncthreads();
        if ((t & ~63) < a.groups) {  // the sums of a wave by shuffles: atomics of 64 lanes are a loop of 64 trips each
            uint32_t lowSum = low, tallSum = tall;
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) {
                lowSum += __shfl_xor(lowSum, d, 64);
                tallSum += __shfl_xor(tallSum, d, 64);
            }
            if ((t & 63) == 0) {
                atomicAdd(&sLow, lowSum);
                atomicAdd(&sTall, tallSum);
            }
        }
        __syncthreads();
        // (neither product overflows: a launch with this choice has at most two rounds of M / kLowTileM rows)
        const uint32_t cus = a.cus, lowTiles = sLow * a.tilesN;
        if (lowTiles <= cus || (lowTiles <= 2 * cus && sTall * a.tilesN > cus)) {
            tileM = kLowTileM;
            // Even tiles, in sixteens: 160 + 20 rows would read the weights twice, at two paces.  The last one is what is left, of many
            // tiles sometimes next to nothing (1441 rows: nine of 160 and one of 1); blocks dealt out exactly measured the same.
            cut = low > 0 ? static_cast<int32_t>(((rows + low - 1) / low + 15) & ~15u) : kLowTileM;
        }
    } else if (a.mayLower) {
        const int32_t last = rows % kLowTileM;
        const bool smallLast = last > 0 && last <= kSmallRows;
        bool lower, narrow = false;
        if (a.mayLower == 1) {
            lower = __syncthreads_count(smallLast) * 8 <= a.groups;
        } else {
            // us; experts, rows each on average at popularity rank^-s, sizes of the launch.
            // Groups of at most kSmallRows rows, nearly all of them: the two-geometry kernel's small run.  One geometry / that: 256
            // of 50, 7168 x 2 x 2048 1285 (wide), 2048 x 7168 736 / 1170, 708.  Half of them, beside groups of
            // several m-tiles: that too, of 80 at s 0.6 875 / 808 (down).  Otherwise one geometry.
            // Wide tiles are half as many, and a launch of a part of a round ends with a tile of twice the length: beside second m-tiles of
            // more than a few groups they are taken where few groups are small and there are four rounds of them, two geometries / that:
            // 7168 x 2 x 2048, 256 of 100 at s 0.4 1541 / 1440; 1024 x 2 x 1024 170 / 147; not 7168 x 2 x 2048, 256 of 128 even, one of
            // 161 rows 1440 / 1463, nor 32 of 100 at s 0.4 245 / 267; and where they fill at most two rounds of the machine well:
            // 4096 x 2 x 1536, 32 of 80 at s 1.2 121 / 88.
            // (Counted by ballots and one round of LDS: four __syncthreads_count took 3 us.)
            __shared__ int4 waveCounts[16];
            const int4 mine = make_int4(__popcll(__ballot(rows > 0)), __popcll(__ballot(rows > 0 && rows <= kSmallRows)),
                                        __popcll(__ballot(rows > kLowTileM)), __popcll(__ballot(rows > kLowTileM && smallLast)));
            if ((t & 63) == 0) waveCounts[t >> 6] = mine;
            __syncthreads();
            int32_t some = 0, small = 0, over = 0, loses = 0;
#pragma unroll
            for (int w = 0; w < 16; ++w) {
                some += waveCounts[w].x;
                small += waveCounts[w].y;
                over += waveCounts[w].z;
                loses += waveCounts[w].w;
            }
            const bool fewSmall = small * 8 < some * 7, manyOver = over * 16 > some;
            const bool offGridOver = a.offGrid != 0 && over > 0, oneOrTwo = a.lowIsWide && !a.maySmall && fewSmall && manyOver;
            if (a.lowIsWide) lower = over == 0 && (fewSmall || a.offGrid);
            else lower = a.offGrid == kOffGridLong || (fewSmall && loses * 8 <= a.groups && (small * 2 < some || over * 32 < a.groups));
            // What asks for sums over the groups asks once more (1.7 us): the m-tiles of the lowest height, and in two geometries the big
            // ones and the cost of all.
            if (!lower && (a.maySmall || offGridOver || oneOrTwo)) {
                __shared__ uint2 waveSums[16];
                const Cut planned = CutOf(rows, tileM, false, false);
                const int32_t lowestHeight = a.maySmall ? kSmallRows : kLowTileM;
                // (the two counts in one register, where a wave's sums stay below 2^16)
                uint32_t countSum = min((rows + lowestHeight - 1) / lowestHeight, 1023) | min(planned.big, 1023) << 16;
                uint32_t costSum = planned.bigCost + planned.small * kSmallCost;
#pragma unroll
                for (int d = 1; d < 64; d <<= 1) {
                    countSum += __shfl_xor(countSum, d, 64);
                    costSum += __shfl_xor(costSum, d, 64);
                }
                if ((t & 63) == 0) waveSums[t >> 6] = make_uint2(countSum, costSum);
                __syncthreads();
                uint32_t lowestSum = 0, bigSum = 0;
                costSum = 0;
#pragma unroll
                for (int w = 0; w < 16; ++w) {
                    lowestSum += waveSums[w].x & 0xffffu;
                    bigSum += waveSums[w].x >> 16;
                    costSum += waveSums[w].y;
                }
                const float perCu = static_cast<float>(a.tilesN) / static_cast<float>(a.cus);  // rounds of the machine that an m-tile's tiles are
                const float wideRounds = static_cast<float>(lowestSum) * static_cast<float>((a.tilesN + 1) / 2) / static_cast<float>(a.cus);
                if (a.maySmall) {
                    // Means that 64-row tiles hold: those for every group, dealt out whole, where the weights that groups of several of them
                    // read again cost less than the change of geometry, 8 k-steps' time, or 12 with more big tiles than workgroups begin
                    // with.  A round that has begun is half a one at least (a quarter behind tiles that are drawn).  64-row tiles / two
                    // geometries: 2048 x 2 x 2048, 64 of 25 at s 0.4 104 / 108, of 32 at s 1.2 119 / 110; 7168 x 2 x 2048, 64 of 25 at
                    // s 0.4 327 / 298.  (The ones of a fixed share took 104 too, drawn ones 111.)
                    auto begun = [](float r, float least) { return floorf(r) + (r > floorf(r) ? fmaxf(r - floorf(r), least) : 0.0f); };
                    const float kSteps = static_cast<float>(a.kSteps), change = static_cast<float>(bigSum) * perCu * 8.0f <= 7.0f ? 8.0f : 12.0f;
                    if (begun(static_cast<float>(lowestSum) * perCu, 0.5f) * kSteps <
                        begun(static_cast<float>(costSum) * perCu * (1.0f / kSmallCost), 0.25f) * kSteps + change) {
                        tileM = cut = kSmallRows;
                        dealt = true;
                    }
                } else if (a.offGrid == kOffGridLong) {
                    lower = true;
                    narrow = wideRounds < 4.0f;
                } else {
                    lower = oneOrTwo && (wideRounds <= 2.0f ? wideRounds * 6.0f >= ceilf(wideRounds) * 5.0f : small * 4 < some && wideRounds >= 4.0f);
                    if (!lower && offGridOver && fewSmall && manyOver) lower = narrow = true;
                }
            }
        }
        if (lower) {
            tileM = cut = kLowTileM;
            wide = a.lowIsWide && !narrow;
            oneList = a.mayLower == 3;
        }
    }
    // big and small m-tiles of this group (with tiles of at most kSmallRows rows every m-tile is small; otherwise only
    // a group's last, partly filled m-tile can be) and the cost of the big ones; two packed prefix sums give every
    // group the positions of its m-tiles in the two runs of the table, and the launch the totals
    const bool allSmall = tileM <= kSmallRows;
    const Cut own = CutOf(rows, cut, allSmall, oneList);
    const int32_t tiles = own.big + own.small, smallCount = own.small, bigCount = own.big, bigCost = own.bigCost;
    uint64_t countsInc = static_cast<uint64_t>(tiles) | (static_cast<uint64_t>(bigCount) << 32);
    uint64_t costInc = static_cast<uint64_t>(bigCost) | (static_cast<uint64_t>(tiles > 0 ? 1 : 0) << 32);
    inclusiveScan64(countsInc, costInc);
    const int32_t tileInc = static_cast<int32_t>(countsInc & 0xffffffffu), bigInc = static_cast<int32_t>(countsInc >> 32);
    // rows covered by the list: the end of the last group, or with a sparse list the furthest end of any expert
    int32_t covered = static_cast<int32_t>(end);
    if (a.isCount == 2) {
        scan[t] = t < a.groups ? static_cast<int32_t>(end) : 0;
        __syncthreads();
        for (int d = 512; d > 0; d >>= 1) {
            if (t < d) scan[t] = max(scan[t], scan[t + d]);
            __syncthreads();
        }
        covered = scan[0];
        __syncthreads();
    }
    __shared__ int32_t sRowStart[kMaxGroups], sRows[kMaxGroups], sCut[kMaxGroups], sBigBefore[kMaxGroups], sSmallBefore[kMaxGroups];
    __shared__ int32_t totals[4];
    sRowStart[t] = static_cast<int32_t>(begin);
    sRows[t] = rows;
    sCut[t] = cut;
    sBigBefore[t] = bigInc - bigCount;
    sSmallBefore[t] = (tileInc - bigInc) - smallCount;
    __shared__ int32_t sCovered;
    if (t == a.groups - 1) sCovered = covered;
    if (t == 1023) {
        totals[0] = bigInc;
        totals[1] = tileInc - bigInc;
        totals[2] = static_cast<int32_t>(costInc & 0xffffffffu);
        totals[3] = static_cast<int32_t>(costInc >> 32);  // groups with rows
    }
    // group of every m-tile: scan[] takes the inclusive m-tile prefix (zero-tile groups repeat their
    // predecessor's value); m-tile m belongs to the first group whose inclusive prefix exceeds m
    scan[t] = t < a.groups ? tileInc : 0x7fffffff;
    __syncthreads();
    const int32_t totalMTiles = scan[a.groups - 1];
    // A well-formed list never needs more than maxMTiles m-tiles: the rows of the launch by the lowest height that MakePlan sizes the table
    // for, and one more per group.  A malformed one whose groups
    // overlap could: the m-tiles beyond the table are dropped, so no kernel indexes past it.
    const int32_t nBig = min(totals[0], a.maxMTiles);
    const int32_t nSmall = min(totals[1], a.maxMTiles - nBig);
    if (t < kQueueCounterInts) a.sched[kQueueHeaderInts + t] = 0;
    // Band width: with two or more m-tiles per group on average, four neighbouring m-tiles (mostly of one group) walk
    // the n-tiles together and share each weight column block through L2; with one m-tile per group the n-tiles of a
    // group follow each other, so that its activation rows are what stays in L2.  A small m-tile is its group's only
    // one of its kind unless every tile is small.
    const int32_t wideBands = totalMTiles >= 2 * totals[3] ? kGroupM : 1;
    if (t < kQueueHeaderInts) {
        a.sched[t] = t == 0 ? nBig : t == 1 ? nSmall : t == 2 ? nSmall * kSmallCost : t == 3 ? totals[2] : t == 4 ? wideBands
                   : t == 5 ? (allSmall ? wideBands : 1) : t == kHdrCoveredRows ? sCovered : t == kHdrTileM ? tileM
                   : t == kHdrWide ? wide
                   : t == kHdrEven ? dealt ? 2 : (totalMTiles * 8 <= totals[3] * 9 && (nSmall * 8 <= totals[3] || nBig == 0) ? 1 : 0) : 0;
    }
    int4* const mTileTable = reinterpret_cast<int4*>(a.sched + kQueueHeaderInts + kQueueCounterInts);
    for (int32_t m = t; m < totalMTiles; m += 1024) {
        int lo = -1, hi = a.groups - 1;  // scan[hi] > m always holds, scan[lo] <= m (lo = -1: nothing before)
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (scan[mid] > m) hi = mid; else lo = mid;
        }
        const int32_t inGroup = m - (hi > 0 ? scan[hi - 1] : 0);
        const int32_t tileRows = min(sCut[hi], sRows[hi] - inGroup * sCut[hi]);
        const bool small = allSmall || (!oneList && tileRows <= kSmallRows);
        const int32_t pos = small ? nBig + sSmallBefore[hi] + (allSmall ? inGroup : 0) : sBigBefore[hi] + inGroup;
        const int32_t limit = small ? nBig + nSmall : nBig;
        if (pos < limit) mTileTable[pos] = make_int4(hi, sRowStart[hi] + inGroup * sCut[hi], tileRows, 0);
    }
}

// ---------------------------------------------------------------------------------------------- requantisation
struct RequantArgs {
    const float* s;          // [rows of the band, halfN]: row r of the problem at index r - rowBegin
    const float* rowMax;     // partial max |S|: entry t of row r at r * maxRowStride + t * maxStride, t < partials
    int32_t partials;
    int64_t maxRowStride, maxStride;
    const int32_t* sched;
    int8_t* y;               // [M, halfN]
    float* yScale;           // [M]
    int32_t halfN;
    int64_t rowBegin;        // first row of the band; the grid covers the band's rows
};

__device__ __forceinline__ int8_t QuantOne(float s, float inv) {
    const __half h = __ushort_as_half(HalfBitsOfRounded(__fmul_rn(s, inv)));
    return static_cast<int8_t>(__float2int_rn(__half2float(h)));
}

// One workgroup per row; rows at or beyond the last group boundary are left untouched.
// Every thread requests its first two packets of S before the row maximum is known, and every wave folds the partial
// maxima for itself (a handful of L2 hits): the row's two dependent memory round trips overlap and there is no barrier.
__global__ __launch_bounds__(256) void RequantKernel(RequantArgs a) {
    const int64_t row = a.rowBegin + blockIdx.x;
    if (row >= a.sched[kHdrCoveredRows]) return;
    const float* src = a.s + static_cast<int64_t>(blockIdx.x) * a.halfN;
    int8_t* dst = a.y + row * a.halfN;
    const bool packets = (a.halfN & 3) == 0;
    constexpr int kAhead = 2;
    Float4 ahead[kAhead];
    if (packets) {
#pragma unroll
        for (int i = 0; i < kAhead; ++i) {
            const int j = (static_cast<int>(threadIdx.x) + 256 * i) * 4;
            // S is read exactly once: a non-temporal load keeps it from displacing anything in the caches
            ahead[i] = j < a.halfN ? __builtin_nontemporal_load(reinterpret_cast<const Float4*>(src + j)) : Float4{0.0f, 0.0f, 0.0f, 0.0f};
        }
    }
    float mx = 0.0f;
    for (int t = threadIdx.x & 63; t < a.partials; t += 64) mx = fmaxf(mx, a.rowMax[row * a.maxRowStride + t * a.maxStride]);
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) mx = fmaxf(mx, __shfl_xor(mx, d, 64));
    const float ys = __fdiv_rn(mx, 127.0f);
    const float inv = __fdiv_rn(1.0f, ys);
    if (threadIdx.x == 0) a.yScale[row] = ys;
    const bool zeroRow = mx == 0.0f;  // reference: 0 * inf; defined here as zeros
    if (packets) {
        auto quantPacket = [&](const Float4 v, int j) __attribute__((always_inline)) {
            char4 q;
            q.x = zeroRow ? 0 : QuantOne(v.x, inv);
            q.y = zeroRow ? 0 : QuantOne(v.y, inv);
            q.z = zeroRow ? 0 : QuantOne(v.z, inv);
            q.w = zeroRow ? 0 : QuantOne(v.w, inv);
            *reinterpret_cast<char4*>(dst + j) = q;  // read again soon, by the down projection: stays cacheable
        };
#pragma unroll
        for (int i = 0; i < kAhead; ++i) {
            const int j = (static_cast<int>(threadIdx.x) + 256 * i) * 4;
            if (j < a.halfN) quantPacket(ahead[i], j);
        }
        // rows longer than 2048 columns: one packet per trip (batching four loads per trip measured 5 % slower on
        // 14336-column rows)
        for (int j = (static_cast<int>(threadIdx.x) + 256 * kAhead) * 4; j < a.halfN; j += 256 * 4) {
            quantPacket(__builtin_nontemporal_load(reinterpret_cast<const Float4*>(src + j)), j);
        }
    } else {
        for (int j = threadIdx.x; j < a.halfN; j += 256) dst[j] = zeroRow ? 0 : QuantOne(src[j], inv);
    }
}

}  // namespace

// ---------------------------------------------------------------------------------------------- dispatch
int DeviceCuCount() {
    static const int count = [] {
        int dev = 0, n = 0;
        if (hipGetDevice(&dev) != hipSuccess) return 256;
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) return 256;
        return n;
    }();
    return count;
}

namespace {
// ---- workgroup spans (opapiGemmWorkgroupSpans*, include/opapi_profile.h): a measurement aid, off by default ----
// The buffers are allocated by opapiGemmWorkgroupSpansEnable(1) on the device that is current then, never on a launch
// path; recording is for one device and one launching thread at a time (the mutex only keeps the bookkeeping whole).
constexpr int kSpanKinds = 3;        // indexed by Epilogue
constexpr int kSpanMaxGrid = 1024;
std::mutex gSpanMutex;
bool gSpansOn = false;
int gSpanDevice = -1;
uint64_t* gSpanBuf[kSpanKinds] = {nullptr, nullptr, nullptr};
int gSpanGrid[kSpanKinds] = {0, 0, 0};   // workgroups of the last recorded launch of the kind; 0: nothing recorded
int gSpanTileM[kSpanKinds] = {0, 0, 0};
}  // namespace

// Device buffer for the next ring-kernel launch of this epilogue kind (every workgroup of the launch writes its own
// entry), or null when recording is off, the launch runs on another device or its grid exceeds the buffer -- the kind's
// earlier record is dropped then, so that a report never shows another launch's figures as the last one's.
uint64_t* SpanBufferFor(Epilogue epi, int grid, int tileM) {
    std::lock_guard<std::mutex> lock(gSpanMutex);
    if (!gSpansOn) return nullptr;
    const int k = static_cast<int>(epi);
    int dev = -1;
    if (gSpanBuf[k] == nullptr || grid > kSpanMaxGrid || hipGetDevice(&dev) != hipSuccess || dev != gSpanDevice) {
        gSpanGrid[k] = 0;
        return nullptr;
    }
    gSpanGrid[k] = grid;
    gSpanTileM[k] = tileM;
    return gSpanBuf[k];
}

namespace {
// The DMA ring needs at least one 128-byte k step, rows and bases on the 16-byte grid, 32-bit offsets inside one expert's weights and one of
// the three weight layouts it knows: K-contiguous rows per channel, the blocked layout, or row-major [K, N].
bool StreamOk(const Problem& p) {
    // blocked: whole 32-channel blocks; row-major: whole 16-byte chunks (per half of a SwiGLU tile)
    const int64_t grain = p.wNz ? 32 : 16;
    const bool layoutOk = p.wKMajor && !p.wNz ? true
                          : (p.N % grain == 0 && (p.epilogue != Epilogue::kSwiglu || (p.N / 2) % grain == 0));
    // One expert's weights must hold at least the kilobyte (64 lanes x 16 bytes) that a drained workgroup's idle issue
    // slots keep re-reading from the start of its last tile's expert: smaller experts go to the byte-wise kernel.
    return layoutOk && p.K % kChunk == 0 && p.K >= 128 && reinterpret_cast<uintptr_t>(p.x) % kChunk == 0 &&
           reinterpret_cast<uintptr_t>(p.w) % kChunk == 0 && p.N * p.K < (1ll << 31) && p.N * p.K >= 64 * kChunk;
}

// Tiles of one launch of the LDS-ring kernels: their numbers, and what the workgroups add to the tile counters past the last
// one, stay below 2^31.
constexpr int64_t kMaxTiles = 1ll << 30;

uint64_t Align256(uint64_t v) { return (v + 255) / 256 * 256; }

// S, the fp32 SwiGLU result that the requantisation reads back, is held for a band of rows at a time: at most 512 MiB of it
// (OPAPI_SWIGLU_WORKSPACE_MB=<n> sets another limit).
uint64_t SwigluWorkspaceCap() {
    if (const char* env = std::getenv("OPAPI_SWIGLU_WORKSPACE_MB")) {
        const long long mb = std::atoll(env);
        if (mb > 0) return static_cast<uint64_t>(mb) << 20;
    }
    return 512ull << 20;
}

// Rows that hold nearly every group of a router's choice whole: group sizes spread like a Poisson variable around their
// mean, so the mean plus 2.5 standard deviations.
double RowsOfNearlyEveryGroup(double meanRows) { return meanRows + 2.5 * std::sqrt(meanRows) + 1.0; }

// Share of the CUs' time that `tiles` like tiles use in whole rounds of one tile per CU.
double RoundEfficiency(int64_t tiles) {
    const int64_t cus = DeviceCuCount();
    return static_cast<double>(tiles) / static_cast<double>((tiles + cus - 1) / cus * cus);
}

// Rows per tile of the kernels for a handful of rows per group, or 0 where they are not the ones to run.  A tile has to hold
// nearly every group whole, since a second tile reads the group's weights again.  This is the height for groups that spread
// like a Poisson variable; the kernel takes taller tiles where the list it finds is more uneven than that.  At 64 rows the LDS-ring kernel's 64-row
// tile, twice as many channels wide, moves less per weight byte: gate/up of 31 rows each for 128 experts, hidden 4096,
// intermediate 1536, takes it 280 us against 300; it is left where its tiles fill the machine's rounds worse by more than
// that (a down projection of 128 of them: 115 us against 78).
// Groups of any size take the 64-row tiles where all of them are at most one round of the machine: taller and wider tiles
// would leave it idle (64 rows each for 8 experts, hidden 1024, intermediate 1024: 64 and 32 tiles of 96 x 256 take 18.8 and
// 16.7 us plus 4.8 us each for their table; 256 and 128 of these 12.6 and 11.3 us), and a group's m-tiles, side by side on
// one XCD, share its weights through L2.
// A forced tile height (OPAPI_GEMM_TILE_M) or tile order (OPAPI_GEMM_PULL) means the kernels those belong to.
int SlimTileRows(const Problem& p, double meanRows) {
    if (!StreamOk(p) || !(p.wKMajor || p.wNz) || p.groups > kSlimMaxGroups || p.M > kSlimMaxRows || p.groupListKind == GroupListKind::kSparse ||
        p.combineIndex != nullptr || p.bias != nullptr || std::getenv("OPAPI_GEMM_TILE_M") != nullptr ||
        std::getenv("OPAPI_GEMM_PULL") != nullptr) {
        return 0;
    }
    if (p.epilogue == Epilogue::kSwiglu && static_cast<uint64_t>(p.M) * static_cast<uint64_t>(p.N / 2) * 4 > SwigluWorkspaceCap()) return 0;
    const int64_t cols = p.epilogue == Epilogue::kSwiglu ? p.N / 2 : p.N;
    const int64_t wide = p.epilogue == Epilogue::kSwiglu ? kTileN / 2 : kTileN, slim = wide * kSlimTileN / kTileN;
    if (cols > kSlimMaxTilesN * slim) return 0;
    const double want = RowsOfNearlyEveryGroup(meanRows);
    if (want <= 16.0) return 16;
    if (want <= 32.0) return 32;
    if (p.groups * static_cast<int64_t>(std::ceil(want / 64.0)) * ((cols + slim - 1) / slim) <= DeviceCuCount()) return 64;
    if (want > 64.0) return 0;
    return RoundEfficiency(p.groups * ((cols + slim - 1) / slim)) > 1.06 * RoundEfficiency(p.groups * ((cols + wide - 1) / wide)) ? 64 : 0;
}

}  // namespace

Plan MakePlan(const Problem& p) {
    Plan plan;
    const int64_t groups = p.groups > 0 ? p.groups : 1;
    const int64_t cols = p.epilogue == Epilogue::kSwiglu ? p.N / 2 : p.N;
    const int64_t colsPerTile = p.epilogue == Epilogue::kSwiglu ? kTileN / 2 : kTileN;
    plan.tilesN = static_cast<int32_t>((cols + colsPerTile - 1) / colsPerTile);
    // tile height: the mean group size plus a quarter, so that almost every group is covered by one m-tile and its
    // weights are streamed exactly once.  A group that still overflows its tile adds a second m-tile, i.e. tilesN more
    // tiles, all in one XCD's share: its workgroups walk one round more than the others.  Where a workgroup walks few
    // rounds (one is more than 4 % of the launch) the headroom is half the mean instead: the taller shapes pay for
    // their extra rows with a shallower activation ring, which costs less than that round.
    const double meanRows = p.expectedRowsPerGroup > 0 ? static_cast<double>(p.expectedRowsPerGroup)
                                                       : static_cast<double>(p.M) / static_cast<double>(groups);
    if (const int slimRows = SlimTileRows(p, meanRows)) {
        plan.slim = true;
        plan.tileM = slimRows;
        const int64_t slimCols = p.epilogue == Epilogue::kSwiglu ? kSlimTileN / 2 : kSlimTileN;
        plan.tilesN = static_cast<int32_t>((cols + slimCols - 1) / slimCols);
        plan.maxMTiles = static_cast<int32_t>(p.M / slimRows + (groups < p.M ? groups : p.M));
        plan.maxTiles = (static_cast<int64_t>(plan.maxMTiles) * plan.tilesN + kXcds - 1) / kXcds * kXcds;
        uint64_t off = Align256(kQueueHeaderInts * 4);
        if (p.epilogue == Epilogue::kSwiglu) {
            plan.offRowMax = off;
            off += Align256(static_cast<uint64_t>(p.M) * static_cast<uint64_t>(plan.tilesN) * 16);
            plan.bandRows = p.M;
            plan.offS = off;
            off += Align256(static_cast<uint64_t>(p.M) * static_cast<uint64_t>(p.N / 2) * 4);
        }
        plan.workspaceBytes = off;
        return plan;
    }
    const double rounds = static_cast<double>(groups) * plan.tilesN / DeviceCuCount();
    double want = meanRows * (rounds <= 24.0 ? 1.5 : 1.25);
    // Without the SwiGLU epilogue 160 rows are better where they hold nearly every group: their activation ring is a stage deeper
    // than that of 192 (K 2048 x N 7168, 64 experts of 128 rows: 232 -> 218 us; K 1536 x N 4096, 128 experts of 112 rows:
    // 220 -> 207).  Groups that spread more than a router's even choice leave many small m-tiles, which the 192-row kernel
    // runs in a geometry of their own (the same shapes, popularity falling as rank^-0.6: 254 us against 276 with 160 rows;
    // 229 / 251): the scheduling kernel decides, where it knows the groups.  A workgroup that walks a few tiles only does
    // not repay the change of geometry, however uneven the groups (K 1024 x N 1024, 128 experts, two rounds of tiles:
    // 85 us with 192 rows, 73 with 160; K 1440 x N 2880, 32 experts, a round and a half: 95 / 82; K 1536 x N 4096, 60
    // experts, four rounds: 141 / 144), nor is there one below eight k-steps.
    // The SwiGLU operator has it the other way round: 379 us with 192 rows, 418 with 160 (N 3072, K 4096, 128 experts).
    const int64_t kSteps = (p.K + 127) / 128;
    const bool lowHolds = p.epilogue != Epilogue::kSwiglu && want > kLowTileM && RowsOfNearlyEveryGroup(meanRows) <= kLowTileM;
    if (lowHolds) want = rounds > 4.0 && kSteps >= 8 ? 192.0 : kLowTileM;
    if (StreamOk(p)) {
        static const int kShapes[] = {32, 64, 96, 128, 160, 192, 256};
        plan.tileM = 256;
        for (int s : kShapes) {
            if (static_cast<double>(s) >= want) { plan.tileM = s; break; }
        }
        // A handful of rows per group (decode): the 64-row shape, whose eight waves keep more of the weight stream in
        // flight than the four of the 32-row shape (measured 0.3 - 0.7 % faster on both GEMMs of a 64-token step).
        // Not beyond the means that ask for it, although it would hold nearly all of evenly chosen groups of up to 45 rows:
        // 45 rows each for 128 experts, hidden 4096, intermediate 1536, take 358 / 185 us (gate/up, down) with 96-row
        // tiles and 295 / 158 us with these, but with popularity falling as rank^-1.2 293 / 163 and 366 / 179.
        if (plan.tileM < 64) plan.tileM = 64;
        // tuning override: OPAPI_GEMM_TILE_M=<one of the shapes above>
        if (const char* env = std::getenv("OPAPI_GEMM_TILE_M")) {
            const int forced = std::atoi(env);
            for (int s : kShapes) {
                if (s == forced) plan.tileM = s;
            }
        }
    } else {
        plan.tileM = want <= 32.0 ? 32 : 128;
    }
    // Workgroups pull their tiles from counters where a tile is long enough to hide the draw: at least eight k-steps
    // (the issue side then never runs more than one tile ahead, which is what the two-tile look-ahead of the draw
    // covers) and more than 64 rows; the handful-of-rows tiles of a decode step keep their fixed shares.
    // OPAPI_GEMM_PULL=0 / 1 switches it off / on for every shape with eight k-steps.
    plan.pullTiles = StreamOk(p) && kSteps >= 8 && plan.tileM > 64;
    if (const char* env = std::getenv("OPAPI_GEMM_PULL")) {
        plan.pullTiles = StreamOk(p) && kSteps >= 8 && std::atoi(env) != 0;
    }
    if (lowHolds && plan.tileM == 192 && plan.pullTiles && std::getenv("OPAPI_GEMM_TILE_M") == nullptr) plan.lowTileM = kLowTileM;
    // Launches of at most two rounds of low tiles: the scheduling kernel decides, where it knows the groups (its figures are
    // there).  Asked and answered with the tall ones, it takes 0.5 us longer.
    if (plan.pullTiles && plan.tileM > kLowTileM && plan.lowTileM == 0 && std::getenv("OPAPI_GEMM_TILE_M") == nullptr &&
        (p.M + kLowTileM - 1) / kLowTileM * plan.tilesN <= 2ll * DeviceCuCount()) {
        plan.lowTileM = kLowTileM;
        plan.lowForRounds = true;
    }
    // The bands that S is held for are cut at the height chosen so far: the two choices below do not change them.  The table is sized
    // for the lowest height that a list may be cut at: this one, or what those put in its place.
    const int sizedFor = plan.lowTileM > 0 ? plan.lowTileM : plan.tileM, bandHeight = plan.tileM;
    // (Row-major weights: two geometries beat 64-row tiles on nearly every uneven list, gate/up 2048 x 2 x 2048, 256 experts of 20 at
    // rank^-0.4 378 / 463 us.)
    const bool maySmall = plan.tileM == kSmallRows && (p.wKMajor || p.wNz);
    // The SwiGLU operator on groups that 160 rows hold nearly all: tiles of 512 channels instead of 256, where that costs no round of the
    // machine, on the two-geometry kernel, which takes the lists that turn out uneven (and did so better than one geometry of 96 to 160
    // rows).  Such launches are bound by what a CU has under way, some 32 KB of lines however deep its ring; wide tiles read the
    // activations half as often.  us, before -> this: 256 experts of 128 rows, 7168 x 2 x 2048 1417 -> 1340; 128 of 128, 4096 x 2 x 1536
    // 325 -> 313; 8 of 110, 4096 x 2 x 14336 204 -> 186; 32 of 120, 2880 x 2 x 1440 90 -> 78; 128 of 80, 4096 x 2 x 1536, popularity
    // rank^-0.6 357 -> 326, rank^-1.2 362 -> 335.  Where they leave a round emptier: 60 of 90, 2816 x 2 x 1408 110 -> 122; 16 of
    // 100, 5440 x 2 x 10080 369 -> 395; where a workgroup walks a few short tiles: 32 of 60, 1344 x 2 x 1280, rank^-1.2 39 -> 51.  The down
    // projection, whose tiles are shorter: 1 % either way.
    if (p.epilogue == Epilogue::kSwiglu && StreamOk(p) && kSteps >= 8 && meanRows >= 16.0 && plan.tileM >= kSmallRows && plan.lowTileM == 0 &&
        plan.tilesN > 1 && rounds * kSteps >= 40.0 && RowsOfNearlyEveryGroup(meanRows) <= kLowTileM && std::getenv("OPAPI_GEMM_TILE_M") == nullptr &&
        std::getenv("OPAPI_GEMM_PULL") == nullptr) {
        const int64_t tiles = groups * plan.tilesN, wideTiles = groups * ((plan.tilesN + 1) / 2), cus = DeviceCuCount();
        const double used = static_cast<double>(tiles) / 2 / static_cast<double>((wideTiles + cus - 1) / cus * cus);
        if (used >= 0.97 * RoundEfficiency(tiles)) {
            plan.tileM = 192;
            plan.pullTiles = true;
            plan.lowTileM = kLowTileM;
            plan.lowBySizes = plan.lowIsWide = true;
            plan.maySmall = maySmall;
        }
    }
    // The others on such groups: 160 rows in one geometry are as good as 96 or 128 where the groups are alike, and the two-geometry kernel
    // better where they are not, if a workgroup walks more than a few tiles.  us, down, before -> this: 256 experts, 7168, 2048: 50 rows
    // 736 -> 708, at rank^-1.2 892 -> 750, 80 at rank^-0.6 875 -> 808; 128, 4096, 1536: 50 rows at rank^-1.2 202 -> 185.  Few tiles each,
    // left alone: 32 of 60, 2880, 1440, rank^-0.6 49 / 62; 60 of 90, 2816, 1408 69 / 74.
    if (p.epilogue != Epilogue::kSwiglu && StreamOk(p) && kSteps >= 8 && meanRows >= 16.0 && plan.tileM >= kSmallRows && plan.tileM <= kLowTileM &&
        plan.lowTileM == 0 && !lowHolds && rounds > 4.0 && std::getenv("OPAPI_GEMM_TILE_M") == nullptr && std::getenv("OPAPI_GEMM_PULL") == nullptr) {
        plan.tileM = 192;
        plan.pullTiles = true;
        plan.lowTileM = kLowTileM;
        plan.lowBySizes = true;
        plan.maySmall = maySmall;
    }
    // Weights whose rows begin inside cache lines -- K-contiguous ones with K off the 128 grid, the two halves of row-major ones for SwiGLU with N
    // off it -- on taller plans than 64 rows: tiles of few rows pay for the lines at the ends of theirs, and one geometry is better for more
    // lists.  Long: a workgroup walks sixty k-steps and more.  us, two geometries / one: 2880 x 2 x 1440, 256 experts of 50 rows even 480 / 439
    // (wide), at rank^-0.4 492 / 476, 128 of these, 277 / 252 (268 wide); down 272 / 263, of 60 296 / 271; 1296 x 2 x 1024, 128 of 60 at
    // rank^-0.8 120 / 112 (125 wide).  Row-major: 2880 x 2 x 1440, 256 of 50 even 553 / 437, of 100 at rank^-0.8 667 / 558; not 1344 x 2 x 1280, of 50 at
    // rank^-0.4 191 / 213 (wide).
    if (plan.lowBySizes && !plan.maySmall && !p.wNz && (p.wKMajor ? p.K : p.epilogue == Epilogue::kSwiglu ? p.N : 0) % 128 != 0) {
        plan.offGrid = rounds * kSteps >= 60.0 ? kOffGridLong : kOffGridShort;
    }
    const int64_t lowest = plan.lowBySizes ? std::min(sizedFor, kLowTileM) : sizedFor;
    // The LDS-ring kernels number the tiles of a launch in 32 bits.  More than kMaxTiles of them (the scatter-add alone can ask for so
    // many: its output has few rows) run as several launches, each over a band of rows.  One expert's weights stay below 2 GB
    // (StreamOk), so that every group's last m-tile is a small part of the limit: 1024 groups x 65536 n-tiles.
    int64_t bandRows = p.M;
    if (StreamOk(p) && (p.M / lowest + groups) * plan.tilesN > kMaxTiles) {
        bandRows = (kMaxTiles / plan.tilesN - groups) * lowest / bandHeight * bandHeight;
    }
    const int64_t maxMTiles = bandRows / lowest + groups;
    plan.maxMTiles = static_cast<int32_t>(maxMTiles);
    // round up so that every XCD's share [xcd * ceil(total/8), ...) is covered by the launch
    plan.maxTiles = (maxMTiles * plan.tilesN + kXcds - 1) / kXcds * kXcds;
    uint64_t off = 0;
    plan.offSched = off;
    off += ScheduleBytes(plan);
    if (p.epilogue == Epilogue::kSwiglu) {
        plan.offRowMax = off;
        off += Align256(static_cast<uint64_t>(p.M) * 4 * static_cast<uint64_t>(plan.tilesN));
        // S is held for one band of rows at a time, in whole m-tiles, at least one.  A launch whose S fits the limit runs as
        // one band; a taller one runs schedule, GEMM and requantisation once per band.  A band of 512 MiB is at least 4096
        // tiles, sixteen rounds of the machine, whatever the shape: measured against a single band on 1.9 GB of S it
        // costs nothing (halving the limit twice costs 2 % and 7 % of the pass).
        const uint64_t capBytes = SwigluWorkspaceCap();
        const uint64_t rowBytes = static_cast<uint64_t>(p.N / 2) * 4;
        int64_t capRows = rowBytes > 0 ? static_cast<int64_t>(capBytes / rowBytes) / bandHeight * bandHeight : p.M;
        if (capRows < bandHeight) capRows = bandHeight;
        if (capRows < bandRows) bandRows = capRows;
        plan.offS = off;
        off += Align256(static_cast<uint64_t>(bandRows) * rowBytes);
    }
    plan.bandRows = bandRows;
    plan.workspaceBytes = off;
    return plan;
}

namespace {
SchedArgs ScheduleArgsOf(const Problem& p, const Plan& plan, int32_t* table) {
    SchedArgs sa{};
    sa.groupList = p.groupList;
    sa.sched = table;
    sa.groups = p.groups;
    sa.groupListIsInt64 = p.groupListIsInt64 ? 1 : 0;
    sa.isCount = static_cast<int32_t>(p.groupListKind);
    sa.tileM = plan.tileM;
    sa.mayLower = plan.lowForRounds ? 2 : plan.lowBySizes ? 3 : plan.lowTileM > 0 ? 1 : 0;
    sa.lowIsWide = plan.lowIsWide ? 1 : 0;
    sa.offGrid = plan.offGrid;
    sa.maySmall = plan.maySmall ? 1 : 0;
    sa.kSteps = static_cast<int32_t>((p.K + 127) / 128);
    sa.cus = DeviceCuCount();
    sa.tilesN = plan.tilesN;
    sa.maxMTiles = plan.maxMTiles;
    sa.M = p.M;
    sa.rowEnd = p.M;
    return sa;
}
}  // namespace

bool SchedulesOnce(const Problem& p, const Plan& plan) {
    return !plan.slim && p.M > 0 && p.N > 0 && p.K > 0 && p.groups > 0 && p.groups <= kMaxGroups && (plan.bandRows == 0 || plan.bandRows >= p.M);
}

uint64_t ScheduleBytes(const Plan& plan) { return Align256(static_cast<uint64_t>(SchedTotalInts(plan.maxMTiles)) * 4); }

hipError_t Enqueue(const Problem& p, const Plan& plan, void* workspace, hipStream_t stream, const SharedSchedule& shared) {
    if (p.M == 0 || p.N == 0 || p.groups == 0) return hipSuccess;
    if (p.groups > kMaxGroups) return hipErrorInvalidValue;
    // K = 0 leaves the other epilogues nothing to do; with kSwiglu it would leave the requantisation an unwritten S
    // (the operator's first phase refuses K = 0, so this is a guard, not a path)
    if (p.K <= 0 && p.epilogue == Epilogue::kSwiglu) return hipErrorInvalidValue;
    char* ws = static_cast<char*>(workspace);
    int32_t* sched = shared.table != nullptr ? shared.table : reinterpret_cast<int32_t*>(ws + plan.offSched);
    const bool swiglu = p.epilogue == Epilogue::kSwiglu;
    float* rowMax = swiglu ? reinterpret_cast<float*>(ws + plan.offRowMax) : nullptr;
    float* sBuf = swiglu ? reinterpret_cast<float*>(ws + plan.offS) : nullptr;

    SchedArgs sa = ScheduleArgsOf(p, plan, sched);

    KernelArgs ka{};
    ka.x = p.x;
    ka.w = p.w;
    ka.wGroupStride = p.K * p.N;
    ka.wStrideN = p.wKMajor ? p.K : 1;
    ka.wStrideK = p.wNz ? 32 : (p.wKMajor ? 1 : p.N);
    ka.wNz = p.wNz ? 1 : 0;
    ka.M = static_cast<int32_t>(p.M);
    ka.K = static_cast<int32_t>(p.K);
    ka.N = static_cast<int32_t>(p.N);
    ka.groups = p.groups;
    ka.tilesN = plan.tilesN;
    ka.halfN = static_cast<int32_t>(p.N / 2);
    ka.out = p.out;
    ka.outDtype = p.outDtype;
    ka.scale = p.scale;
    ka.scaleDtype = p.scaleDtype;
    ka.rowScale = p.rowScale;
    ka.sOut = sBuf;
    ka.rowMax = rowMax;
    ka.combineIndex = p.combineIndex;
    ka.combineIndexIsInt64 = p.combineIndexIsInt64 ? 1 : 0;
    ka.combineRows = static_cast<int32_t>(p.combineRows);
    ka.combineWeight = p.combineWeight;
    ka.bias = p.bias;
    ka.biasDtype = p.biasDtype;
    ka.wgSpans = nullptr;
    ka.queueCounters = sched + kQueueHeaderInts;
    ka.pullTiles = plan.pullTiles ? 1 : 0;

    hipError_t e = hipSuccess;
    // One band covers every row unless S is held for a band of rows at a time (kSwiglu with a capped workspace) or the rows
    // have more tiles than a launch can number: then schedule, GEMM and requantisation run once per band, the schedule
    // handing out only the band's rows, and S is addressed as if the band's first row were at sBuf (the kernels index S by the
    // row of the problem).
    const int64_t bandRows = plan.bandRows > 0 ? plan.bandRows : p.M;
    for (int64_t rowBegin = 0; rowBegin < p.M; rowBegin += bandRows) {
        const int64_t rowEnd = rowBegin + bandRows < p.M ? rowBegin + bandRows : p.M;
        sa.rowBegin = rowBegin;
        sa.rowEnd = rowEnd;
        if (!plan.slim && shared.table == nullptr) {
            opapi::KernelTimer timer("gmm_schedule", stream);
            const bool both = shared.nextTable != nullptr;
            hipLaunchKernelGGL(ScheduleKernel, dim3(both ? 2 : 1), dim3(1024), 0, stream, sa,
                               both ? ScheduleArgsOf(*shared.nextProblem, *shared.nextPlan, shared.nextTable) : sa);
        }
        if (swiglu) {
            ka.sOut = reinterpret_cast<float*>(reinterpret_cast<uintptr_t>(sBuf) -
                                               static_cast<uintptr_t>(rowBegin) * static_cast<uintptr_t>(p.N / 2) * 4);
        }
        if (p.K > 0) {
            const bool fast = !plan.slim && StreamOk(p), tail = p.K % 128 != 0;
            opapi::KernelTimer timer(p.epilogue == Epilogue::kSwiglu ? "gmm_swiglu"
                                     : p.epilogue != Epilogue::kDequant ? "gmm_int32"
                                     : p.combineIndex != nullptr ? "gmm_combine" : "gmm_dequant", stream);
            if (plan.slim) {
                if (p.epilogue == Epilogue::kInt32) ka.scale = nullptr;  // raw accumulators
                const SlimList list{p.groupList, sa.groupListIsInt64, sa.isCount, p.groups, plan.tileM == 16 ? 0 : plan.tileM == 32 ? 1 : 2,
                                    sched + kHdrCoveredRows};
                e = swiglu ? LaunchSlimSwiglu(plan, ka, list, stream) : LaunchSlimPlain(plan, ka, list, stream);
            } else switch (p.epilogue) {
                case Epilogue::kInt32:
                    e = !fast ? LaunchGenericInt32(plan, ka, sched, stream) : tail ? LaunchRingTailInt32(plan, ka, sched, stream)
                         : LaunchRingInt32(plan, ka, sched, stream);
                    break;
                case Epilogue::kDequant:
                    e = !fast ? LaunchGenericDequant(plan, ka, sched, stream) : tail ? LaunchRingTailDequant(plan, ka, sched, stream)
                         : LaunchRingDequant(plan, ka, sched, stream);
                    break;
                case Epilogue::kSwiglu:
                    e = !fast ? LaunchGenericSwiglu(plan, ka, sched, stream) : tail ? LaunchRingTailSwiglu(plan, ka, sched, stream)
                         : LaunchRingSwiglu(plan, ka, sched, stream);
                    break;
            }
            if (e != hipSuccess) return e;
        }
        if (swiglu) {
            RequantArgs ra{sBuf, rowMax, plan.slim ? 4 * plan.tilesN : plan.tilesN, plan.slim ? 4 * plan.tilesN : 1,
                           plan.slim ? 1 : p.M, sched, p.quantOut, p.quantScaleOut, static_cast<int32_t>(p.N / 2),
                           rowBegin};
            opapi::KernelTimer timer("gmm_requant", stream);
            hipLaunchKernelGGL(RequantKernel, dim3(static_cast<unsigned>(rowEnd - rowBegin)), dim3(256), 0, stream, ra);
            e = hipGetLastError();
            if (e != hipSuccess) return e;
        }
    }
    return e;
}

}  // namespace gemm

extern "C" __attribute__((visibility("default"))) void opapiGemmWorkgroupSpansEnable(int enable) {
    using namespace gemm;
    std::lock_guard<std::mutex> lock(gSpanMutex);
    gSpansOn = false;
    for (int k = 0; k < kSpanKinds; ++k) gSpanGrid[k] = 0;  // records of an earlier recording period are not reported
    if (!enable) return;
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess) return;
    if (dev != gSpanDevice) {
        // buffers of another device stay allocated until the process ends (a few KB); this device gets its own
        for (int k = 0; k < kSpanKinds; ++k) gSpanBuf[k] = nullptr;
        gSpanDevice = dev;
    }
    for (int k = 0; k < kSpanKinds; ++k) {
        if (gSpanBuf[k] == nullptr && hipMalloc(&gSpanBuf[k], kSpanMaxGrid * 3 * sizeof(uint64_t)) != hipSuccess) {
            gSpanBuf[k] = nullptr;
            return;
        }
    }
    gSpansOn = true;
}

extern "C" __attribute__((visibility("default"))) int opapiGemmWorkgroupSpansReport(char* buf, size_t cap) {
    using namespace gemm;
    if (buf == nullptr || cap == 0) return -1;
    if (hipDeviceSynchronize() != hipSuccess) return -1;
    std::lock_guard<std::mutex> lock(gSpanMutex);
    static const char* const kNames[kSpanKinds] = {"gmm_int32", "gmm_dequant", "gmm_swiglu"};
    size_t used = 0;
    int lines = 0;
    buf[0] = 0;
    std::vector<uint64_t> host(kSpanMaxGrid * 3);
    for (int k = 0; k < kSpanKinds; ++k) {
        const int grid = gSpanGrid[k];
        if (gSpanBuf[k] == nullptr || grid <= 0) continue;
        if (hipMemcpy(host.data(), gSpanBuf[k], static_cast<size_t>(grid) * 3 * sizeof(uint64_t), hipMemcpyDeviceToHost) != hipSuccess) return -1;
        uint64_t first = ~0ull, last = 0;
        const int tileRows = host[2] >> 32 != 0 ? static_cast<int>(host[2] >> 32) : gSpanTileM[k];
        for (int b = 0; b < grid; ++b) {
            first = std::min(first, host[3 * b]);
            last = std::max(last, host[3 * b + 1]);
        }
        const double span = static_cast<double>(last - first) / 100.0;  // 100 MHz counter -> microseconds
        int n = snprintf(buf + used, cap - used, "%s workgroups %d tile_rows %d span_us %.1f", kNames[k], grid, tileRows, span);
        if (n < 0 || static_cast<size_t>(n) >= cap - used) break;
        used += static_cast<size_t>(n);
        // per XCD (workgroup b runs on XCD b % 8): when its last workgroup ended, relative to the launch's first start,
        // the mean busy fraction of its workgroups over the whole span, and the fewest / most tiles one of them took
        for (int x = 0; x < kXcds; ++x) {
            uint64_t xLast = 0, tMin = ~0ull, tMax = 0;
            double busy = 0.0;
            int count = 0;
            for (int b = x; b < grid; b += kXcds) {
                xLast = std::max(xLast, host[3 * b + 1]);
                busy += static_cast<double>(host[3 * b + 1] - host[3 * b]);
                tMin = std::min(tMin, host[3 * b + 2] & 0xffffffffu);
                tMax = std::max(tMax, host[3 * b + 2] & 0xffffffffu);
                ++count;
            }
            n = snprintf(buf + used, cap - used, " xcd%d end_us %.1f busy %.3f tiles %llu-%llu", x,
                         static_cast<double>(xLast - first) / 100.0,
                         span > 0 && count > 0 ? busy / 100.0 / count / span : 0.0, (unsigned long long)tMin, (unsigned long long)tMax);
            if (n < 0 || static_cast<size_t>(n) >= cap - used) break;
            used += static_cast<size_t>(n);
        }
        if (used + 2 < cap) {
            buf[used++] = '\n';
            buf[used] = 0;
        }
        ++lines;
    }
    return lines;
}
