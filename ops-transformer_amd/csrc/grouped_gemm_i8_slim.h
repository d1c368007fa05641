// Expert-grouped int8 GEMM for a handful of rows per expert (decode steps, short prompts over many experts): the weights
// of every expert with a row are streamed from HBM once, and everything else has to stay out of that stream's way.
// Included by the two translation units that instantiate its epilogues.
//
// What bounds it: the HBM, and below some hundred megabytes of weights the latency of getting going.  On one MI355X a bare
// DMA stream of this access pattern reaches 6.75 TB/s on random bytes.  Measured per operator call, weights only, before
// (tiles of 64 rows x 256 channels behind a scheduling kernel) and now:
//   hidden 4096, intermediate 1536, 128 experts, top-8     gate/up (with requantisation)    down
//     1 token    (8 experts touched, 151 MB)                40 -> 23 us                      22 -> 14 us
//     4 tokens   (29)                                        76 -> 63                         39 -> 33
//     64 tokens  (127, 2.4 GB)                               255 -> 254                       139 -> 125 (6.4 TB/s)
//   hidden 4096, intermediate 14336, 8 experts, top-2, 64 tokens     178 -> 168               113 -> 77
// The split:
//   * A tile is 16 / 32 / 64 rows x 128 channels (the lowest that holds the mean group nearly whole, or a taller one where
//     the list at hand needs it: SlimGroupTable), a workgroup four waves of 32 channels on v_mfma_i32_16x16x64_i8, one
//     workgroup per CU with a ring of six to eight stages of 16 KB of weights.  (Two workgroups per CU with half the ring
//     each measured the same within 1 % on everything but launches of few tiles, where they lose up to 15 %.)  Half the
//     channels of the 256-wide tiles: twice the tiles, so the last round of a launch leaves less of the machine idle.
//   * A CU pulls at most 50 GB/s out of HBM however deep its ring, so that fewer than about 140 of them cannot use it up:
//     where a launch has fewer tiles than workgroups, tiles are cut into parts of 64 or 32 channels.
//   * The tile table of the other kernels is a kernel of its own in front of every launch (5 us).  Here every workgroup
//     reads the group list for itself -- at most 512 groups, two per thread -- into a prefix table in LDS and finds a tile
//     with two ballots.
//   * The scales of a tile travel with its first stage, by DMA into LDS: an epilogue that loaded them would wait behind
//     every stage in flight (loads return in issue order), which is the ring's whole depth.
//   * Row maxima leave the SwiGLU epilogue per wave, [row][n-tile x wave]: no barrier in the epilogue.
// Row-major [K, N] weights stay with the 256-channel tiles: 128 channels of a SwiGLU tile are 64-byte pieces of two runs
// there, and the stream drops to 4.4 TB/s (the 256-wide tiles: 5.7).
#pragma once
#include "grouped_gemm_i8_kernels.h"

namespace gemm {

namespace {

constexpr int kSlimThreads = 256;
constexpr int kSlimCols = kSlimTileN;     // channels per tile
constexpr int kSlimTable = kSlimMaxGroups;
constexpr int kSlimTableBytes = 3328;     // prefix, first row and rows of every group (16 bits each), four totals per wave
static_assert(3 * kSlimTable * 2 + 16 * 4 <= kSlimTableBytes && kSlimTableBytes % 256 == 0, "the table in front of the ring");

template <int kMi, int kStages>
struct SlimCfg {
    static constexpr int kRows = 16 * kMi;
    static constexpr int kStageA = kRows * 128;
    static constexpr int kStageB = kSlimCols * 128;
    static constexpr int kInstrA = kRows / 8;              // DMA instructions of 1 KB (eight rows) in the activation part
    static constexpr int kSlotsA = (kInstrA + 3) / 4;      // per wave (16 rows: waves 2 and 3 repeat waves 0 and 1)
    static constexpr int kSlotsB = kStageB / 1024 / 4;
    static constexpr int kPerWave = kSlotsA + kSlotsB;
    static constexpr int kScaleFloats = kSlimCols + 64;    // per tile: channel scales, then row scales
    static constexpr int kOffScales = kSlimTableBytes + kStages * (kStageA + kStageB);  // the ring is behind the table
    static constexpr int kLdsBytes = kOffScales + kStages * kScaleFloats * 4;
    static_assert(kSlotsA + kSlotsB <= 8 && (kStages - 2) * kPerWave <= 63, "vmcnt is a 6-bit counter");
    static_assert(kLdsBytes <= kLdsBudget, "LDS of one workgroup");
};

// Relative cost of a tile of 16, 32 or 64 rows: its weights are the same, but a taller one leaves the ring fewer stages (64
// tokens evenly over 128 experts, hidden 4096, intermediate 1536: 247 / 251 / 262 us gate/up).  A launch costs its rounds of
// tiles times that.  What speaks for a taller tile is groups that need several of the lower ones; how many there are is known
// here and not to the planner, which has only the mean.  Kernel time on the planner's height and on the one chosen here, and
// the ring kernel's 64-row tiles beside them (1024 rows, all on eight of 256 experts, hidden 7168, intermediate 2048,
// 16-row tiles planned): 143 -> 64 us, ring 67; popularity falling as rank^-1.2, 128 tokens: gate/up 347 -> 275, ring 308;
// 512 tokens (32 rows planned): 630 -> 555, ring 689.
__device__ constexpr uint32_t kSlimTileCost[3] = {50, 51, 62};

// Inclusive sum over the wave, without LDS: inside the rows of sixteen lanes, then the rows' totals into those behind them.
// (As six shuffles, three of these sums put 0.5 us more into the head of every launch.)
__device__ __forceinline__ int32_t WaveInclusiveSum(int32_t v) {
    auto add = [&](auto ctl, auto rows) __attribute__((always_inline)) {
        v += __builtin_amdgcn_update_dpp(0, v, decltype(ctl)::value, decltype(rows)::value, 0xF, false);
    };
    using All = std::integral_constant<int, 0xF>;
    add(std::integral_constant<int, 0x111>{}, All{});  // row_shr:1, 2, 4, 8
    add(std::integral_constant<int, 0x112>{}, All{});
    add(std::integral_constant<int, 0x114>{}, All{});
    add(std::integral_constant<int, 0x118>{}, All{});
    add(std::integral_constant<int, 0x142>{}, std::integral_constant<int, 0xA>{});  // row_bcast:15 into rows 1 and 3
    add(std::integral_constant<int, 0x143>{}, std::integral_constant<int, 0xC>{});  // row_bcast:31 into rows 2 and 3
    return v;
}

struct SlimTile {
    int32_t valid;
    int32_t group;
    int32_t rowBase;
    int32_t rows;
    int32_t tileN;
    int32_t part;  // of the tile's four 32-channel columns, this workgroup computes (4 >> cut) from part * (4 >> cut) on
    int32_t shared;  // its weights are another m-tile's as well
    int32_t kStart;  // k-step that its walk starts from
};

// The table of a launch, in LDS: m-tiles of groups 0 .. g, first row and rows of group g.
struct SlimGroups {
    uint16_t* incl;
    uint16_t* start;
    uint16_t* rows;
};

// Workgroup-wide: the group list becomes the prefix table.  Thread t owns groups 2t and 2t + 1.  Boundaries are clamped into
// [0, M] and the prefix saturates, so that a malformed list cannot push an access out of bounds.  Returns the tile height,
// as log2(rows / 16): the lowest from sl.minHeight on unless a taller one is the cheaper for this list.
__device__ __forceinline__ int SlimGroupTable(const KernelArgs& a, const SlimList& sl, char* const lds, const SlimGroups& table) {
    int32_t* const waveTotal = reinterpret_cast<int32_t*>(lds + 3 * kSlimTable * 2);  // [4][4]
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g0 = 2 * tid, g1 = g0 + 1;
    // entries g0 - 1, g0 and g1 in one round trip (indices clamped into the list)
    int32_t vPrev, v0, v1;
    {
        const int last = sl.groups - 1;
        const int iPrev = min(max(g0 - 1, 0), last), i0 = min(g0, last), i1 = min(g1, last);
        auto clamped = [&](int64_t v) { return static_cast<int32_t>(v < 0 ? 0 : (v > a.M ? a.M : v)); };
        if (sl.isInt64) {
            const int64_t* const p = static_cast<const int64_t*>(sl.list);
            const int64_t w0 = p[iPrev], w1 = p[i0], w2 = p[i1];
            vPrev = clamped(w0);
            v0 = clamped(w1);
            v1 = clamped(w2);
        } else {
            const int32_t* const p = static_cast<const int32_t*>(sl.list);
            const int32_t w0 = p[iPrev], w1 = p[i0], w2 = p[i1];
            vPrev = clamped(w0);
            v0 = clamped(w1);
            v1 = clamped(w2);
        }
    }
    // a wave's sums to the workgroup's: slot is the wave's of four totals that it leaves for the others
    auto leaveTotal = [&](int32_t inclusive, int slot) __attribute__((always_inline)) {
        if (lane == 63) waveTotal[4 * slot + wave] = inclusive;
    };
    auto wavesBefore = [&](int slot, int waves) __attribute__((always_inline)) {
        const int4 t = *reinterpret_cast<const int4*>(waveTotal + 4 * slot);
        return (waves > 0 ? t.x : 0) + (waves > 1 ? t.y : 0) + (waves > 2 ? t.z : 0) + (waves > 3 ? t.w : 0);
    };
    int32_t b0 = 0, e0 = 0, b1 = 0, e1 = 0;
    if (sl.isCount) {
        const int32_t c0 = g0 < sl.groups ? v0 : 0, c1 = g1 < sl.groups ? v1 : 0;
        // counts may add up to more than M: 256 x 2 x 65535 still fits
        const int32_t incl = WaveInclusiveSum(c0 + c1);
        leaveTotal(incl, 3);
        __syncthreads();
        const int32_t before = incl - c0 - c1 + wavesBefore(3, wave);
        b0 = min(before, a.M);
        e0 = min(before + c0, a.M);
        b1 = e0;
        e1 = min(before + c0 + c1, a.M);
    } else {
        b0 = g0 > 0 ? vPrev : 0;
        e0 = v0;
        b1 = e0;
        e1 = v1;
    }
    const int32_t r0 = g0 < sl.groups ? max(e0 - b0, 0) : 0, r1 = g1 < sl.groups ? max(e1 - b1, 0) : 0;
    // m-tiles of 16, 32 and 64 rows
    auto mTiles = [](int32_t rows, int height) { return (rows + (16 << height) - 1) >> (4 + height); };
    int32_t incl[3];
#pragma unroll
    for (int h = 0; h < 3; ++h) {
        incl[h] = WaveInclusiveSum(mTiles(r0, h) + mTiles(r1, h));
        leaveTotal(incl[h], h);
    }
    __syncthreads();
    auto all = [&](int h) __attribute__((always_inline)) { return static_cast<uint32_t>(min(__builtin_amdgcn_readfirstlane(wavesBefore(h, 4)), 65535)); };
    const uint32_t total[3] = {all(0), all(1), all(2)};
    int height = sl.minHeight;
    if ((height == 0 ? total[0] : total[1]) != total[2] && height < 2) {
        const uint32_t grid = gridDim.x;
        auto cost = [&](int h) __attribute__((always_inline)) { return (total[h] * a.tilesN + grid - 1) / grid * kSlimTileCost[h]; };
        const uint32_t cost16 = cost(0), cost32 = cost(1), cost64 = cost(2);
        if (height == 0 && cost32 < cost16) height = 1;
        if (cost64 < (height == 0 ? cost16 : cost32)) height = 2;
    }
    const int32_t mt1 = height == 0 ? mTiles(r1, 0) : height == 1 ? mTiles(r1, 1) : mTiles(r1, 2);
    const int32_t incl1 = (height == 0 ? incl[0] : height == 1 ? incl[1] : incl[2]) + wavesBefore(height, wave);
    table.incl[g0] = static_cast<uint16_t>(min(incl1 - mt1, 65535));
    table.incl[g1] = static_cast<uint16_t>(min(incl1, 65535));
    table.start[g0] = static_cast<uint16_t>(b0);
    table.start[g1] = static_cast<uint16_t>(b1);
    table.rows[g0] = static_cast<uint16_t>(r0);
    table.rows[g1] = static_cast<uint16_t>(r1);
    if (blockIdx.x == 0 && (g0 == sl.groups - 1 || g1 == sl.groups - 1)) {
        *sl.coveredRows = g1 == sl.groups - 1 ? max(e1, b1) : max(e0, b0);
    }
    __syncthreads();
    return height;
}

// kNz: weights in the blocked layout instead of K-contiguous channels.
template <int kMi, int kStages, bool kSwiglu, bool kNz>
__device__ __forceinline__ void SlimGemmBody(const KernelArgs& a, const SlimGroups& table, char* const lds, uint64_t& spanTiles) {
    using Cfg = SlimCfg<kMi, kStages>;
    const uint16_t* const tabIncl = table.incl;
    const uint16_t* const tabStart = table.start;
    const uint16_t* const tabRows = table.rows;
    char* const ringBase = lds + kSlimTableBytes;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l16 = lane & 15;
    const int quad = lane >> 4;

    // ---- this workgroup's tiles: the list of (group, n-tile, m-tile) is cut into eight contiguous shares, one per XCD,
    // which the workgroups of an XCD walk side by side: the m-tiles of a group follow each other at one n-tile and share
    // its weights through L2, the n-tiles of a group share its rows.
    // Fewer tiles than workgroups: a tile is cut into two or four parts of 64 or 32 channels (a part runs as a whole tile
    // whose other channels' loads re-read one chunk; leaving those loads out measured no faster, 42 against 39 us on a
    // down projection of 64 tiles of K 14336).
    const int64_t wholeTiles = static_cast<int64_t>(__builtin_amdgcn_readfirstlane(tabIncl[kSlimTable - 1])) * a.tilesN;
    constexpr int kMaxCut = kNz && kSwiglu ? 1 : 2;  // a 32-channel block is loaded whole
    int cut = 0;
    while (cut < kMaxCut && (wholeTiles << (cut + 1)) <= gridDim.x) ++cut;
    const int64_t totalTiles = wholeTiles << cut;
    const int64_t perXcd = (totalTiles + kXcds - 1) / kXcds;
    const int64_t xcdFirst = (blockIdx.x % kXcds) * perXcd;
    const int64_t xcdTiles = min(perXcd, totalTiles - xcdFirst);  // may be negative: nothing to do
    const int32_t slots = gridDim.x / kXcds, slot = blockIdx.x / kXcds;
    const int kSteps = (a.K + 127) / 128;  // K off the step grid: the last step overlaps the one before (see kTail of StreamGemmBody)
    // Every workgroup walks its tiles' k-steps from a start of its own and wraps (integer sums do not depend on the order):
    // with rows a multiple of 4096 bytes apart the memory channel depends on the k offset alone, and workgroups at the
    // same k-step would all queue on the same channels.  The m-tiles of a group have to meet in L2 instead: their start is
    // that of the weight block they share.  (Not so where rows do not start on a cache line: they are spread over the
    // channels as they are, and 320 rows at most for 32 experts, K 2880, take 96.6 us with a common start, 94.1 without.)
    const bool splitLines = !kNz && a.K % 128 != 0;
    const int32_t ownStart = static_cast<int32_t>((blockIdx.x * 7u + blockIdx.x / kXcds) % static_cast<unsigned>(kSteps));
    auto tileAt = [&](int32_t n) __attribute__((always_inline)) -> SlimTile {
        const int64_t local = slot + static_cast<int64_t>(n) * slots;
        SlimTile t{};
        if (local >= xcdTiles) return t;
        const int32_t logicalPart = static_cast<int32_t>(xcdFirst + local);
        const int32_t logical = logicalPart >> cut;
        const int32_t q = logical / a.tilesN;
        // the group is the first whose prefix exceeds q: lane i looks at the last of groups 8i .. 8i + 7, then the first
        // eight lanes at those of the first such lane
        const uint64_t coarse = __ballot(tabIncl[8 * lane + 7] > q);
        const int blk = __ffsll(static_cast<unsigned long long>(coarse)) - 1;
        const uint64_t fine = __ballot(tabIncl[8 * blk + (lane & 7)] > q);
        const int g = 8 * blk + __ffsll(static_cast<unsigned long long>(fine)) - 1;
        const int32_t before = g > 0 ? __builtin_amdgcn_readfirstlane(tabIncl[g - 1]) : 0;
        const int32_t mTiles = __builtin_amdgcn_readfirstlane(tabIncl[g]) - before;
        const int32_t idx = logical - before * a.tilesN;
        const int32_t mIn = idx % mTiles;
        t.valid = 1;
        t.group = g;
        t.tileN = idx / mTiles;
        t.part = logicalPart & ((1 << cut) - 1);
        t.shared = mTiles > 1;
        t.kStart = t.shared && !splitLines ? static_cast<int32_t>((g * 5u + t.tileN * 7u) % static_cast<unsigned>(kSteps)) : ownStart;
        t.rowBase = __builtin_amdgcn_readfirstlane(tabStart[g]) + mIn * Cfg::kRows;
        t.rows = min(Cfg::kRows, __builtin_amdgcn_readfirstlane(tabRows[g]) - mIn * Cfg::kRows);
        return t;
    };

    SlimTile cur = tileAt(0);
    if (!cur.valid) return;
    const bool hasRowScale = a.rowScale != nullptr;
    const bool hasScale = a.scale != nullptr;
    const bool scaleByDma = hasScale && a.scaleDtype == 0;

    // ---- issue side
    const uint32_t ldsBase = LdsAddress(lds);
    SlimTile iss = cur;
    int32_t issNo = 0;
    int issStep = 0, issK = cur.kStart, issSlot = 0, issScaleSlot = 0;
    bool drained = false;
    const char* issBaseA = nullptr;
    const char* issBaseB = nullptr;
    uint32_t offA[Cfg::kSlotsA], offB[Cfg::kSlotsB];
    // in registers: a per-lane choice between the two as kernel arguments becomes a vector load of the chosen one
    const int32_t halfN = __builtin_amdgcn_readfirstlane(a.halfN), allN = __builtin_amdgcn_readfirstlane(a.N);
    auto channelOf = [&](const SlimTile& t, int r) __attribute__((always_inline)) {  // of weight row r of the tile, clamped
        int32_t n;
        if (kSwiglu) n = r < kSlimCols / 2 ? min(t.tileN * (kSlimCols / 2) + r, halfN - 1)
                                           : min(halfN + t.tileN * (kSlimCols / 2) + r - kSlimCols / 2, allN - 1);
        else n = min(t.tileN * kSlimCols + r, allN - 1);
        return n;
    };
    auto setupIssue = [&](const SlimTile& t) __attribute__((always_inline)) {
        issBaseA = reinterpret_cast<const char*>(a.x) + static_cast<int64_t>(t.rowBase) * a.K;
        issBaseB = reinterpret_cast<const char*>(a.w) + static_cast<int64_t>(t.group) * a.wGroupStride;
        const int rowIn = lane >> 3, chunkSlot = lane & 7;
        const int columns = 4 >> cut, firstColumn = t.part * columns;  // a column: the channels of one wave
        auto wanted = [&](int column) __attribute__((always_inline)) { return column >= firstColumn && column < firstColumn + columns; };
#pragma unroll
        for (int q = 0; q < Cfg::kSlotsA; ++q) {
            const int j = (wave + 4 * q) % Cfg::kInstrA;
            const int r = 8 * j + rowIn;
            const int c = chunkSlot ^ ((r >> 1) & 7);
            // rows past the last re-read it; an instruction wholly past it reads one chunk
            offA[q] = 8 * j >= t.rows ? 0u : static_cast<uint32_t>(min(r, t.rows - 1) * a.K + c * kChunk);
        }
#pragma unroll
        for (int q = 0; q < Cfg::kSlotsB; ++q) {
            const int j = wave + 4 * q;
            if (kNz) {
                // 32 k of channel block j / 4: 1 KB, contiguous in memory and in LDS
                const int32_t block = channelOf(t, 32 * (j / 4)) >> 5;
                const bool want = kSwiglu ? wanted(2 * ((j / 4) & 1)) || wanted(2 * ((j / 4) & 1) + 1) : wanted(j / 4);
                offB[q] = want ? static_cast<uint32_t>(block * a.K * 32 + ((j % 4) * 32 + lane / 2) * 32 + (lane % 2) * kChunk) : 0u;
            } else {
                const int r = 8 * j + rowIn;
                const int c = chunkSlot ^ ((r >> 1) & 7);
                const bool want = wanted(kSwiglu ? (j & 7) / 2 : j / 4);
                offB[q] = want ? static_cast<uint32_t>(channelOf(t, r) * a.K + c * kChunk) : 0u;
            }
        }
    };
    auto issueStage = [&]() __attribute__((always_inline)) {
        if (issStep == 0 && !drained) {
            // the tile's scales, ahead of its first stage: whatever certifies that stage certifies them
            const uint32_t dst = ldsBase + Cfg::kOffScales + issScaleSlot * (Cfg::kScaleFloats * 4);
            if (wave < 2) {
                if (scaleByDma) {
                    DmaToLdsAddr4(static_cast<const char*>(a.scale) + static_cast<int64_t>(iss.group) * allN * 4,
                                  static_cast<uint32_t>(channelOf(iss, 64 * wave + lane)) * 4u, dst + 256 * wave);
                }
            } else if (wave == 2) {
                if (hasRowScale) {
                    DmaToLdsAddr4(reinterpret_cast<const char*>(a.rowScale) + static_cast<int64_t>(iss.rowBase) * 4,
                                  static_cast<uint32_t>(min(lane, iss.rows - 1)) * 4u, dst + kSlimCols * 4);
                }
            }
        }
        const int kOff = drained ? 0 : min(issK * 128, a.K - 128);
        const int64_t kOffW = static_cast<int64_t>(kOff) * (kNz ? 32 : 1);
        const uint32_t dst = ldsBase + kSlimTableBytes + issSlot * (Cfg::kStageA + Cfg::kStageB);
#pragma unroll
        for (int q = 0; q < Cfg::kSlotsA; ++q) {
            DmaToLdsAddr16<false>(issBaseA + kOff, offA[q], dst + ((wave + 4 * q) % Cfg::kInstrA) * 1024);
        }
        // The weights of a group with one m-tile are used once: past the caches.  Not so those that other m-tiles want as
        // well, at about the same time on the same XCD: past the caches every m-tile fetched them from HBM (512 tokens of 256
        // experts, top-8, popularity falling as rank^-1.2, hidden 7168, intermediate 2048, on 32-row tiles: 700 -> 630 us
        // gate/up, 414 -> 336 us down).  And rows that do not start on a line
        // have their 128 bytes of a k-step in two, each wanted again by the next step (K 2880 / 1440, 37 rows each for 32
        // experts: 68.8 -> 64.6 us gate/up, 41.8 -> 39.0 us down).
        if (splitLines || iss.shared) {
#pragma unroll
            for (int q = 0; q < Cfg::kSlotsB; ++q) {
                DmaToLdsAddr16<false>(issBaseB + kOffW, offB[q], dst + Cfg::kStageA + (wave + 4 * q) * 1024);
            }
        } else {
#pragma unroll
            for (int q = 0; q < Cfg::kSlotsB; ++q) {
                DmaToLdsAddr16<true>(issBaseB + kOffW, offB[q], dst + Cfg::kStageA + (wave + 4 * q) * 1024);
            }
        }
        issSlot = issSlot + 1 == kStages ? 0 : issSlot + 1;
        issK = issK + 1 == kSteps ? 0 : issK + 1;
        if (++issStep == kSteps) {
            issStep = 0;
            const SlimTile next = tileAt(issNo + 1);
            if (next.valid) {
                iss = next;
                issK = next.kStart;
                ++issNo;
                issScaleSlot = issScaleSlot + 1 == kStages ? 0 : issScaleSlot + 1;
                setupIssue(iss);
            } else if (!drained) {
                // past the last tile the slots still go out, to keep the count of outstanding DMAs, and re-read one kilobyte
                drained = true;
                issBaseA = issBaseB = reinterpret_cast<const char*>(a.w) + static_cast<int64_t>(iss.group) * a.wGroupStride;
#pragma unroll
                for (int q = 0; q < Cfg::kSlotsA; ++q) offA[q] = static_cast<uint32_t>(lane) * kChunk;
#pragma unroll
                for (int q = 0; q < Cfg::kSlotsB; ++q) offB[q] = static_cast<uint32_t>(lane) * kChunk;
            }
        }
    };
    setupIssue(cur);
#pragma unroll 1
    for (int s = 0; s < kStages - 1; ++s) issueStage();

    int ring = 0, scaleSlot = 0;
    int32_t curNo = 0;
    v4i acc[kMi][2];
    // weight rows of the wave's two 16-channel blocks: neighbours, or an activated block and its linear partner
    const int bRow0 = kSwiglu ? 16 * wave : 32 * wave;
    const int bRow1 = kSwiglu ? kSlimCols / 2 + 16 * wave : 32 * wave + 16;
    while (true) {
        int curK = cur.kStart;
#pragma unroll
        for (int mi = 0; mi < kMi; ++mi) acc[mi][0] = acc[mi][1] = v4i{0, 0, 0, 0};
#pragma unroll 1
        for (int step = 0; step < kSteps; ++step) {
            // the oldest stage has landed once at most the younger stages' share of this wave is outstanding (stores and
            // scales in flight only make that stricter); the barrier: for every wave, and the stage before is no longer read
            WaitVmcnt<(kStages - 2) * Cfg::kPerWave>();
            __syncthreads();
            const char* const A = ringBase + ring * (Cfg::kStageA + Cfg::kStageB);
            const char* const B = A + Cfg::kStageA;
            const uint32_t bAddr = ldsBase + kSlimTableBytes + ring * (Cfg::kStageA + Cfg::kStageB) + Cfg::kStageA;
            const int covered = curK + 1 == kSteps ? kSteps * 128 - a.K : 0;  // leading k of this stage that another one has
            curK = curK + 1 == kSteps ? 0 : curK + 1;
            v4i bf[2][2], af[2][kMi];
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) {
                const int chunk = 4 * ks + quad;
                if constexpr (!kNz) {
                    bf[ks][0] = *reinterpret_cast<const v4i*>(B + LdsOffset(bRow0 + l16, chunk));
                    bf[ks][1] = *reinterpret_cast<const v4i*>(B + LdsOffset(bRow1 + l16, chunk));
                } else {
                    // lane j of a 16-lane group supplies bytes (k = kBase + j / 2, channels 8 * (j % 2) .. + 7) and receives
                    // eight consecutive k of channel j
                    const int k = 64 * ks + 16 * quad + (l16 >> 1);
#pragma unroll
                    for (int ni = 0; ni < 2; ++ni) {
                        const int row = ni ? bRow1 : bRow0;
                        const uint32_t lo = bAddr + (row >> 5) * 4096 + k * 32 + (row & 16) + 8 * (l16 & 1);
                        const uint32_t hi = lo + 8 * 32;
                        const v2i vlo = __builtin_amdgcn_ds_read_tr8_b64_v2i32(reinterpret_cast<LdsV2iPtr>(lo));
                        const v2i vhi = __builtin_amdgcn_ds_read_tr8_b64_v2i32(reinterpret_cast<LdsV2iPtr>(hi));
                        bf[ks][ni] = v4i{vlo[0], vlo[1], vhi[0], vhi[1]};
                    }
                }
#pragma unroll
                for (int mi = 0; mi < kMi; ++mi) af[ks][mi] = *reinterpret_cast<const v4i*>(A + LdsOffset(16 * mi + l16, chunk));
            }
            // The refill goes out while the fragments are on their way (in front of them, the wave would wait for the address
            // unit first, which takes sixteen clocks per DMA), into the buffer that the step before read.
            issueStage();
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) {
                const bool counts = 64 * ks + 16 * quad >= covered;
#pragma unroll
                for (int mi = 0; mi < kMi; ++mi) {
                    v4i av = af[ks][mi];
                    if (!counts) av = v4i{0, 0, 0, 0};
                    acc[mi][0] = __builtin_amdgcn_mfma_i32_16x16x64_i8(av, bf[ks][0], acc[mi][0], 0, 0, 0);
                    acc[mi][1] = __builtin_amdgcn_mfma_i32_16x16x64_i8(av, bf[ks][1], acc[mi][1], 0, 0, 0);
                }
            }
            ring = ring + 1 == kStages ? 0 : ring + 1;
        }

        // ---- epilogue: acc[mi][ni][v] is C[16 mi + 4 quad + v, channel l16 of block ni]
        const float* const ldsScale = reinterpret_cast<const float*>(lds + Cfg::kOffScales + scaleSlot * (Cfg::kScaleFloats * 4));
        const float* const ldsRowScale = ldsScale + kSlimCols;
        const bool mine = wave >= cur.part * (4 >> cut) && wave < (cur.part + 1) * (4 >> cut);  // this wave's channels are of the part
        const int32_t colBase = cur.tileN * (kSwiglu ? kSlimCols / 2 : kSlimCols);
        const int32_t c0 = channelOf(cur, bRow0 + l16), c1 = channelOf(cur, bRow1 + l16);
        float sc0 = 1.0f, sc1 = 1.0f;
        if (scaleByDma) {
            sc0 = ldsScale[bRow0 + l16];
            sc1 = ldsScale[bRow1 + l16];
        } else if (hasScale) {
            sc0 = LoadScale(a.scale, static_cast<int64_t>(cur.group) * a.N + c0, a.scaleDtype);
            sc1 = LoadScale(a.scale, static_cast<int64_t>(cur.group) * a.N + c1, a.scaleDtype);
            // waited for here: were they still pending on some path into the k loop, the compiler would drain every DMA there
            asm volatile("" : "+v"(sc0), "+v"(sc1));
        }
        if constexpr (kSwiglu) {
            const int32_t j = colBase + 16 * wave + l16;  // column of S
            const bool jValid = j < a.halfN;
            const int32_t partials = a.tilesN * 4;
#pragma unroll
            for (int mi = 0; mi < kMi; ++mi) {
                if (!mine || 16 * mi >= cur.rows) continue;  // wave-uniform
                const float4 xs4 = *reinterpret_cast<const float4*>(ldsRowScale + 16 * mi + 4 * quad);
                const float xs[4] = {xs4.x, xs4.y, xs4.z, xs4.w};
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int r = 16 * mi + 4 * quad + v;
                    const float ca = __fmul_rn(__fmul_rn(static_cast<float>(acc[mi][0][v]), xs[v]), sc0);
                    const float cb = __fmul_rn(__fmul_rn(static_cast<float>(acc[mi][1][v]), xs[v]), sc1);
                    const float s = __fmul_rn(__fmul_rn(ca, __builtin_amdgcn_rcpf(__fadd_rn(1.0f, __expf(-ca)))), cb);
                    const bool ok = r < cur.rows && jValid;
                    if (ok) a.sOut[static_cast<int64_t>(cur.rowBase + r) * a.halfN + j] = s;
                    const float m = MaxOver16(jValid ? fabsf(s) : 0.0f);
                    if (l16 == 0 && r < cur.rows) {
                        a.rowMax[static_cast<int64_t>(cur.rowBase + r) * partials + 4 * cur.tileN + wave] = m;
                    }
                }
            }
        } else {
            const int32_t n0 = colBase + 32 * wave + l16, n1 = n0 + 16;
            const bool valid0 = n0 < a.N, valid1 = n1 < a.N;
            const bool oddLane = (l16 & 1) != 0;
            const bool pairs = (a.N & 1) == 0 && colBase + 32 * wave + 32 <= a.N;  // wave-uniform
#pragma unroll
            for (int mi = 0; mi < kMi; ++mi) {
                if (!mine || 16 * mi >= cur.rows) continue;
                float rs[4] = {1.0f, 1.0f, 1.0f, 1.0f};  // multiplying by 1 is exact
                if (hasRowScale) {
                    const float4 rs4 = *reinterpret_cast<const float4*>(ldsRowScale + 16 * mi + 4 * quad);
                    rs[0] = rs4.x; rs[1] = rs4.y; rs[2] = rs4.z; rs[3] = rs4.w;
                }
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int r = 16 * mi + 4 * quad + v;
                    const bool rowOk = r < cur.rows;
                    const int64_t rowOff = static_cast<int64_t>(cur.rowBase + r) * a.N;
                    if (!hasScale) {
                        int32_t* const out = static_cast<int32_t*>(a.out) + rowOff;
                        if (rowOk && valid0) out[n0] = acc[mi][0][v];
                        if (rowOk && valid1) out[n1] = acc[mi][1][v];
                        continue;
                    }
                    const float y0 = __fmul_rn(__fmul_rn(static_cast<float>(acc[mi][0][v]), sc0), rs[v]);
                    const float y1 = __fmul_rn(__fmul_rn(static_cast<float>(acc[mi][1][v]), sc1), rs[v]);
                    uint32_t pk;
                    if (a.outDtype == 27) {
                        const Float2 f = {y0, y1};
                        pk = __builtin_bit_cast(uint32_t, __builtin_convertvector(f, Bf16x2));
                    } else {
                        pk = static_cast<uint32_t>(HalfBitsOfRounded(y0)) | (static_cast<uint32_t>(HalfBitsOfRounded(y1)) << 16);
                    }
                    uint16_t* const out = static_cast<uint16_t*>(a.out) + rowOff;
                    if (pairs) {
                        // an even lane stores columns (c, c + 1) of block 0, the odd lane next to it those of block 1
                        const uint32_t got = static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(static_cast<int>(pk), 0xB1, 0xF, 0xF, true));
                        const uint32_t word = __builtin_amdgcn_perm(got, pk, oddLane ? 0x03020706u : 0x05040100u);
                        if (rowOk) *reinterpret_cast<uint32_t*>(out + (oddLane ? n0 + 15 : n0)) = word;
                    } else {
                        if (rowOk && valid0) out[n0] = static_cast<uint16_t>(pk & 0xffffu);
                        if (rowOk && valid1) out[n1] = static_cast<uint16_t>(pk >> 16);
                    }
                }
            }
        }
        ++spanTiles;
        cur = tileAt(++curNo);
        if (!cur.valid) break;
        scaleSlot = scaleSlot + 1 == kStages ? 0 : scaleSlot + 1;
    }
    // the drained slots' DMAs write this workgroup's LDS: none may be outstanding when it is given to another
    WaitVmcnt<0>();
}

// The three tile heights with as many stages as LDS holds.
template <bool kSwiglu, bool kNz>
__global__ __launch_bounds__(kSlimThreads) void SlimGemmKernel(KernelArgs a, SlimList sl) {
    extern __shared__ __attribute__((aligned(16))) char lds[];
    const uint64_t spanStart = a.wgSpans != nullptr ? __builtin_amdgcn_s_memrealtime() : 0;
    uint64_t spanTiles = 0;
    uint16_t* const entries = reinterpret_cast<uint16_t*>(lds);
    const SlimGroups table{entries, entries + kSlimTable, entries + 2 * kSlimTable};
    const int height = SlimGroupTable(a, sl, lds, table);
    if (height == 0) SlimGemmBody<1, 8, kSwiglu, kNz>(a, table, lds, spanTiles);
    else if (height == 1) SlimGemmBody<2, 7, kSwiglu, kNz>(a, table, lds, spanTiles);
    else SlimGemmBody<4, 6, kSwiglu, kNz>(a, table, lds, spanTiles);
    WriteSpan(a, spanStart, spanTiles);
}

template <bool kSwiglu, bool kNz>
hipError_t LaunchSlimKernel(const Plan& plan, const KernelArgs& args, const SlimList& list, hipStream_t stream) {
    constexpr int kLdsBytes = std::max({SlimCfg<1, 8>::kLdsBytes, SlimCfg<2, 7>::kLdsBytes, SlimCfg<4, 6>::kLdsBytes});
    auto kernel = SlimGemmKernel<kSwiglu, kNz>;
    static std::atomic<uint64_t> optedIn{0};
    const hipError_t attr = opapi::EnsureDynamicLds(reinterpret_cast<const void*>(kernel), kLdsBytes, optedIn);
    if (attr != hipSuccess) return attr;
    int64_t grid = DeviceCuCount();
    if (grid > 4 * plan.maxTiles) grid = 4 * plan.maxTiles;  // a tile may be cut in four
    grid = grid / kXcds * kXcds;
    if (grid < kXcds) grid = kXcds;
    KernelArgs launchArgs = args;
    launchArgs.wgSpans = SpanBufferFor(kSwiglu ? Epilogue::kSwiglu : args.scale == nullptr ? Epilogue::kInt32 : Epilogue::kDequant,
                                       static_cast<int>(grid), plan.tileM);
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(grid)), dim3(kSlimThreads), kLdsBytes, stream, launchArgs, list);
    return hipGetLastError();
}

template <bool kSwiglu>
hipError_t LaunchSlimLayout(const Plan& plan, const KernelArgs& args, const SlimList& list, hipStream_t stream) {
    if (args.wNz) return LaunchSlimKernel<kSwiglu, true>(plan, args, list, stream);
    return LaunchSlimKernel<kSwiglu, false>(plan, args, list, stream);
}

}  // namespace
}  // namespace gemm
