// Device side of the expert-grouped int8 GEMM (see grouped_gemm_i8.hip for the overview): the LDS-ring kernels, the
// byte-wise kernel, their epilogues and launchers.  Included by grouped_gemm_i8.hip (scheduling, requantisation, planning)
// and by one translation unit per epilogue (grouped_gemm_i8_int32.hip, _dequant.hip, _swiglu.hip), each of which
// instantiates the kernels of its epilogue only, so that the three compile side by side.
#pragma once
#include "grouped_gemm_i8.h"

#include <hip/hip_fp16.h>

#include <algorithm>
#include <atomic>
#include <cstdlib>
#include <type_traits>

#include "opapi_common.h"

#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Wunused-function"

namespace gemm {

// Arguments of the GEMM kernels (one type for every translation unit of the engine).
struct KernelArgs {
    const int8_t* x;
    const int8_t* w;
    int64_t wGroupStride;  // bytes between experts
    int64_t wStrideN;      // bytes between consecutive output channels
    int64_t wStrideK;      // bytes between consecutive k
    int32_t wNz;           // weights in 32-channel x 16-k blocks ([N/32][K/16][16][32] per expert), see Problem::wNz
    int32_t M, K, N;
    int32_t groups;
    int32_t tilesN;
    int32_t halfN;  // N / 2 (kSwiglu)
    void* out;
    int32_t outDtype;
    const void* scale;
    int32_t scaleDtype;
    const float* rowScale;
    float* sOut;
    float* rowMax;  // partial max |S|: [tilesN][M], one per n-tile; grouped_gemm_i8_slim.h: [M][4 tilesN], one per wave
    // scatter-add mode of the fp32 kDequant epilogue (Problem::combineIndex)
    const void* combineIndex;
    int32_t combineIndexIsInt64;
    int32_t combineRows;
    const float* combineWeight;
    const void* bias;
    int32_t biasDtype;
    // workgroup spans (include/opapi_profile.h): per workgroup what WriteSpan leaves, times of the 100 MHz real-time counter;
    // null unless span recording is on
    uint64_t* wgSpans;
    // LDS-ring kernels: the tile counters of the scheduling table as a pointer the kernel may write through (the table
    // itself is a read-only kernel parameter), and whether workgroups pull their tiles from the counters (1) or walk a
    // fixed share (0)
    int32_t* queueCounters;
    int32_t pullTiles;
};

// The group list (cumsum or counts) as the kernels of grouped_gemm_i8_slim.h read it.
struct SlimList {
    const void* list;
    int32_t isInt64;
    int32_t isCount;
    int32_t groups;
    int32_t minHeight;     // lowest tiles to consider, as log2(rows / 16)
    int32_t* coveredRows;  // written by workgroup 0: rows covered by the list (the requantisation reads it)
};

// Defined in grouped_gemm_i8.hip.
int DeviceCuCount();
uint64_t* SpanBufferFor(Epilogue epi, int grid, int tileM);

// The launchers of each epilogue: the LDS-ring kernels for K a multiple of 128, those for the other K on the 16-byte grid
// (Tail; each of the two in a translation unit of its own, so that they compile side by side), and the byte-wise kernel.
hipError_t LaunchRingInt32(const Plan& plan, const KernelArgs& args, const int32_t* sched, hipStream_t stream);
hipError_t LaunchRingDequant(const Plan& plan, const KernelArgs& args, const int32_t* sched, hipStream_t stream);
hipError_t LaunchRingSwiglu(const Plan& plan, const KernelArgs& args, const int32_t* sched, hipStream_t stream);
hipError_t LaunchRingTailInt32(const Plan& plan, const KernelArgs& args, const int32_t* sched, hipStream_t stream);
hipError_t LaunchRingTailDequant(const Plan& plan, const KernelArgs& args, const int32_t* sched, hipStream_t stream);
hipError_t LaunchRingTailSwiglu(const Plan& plan, const KernelArgs& args, const int32_t* sched, hipStream_t stream);
hipError_t LaunchSlimPlain(const Plan& plan, const KernelArgs& args, const SlimList& list, hipStream_t stream);
hipError_t LaunchSlimSwiglu(const Plan& plan, const KernelArgs& args, const SlimList& list, hipStream_t stream);
hipError_t LaunchGenericInt32(const Plan& plan, const KernelArgs& args, const int32_t* sched, hipStream_t stream);
hipError_t LaunchGenericDequant(const Plan& plan, const KernelArgs& args, const int32_t* sched, hipStream_t stream);
hipError_t LaunchGenericSwiglu(const Plan& plan, const KernelArgs& args, const int32_t* sched, hipStream_t stream);

namespace {

typedef int v2i __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) v2i* LdsV2iPtr;
typedef int v4i __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) const v4i* LdsV4iPtr;
typedef float Float2 __attribute__((ext_vector_type(2)));
typedef float Float4 __attribute__((ext_vector_type(4)));
// Vectors that begin on any element: a global store of several dwords may begin on any byte.
typedef uint32_t Uint2Half __attribute__((ext_vector_type(2), aligned(2)));
typedef int Int4Dword __attribute__((ext_vector_type(4), aligned(4)));
typedef float Float4Dword __attribute__((ext_vector_type(4), aligned(4)));
typedef __bf16 Bf16x2 __attribute__((ext_vector_type(2)));

constexpr int kTileN = 256;
constexpr int kWavesN = 4;
constexpr int kChunk = 16;
constexpr int kXcds = 8;
constexpr int kGroupM = 4;  // m-tiles walked together per n-tile for L2 reuse of weight columns
constexpr int kMaxGroups = 1024;
constexpr int kLdsBudget = 160 * 1024;

// ---------------------------------------------------------------------------------------------- scheduling table
// int32 layout, all written by the scheduling kernel:
//   header, 32 ints: [0] big m-tiles, [1] small m-tiles, [2] cost of the small ones, [3] cost of the big ones (see below),
//                    [4] / [5] band width of the big / small run, [6] total rows covered by the groups, [7] rows per m-tile, [8] 1: nearly every group is one m-tile, of one kind, 2: every tile is dealt out, [9] 1: tiles are 512 channels wide;
//   16 tile counters in one 128-byte line (32 ints): counter [2 * xcd + list], zeroed;
//   the m-tile table, 4 ints per m-tile {group, first row, rows, 0} (at most maxMTiles of them): the big m-tiles in group
//   order, then the small ones.  A GEMM kernel finds everything about a tile with one 16-byte load.
// An m-tile is small when it holds at most kSmallRows rows: its time is the weight stream's (the whole K x 256 weight
// block for a handful of rows), not the matrix pipe's.  The two kinds are kept apart so that a launch which holds both
// (a skewed routing: a few experts with thousands of rows, many with a few) can run them side by side -- some
// workgroups streaming small tiles while the others multiply big ones -- instead of a compute-bound phase followed by
// a bandwidth-bound one.  Costs are in units of one 32-row MFMA tile over the whole K: a big m-tile costs its count of
// occupied 32-row tiles (at least kSmallCost), a small one kSmallCost (what the weight stream of a tile takes when
// only a part of the workgroups stream).
constexpr int kSmallRows = 64;
constexpr int kSmallCost = 3;
constexpr int kQueueHeaderInts = 32;
constexpr int kQueueCounterInts = 32;
constexpr int kHdrCoveredRows = 6;
constexpr int kHdrTileM = 7;
constexpr int kHdrEven = 8;
constexpr int kHdrWide = 9;
// A height that the scheduling kernel may choose instead of 192 or 256 rows (Plan::lowTileM), maybe with wide tiles (Plan::lowIsWide).
constexpr int kLowTileM = 160;
__host__ __device__ inline int SchedTotalInts(int maxMTiles) { return kQueueHeaderInts + kQueueCounterInts + 4 * maxMTiles; }


// One output tile of one group, decoded from the scheduling table (all fields are wave-uniform).
struct TileInfo {
    int32_t valid;
    int32_t group;
    int32_t rowBase;  // first row of the tile in x / out
    int32_t rows;     // 1..tileM real rows
    int32_t tileN;
    int32_t colBase;  // first output channel (kSwiglu: first column of S)
};

// An entry of the m-tile table, which nothing writes while a GEMM kernel runs: where the index is the wave's, through the scalar
// cache, past the DMAs that a vector load would wait behind.
__device__ __forceinline__ v4i ConstantEntry(const int4* table, int32_t i) {
    typedef __attribute__((address_space(4))) const v4i* EntryPtr;
    return ((EntryPtr)(reinterpret_cast<uintptr_t>(table)))[i];
}

// What the header says of the two runs.  Read again wherever it is wanted: held in scalar registers across the k loop it would push out
// what that needs there.
struct RunTable {
    const int4* entries;
    int32_t countBig, countSmall;  // m-tiles
    int32_t bandBig, bandSmall;
};
__device__ __forceinline__ RunTable ReadRunTable(const int32_t* sched) {
    typedef __attribute__((address_space(4))) const int32_t* HeaderPtr;
    auto h = (HeaderPtr)(reinterpret_cast<uintptr_t>(sched));
    asm volatile("" : "+s"(h));
    return RunTable{reinterpret_cast<const int4*>(reinterpret_cast<uintptr_t>(h) + (kQueueHeaderInts + kQueueCounterInts) * sizeof(int32_t)),
                    h[0], h[1], h[4], h[5]};
}

// Tile `logical` of one run of the m-tile table (`count` m-tiles from entry `first` on).  Bands of bandWidth m-tiles walk
// the n-tiles together: consecutive tiles are the band's m-tiles at one n-tile, then the next n-tile.
template <bool kSwiglu>
__device__ __forceinline__ TileInfo DecodeListTile(int32_t tilesN, const int4* __restrict__ table, int32_t first,
                                                   int32_t count, int32_t bandWidth, int32_t logical) {
    TileInfo t{};
    const int32_t perBand = bandWidth * tilesN;
    const int32_t band = logical / perBand;
    const int32_t rem = logical - band * perBand;
    const int32_t bandTiles = min(bandWidth, count - bandWidth * band);
    const int32_t tileN = rem / bandTiles;
    const v4i e = ConstantEntry(table, first + bandWidth * band + rem - tileN * bandTiles);
    t.valid = 1;
    t.group = e[0];
    t.rowBase = e[1];
    t.rows = e[2];
    t.tileN = tileN;
    t.colBase = kSwiglu ? t.tileN * (kTileN / 2) : t.tileN * kTileN;
    return t;
}

// ---- tile counters: workgroups pull their tiles instead of walking a fixed share ----
// Each of the two runs of the m-tile table (big, small) is cut into eight contiguous shares of tiles, one per XCD, so
// that the workgroups of an XCD sit on neighbouring tiles and share operands through that XCD's L2.  Counter
// [2 * xcd + list] hands out the tiles of a share in order.  A workgroup draws from its own XCD first -- the list it
// prefers, then the other -- and, when both are used up, from the other XCDs' shares in ring order, so nobody idles
// while tiles are left anywhere.  The counters are only ever added to (values past a share's size mean "used up").
// The first `seated` tiles of every share are not drawn but dealt out (see the seats).
// (The lists' sizes travel as plain values: a structure handed round by reference, or an array indexed at run time,
// ends up in scratch memory.)
struct QueueLists {
    int32_t tilesBig, tilesSmall;
    int32_t seatedBig, seatedSmall;  // tiles of a share that workgroups begin with
};
__device__ __forceinline__ void QueueShare(const QueueLists q, int counter, int32_t* first, int32_t* size) {
    const int32_t total = (counter & 1) ? q.tilesSmall : q.tilesBig;
    const int32_t per = (total + kXcds - 1) / kXcds;
    const int32_t begin = (counter >> 1) * per;
    const int32_t all = max(min(total - begin, per), 0), seated = min((counter & 1) ? q.seatedSmall : q.seatedBig, all);
    *first = begin + seated;
    *size = all - seated;
}
// Workgroups of an XCD's `slots` that begin with the small m-tiles: the share that their cost is of the whole, so that lists of many
// rounds run dry at about the same time; until then a part of the machine streams weights for a handful of rows each while
// the rest multiplies.  But in two geometries, where the tiles of the big ones are no more than seven eighths of the workgroups, all of these begin with: those
// left over would each be a whole tile behind the last small one.  us, by cost -> this: gate/up 2048 x 2 x 2048, 64 experts of 25 rows on average,
// popularity rank^-0.8 (112 big tiles) 127 -> 108; 7168 x 2 x 2048, 32 of 80, rank^-1.2 (224) 238 -> 197; down 1536 x 4096, 128 of 20,
// rank^-0.4 (16) 167 -> 155.  With 240 and 256 of them, which leaves the small ones' weights for a round of their own: 64 of 60,
// rank^-0.4 115 -> 125, 256 of 50, 2048 x 2 x 768 161 -> 172.  Row-major weights for SwiGLU are left with the share of the cost (7168 x 2 x 2048,
// 32 of 25, rank^-0.4 176 against 192 us), and so is one geometry for both (int32, 59 experts of 68 rows, rank^-0.4, 1536 x 2048 51 against 59 us;
// bf16, 99 of 62 even, 1024 x 1024 36 against 40).
template <Epilogue kEpi, bool kNMajor, bool kTwoGeometries>
__device__ __forceinline__ int32_t SlotsForSmall(const int32_t* __restrict__ hdr, int32_t slots, int32_t tilesN) {
    const int64_t costSmall = hdr[2], costAll = costSmall + hdr[3];
    int32_t forSmall = static_cast<int32_t>(costAll > 0 ? (slots * costSmall + costAll / 2) / costAll : 0);
    if (forSmall == 0 && hdr[1] > 0 && slots > 1) forSmall = 1;
    if (!kTwoGeometries || (kNMajor && kEpi == Epilogue::kSwiglu)) return forSmall;
    const int32_t forBig = (hdr[0] * tilesN + kXcds - 1) / kXcds;
    return 8 * forBig <= 7 * slots ? min(forSmall, slots - forBig) : forSmall;
}
// Counter i-th in the preference order of a workgroup on XCD `home` that prefers list `prefer`.
__device__ __forceinline__ int QueueCandidate(int i, int home, int prefer) {
    return 2 * ((home + (i >> 1)) & (kXcds - 1)) + ((i & 1) ? 1 - prefer : prefer);
}
// onlyPreferred: the other run's counters are not candidates at all (a workgroup that serves one run at a time).
__device__ __forceinline__ int QueueFirstOpen(uint32_t usedUp, int home, int prefer, bool onlyPreferred = false) {
#pragma unroll
    for (int i = 0; i < 2 * kXcds; ++i) {
        if (onlyPreferred && (i & 1)) continue;
        const int c = QueueCandidate(i, home, prefer);
        if (((usedUp >> c) & 1u) == 0) return c;
    }
    return -1;
}
// (One lane's.  The zero keeps the address out of the compiler's sight: seen to be the same in every lane, it adds the wave's lanes up
// first and waits for the answer on the spot to deal it out, microseconds in which the caller has other work to do.)
__device__ __forceinline__ int32_t QueueTake(int32_t* counters, int c) {
    int32_t zero;
    asm volatile("v_mov_b32 %0, 0" : "=v"(zero));
    return __hip_atomic_fetch_add(counters + c + zero, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Completes a draw that began with QueueTake on counter c (value v; c < 0: nothing was open): returns the list (0 big,
// 1 small) and the tile inside that list's run, or list -1 when every share is used up.  One thread of the workgroup.
struct QueueDraw {
    int32_t list;     // 0 big, 1 small, -1 none
    int32_t logical;  // tile inside that list's run
    uint32_t usedUp;  // the caller's mask of used-up counters, updated
};
__device__ __forceinline__ QueueDraw QueueResolve(const QueueLists q, int32_t* counters, int home, int prefer,
                                                  uint32_t usedUp, int c, int32_t v, bool onlyPreferred = false) {
    while (c >= 0) {
        int32_t first, size;
        QueueShare(q, c, &first, &size);
        if (v < size) return QueueDraw{c & 1, first + v, usedUp};
        usedUp |= 1u << c;
        // a look at all sixteen counters at once (one round trip) spares a failed draw, i.e. a round trip, per used-up share
        int32_t now[2 * kXcds];  // fully unrolled below: stays in registers
#pragma unroll
        for (int i = 0; i < 2 * kXcds; ++i) now[i] = __hip_atomic_load(counters + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
        for (int i = 0; i < 2 * kXcds; ++i) {
            QueueShare(q, i, &first, &size);
            if (now[i] >= size) usedUp |= 1u << i;
        }
        c = QueueFirstOpen(usedUp, home, prefer, onlyPreferred);
        if (c >= 0) v = QueueTake(counters, c);
    }
    return QueueDraw{-1, 0, usedUp};
}

// ---------------------------------------------------------------------------------------------- tiles and their waves
// A tile is up to kRows rows x 256 channels, computed by eight waves: two wave rows x four wave columns.  The matrix
// instruction is v_mfma_i32_16x16x64_i8: per operation it costs the power of 0.85 to 0.9 of a 32x32x32 one -- eight waves per CU
// on register operands sustain 3.7 to 4.1 POP/s with it, depending on the card, and 3.4 to 3.5 with that, uniform random bytes,
// both at the power limit (4.8 to 4.9 both with zeros; opapiInt8MfmaRateProbe) -- and it splits a tile's rows in sixteens.
//   Rows: 16-row block b of the tile belongs to wave row b & 1, and there to its first half (b & 2 == 0) or its second, as
//   number b >> 2: whatever the tile's row count, the four (wave row, half) pairs hold the same number of blocks but for one.
//   Channels: the 256 channels are two halves of 128 rows in LDS, 32 of each belonging to each wave column, as two blocks
//   of sixteen.  kSwiglu: the first half is activated, the second linear.
constexpr int kWaves = 8;
constexpr int kThreads = 64 * kWaves;

// Which channel a row of a weight half is.  Weights by channel (K-contiguous) may lie in LDS in any order, and they lie so
// that the accumulators of a lane are neighbouring channels: four (kSwiglu: two of S), one store.  The two layouts with the
// channels side by side in memory hand sixteen neighbours to sixteen lanes.
constexpr int kOrderLane = 0;   // K-contiguous: wave column w, block n, lane l: channel 64 w + 4 l + n
constexpr int kOrderBlock = 1;  // blocked and row-major: 64 w + 16 n + l
template <bool kNz, bool kNMajor>
constexpr int kOrderOf = kNz || kNMajor ? kOrderBlock : kOrderLane;

// Scatter-add of the rows wants neighbouring lanes on neighbouring channels: the order of the blocked layout.
__device__ __forceinline__ bool LanesHoldNeighbours(const KernelArgs& a) { return a.combineIndex == nullptr; }

// Channel of column block n = 2 * half + j (j = 0, 1) and lane l of wave column w, from the tile's first on
// (kSwiglu: column of S, the same for both halves).
template <int kOrder, bool kSwiglu>
__device__ __forceinline__ int ColumnInTile(int w, int n, int l, bool neighbours) {
    if (kSwiglu) return 32 * w + (kOrder == kOrderLane ? 2 * l + (n & 1) : 16 * (n & 1) + l);
    return 64 * w + (kOrder == kOrderLane && neighbours ? 4 * l + n : 16 * n + l);
}

// Channel held in row r of weight half `half`, rows by channel (clamped: channels past N are loaded but never stored).
template <int kOrder, bool kSwiglu>
__device__ __forceinline__ int32_t ChannelOfRow(const KernelArgs& a, const TileInfo& t, int half, int r) {
    const int32_t col = t.colBase + ColumnInTile<kOrder, kSwiglu>(r >> 5, 2 * half + ((r >> 4) & 1), r & 15, LanesHoldNeighbours(a));
    return min(kSwiglu && half ? a.halfN + col : col, a.N - 1);
}

__device__ __forceinline__ float LoadScale(const void* p, int64_t i, int dtype) {
    if (dtype == 0) return static_cast<const float*>(p)[i];
    const uint16_t raw = static_cast<const uint16_t*>(p)[i];
    if (dtype == 1) return __half2float(__ushort_as_half(raw));
    return __uint_as_float(static_cast<uint32_t>(raw) << 16);
}

// fp32 -> fp16, round to nearest even, of a value that is itself an fp32 result.  The reference rounds its products to
// fp32 and then casts; left in sight of each other, a multiply and this conversion are merged by the compiler into one
// v_fma_mixlo_f16, which rounds the exact product once -- a different value in the rare double-rounding cases.  The
// empty statement hides the value's origin.
__device__ __forceinline__ uint16_t HalfBitsOfRounded(float f) {
    asm("" : "+v"(f));
    return __half_as_ushort(__float2half_rn(f));
}

// Two values to bf16 (else fp16), the first in the low half.
template <bool kToBf16>
__device__ __forceinline__ uint32_t PackHalves(float lo, float hi) {
    if constexpr (kToBf16) {
        const Float2 f = {lo, hi};
        return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, Bf16x2));  // v_cvt_pk_bf16_f32
    } else {
        return static_cast<uint32_t>(HalfBitsOfRounded(lo)) | (static_cast<uint32_t>(HalfBitsOfRounded(hi)) << 16);
    }
}

// The value of another lane of the row of sixteen (kCtl: a DPP control).
template <int kCtl>
__device__ __forceinline__ float RowLane(float v) {
    return __uint_as_float(static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(static_cast<int>(__float_as_uint(v)), kCtl, 0xF, 0xF, true)));
}

template <int kCtl>
__device__ __forceinline__ uint32_t RowLane(uint32_t v) {
    return static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(static_cast<int>(v), kCtl, 0xF, 0xF, true));
}

// kOrderBlock, 16-bit values: a lane holds channel l of each of its four blocks, 0 and 1 in the first word, 2 and 3 in the second.
// In every four lanes side by side, lane i (l & 3) gets the four lanes' channels of block i: one store of eight bytes, and sixteen
// lanes fill a cache line.  (Of int32 results, where this is sixteen instructions for four values, it measured 1 to 3 % slower than
// stores of a block each: 16 groups of 1000 rows, K 2048 x N 4096 163 against 159 us.)
__device__ __forceinline__ void BlockOfLane(uint32_t (&word)[2], int l16) {
    const bool odd = (l16 & 1) != 0, far = (l16 & 2) != 0;
#pragma unroll
    for (int p = 0; p < 2; ++p) word[p] = __builtin_amdgcn_perm(RowLane<0xB1>(word[p]), word[p], odd ? 0x03020706u : 0x05040100u);
    const uint32_t got = RowLane<0x4E>(far ? word[0] : word[1]);
    word[0] = far ? got : word[0];
    word[1] = far ? word[1] : got;
}

// Maximum over the 16 lanes of a row group, in every lane (rotations inside the row: no LDS).
__device__ __forceinline__ float MaxOver16(float v) {
    v = fmaxf(v, RowLane<0x128>(v));  // row_ror:8
    v = fmaxf(v, RowLane<0x124>(v));
    v = fmaxf(v, RowLane<0x122>(v));
    return fmaxf(v, RowLane<0x121>(v));
}

// Raises a maximum in LDS, kept as the bits of a float that is not negative, to m (NaN counts as nothing, as it does with fmaxf).
__device__ __forceinline__ void RaiseRowMax(uint32_t* ldsMax, float m) { atomicMax(ldsMax, __float_as_uint(fmaxf(m, 0.0f))); }

// Maxima of four values over the 16 lanes of a row group: lane l gets that of value l >> 2.  A halving butterfly: a lane
// gives its partner the values that it drops.
__device__ __forceinline__ float FourMaxOver16(const float (&m)[4], int l16) {
    const bool b3 = (l16 & 8) != 0, b2 = (l16 & 4) != 0;
    const float k0 = fmaxf(b3 ? m[2] : m[0], RowLane<0x140>(b3 ? m[0] : m[2]));  // row_mirror: lane 15 - l
    const float k1 = fmaxf(b3 ? m[3] : m[1], RowLane<0x140>(b3 ? m[1] : m[3]));
    float k = fmaxf(b2 ? k1 : k0, RowLane<0x141>(b2 ? k0 : k1));                 // row_half_mirror: 7 - l in each eight
    k = fmaxf(k, RowLane<0x4E>(k));                                              // quad_perm [2,3,0,1], [1,0,3,2]
    return fmaxf(k, RowLane<0xB1>(k));
}

// Byte offset of (channel n, k = 0) inside one expert's weights; consecutive k are a.wStrideK bytes apart (32 in the
// blocked layout: a 32-channel block holds its K rows of 32 channel bytes back to back).
__device__ __forceinline__ int64_t WeightRowBase(const KernelArgs& a, int32_t n) {
    return a.wNz ? static_cast<int64_t>(n >> 5) * a.K * 32 + (n & 31) : static_cast<int64_t>(n) * a.wStrideN;
}

// Blocks of a wave in the first and in the second half of its rows, tile of kRows rows.
template <int kRows>
struct RowBlocks {
    static_assert(kRows % 32 == 0, "both wave rows hold the same number of 16-row blocks");
    static constexpr int kFirst = (kRows + 63) / 64, kSecond = kRows / 64, kAll = kFirst + kSecond;
    // first tile row of block m (first half, then second half) of wave row `waveM`
    __device__ static __forceinline__ int RowOf(int m, int waveM) {
        return 16 * (m < kFirst ? 4 * m + waveM : 4 * (m - kFirst) + 2 + waveM);
    }
};

// Epilogue of one tile.  acc[m][n][v] is C[row, col] with row = RowOf(m) + 4 * quad + v and col = ColumnInTile(n) of lane l16.
// ldsRowScale holds the tile's per-row scales, ldsChannelScale those of its 256 channels by their place in the tile (null: they are
// loaded here).  kSwiglu: ldsRowMax, zero before, takes the tile's row maxima of |S| as float bits (TileEpilogueStoreMax).
// beforeStores() is called between the arithmetic and the stores of whole column blocks, in front of both elsewhere.  Not so without
// kAllAtOnce: a block's results are stored before the next one's are worked out, and beforeStores() comes behind them all, where the DMAs
// have landed.  The tallest and the wide tiles have no registers for all results beside the accumulators of those to come (and the SwiGLU
// of 256 rows, which has, is slower for them on short K: 64 groups of 2000 rows, K 1024 x 2 x 512, 187 / 181 us).
// Row checks are made per 16-row block, wave-uniformly: a block wholly inside the expert's rows takes a copy of the code
// without checks, a block wholly outside is skipped, and only the one that straddles the last row tests every lane.  (A
// per-lane test makes every element a predicated basic block of its own, and their independent chains no longer interleave.)
// Values that may have been loaded are waited for here: were they still pending on some path into the k loop, the compiler would
// drain every DMA there.
template <int kCount>
__device__ __forceinline__ void SettleLoads(float (&v)[kCount]) {
#pragma unroll
    for (int i = 0; i < kCount; ++i) asm volatile("" : "+v"(v[i]));
}

struct NoHook {
    __device__ __forceinline__ void operator()() const {}
};
template <int kRows, Epilogue kEpi, int kOrder, bool kAllAtOnce = (kRows < 256), typename Hook = NoHook>
__device__ __forceinline__ void TileEpilogueWave(const KernelArgs& a, const TileInfo& t, v4i (&acc)[RowBlocks<kRows>::kAll][4], int waveM,
                                                 int waveN, int l16, int quad, const float* ldsChannelScale, const float* ldsRowScale,
                                                 uint32_t* ldsRowMax, Hook beforeStores = NoHook{}) {
    using Blocks = RowBlocks<kRows>;
    constexpr bool kSwiglu = kEpi == Epilogue::kSwiglu;
    const int32_t rows = t.rows, rowBase = t.rowBase, group = t.group;
    // The row / address arithmetic below depends only on the lane; hoisted out of the persistent tile loop it would
    // stay alive across the whole kernel and spill, and a reload in here waits for every store issued so far.  An
    // opaque per-call zero folded into the lane index keeps the arithmetic inside the epilogue.
    int opaqueZero;
    asm volatile("v_mov_b32 %0, 0" : "=v"(opaqueZero));
    quad += opaqueZero;
    l16 += opaqueZero;
    const bool neighbours = kOrder == kOrderLane && LanesHoldNeighbours(a);
    if constexpr (!kSwiglu) {
        const bool hasRowScale = a.rowScale != nullptr;
        int32_t col[4];
        bool valid[4];
        float sc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int n = 0; n < 4; ++n) {
            col[n] = t.colBase + ColumnInTile<kOrder, false>(waveN, n, l16, neighbours);
            valid[n] = col[n] < a.N;
            if (kEpi == Epilogue::kDequant) {
                if (ldsChannelScale != nullptr) sc[n] = ldsChannelScale[ColumnInTile<kOrder, false>(waveN, n, l16, neighbours)];
                else if (valid[n]) sc[n] = LoadScale(a.scale, static_cast<int64_t>(group) * a.N + col[n], a.scaleDtype);
            }
        }
        SettleLoads(sc);
        // wave-uniform: every channel of the wave exists
        const bool whole = t.colBase + ColumnInTile<kOrder, false>(waveN, 3, 15, neighbours) < a.N;
        // Where a lane's four 16-bit results begin, which it stores at once (kOrderBlock: behind BlockOfLane).  us, stores of a block's half
        // lines -> this, bf16, row-major / blocked: 16 groups of 500 rows, K 128 x N 4096 29.3 -> 23.7 / 28.8 -> 23.7; 32 of 400,
        // K 512 x N 2048 32.4 -> 28.3 / 32.5 -> 28.7; 16 of 1000, K 2048 x N 4096 141 -> 131 / 140 -> 133.
        const int32_t vectorCol = kOrder == kOrderLane ? col[0] : t.colBase + 64 * waveN + 16 * (l16 & 3) + 4 * (l16 >> 2);
        // Rows of 16-bit results start on whole dwords, if the output does; 32-bit results always do.  us, K 2048 x N 4098, with vectors
        // only where rows start on 16 bytes -> on any dword: 16 groups of 128 rows bf16 71 -> 63, int32 74 -> 61; of 1000 rows
        // 210 -> 195, 231 -> 180.
        const bool pairs = (a.N & 1) == 0;
        // 16-bit results of whole column blocks, without per-element dtype dispatch; stores through a (uniform row pointer
        // + 32-bit lane offset) address.  Past the caches: nothing reads them back before they have left these.
        const bool halves = kEpi == Epilogue::kDequant && (a.outDtype == 27 || a.outDtype == 1) && whole && pairs;
        const bool toBf16 = a.outDtype == 27;  // wave-uniform: bf16, else fp16
        uint32_t word[kAllAtOnce ? Blocks::kAll : 1][4][2];
        auto results = [&](int m, uint32_t (&w)[4][2], auto bf16Tag) __attribute__((always_inline)) {
            constexpr bool kToBf16 = decltype(bf16Tag)::value;  // compile-time: a run-time choice per element splits the block
            const int rTop = Blocks::RowOf(m, waveM);
            float4 rs = make_float4(1.0f, 1.0f, 1.0f, 1.0f);  // multiplying by 1 is exact
            if (hasRowScale) rs = *reinterpret_cast<const float4*>(ldsRowScale + rTop + 4 * quad);
            const float rsv[4] = {rs.x, rs.y, rs.z, rs.w};
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                float y[4];
#pragma unroll
                for (int n = 0; n < 4; ++n) y[n] = __fmul_rn(__fmul_rn(static_cast<float>(acc[m][n][v]), sc[n]), rsv[v]);
                w[v][0] = PackHalves<kToBf16>(y[0], y[1]);
                w[v][1] = PackHalves<kToBf16>(y[2], y[3]);
            }
        };
        auto forBlocks = [&](auto f) __attribute__((always_inline)) {
#pragma unroll
            for (int m = 0; m < Blocks::kAll; ++m) {
                const int rTop = Blocks::RowOf(m, waveM);
                if (rTop >= rows) continue;
                if (rTop + 16 <= rows) f(m, std::true_type{});
                else f(m, std::false_type{});
            }
        };
        if constexpr (kAllAtOnce) {
            if (halves) {
                if (toBf16) forBlocks([&](int m, auto) __attribute__((always_inline)) { results(m, word[m], std::true_type{}); });
                else forBlocks([&](int m, auto) __attribute__((always_inline)) { results(m, word[m], std::false_type{}); });
            }
        }
        if constexpr (kAllAtOnce) beforeStores();
        if (halves) {
            uint16_t* const outTile = static_cast<uint16_t*>(a.out) + static_cast<int64_t>(rowBase) * a.N;
            const int32_t laneOff = 4 * quad * a.N + vectorCol;
            auto store = [&](int m, uint32_t (&w)[4][2], auto fullTag) __attribute__((always_inline)) {
                constexpr bool kFull = decltype(fullTag)::value;
                const int rTop = Blocks::RowOf(m, waveM);
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    uint16_t* const rowPtr = outTile + static_cast<int64_t>(rTop + v) * a.N;
                    const bool ok = kFull || rTop + 4 * quad + v < rows;
                    if constexpr (kOrder == kOrderBlock) BlockOfLane(w[v], l16);
                    if (ok) __builtin_nontemporal_store(Uint2Half{w[v][0], w[v][1]}, reinterpret_cast<Uint2Half*>(rowPtr + laneOff));
                }
            };
            if constexpr (kAllAtOnce) {
                forBlocks([&](int m, auto fullTag) __attribute__((always_inline)) { store(m, word[m], fullTag); });
            } else {
                forBlocks([&](int m, auto fullTag) __attribute__((always_inline)) {
                    if (toBf16) results(m, word[0], std::true_type{});
                    else results(m, word[0], std::false_type{});
                    store(m, word[0], fullTag);
                });
                beforeStores();
            }
            return;
        }
        if constexpr (!kAllAtOnce) beforeStores();
        const bool vectorStores = neighbours && whole;
        float bias[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        if (kEpi == Epilogue::kDequant && a.bias != nullptr) {
#pragma unroll
            for (int n = 0; n < 4; ++n) {
                if (valid[n]) bias[n] = LoadScale(a.bias, static_cast<int64_t>(group) * a.N + col[n], a.biasDtype);
            }
            SettleLoads(bias);
        }
#pragma unroll
        for (int m = 0; m < Blocks::kAll; ++m) {
            const int rTop = Blocks::RowOf(m, waveM);
            if (rTop >= rows) continue;
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int r = rTop + 4 * quad + v;
                if (r >= rows) continue;
                const int64_t rowOff = static_cast<int64_t>(rowBase + r) * a.N;
                if constexpr (kEpi == Epilogue::kInt32) {
                    int32_t* const out = static_cast<int32_t*>(a.out) + rowOff;
                    if (vectorStores) {
                        *reinterpret_cast<Int4Dword*>(out + col[0]) = Int4Dword{acc[m][0][v], acc[m][1][v], acc[m][2][v], acc[m][3][v]};
                    } else {
#pragma unroll
                        for (int n = 0; n < 4; ++n) {
                            if (valid[n]) out[col[n]] = acc[m][n][v];
                        }
                    }
                    continue;
                }
                const float rs = hasRowScale ? ldsRowScale[r] : 1.0f;
                float y[4];
#pragma unroll
                for (int n = 0; n < 4; ++n) {
                    y[n] = __fmul_rn(static_cast<float>(acc[m][n][v]), sc[n]);
                    if (hasRowScale) y[n] = __fmul_rn(y[n], rs);
                }
                if (a.outDtype == 0) {
                    if (a.combineIndex != nullptr) {
                        const int64_t src = rowBase + r;
                        const int64_t dst = a.combineIndexIsInt64 ? static_cast<const int64_t*>(a.combineIndex)[src]
                                                                  : static_cast<const int32_t*>(a.combineIndex)[src];
                        if (dst < 0 || dst >= a.combineRows) continue;
                        if (a.bias != nullptr) {
                            const float wgt = a.combineWeight != nullptr ? a.combineWeight[src] : 1.0f;
#pragma unroll
                            for (int n = 0; n < 4; ++n) y[n] = __fadd_rn(y[n], __fmul_rn(wgt, bias[n]));
                        }
                        float* const dstRow = static_cast<float*>(a.out) + dst * a.N;
#pragma unroll
                        for (int n = 0; n < 4; ++n) {
                            if (valid[n]) unsafeAtomicAdd(dstRow + col[n], y[n]);
                        }
                        continue;
                    }
                    float* const out = static_cast<float*>(a.out) + rowOff;
                    if (vectorStores) {
                        *reinterpret_cast<Float4Dword*>(out + col[0]) = Float4Dword{y[0], y[1], y[2], y[3]};
                    } else {
#pragma unroll
                        for (int n = 0; n < 4; ++n) {
                            if (valid[n]) out[col[n]] = y[n];
                        }
                    }
                    continue;
                }
                uint16_t* const out = static_cast<uint16_t*>(a.out) + rowOff;
#pragma unroll
                for (int n = 0; n < 4; ++n) {
                    const uint32_t bits = a.outDtype == 27 ? PackHalves<true>(y[n], 0.0f) : PackHalves<false>(y[n], 0.0f);
                    if (valid[n]) out[col[n]] = static_cast<uint16_t>(bits & 0xffffu);
                }
            }
        }
    } else {
        float scA[2], scB[2];
        int32_t col[2];  // columns of S
        bool valid[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            col[j] = t.colBase + ColumnInTile<kOrder, true>(waveN, j, l16, true);
            valid[j] = col[j] < a.halfN;
            scA[j] = scB[j] = 0.0f;
            if (ldsChannelScale != nullptr) {
                const int c = ColumnInTile<kOrder, true>(waveN, j, l16, true);
                scA[j] = ldsChannelScale[c];
                scB[j] = ldsChannelScale[kTileN / 2 + c];
            } else if (valid[j]) {
                scA[j] = LoadScale(a.scale, static_cast<int64_t>(group) * a.N + col[j], a.scaleDtype);
                scB[j] = LoadScale(a.scale, static_cast<int64_t>(group) * a.N + a.halfN + col[j], a.scaleDtype);
            }
        }
        SettleLoads(scA);
        SettleLoads(scB);
        // swish(ca) * cb with the hardware exp2 / reciprocal: a few ulp from the correctly rounded value, far inside the
        // +-1 LSB the int8 requantisation is held to
        auto activated = [&](int m, int j, int v, float xs) __attribute__((always_inline)) {
            const float ca = __fmul_rn(__fmul_rn(static_cast<float>(acc[m][j][v]), xs), scA[j]);
            const float cb = __fmul_rn(__fmul_rn(static_cast<float>(acc[m][2 + j][v]), xs), scB[j]);
            return __fmul_rn(__fmul_rn(ca, __builtin_amdgcn_rcpf(__fadd_rn(1.0f, __expf(-ca)))), cb);
        };
        // wave-uniform: every column of the wave exists, and S rows start on a lane's pair
        const bool whole = t.colBase + 32 * waveN + 32 <= a.halfN && (kOrder != kOrderLane || (a.halfN & 1) == 0);
        Float2 s[kAllAtOnce ? Blocks::kAll : 1][4];
        auto results = [&](int m, Float2 (&out)[4], auto fullTag) __attribute__((always_inline)) {
            constexpr bool kFull = decltype(fullTag)::value;
            const int rTop = Blocks::RowOf(m, waveM);
            const float4 xs4 = *reinterpret_cast<const float4*>(ldsRowScale + rTop + 4 * quad);
            const float xs[4] = {xs4.x, xs4.y, xs4.z, xs4.w};
            float top[4];
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                out[v] = Float2{activated(m, 0, v, xs[v]), activated(m, 1, v, xs[v])};
                const bool ok = kFull || rTop + 4 * quad + v < rows;
                top[v] = ok ? fmaxf(fabsf(out[v][0]), fabsf(out[v][1])) : 0.0f;
            }
            const float m16 = FourMaxOver16(top, l16);
            if ((l16 & 3) == 0) RaiseRowMax(ldsRowMax + rTop + 4 * quad + (l16 >> 2), m16);
        };
        auto forBlocks = [&](auto f) __attribute__((always_inline)) {
#pragma unroll
            for (int m = 0; m < Blocks::kAll; ++m) {
                const int rTop = Blocks::RowOf(m, waveM);
                if (rTop >= rows) continue;
                if (rTop + 16 <= rows) f(m, std::true_type{});
                else f(m, std::false_type{});
            }
        };
        if constexpr (kAllAtOnce) {
            if (whole) forBlocks([&](int m, auto fullTag) __attribute__((always_inline)) { results(m, s[m], fullTag); });
            beforeStores();
        }
        if (whole) {
            float* const sTile = a.sOut + static_cast<int64_t>(rowBase) * a.halfN;
            const int32_t laneOff = 4 * quad * a.halfN + col[0];
            auto store = [&](int m, const Float2 (&v2)[4], auto fullTag) __attribute__((always_inline)) {
                constexpr bool kFull = decltype(fullTag)::value;
                const int rTop = Blocks::RowOf(m, waveM);
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    float* const sRow = sTile + static_cast<int64_t>(rTop + v) * a.halfN;
                    const bool ok = kFull || rTop + 4 * quad + v < rows;
                    if constexpr (kOrder == kOrderLane) {
                        if (ok) __builtin_nontemporal_store(v2[v], reinterpret_cast<Float2*>(sRow + laneOff));
                    } else {
                        if (ok) __builtin_nontemporal_store(v2[v][0], sRow + laneOff);
                        if (ok) __builtin_nontemporal_store(v2[v][1], sRow + laneOff + 16);
                    }
                }
            };
            forBlocks([&](int m, auto fullTag) __attribute__((always_inline)) {
                if constexpr (!kAllAtOnce) results(m, s[0], fullTag);
                store(m, s[kAllAtOnce ? m : 0], fullTag);
            });
            if constexpr (!kAllAtOnce) beforeStores();
            return;
        }
        if constexpr (!kAllAtOnce) beforeStores();
#pragma unroll
        for (int m = 0; m < Blocks::kAll; ++m) {
            const int rTop = Blocks::RowOf(m, waveM);
            if (rTop >= rows) continue;
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int r = rTop + 4 * quad + v;
                float top = 0.0f;
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    if (r < rows && valid[j]) {
                        const float s = activated(m, j, v, ldsRowScale[r]);
                        a.sOut[static_cast<int64_t>(rowBase + r) * a.halfN + col[j]] = s;
                        top = fmaxf(top, fabsf(s));
                    }
                }
                top = MaxOver16(top);
                if (l16 == 0) RaiseRowMax(ldsRowMax + r, top);
            }
        }
    }
}

// The part of the kSwiglu epilogue behind a barrier: one partial maximum per (256 channels, row) goes to memory -- no atomics there and
// nothing to pre-zero; the requantisation folds them -- and the LDS copies start at zero again.  (The workgroup has at least kRows threads.)
template <int kRows>
__device__ __forceinline__ void TileEpilogueStoreMax(const KernelArgs& a, const TileInfo& t, int32_t unit, int32_t units, int tid, uint32_t* ldsRowMax) {
    if (tid < t.rows) {
        const float m = __uint_as_float(ldsRowMax[tid]);
        for (int32_t u = unit; u < unit + units; ++u) a.rowMax[static_cast<int64_t>(u) * a.M + t.rowBase + tid] = m;
        ldsRowMax[tid] = 0;
    }
}

// Calls f(std::integral_constant<int, n>) for n = count clamped into 0..kMax.
template <int kMax, typename F>
__device__ __forceinline__ void ForCount(int count, F& f) {
    if constexpr (kMax == 0) {
        f(std::integral_constant<int, 0>{});
    } else {
        if (count >= kMax) f(std::integral_constant<int, kMax>{});
        else ForCount<kMax - 1>(count, f);
    }
}

// ---------------------------------------------------------------------------------------------- fast path: LDS-DMA ring
// k-bytes per ring stage: 128 streams weights in whole lines (best HBM efficiency).
constexpr int kStep = 128;

// A stage is kRows activation rows and 256 weight channels of 128 k-bytes each; the two kinds have rings of their own depth in
// LDS.  A k-step multiplies a stage in four products, two halves of the wave's rows times two slices of 64 k, and the fragments
// of a product are read from LDS while the one before it is multiplied (fragment double buffers).  The buffers that a step reads
// are refilled in two goes, each behind a barrier:
//     product    first half x 0    first half x 1     second half x 0    second half x 1
//     reads      weights, 1        second half, 0     second half, 1     of the next step: weights and first half, 0
//                first half, 1
//     requests                                        even slots         odd slots
// The barrier in the middle says that every wave has read the weights and the first half of the rows, the one in front of the
// last product that it has read the second half, and that the next stage has landed.  The requests go out one at a time between
// the matrix instructions.
// What bounds it: with few experts of thousands of rows the matrix unit's power; with about a hundred rows each, the HBM and the
// latency under it.  Gate/up and down in us, as 32x32x32 instructions on whole stages refilled in one burst behind a step's
// barrier, and now: 16384 tokens top-2 of 8 experts, hidden 4096, intermediate 14336: 3922 / 1761 -> 3367 / 1515 (2.29 and 2.54
// POP/s); 4096 top-8 of 256, 7168, 2048: 1526 / 876 -> 1461 / 836; 8192 of these at popularity rank^-1.2: 2278 / 1305 -> 2031 /
// 1152; 2047 top-8 of 128, 4096, 1536: 360 / 230 -> 352 / 223.
// (With the first barrier a quarter of a step earlier, so that every part had as long to land, its wait for the fragments just
// requested showed: 16384 tokens, 8 experts, hidden 4096, intermediate 14336, 3716 against 3418 us gate/up and 1685 / 1578 down.
// Eight barriers a step, the two wave rows half a phase apart: 3400 / 1480 there, but 254 against 219 us where a tile has 128 rows
// and twelve steps.)
//
// Wave row 0 requests the weights, wave row 1 the activation rows.  A wave's loads return in issue order, so a wave that had
// to wait for activation rows, which come out of L2 and need one or two stages in flight, would wait for all weights
// requested before them, which come out of HBM and want to be three stages ahead.
//
// One DMA instruction moves 64 lanes x 16 bytes = 8 rows of 128 k-bytes.  Slot q of wave column w is instruction w + 4 q of
// its kind, i.e. 32 rows per slot: even slots of the activation rows are the first half of the wave rows' blocks.
template <int kRows, Epilogue kEpi, int kUnits = 1>
struct StreamCfg {
    using Blocks = RowBlocks<kRows>;
    static constexpr int kStageBytesA = kRows * kStep;
    static constexpr int kStageBytesB = kTileN * kStep;
    static constexpr int kHalfBytesB = kStageBytesB / 2;
    static constexpr int kQueueLdsInts = 40;  // the workgroup's next eight tiles and how it comes by them
    static constexpr int kRowScales = (kRows + 63) / 64 * 64;  // in whole DMA instructions
    // SwiGLU tiles of 256 rows, whose rings are two stages deep, hold the next tile's scales too (see requestScales).
    static constexpr int kScaleSets = kRows == 256 && kEpi == Epilogue::kSwiglu ? 2 : 1;
    // channel scales, row scales, row maxima, tiles
    static constexpr int kScratchBytes = (kScaleSets * (kUnits * kTileN + kRowScales) + kRows + kQueueLdsInts) * 4;
    static constexpr int kRingBytes = kLdsBudget - kScratchBytes;
    // as many weight stages as leave room for two of activation rows, then as many of those as fit
    static constexpr int kFitB = (kRingBytes - 2 * kStageBytesA) / kStageBytesB;
    // (64 rows: a fourth only puts off the first one's requests in a launch of a tile or two.  us, 8 experts of 20 rows, K 1024 x N 2048,
    // row-major 16.3 -> 15.8; 16 of 30, K 512 x N 1024 13.4 -> 12.8; 60 of 24, K 768 x N 2048 26.8 -> 26.0; long launches the same.)
    static constexpr int kStagesB = kRows == 64 ? 3 : kFitB > 4 ? 4 : kFitB;
    static constexpr int kFitA = (kRingBytes - kStagesB * kStageBytesB) / kStageBytesA;
    static constexpr int kStagesA = kFitA > kStagesB ? kStagesB : kFitA;
    static constexpr int kFirstB = kStagesA * kStageBytesA;  // the ring of weight stages, behind that of the activation rows
    static constexpr int kLdsBytes = kFirstB + kStagesB * kStageBytesB + kScratchBytes;
    static constexpr int kSlotsA = kRows / 32, kSlotsB = kTileN / 32;  // a wave's DMA instructions per stage
    static_assert(kSlotsA <= kSlotsB && kStagesA >= 2 && kStagesB >= 2 && kThreads >= kRows, "");
    // a wave's DMA instructions younger than the next stage's last one, in front of the last product of a step
    static constexpr int kYoungerA = (kStagesA - 2) * kSlotsA + (kSlotsA + 1) / 2;
    static constexpr int kYoungerB = (kStagesB - 2) * kSlotsB + (kSlotsB + 1) / 2;
    static_assert(kStagesB * kSlotsB <= 63, "vmcnt is a 6-bit counter");
};

// Byte offset of 16-byte chunk `chunk` of row `row` in a stage whose rows are 128 bytes.  The LDS serves 16 lanes per
// clock out of 64 banks (256 bytes): the chunk index is XOR-ed with row bits such that 16 consecutive rows reading the
// same logical chunk land in 16 different 16-byte bank groups.
__device__ __forceinline__ int LdsOffset(int row, int chunk) { return row * 128 + ((chunk ^ ((row >> 1) & 7)) << 4); }

// What the 16-byte chunk index of k-row k of a row-major weight half (rows of 128 channel bytes) is XOR-ed with: the 32
// lanes that the LDS serves together read one chunk of eight consecutive k-rows and of those sixteen further on, and these
// sixteen pieces land in different bank groups.
__device__ __forceinline__ int RowMajorSwizzle(int k) { return ((k >> 1) & 3) | (((k >> 4) & 1) << 2); }
// The same for rows of 256 channel bytes, which begin on the same bank each.
__device__ __forceinline__ int RowMajorWideSwizzle(int k) { return (k & 7) | (((k >> 4) & 1) << 3); }

// A wave-uniform pointer, forced into scalar registers.
__device__ __forceinline__ const char* UniformPtr(const char* p) {
    const uint64_t b = reinterpret_cast<uint64_t>(p);
    const uint32_t lo = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(static_cast<uint32_t>(b))));
    const uint32_t hi = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(static_cast<uint32_t>(b >> 32))));
    return reinterpret_cast<const char*>(static_cast<uint64_t>(lo) | (static_cast<uint64_t>(hi) << 32));
}

// The 32-bit LDS address of a generic pointer into LDS (wave-uniform).
__device__ __forceinline__ uint32_t LdsAddress(const char* p) {
    typedef __attribute__((address_space(3))) const char* LdsPtr;
    return static_cast<uint32_t>(
        __builtin_amdgcn_readfirstlane(static_cast<int>(static_cast<uint32_t>(reinterpret_cast<size_t>((LdsPtr)p)))));
}

// 16 bytes of LDS at a 32-bit address and a constant (in the instruction's offset field).
__device__ __forceinline__ v4i LdsRead16(uint32_t addr, int offset) {
    typedef __attribute__((address_space(3))) const char* LdsPtr;
    return *(LdsV4iPtr)(reinterpret_cast<LdsPtr>(addr) + offset);
}

// Sixteen consecutive k of one channel, from two transposing loads of eight k-rows each.
__device__ __forceinline__ v4i LdsReadTransposed(uint32_t addr, int offset, int eightK) {
    typedef __attribute__((address_space(3))) char* LdsPtr;
    const v2i lo = __builtin_amdgcn_ds_read_tr8_b64_v2i32((LdsV2iPtr)(reinterpret_cast<LdsPtr>(addr) + offset));
    const v2i hi = __builtin_amdgcn_ds_read_tr8_b64_v2i32((LdsV2iPtr)(reinterpret_cast<LdsPtr>(addr) + offset + eightK));
    return v4i{lo[0], lo[1], hi[0], hi[1]};
}

// 16 bytes per lane from (uniform base + 32-bit lane offset) straight into LDS at ldsAddr + lane * 16 (ldsAddr is the
// 32-bit LDS address, see LdsAddress).  The compiler does not see this as a memory instruction: completion is awaited
// with WaitVmcnt below.
// kStreaming marks the load non-temporal: the bytes are used once (weights), so they should not push the operands
// that are re-read from L2 (activation rows) out of the caches.
// The instruction takes its LDS base from m0, which the statement sets itself.  m0 is a reserved register that cannot
// be named as a clobber; nothing else in these kernels uses it (no LDS-direct or register-indexed code is generated
// for them), and the compiler sets m0 afresh before any use of its own.
template <bool kStreaming>
__device__ __forceinline__ void DmaToLdsAddr16(const char* base, uint32_t laneOffset, uint32_t ldsAddr) {
    const uint32_t m0 = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(ldsAddr)));
    const char* const sbase = UniformPtr(base);
    if (kStreaming) {
        asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, %2 nt" ::"s"(m0), "v"(laneOffset), "s"(sbase) : "memory");
    } else {
        asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(m0), "v"(laneOffset), "s"(sbase) : "memory");
    }
}

// 4 bytes per lane from (uniform base + lane offset) into LDS at ldsAddr + lane * 4 (see DmaToLdsAddr16).
__device__ __forceinline__ void DmaToLdsAddr4(const char* base, uint32_t laneOffset, uint32_t ldsAddr) {
    const uint32_t m0 = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(ldsAddr)));
    const char* const sbase = UniformPtr(base);
    asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dword %1, %2" ::"s"(m0), "v"(laneOffset), "s"(sbase) : "memory");
}

// The value itself, through a statement the optimiser cannot see through: what is computed from the copy stays where it
// is written.  Used on lane indices at the head of per-tile code, so that the per-lane offsets and addresses of that code
// are recomputed once per tile instead of being hoisted out of the tile loop and held in registers (or spilled) across the
// k loop, where the accumulators and fragments of the tallest tiles leave no room for them.
__device__ __forceinline__ int Opaque(int v) {
    asm volatile("" : "+v"(v));
    return v;
}

// The kernel's arguments (its first parameter), read again from memory.  What only the epilogue wants of them would otherwise stay
// in scalar registers across the k loop, and those of the tallest tiles, once spilled, cost vector registers that are not there.
// (Through the address space of constants, i.e. the scalar cache: vector loads, which is what a plain pointer gives here, would wait
// behind every DMA in flight.)
__device__ __forceinline__ KernelArgs ReloadArgs() {
    typedef __attribute__((address_space(4))) const KernelArgs* ArgsPtr;
    auto p = (ArgsPtr)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    KernelArgs a;
    __builtin_memcpy(&a, p, sizeof(a));
    return a;
}

template <int kCount>
__device__ __forceinline__ void WaitVmcnt() {  // s_waitcnt vmcnt(kCount), leaving expcnt / lgkmcnt untouched
    __builtin_amdgcn_s_waitcnt(0x0f70 | (kCount & 15) | ((kCount >> 4) << 14));
}

// This wave's LDS reads and writes have been carried out, all but the youngest kPending (they are carried out in order;
// s_waitcnt lgkmcnt(kPending) alone).
template <int kPending = 0>
__device__ __forceinline__ void WaitLds() {
    static_assert(kPending < 16, "lgkmcnt is a 4-bit counter");
    __builtin_amdgcn_s_waitcnt(0xc07f | (kPending << 8));
}

// The workgroup's barrier, and nothing crosses it in the compiler's order.  Unlike __syncthreads() it waits for no memory
// request: what has to have landed in front of it is waited for by count.
__device__ __forceinline__ void PhaseBarrier() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
}

// Persistent: the grid is one workgroup per CU (a multiple of 8); workgroup b serves XCD b % 8 and walks that XCD's
// share of the tile list with stride gridDim / 8.
//
// kNz: the weights come in the 32-channel x 16-k blocked layout.  A 32-channel block is then one contiguous stream of
// K x 32 bytes, so a stage's weight part is eight 4 KB pieces that land in LDS as [block][k][32 channels]; the MFMA
// operand (16 consecutive k of one channel per lane) is read back with the transposing LDS load ds_read_b64_tr_b8:
// per 16 lanes, lanes 2r and 2r + 1 supply the two 8-byte halves of row r (r = 0..7) and lane i receives column i,
// i.e. with rows = 8 consecutive k and columns = 16 channels each lane gets 8 consecutive k of its channel.  (The two
// sixteen-channel halves of a k-row lie swapped where bit 4 of k is set: the 32 lanes served together read k-rows sixteen
// apart.)
//
// kNMajor: the weights are row-major [K, N] per expert (N contiguous), the reference's plain ND layout of the grouped
// matmul.  A stage's weight half is then 128 k-rows of 128 channel bytes (kSwiglu: of the gate or of the up half); it lies
// in LDS as [k][128] with the chunks of row k swizzled (RowMajorSwizzle), and the operands come out through the same
// transposing load as for the blocked layout.
//
// kRun: which runs of the m-tile table the body serves.  kBothRuns: all of it (pulled or in fixed shares).  kBigRun /
// kSmallRun: that run only, pulled, until its counters are used up on every XCD -- the form in which MixedGemmKernel
// calls the body twice, once per run with a stage geometry of that run's own; `begins` says for which of them.
//
// kUnits: how many times 256 channels a tile is wide.  With two, a k-step is one stage of activation rows and two of weights, multiplied in
// turn, and the ring of the rows moves on at every other stage of the weights'.  The accumulators of 160 rows and the fragments are what
// the registers hold.
//
// kTail: K is a multiple of 16 and at least one k-step, but no multiple of a k-step.  The last k-step then starts kStep
// bytes before the end of K instead of behind the step before it: every DMA stays inside its row and is as wide as any
// other, and the k that the step before has already covered are multiplied by zero (the weight fragments of that one
// step are masked).
// Before, such K went through the byte-wise kernel: a 301-token pass over 32 experts with hidden 2880 and intermediate
// 1440 took 1.396 ms and takes 0.126 ms (its 398 MB of weights alone are 0.06 ms at the HBM's streaming rate).
constexpr int kBigRun = 0, kSmallRun = 1, kBothRuns = 2;
template <int kRows, Epilogue kEpi, bool kNz, bool kNMajor, int kRun, bool kTail, int kUnits = 1>
__device__ __forceinline__ void StreamGemmBody(const KernelArgs& a, const int32_t* __restrict__ sched, char* const lds,
                                               uint64_t& spanTiles, bool begins = true) {
    static_assert(!(kNz && kNMajor), "one weight layout at a time");
    using Cfg = StreamCfg<kRows, kEpi, kUnits>;
    using Blocks = RowBlocks<kRows>;
    constexpr bool kSwiglu = kEpi == Epilogue::kSwiglu;
    constexpr int kUnitCols = kSwiglu ? kTileN / 2 : kTileN;  // output columns of 256 channels
    float* const ldsScales = reinterpret_cast<float*>(lds + Cfg::kFirstB + Cfg::kStagesB * Cfg::kStageBytesB);
    constexpr int kScaleSet = kUnits * kTileN + Cfg::kRowScales;  // of a tile: [kUnits][kTileN] of channels, [kRowScales] of rows
    uint32_t* const ldsRowMax = reinterpret_cast<uint32_t*>(ldsScales + Cfg::kScaleSets * kScaleSet);  // [kRows]

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int waveN = wave % kWavesN;
    const int waveM = wave / kWavesN;

    // ---- this workgroup's sequence of tiles ----
    // Workgroup b serves XCD b % 8 as its slot b / 8.  Wave 0 finds the tiles and leaves them, decoded, in an eight-entry ring
    // in LDS.  With a.pullTiles the first ones are its seat's and the others come out of the tile counters (see QueueShare): tile n + 2 is
    // drawn while tile n's epilogue runs, because the issue side already reads tile n + 1's operands during tile n.  Otherwise (tiles of 256 channels only) the two runs of the m-tile table are one list cut into eight fixed
    // shares, which the workgroups of an XCD walk with stride gridDim / 8, and the ring holds six tiles (tiles of one k-step
    // have the issue side five tiles ahead).
    const int xcd = blockIdx.x % kXcds;
    const int32_t slots = gridDim.x / kXcds;
    const int32_t slot = blockIdx.x / kXcds;
    constexpr bool kOneRun = kRun != kBothRuns;
    const bool pull = kOneRun || kUnits > 1 || a.pullTiles != 0;
    int32_t* const ldsSeq = reinterpret_cast<int32_t*>(ldsRowMax + kRows);
    // wave 0's state, behind the ring: used-up counters, tiles of a share that are dealt out (big, small), this workgroup's next tile of those,
    // how many it has left, and how far apart they are
    constexpr int kSeqUsedUp = 32, kSeqSeated = 33, kSeqSeatNext = 35, kSeqSeatLeft = 36, kSeqSeatStride = 37;
    constexpr int kTilesAhead = 6;
    // Which list this workgroup draws from first.
    const int32_t forSmall = sched[0] == 0 ? slots : SlotsForSmall<kEpi, kNMajor, kOneRun>(sched, slots, a.tilesN);
    const int prefer = kOneRun ? kRun : (slot < forSmall ? 1 : 0);
    auto tilesAcross = [](const KernelArgs& args) __attribute__((always_inline)) { return (args.tilesN + kUnits - 1) / kUnits; };
    // tile `logical` of a run (list < 0: none), decoded
    auto decodeTile = [&](const KernelArgs& args, const RunTable& r, int32_t list, int32_t logical) __attribute__((always_inline)) -> v4i {
        if (list < 0) return v4i{0, 0, 0, 0};
        const TileInfo t = DecodeListTile<kSwiglu>(tilesAcross(args), r.entries, list ? r.countBig : 0, list ? r.countSmall : r.countBig,
                                                   list ? r.bandSmall : r.bandBig, logical);
        return v4i{t.group, t.rowBase, t.rows, t.tileN};
    };
    // the n-th tile of this workgroup in fixed shares
    auto shareTile = [&](const KernelArgs& args, const RunTable& r, int32_t n) __attribute__((always_inline)) -> v4i {
        const int32_t big = r.countBig * args.tilesN, total = big + r.countSmall * args.tilesN;
        const int32_t perXcd = (total + kXcds - 1) / kXcds, local = slot + n * slots, logical = xcd * perXcd + local;
        const bool none = local >= perXcd || logical >= total;
        return decodeTile(args, r, none ? -1 : logical < big ? 0 : 1, logical < big ? logical : logical - big);
    };
    auto leaveTile = [&](int32_t n, v4i e) __attribute__((always_inline)) { *reinterpret_cast<v4i*>(ldsSeq + 4 * (n & 7)) = e; };
    // the n-th tile of this workgroup, out of the ring
    auto tileAt = [&](int32_t n) __attribute__((always_inline)) -> TileInfo {
        const int4 e = *reinterpret_cast<const int4*>(ldsSeq + 4 * (n & 7));
        TileInfo t;
        t.group = __builtin_amdgcn_readfirstlane(e.x);
        t.rowBase = __builtin_amdgcn_readfirstlane(e.y);
        t.rows = __builtin_amdgcn_readfirstlane(e.z);
        t.tileN = __builtin_amdgcn_readfirstlane(e.w);
        t.valid = t.rows > 0;
        t.colBase = t.tileN * kUnits * kUnitCols;
        return t;
    };
    // 256-channel units of a tile, and the first column of its second: where that would end behind the last column it begins earlier, over
    // columns of the first, which then are computed, and stored, twice
    auto unitsOf = [&](const TileInfo& t) __attribute__((always_inline)) { return min(kUnits, a.tilesN - kUnits * t.tileN); };
    auto secondUnit = [&](const TileInfo& t) __attribute__((always_inline)) { return min(t.colBase + kUnitCols, (kSwiglu ? a.halfN : a.N) - kUnitCols); };
    // Side by side: their table entries are one round trip (0.3 to 1.2 us of a launch of shares, as one thread's loop).
    if (!pull && tid < kTilesAhead) leaveTile(tid, shareTile(a, ReadRunTable(sched), tid));
    if (kSwiglu && tid < kRows) ldsRowMax[tid] = 0;
    // Seats: the first `each` tiles of a workgroup are not drawn but dealt out, those of seats side by side neighbours.  Two, so that no
    // draw stands in front of the launch, and an XCD's workgroups walk neighbouring tiles from the start (two draws at once handed
    // each of them two neighbours, its first round being every other tile of twice as many groups).  All whole rounds where the tiles are
    // alike (kHdrEven): those launches are bound by memory, where a workgroup that lags gets the bandwidth that others leave, while one
    // that is ahead and draws a tile more ends the launch alone.  us, 128 experts of 128 rows, gate/up 4096 x 2 x 1536 and down, six
    // and eight rounds: drawn 344 / 207, two dealt out 334 / 204, all 327 / 194; 256 experts, 7168, 2048: 1441 / 800, 1425 / 772,
    // 1427 / 762.  Not so where tiles differ: 65536 rows at popularity rank^-1.2, all dealt out, 2264 / 1220 against 1940 / 1080.
    // A run of no more tiles than there are workgroups: one tile each.  A second one taken along with it would be missing
    // where another workgroup is idle (128 tiles of K 14336: 200 us, or 400 where one had two).  In the two-geometry
    // form fewer workgroups than that begin with the run; they go on to the other run after their one tile, and the tiles
    // left of this one fill the last round of that.  us, drawing on until the run is used up -> one each: 8 experts of 1000
    // rows, gate/up 7168 x 2 x 2048 with 4 of 40 rows 303 -> 262, K 14336 x N 4096 with 4 of 60 514 -> 448; K 1408 x
    // N 2048, 216 big and 104 small tiles 67 -> 52; the other way round 830 -> 858 at most (of sixty launches).
    if (wave == 0 && pull) {
        const RunTable runs = ReadRunTable(sched);
        const int32_t bigTiles = runs.countBig * tilesAcross(a), smallTiles = runs.countSmall * tilesAcross(a);
        auto eachOf = [&](int32_t tiles) __attribute__((always_inline)) {
            return (kOneRun ? tiles : bigTiles + smallTiles) <= static_cast<int32_t>(gridDim.x) ? 1 : 2;
        };
        int32_t eachBig = eachOf(bigTiles), eachSmall = eachOf(smallTiles);
        if (sched[kHdrEven] != 0) {
            if (eachBig > 1 && slots > forSmall) eachBig = max(eachBig, bigTiles / kXcds / (slots - forSmall));
            // (2: the part of a round that is left too; drawn, it would cost every workgroup a draw that finds nothing, some 6 us)
            const int32_t lastRound = sched[kHdrEven] == 2 ? kXcds * slots - 1 : 0;
            if (eachSmall > 1 && bigTiles == 0) eachSmall = max(eachSmall, (smallTiles + lastRound) / kXcds / slots);
        }
        const QueueLists lists{bigTiles, smallTiles, eachBig * (slots - forSmall), eachSmall * forSmall};
        const int32_t seats = prefer ? forSmall : slots - forSmall, seat = prefer ? slot : slot - forSmall;
        const int32_t each = prefer ? eachSmall : eachBig;
        int32_t first, size;
        QueueShare(QueueLists{bigTiles, smallTiles, 0, 0}, 2 * xcd + prefer, &first, &size);
        // tiles that this workgroup is dealt: seat, seat + seats, ... of the share
        const int32_t dealt = begins && seat < size ? min(each, (size - seat + seats - 1) / seats) : 0;
        int32_t drawnFirst, drawn;
        QueueShare(lists, tid & (2 * kXcds - 1), &drawnFirst, &drawn);
        const uint32_t allSeated = static_cast<uint32_t>(__ballot(tid < 2 * kXcds && drawn <= 0));  // shares without a tile to draw
        if (tid == 0) {
            ldsSeq[kSeqUsedUp] = static_cast<int32_t>(allSeated);
            ldsSeq[kSeqSeated] = lists.seatedBig;
            ldsSeq[kSeqSeated + 1] = lists.seatedSmall;
            ldsSeq[kSeqSeatNext] = first + seat + 2 * seats;
            ldsSeq[kSeqSeatLeft] = dealt - 2;
            ldsSeq[kSeqSeatStride] = seats;
        }
        if (dealt >= min(each, 2)) {
            const v4i tile0 = decodeTile(a, runs, prefer, first + seat), tile1 = decodeTile(a, runs, each == 1 ? -1 : prefer, first + seat + seats);
            if (tid == 0) {
                leaveTile(0, tile0);
                leaveTile(1, tile1);
            }
        } else if (tid == 0) {  // both draws, if there are two, go out together
            const int c = QueueFirstOpen(allSeated, xcd, prefer, kOneRun);
            int32_t v[2] = {0, 0};
            if (c >= 0) {
                if (dealt < 1) v[0] = QueueTake(a.queueCounters, c);
                if (each > 1) v[1] = QueueTake(a.queueCounters, c);
            }
            QueueDraw d{prefer, first + seat, allSeated};
#pragma unroll 1
            for (int n = 0; n < 2; ++n) {
                if (n >= each) d.list = -1;
                else if (n >= dealt && d.list >= 0) d = QueueResolve(lists, a.queueCounters, xcd, prefer, d.usedUp, c, n == 0 ? v[0] : v[1], kOneRun);
                leaveTile(n, decodeTile(a, runs, d.list, d.logical));
            }
            ldsSeq[kSeqUsedUp] = static_cast<int32_t>(d.usedUp);
        }
    }
    __syncthreads();

    int32_t curNo = 0;  // position of the tile being computed in this workgroup's sequence
    TileInfo cur = tileAt(0);
    if (!cur.valid) return;
    const int kSteps = kTail ? (a.K + kStep - 1) / kStep : a.K / kStep;
    // Small tiles are the decode shapes: a handful of rows per expert, every weight byte used once, pure streaming.
    constexpr bool kSmallTile = kRows <= 64;
    // The k-steps of a tile are walked from a start of its own (integer accumulation does not care about the order; not with
    // kTail, whose last step is masked).  When rows lie a power-of-two stride apart (K = 4096 with K-contiguous weights), the low
    // address bits of every row of every expert depend on the k offset alone: workgroups that all sit at the same k-step all
    // queue on the same memory channels.  Small tiles, where every weight byte is used once, start where their workgroup says;
    // taller ones where their group says: the tiles of a group share operands through L2, and walking k in step is what makes
    // those hits.  us from one start for all -> a start per group, K 4096:
    //   128 experts of 100 rows, N 3072 with SwiGLU 345 -> 322; 8 of 180, N 28672 with SwiGLU 252 -> 230; 16 of 100, N 4096 79 -> 64.
    //   K 2048, 7168, 14336, the two other weight layouts, and groups of many m-tiles: the same within 1 %.
    // A start per workgroup instead on tall tiles cost 3 to 8 %.
    const int blockRotate = kSmallTile && !kTail ? static_cast<int>((blockIdx.x * 7u + blockIdx.x / kXcds) % static_cast<unsigned>(kSteps)) : 0;
    auto rotateOf = [&](const TileInfo& t) __attribute__((always_inline)) {
        if (kTail) return 0;
        if (kSmallTile) return blockRotate;
        // the golden ratio spreads any arithmetic sequence of groups
        return static_cast<int>(((static_cast<uint32_t>(t.group) * 0x9e3779b1u) >> 16) * static_cast<uint32_t>(kSteps) >> 16);
    };

    // ---- issue side: runs ahead of the compute side by the depth of the ring, across tile boundaries ----
    // The cursor walks this workgroup's tiles k-step by k-step, for the kind of operand that this wave requests.
    const bool forWeights = waveM == 0;
    const uint32_t ldsBase = LdsAddress(lds);
    TileInfo issTile = cur;
    int32_t issNo = 0;        // position of the cursor's tile in the sequence
    int issStep = 0;          // k-step of the tile that goes out next
    int issRotate = rotateOf(cur);
    bool issDrained = false;  // no further tile: the issue slots re-read one hot kilobyte (see advance)
    const uint32_t issFirst = ldsBase + (forWeights ? Cfg::kFirstB : 0) + 1024 * waveN;  // where slot 0 goes, first buffer of the ring
    const uint32_t issStride = forWeights ? Cfg::kStageBytesB : Cfg::kStageBytesA;
    const uint32_t issEnd = issFirst + (forWeights ? Cfg::kStagesB * Cfg::kStageBytesB : Cfg::kStagesA * Cfg::kStageBytesA);
    uint32_t issAddr = issFirst;
    const char* issBase = nullptr;  // the tile's activation rows, or its expert's weights
    uint32_t laneOff[Cfg::kSlotsB];
    int32_t issUnit = 0, issUnits = 1;  // weights: unit of the k-step that goes out next
    int64_t issUnitShift = 0;           // from the first unit's weights to the second's, bytes

    // The lambdas below are forced inline: left to the inliner's size heuristics, one of them staying a real call puts
    // the whole issue state (captured by reference) into scratch memory and the kernel runs three times slower.
    // Base (in scalar registers: a DMA is then three instructions, LDS address, m0 and the load) and lane offsets for tile t.
    auto setupIssue = [&](const TileInfo& t) __attribute__((always_inline)) {
        const int lane = Opaque(tid) & 63;
        const int rowIn = lane >> 3, slot = lane & 7;  // row inside the instruction, LDS chunk slot
        if (!forWeights) {
            issBase = UniformPtr(reinterpret_cast<const char*>(a.x) + static_cast<int64_t>(t.rowBase) * a.K);
#pragma unroll
            for (int q = 0; q < Cfg::kSlotsA; ++q) {
                // rows past the tile's last row are never used: such lanes re-read the last real row (same cache
                // lines as its own lanes), and an instruction wholly past it reads one chunk, so the number of DMAs
                // per stage stays constant while the activation traffic follows the real row count
                const int firstRow = 8 * (waveN + kWavesN * q), r = firstRow + rowIn;
                laneOff[q] = firstRow >= t.rows ? 0u : static_cast<uint32_t>(min(r, t.rows - 1) * a.K + (slot ^ ((r >> 1) & 7)) * kChunk);
            }
            return;
        }
        issBase = UniformPtr(reinterpret_cast<const char*>(a.w) + static_cast<int64_t>(t.group) * a.wGroupStride);
        if constexpr (kUnits > 1) {
            issUnits = unitsOf(t);
            issUnitShift = static_cast<int64_t>(secondUnit(t) - t.colBase) * (kNMajor ? 1 : a.K);  // (blocked: 32 channels, K x 32 bytes)
        }
#pragma unroll
        for (int q = 0; q < Cfg::kSlotsB; ++q) {
            constexpr int kPerHalf = Cfg::kSlotsB / 2;
            const int half = q / kPerHalf, j = waveN + kWavesN * (q % kPerHalf);  // instruction j of its half of the channels
            if (kNMajor) {
                // Instruction j moves k-rows 4 * j .. + 3 of the stage, 256 channel bytes each (kSwiglu, whose halves lie apart: of its
                // half k-rows 8 * j .. + 7, 128 bytes each); chunks past the last channel are never stored: such lanes re-read the
                // last real chunk.  us, 128-byte pieces of each half in all epilogues -> this: 32 experts of 37 rows, K 1440 x N 2880 (rows
                // that begin inside a line) 42.5 -> 38.8; 128 of 4, 1536 x 4096 141 -> 139; 256 of 4, 2048 x 7168 631 -> 626.
                const int k = kSwiglu ? 8 * j + rowIn : 4 * (waveN + kWavesN * q) + (lane >> 4);
                const int c = kSwiglu ? slot ^ RowMajorSwizzle(k) : (lane & 15) ^ RowMajorWideSwizzle(k);
                const int32_t col = !kSwiglu ? min(t.colBase + 16 * c, a.N - 16)
                                    : half ? min(a.halfN + t.colBase + 16 * c, a.N - 16) : min(t.colBase + 16 * c, a.halfN - 16);
                laneOff[q] = static_cast<uint32_t>(k * a.N + col);
            } else if (kNz) {
                // instruction j moves 32 k-rows (x 32 channel bytes) of channel block j / 4: 1 KB, contiguous in memory and
                // in LDS; lane -> (k-row lane / 2, 16-byte half, swapped with bit 4 of k)
                const int k = (j % 4) * 32 + lane / 2;
                const int32_t col = t.colBase + (kSwiglu ? (half ? a.halfN : 0) + 32 * (j / 4) : 64 * (j / 4) + 32 * half);
                const int32_t block = min(col, a.N - 1) >> 5;
                laneOff[q] = static_cast<uint32_t>(block * a.K * 32 + k * 32 + ((lane ^ (k >> 4)) & 1) * kChunk);
            } else {
                const int r = 8 * j + rowIn;
                laneOff[q] = static_cast<uint32_t>(ChannelOfRow<kOrderLane, kSwiglu>(a, t, half, r) * a.K + (slot ^ ((r >> 1) & 7)) * kChunk);
            }
        }
    };
    // Moves the cursor to the next k-step (or, with two units, the weights' to the other one).
    auto advance = [&]() __attribute__((always_inline)) {
        issAddr = issAddr + issStride == issEnd ? issFirst : issAddr + issStride;
        if constexpr (kUnits > 1) {
            if (issUnit + 1 < issUnits) {
                ++issUnit;
                return;
            }
            issUnit = 0;
        }
        if (__builtin_expect(++issStep == kSteps, 0)) {
            // move to this workgroup's next tile.  Past the last one the issue slots still go out (that keeps the number
            // of outstanding DMAs per stage, hence the vmcnt arithmetic, constant) into ring buffers nobody reads -- but
            // every one of them then re-reads the same first kilobyte of the last tile's weights, which stays in L2,
            // instead of pulling more stages of weights from HBM per workgroup.
            issStep = 0;
            const TileInfo next = tileAt(issNo + 1);
            if (next.valid) {
                issTile = next;
                ++issNo;
                issRotate = rotateOf(issTile);
                setupIssue(issTile);
            } else if (!issDrained) {
                issDrained = true;
                issUnitShift = 0;
                // any mapped, 16-byte aligned kilobyte will do: the start of the last tile's expert's weights
                issBase = UniformPtr(reinterpret_cast<const char*>(a.w) + static_cast<int64_t>(issTile.group) * a.wGroupStride);
#pragma unroll
                for (int q = 0; q < Cfg::kSlotsB; ++q) laneOff[q] = static_cast<uint32_t>(Opaque(tid) & 63) * kChunk;
            }
        }
    };
    // This wave's DMA instruction of slot q of the stage at the cursor.  Activation rows always stay cacheable (the
    // n-tiles of a group re-read them from L2); on small tiles (every weight byte is used exactly once) the weights stream
    // past the caches.  On large tiles the m-tiles of a group share their weight columns through L2 and must not, nor must K-contiguous rows
    // with K off the 128 grid: a k-step of such a row ends inside a line, and the next one asks for that again.  us, past the caches ->
    // this: 256 experts of 20 rows, 2880 x 2 x 1440 511 -> 446, down 312 -> 245; of 25, rank^-0.8 577 -> 476, 353 -> 269.
    auto request = [&](int q) __attribute__((always_inline)) {
        const int kIdx = issStep + issRotate;
        const int kOff = issDrained ? 0 : kTail ? min(kIdx * kStep, a.K - kStep) : (kIdx >= kSteps ? kIdx - kSteps : kIdx) * kStep;
        // weights -- blocked layout: one k is 32 bytes further; row-major: N bytes
        const char* const base = issBase + ((kNz || kNMajor) && forWeights ? static_cast<int64_t>(kOff) * (kNz ? 32 : a.N) : kOff) +
                                 (kUnits > 1 && issUnit != 0 ? issUnitShift : 0);
        const uint32_t dst = issAddr + 1024 * kWavesN * q;
        if constexpr (kSmallTile) {
            if (forWeights) DmaToLdsAddr16<!kTail || kNz || kNMajor>(base, laneOff[q], dst);
            else if (q < Cfg::kSlotsA) DmaToLdsAddr16<false>(base, laneOff[q], dst);
        } else {
            if (q < Cfg::kSlotsA || forWeights) DmaToLdsAddr16<false>(base, laneOff[q], dst);
        }
    };
    using FirstHalf = std::integral_constant<int, 0>;
    using SecondHalf = std::integral_constant<int, 1>;

    // The scales of a tile come by DMA into LDS (4 bytes a lane: the wave rows' waves take 64 channels, or rows, each): loaded in the
    // epilogue they would come behind every stage in flight.  They travel with the tile's first k-step, and the k loop certifies them with
    // the stages it requests itself, where it is as long as the ring.  Where that is two stages deep, the wait of the first k-step is for
    // them, and it shows on SwiGLU tiles of a few: there they are asked for behind the k loop of the tile before, with its draw, and settled
    // with it.  us, loaded in the epilogue / with the first k-step / this: gate/up, 64 groups of 500 rows, K x 2 x 1024: K 128 40.6 / 42.9 / 41.1,
    // 256 44.8 / 45.9 / 45.6, 384 49.9 / 50.4 / 50.1, 768 63.2 / 63.9 / 63.6, 1024 87.4 / 77.2 / 76.7 (what is left of the loss is the wait for
    // the stores of the tile before); 8 groups of 4000, K 4096 x 2 x 2048 421 / 417 / 414.  16-bit results
    // gain nothing by it: 29 groups of 1212 rows, 1024 x 4096 185 / 184 / 191; 8 of 4000, 2048 x 4096 228 / 220 / 222.
    constexpr bool kScalesAhead = Cfg::kScaleSets == 2;
    const bool scalesByDma = kScalesAhead || kSteps >= Cfg::kStagesB;
    const bool rowScalesByDma = scalesByDma && reinterpret_cast<uintptr_t>(a.rowScale) % 4 == 0;
    const bool channelScalesByDma = kEpi != Epilogue::kInt32 && scalesByDma && a.scaleDtype == 0 && reinterpret_cast<uintptr_t>(a.scale) % 4 == 0;
    // those of the n-th tile of this workgroup
    auto scalesOf = [&](int32_t n) __attribute__((always_inline)) -> float* { return kScalesAhead ? ldsScales + (n & 1) * kScaleSet : ldsScales; };
    auto requestScales = [&](const TileInfo& t, int32_t n) __attribute__((always_inline)) {
        const int lane = Opaque(tid) & 63;
        float* const channelScales = scalesOf(n);
        float* const rowScales = channelScales + kUnits * kTileN;
        if (forWeights) {
            if (channelScalesByDma) {
#pragma unroll
                for (int u = 0; u < kUnits; ++u) {
                    if (u > 0 && unitsOf(t) == 1) break;
                    const int c = 64 * waveN + lane, base = u ? secondUnit(t) : t.colBase;  // of the unit; the unit's
                    const int32_t col = kSwiglu ? (waveN >= 2 ? min(a.halfN + base + c - kTileN / 2, a.N - 1) : min(base + c, a.halfN - 1))
                                                : min(base + c, a.N - 1);
                    DmaToLdsAddr4(static_cast<const char*>(a.scale) + static_cast<int64_t>(t.group) * a.N * 4, static_cast<uint32_t>(col) * 4u,
                                  LdsAddress(reinterpret_cast<const char*>(channelScales + u * kTileN + 64 * waveN)));
                }
            }
        } else if (a.rowScale != nullptr && rowScalesByDma && 64 * waveN < kRows) {
            DmaToLdsAddr4(reinterpret_cast<const char*>(a.rowScale) + static_cast<int64_t>(t.rowBase) * 4,
                          static_cast<uint32_t>(min(64 * waveN + lane, t.rows - 1)) * 4u,
                          LdsAddress(reinterpret_cast<const char*>(rowScales + 64 * waveN)));
        } else if (a.rowScale != nullptr && !rowScalesByDma && tid - kThreads / 2 < kRows) {
            rowScales[tid - kThreads / 2] = a.rowScale[t.rowBase + min(tid - kThreads / 2, t.rows - 1)];
        }
    };

    if (kScalesAhead) requestScales(cur, 0);
    setupIssue(cur);
#pragma unroll 1
    for (int s = 0; s < (forWeights ? Cfg::kStagesB : Cfg::kStagesA); ++s) {
#pragma unroll
        for (int q = 0; q < Cfg::kSlotsB; ++q) request(q);
        advance();
    }
    // the first stage has landed
    if (forWeights) WaitVmcnt<(Cfg::kStagesB - 1) * Cfg::kSlotsB>();
    else WaitVmcnt<(Cfg::kStagesA - 1) * Cfg::kSlotsA>();
    __syncthreads();

    uint32_t ringA = ldsBase, ringB = ldsBase + Cfg::kFirstB;  // buffers that the compute side reads
    // Lane part of the fragment addresses.  Rows sixteen apart swizzle alike.
    const int l16 = Opaque(tid) & 15, quad = (Opaque(tid) >> 4) & 3;
    const uint32_t rowChunk = l16 * 128 + ((quad ^ ((l16 >> 1) & 7)) << 4);
    const uint32_t laneA = rowChunk + waveM * 16 * 128;  // slice 1 of a k-step is 64 bytes on, or back: buffers and rows begin on 128
    // Weights of the wave's column.  K-contiguous: as the rows (the second block is sixteen rows on).  Otherwise: the first block,
    // the others being chunks beside it (slice 1 is 64 k-rows on and swizzles alike; with the transposing loads this lane supplies
    // half a chunk of k-row k).
    constexpr bool kWide = kNMajor && !kSwiglu;  // a k-row of a stage is 256 channels side by side, not 128 of each half
    uint32_t laneB;
    {
        const int k = 16 * quad + (l16 >> 1);
        if (kWide) laneB = k * 256 + (((4 * waveN) ^ RowMajorWideSwizzle(k)) << 4) + 8 * (l16 & 1);
        else if (kNMajor) laneB = k * 128 + (((2 * waveN) ^ RowMajorSwizzle(k)) << 4) + 8 * (l16 & 1);
        else if (kNz) laneB = waveN * 4096 + k * 32 + 16 * (quad & 1) + 8 * (l16 & 1);
        else laneB = rowChunk + 32 * waveN * 128;
    }
    // the wave's four blocks of weights, slice ks
    auto readB = [&](v4i (&b)[4], uint32_t buffer, int ks) __attribute__((always_inline)) {
#pragma unroll
        for (int n = 0; n < 4; ++n) {
            const int half = kWide ? 0 : (n >> 1) * Cfg::kHalfBytesB, j = kWide ? n : n & 1;
            if constexpr (kNz || kNMajor) {
                constexpr int kEightK = kNz ? 8 * 32 : kWide ? 8 * 256 : 8 * 128;  // the swizzles of k and k + 8 are the same
                b[n] = LdsReadTransposed((buffer + laneB) ^ (16 * j), half + ks * 8 * kEightK, kEightK);
            } else {
                b[n] = LdsRead16((buffer + laneB) ^ (64 * ks), half + j * 16 * 128);
            }
        }
    };

    v4i acc[kUnits][Blocks::kAll][4];
    while (true) {
        const TileInfo following = tileAt(curNo + 1);
        if (!kScalesAhead && kEpi != Epilogue::kInt32) requestScales(cur, curNo);
#pragma unroll
        for (int u = 0; u < kUnits; ++u) {
#pragma unroll
            for (int m = 0; m < Blocks::kAll; ++m) {
#pragma unroll
                for (int n = 0; n < 4; ++n) acc[u][m][n] = v4i{0, 0, 0, 0};
            }
        }
        const int32_t units = unitsOf(cur);

        // The k loop of a wave with kMy row blocks (the loop is instantiated once per count, so that its body stays
        // straight-line code: blocks that hold no real row are never multiplied -- on the memory-bound shapes the matrix
        // pipe's power is what is worth saving).
        auto runTile = [&](auto myTag) __attribute__((always_inline)) {
            constexpr int kMy = decltype(myTag)::value;
            constexpr int kMy0 = (kMy + 1) / 2, kMy1 = kMy / 2;
            v4i af[2][kMy0 > 0 ? kMy0 : 1];  // [slice][block]
            v4i bf[2][4];                    // [slice][block]
            auto readA = [&](v4i (&f)[kMy0 > 0 ? kMy0 : 1], uint32_t buffer, auto halfTag, int ks) __attribute__((always_inline)) {
                constexpr int kHalf = decltype(halfTag)::value;
#pragma unroll
                for (int i = 0; i < (kHalf ? kMy1 : kMy0); ++i) f[i] = LdsRead16((buffer + laneA) ^ (64 * ks), (4 * i + 2 * kHalf) * 16 * 128);
            };
            // The product of one half of the rows with one slice, and between its instructions, if asked for, the requests of the even
            // or the odd slots.  From one row block to the next the weight blocks are walked back and forth: consecutive instructions
            // share an operand, which costs the matrix unit 2 to 3 % less power.
            auto multiply = [&](auto unitTag, auto halfTag, int ks, bool requests, int odd = 0) __attribute__((always_inline)) {
                constexpr int kHalf = decltype(halfTag)::value;
                constexpr int kCount = kHalf ? kMy1 : kMy0, kOnes = kCount > 0 ? kCount : 1;
#pragma unroll
                for (int i = 0; i < kOnes; ++i) {
                    if constexpr (kCount > 0) {
#pragma unroll
                        for (int step = 0; step < 4; ++step) {
                            const int n = i & 1 ? 3 - step : step;
                            v4i& c = acc[decltype(unitTag)::value][kHalf * Blocks::kFirst + i][n];
                            c = __builtin_amdgcn_mfma_i32_16x16x64_i8(af[ks][i], bf[ks][n], c, 0, 0, 0);
                        }
                    }
                    if (requests) {
                        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                        for (int r = 4 * i / kOnes; r < 4 * (i + 1) / kOnes; ++r) request(2 * r + odd);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
            };
            // last step of kTail: the weights of the k that the step before has covered count zero (a lane's fragments hold
            // k 64 * ks + 16 * quad .. + 15 of the stage)
            auto maskB = [&](int ks, bool last) __attribute__((always_inline)) {
                if (kTail && last) {
                    if (64 * ks + 16 * ((Opaque(tid) >> 4) & 3) < kSteps * kStep - a.K) {
#pragma unroll
                        for (int n = 0; n < 4; ++n) bf[ks][n] = v4i{0, 0, 0, 0};
                    }
                }
            };
            auto kStepOf = [&](auto unit, bool last, bool lastUnit) __attribute__((always_inline)) {
                const uint32_t nextA = !lastUnit ? ringA : ringA + Cfg::kStageBytesA == ldsBase + Cfg::kFirstB ? ldsBase : ringA + Cfg::kStageBytesA;
                // a stage of activation rows is read once per unit, and refilled with the last
                const bool refills = forWeights || lastUnit;
                const uint32_t nextB = ringB + Cfg::kStageBytesB == ldsBase + Cfg::kFirstB + Cfg::kStagesB * Cfg::kStageBytesB
                                           ? ldsBase + Cfg::kFirstB : ringB + Cfg::kStageBytesB;
                if (kMy > 0) readB(bf[1], ringB, 1);
                readA(af[1], ringA, FirstHalf{}, 1);
                __builtin_amdgcn_sched_barrier(0);
                maskB(0, last);
                multiply(unit, FirstHalf{}, 0, false);
                __builtin_amdgcn_sched_barrier(0);
                readA(af[0], ringA, SecondHalf{}, 0);
                __builtin_amdgcn_sched_barrier(0);
                maskB(1, last);
                multiply(unit, FirstHalf{}, 1, false);
                // This wave's reads of weights and first half have returned: the products above used them, so the compiler has
                // waited for them already.  But nothing orders those register instructions against the barrier, behind which DMAs
                // that the compiler does not see overwrite what was read.  The kMy1 reads of the second half may be outstanding.
                __builtin_amdgcn_sched_barrier(0);
                WaitLds<kMy1>();
                PhaseBarrier();
                readA(af[1], ringA, SecondHalf{}, 1);
                __builtin_amdgcn_sched_barrier(0);
                multiply(unit, SecondHalf{}, 0, refills, 0);
                __builtin_amdgcn_sched_barrier(0);
                WaitLds();
                if (forWeights) WaitVmcnt<Cfg::kYoungerB>();  // (stores of the tile before, still under way, make it only stricter)
                else if (refills) WaitVmcnt<Cfg::kYoungerA>();
                PhaseBarrier();
                if (kMy > 0 && !(last && lastUnit)) {
                    readB(bf[0], nextB, 0);
                    readA(af[0], nextA, FirstHalf{}, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
                multiply(unit, SecondHalf{}, 1, refills, 1);
                __builtin_amdgcn_sched_barrier(0);
                if (refills) advance();
                ringA = nextA;
                ringB = nextB;
            };
            // the tile's first stage was certified in front of the loop
            if (kMy > 0) readB(bf[0], ringB, 0);
            readA(af[0], ringA, FirstHalf{}, 0);
#pragma unroll 1
            for (int step = 0; step < kSteps; ++step) {
                kStepOf(std::integral_constant<int, 0>{}, step + 1 == kSteps, kUnits == 1 || units == 1);
                if constexpr (kUnits > 1) {
                    if (units > 1) kStepOf(std::integral_constant<int, 1>{}, step + 1 == kSteps, true);
                }
            }
        };
        const int active = (cur.rows + 15) >> 4;  // blocks with real rows
        auto runOne = [&](auto myTag) __attribute__((always_inline)) { runTile(myTag); };
        ForCount<Blocks::kAll>((active + 1 - waveM) >> 1, runOne);

        // Between the k loop and the next tile's a workgroup asks for nothing, its ring being full, so nothing in here waits for memory
        // but once, when it has had the tile's arithmetic to answer:
        //   * the draw for the tile after the next, an atomic that is settled at the memory side, goes out first.  (In front of the k
        //     loop it would hold up the count of every operand part issued after it: loads return in issue order.)
        //   * the arithmetic, on scales that are in LDS.
        //   * every DMA in flight and the draw have landed.  What the ring holds is then certified for the next tile's first steps,
        //     which need no count of their own, so that the stores may still be under way in them.
        //   * the drawn tile's entry of the table: one wave, through the scalar cache, while the others store.
        // us, scales and arguments loaded here, stores drained, draw and entry as two round trips in a row -> this, gate/up / down, two tiles
        // of a workgroup dealt out on both sides: 128 experts of 128 rows, 4096, 1536 336 / 208 -> 334 / 204; 256, 7168, 2048 1431 / 786 ->
        // 1425 / 772; 16 of 2000, 4224, 896 216 / 175 -> 208 / 167; 8 of 155, 4096, 14336 215 / 148 -> 211 / 147.
        v4i next = v4i{0, 0, 0, 0};  // wave 0: the tile that it finds for the ring
        int32_t drawCounter = -1, drawValue = 0, seatLeft = 0;
        if (wave == 0 && pull && following.valid) {
            seatLeft = __builtin_amdgcn_readfirstlane(ldsSeq[kSeqSeatLeft]);
            if (seatLeft <= 0) {
                drawCounter = __builtin_amdgcn_readfirstlane(
                    QueueFirstOpen(static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(ldsSeq[kSeqUsedUp])), xcd, prefer, kOneRun));
                if (drawCounter >= 0 && tid == 0) drawValue = QueueTake(a.queueCounters, drawCounter);
            }
        }
        if (kScalesAhead && following.valid) requestScales(following, curNo + 1);
        const KernelArgs epilogueArgs = ReloadArgs();
        auto beforeStores = [&]() __attribute__((always_inline)) {
            __builtin_amdgcn_sched_barrier(0);
            WaitVmcnt<0>();
            __builtin_amdgcn_sched_barrier(0);
            if (wave == 0 && following.valid) {
                const RunTable runs = ReadRunTable(sched);
                if (!pull) {
                    next = shareTile(epilogueArgs, runs, curNo + kTilesAhead);
                } else if (seatLeft > 0) {
                    const int32_t logical = __builtin_amdgcn_readfirstlane(ldsSeq[kSeqSeatNext]);
                    next = decodeTile(epilogueArgs, runs, prefer, logical);
                    if (tid == 0) {
                        ldsSeq[kSeqSeatNext] = logical + ldsSeq[kSeqSeatStride];
                        ldsSeq[kSeqSeatLeft] = seatLeft - 1;
                    }
                } else if (drawCounter >= 0) {
                    const int32_t v = __builtin_amdgcn_readfirstlane(drawValue);
                    const QueueLists lists{runs.countBig * tilesAcross(epilogueArgs), runs.countSmall * tilesAcross(epilogueArgs),
                                           __builtin_amdgcn_readfirstlane(ldsSeq[kSeqSeated]), __builtin_amdgcn_readfirstlane(ldsSeq[kSeqSeated + 1])};
                    int32_t first, size;
                    QueueShare(lists, drawCounter, &first, &size);
                    int32_t list = drawCounter & 1, logical = first + v;
                    if (v >= size) {
                        if (tid == 0) {
                            const QueueDraw d = QueueResolve(lists, a.queueCounters, xcd, prefer, static_cast<uint32_t>(ldsSeq[kSeqUsedUp]),
                                                             drawCounter, v, kOneRun);
                            ldsSeq[kSeqUsedUp] = static_cast<int32_t>(d.usedUp);
                            list = d.list;
                            logical = d.logical;
                        }
                        list = __builtin_amdgcn_readfirstlane(list);
                        logical = __builtin_amdgcn_readfirstlane(logical);
                    }
                    next = decodeTile(epilogueArgs, runs, list, logical);
                }
            }
        };
        constexpr int kOrder = kOrderOf<kNz, kNMajor>;
        const float* const channelScales = channelScalesByDma ? scalesOf(curNo) : nullptr;
        const float* const ldsRowScale = scalesOf(curNo) + kUnits * kTileN;
        if constexpr (kUnits == 1) {
            TileEpilogueWave<kRows, kEpi, kOrder>(epilogueArgs, cur, acc[0], waveM, waveN, Opaque(tid) & 15, (Opaque(tid) >> 4) & 3, channelScales,
                                                  ldsRowScale, ldsRowMax, beforeStores);
        } else {  // two units' accumulators leave no room for the results of one
            TileEpilogueWave<kRows, kEpi, kOrder, false>(epilogueArgs, cur, acc[0], waveM, waveN, Opaque(tid) & 15, (Opaque(tid) >> 4) & 3, channelScales,
                                                         ldsRowScale, ldsRowMax);
            beforeStores();
            if (units > 1) {
                TileInfo second = cur;
                second.colBase = secondUnit(cur);
                TileEpilogueWave<kRows, kEpi, kOrder, false>(epilogueArgs, second, acc[1], waveM, waveN, Opaque(tid) & 15, (Opaque(tid) >> 4) & 3,
                                                             channelScalesByDma ? channelScales + kTileN : nullptr, ldsRowScale, ldsRowMax);
            }
        }
        if (tid == 0 && following.valid) leaveTile(curNo + (pull ? 2 : kTilesAhead), next);
        ++spanTiles;
        if (!kSwiglu && !following.valid) break;
        WaitLds();
        PhaseBarrier();  // the reads of the scales are done, the row maxima are complete and the drawn tile is in the ring
        if constexpr (kSwiglu) {
            TileEpilogueStoreMax<kRows>(epilogueArgs, cur, kUnits * cur.tileN, units, Opaque(tid), ldsRowMax);
            if (!following.valid) break;
        }
        cur = following;
        ++curNo;
    }
}

// Workgroup span record (include/opapi_profile.h): start, end, tiles computed, and above those, in the upper half of the word,
// the rows of a tile where the scheduling kernel has chosen other ones than planned (else 0).
__device__ __forceinline__ void WriteSpan(const KernelArgs& a, uint64_t start, uint64_t tiles, uint32_t otherRows = 0) {
    if (a.wgSpans != nullptr && threadIdx.x == 0) {
        a.wgSpans[3 * blockIdx.x] = start;
        a.wgSpans[3 * blockIdx.x + 1] = __builtin_amdgcn_s_memrealtime();
        a.wgSpans[3 * blockIdx.x + 2] = tiles | static_cast<uint64_t>(otherRows) << 32;
    }
}

template <int kRows, Epilogue kEpi, bool kNz, bool kNMajor, bool kTail>
__global__ __launch_bounds__(kThreads) void StreamGemmKernel(KernelArgs a, const int32_t* __restrict__ sched) {
    extern __shared__ __attribute__((aligned(128))) char lds[];
    const uint64_t spanStart = a.wgSpans != nullptr ? __builtin_amdgcn_s_memrealtime() : 0;
    uint64_t spanTiles = 0;
    StreamGemmBody<kRows, kEpi, kNz, kNMajor, kBothRuns, kTail>(a, sched, lds, spanTiles);
    WriteSpan(a, spanStart, spanTiles);
}

// Tall tiles (192 and 256 rows) with pulled tiles: the two runs of the m-tile table, each with a stage geometry of its
// own.  A big m-tile of 256 rows needs 256 activation rows per stage and leaves LDS room for two stages; a small one (at
// most 64 rows: the whole K x 256 weight block for a handful of rows) needs 64 and runs as a pure weight stream, for
// which two stages in flight per CU are too few -- with the geometry of the 64-row tiles it has three, the rotated k
// walk and the non-temporal weight loads of the decode shapes.  A workgroup serves the run it prefers (SlotsForSmall) until that run's counters are used up on every XCD, lets its
// ring drain, and serves the other; a launch without small m-tiles costs the workgroups that looked for them one draw.
//
// The scheduling kernel may have cut the groups into m-tiles of at most kLowTileM rows instead; these run in one geometry, in tiles of 256
// or of 512 channels.

template <int kRows, Epilogue kEpi, bool kNz, bool kNMajor, bool kTail>
__global__ __launch_bounds__(kThreads) void MixedGemmKernel(KernelArgs a, const int32_t* __restrict__ sched) {
    extern __shared__ __attribute__((aligned(128))) char lds[];
    const uint64_t spanStart = a.wgSpans != nullptr ? __builtin_amdgcn_s_memrealtime() : 0;
    uint64_t spanTiles = 0;
    if constexpr (kEpi == Epilogue::kSwiglu) {
        if (sched[kHdrWide] != 0) {
            StreamGemmBody<kLowTileM, kEpi, kNz, kNMajor, kBothRuns, kTail, 2>(a, sched, lds, spanTiles);
            WriteSpan(a, spanStart, spanTiles, kLowTileM);
            return;
        }
    }
    if (sched[kHdrTileM] == kLowTileM) {
        StreamGemmBody<kLowTileM, kEpi, kNz, kNMajor, kBothRuns, kTail>(a, sched, lds, spanTiles);
        WriteSpan(a, spanStart, spanTiles, kLowTileM);
        return;
    }
    const int32_t slots = gridDim.x / kXcds, slot = blockIdx.x / kXcds;
    const int32_t forSmall = sched[0] == 0 ? slots : SlotsForSmall<kEpi, kNMajor, true>(sched, slots, a.tilesN);
    if (slot < forSmall) {
        StreamGemmBody<kSmallRows, kEpi, kNz, kNMajor, kSmallRun, kTail>(a, sched, lds, spanTiles);
        if (sched[0] != 0) {
            __syncthreads();  // the other geometry lays LDS out anew
            StreamGemmBody<kRows, kEpi, kNz, kNMajor, kBigRun, kTail>(a, sched, lds, spanTiles, false);
        }
    } else {
        StreamGemmBody<kRows, kEpi, kNz, kNMajor, kBigRun, kTail>(a, sched, lds, spanTiles);
        if (sched[1] != 0) {
            __syncthreads();
            StreamGemmBody<kSmallRows, kEpi, kNz, kNMajor, kSmallRun, kTail>(a, sched, lds, spanTiles, false);
        }
    }
    WriteSpan(a, spanStart, spanTiles, sched[kHdrTileM]);
}

// ---------------------------------------------------------------------------------------------- generic path
// One tile per workgroup (grid = static upper bound of tiles), operands gathered byte by byte through
// registers into a single LDS buffer.  Handles any K and every weight layout.
template <int kRows, Epilogue kEpi>
__global__ __launch_bounds__(kThreads) void GenericGemmKernel(KernelArgs a, const int32_t* __restrict__ sched) {
    using Blocks = RowBlocks<kRows>;
    constexpr int kChunksPerRow = kStep / kChunk;
    constexpr int kBLoads = kTileN * kChunksPerRow / kThreads;
    constexpr bool kSwiglu = kEpi == Epilogue::kSwiglu;
    __shared__ __attribute__((aligned(16))) char ldsA[kRows * kStep];
    __shared__ __attribute__((aligned(16))) char ldsB[kTileN * kStep];
    __shared__ __attribute__((aligned(16))) float ldsRowScale[kRows];
    __shared__ uint32_t ldsRowMax[kRows];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int waveN = (tid >> 6) % kWavesN, waveM = __builtin_amdgcn_readfirstlane((tid >> 6) / kWavesN);
    const int l16 = lane & 15;
    const int quad = lane >> 4;

    // one tile per workgroup: the two runs of the m-tile table as one list, cut into eight contiguous shares
    const int32_t* const queueHdr = sched;
    const int4* const mTileTable = reinterpret_cast<const int4*>(queueHdr + kQueueHeaderInts + kQueueCounterInts);
    const int32_t countBig = queueHdr[0], countSmall = queueHdr[1];
    const int32_t bigTiles = countBig * a.tilesN;
    const int32_t totalTiles = bigTiles + countSmall * a.tilesN;
    const int32_t perXcd = (totalTiles + kXcds - 1) / kXcds;
    const int32_t local = blockIdx.x / kXcds;
    const int32_t logical = static_cast<int32_t>(blockIdx.x % kXcds) * perXcd + local;
    if (local >= perXcd || logical >= totalTiles) return;
    const TileInfo t = logical < bigTiles
        ? DecodeListTile<kSwiglu>(a.tilesN, mTileTable, 0, countBig, queueHdr[4], logical)
        : DecodeListTile<kSwiglu>(a.tilesN, mTileTable, countBig, countSmall, queueHdr[5], logical - bigTiles);
    if (kEpi != Epilogue::kInt32 && a.rowScale != nullptr && tid < kRows) {
        ldsRowScale[tid] = a.rowScale[t.rowBase + (tid < t.rows ? tid : t.rows - 1)];
    }
    if (kSwiglu && tid < kRows) ldsRowMax[tid] = 0;
    const int8_t* const wGroup = a.w + static_cast<int64_t>(t.group) * a.wGroupStride;

    v4i acc[Blocks::kAll][4];
#pragma unroll
    for (int m = 0; m < Blocks::kAll; ++m) {
#pragma unroll
        for (int n = 0; n < 4; ++n) acc[m][n] = v4i{0, 0, 0, 0};
    }

    for (int k0 = 0; k0 < a.K; k0 += kStep) {
        // consecutive threads take consecutive tile rows, and those of the weights consecutive channels (kOrderBlock), so that
        // N-contiguous weights still coalesce
        for (int p = tid; p < kRows * kChunksPerRow; p += kThreads) {
            const int r = p % kRows;
            const int chunk = p / kRows;
            const int8_t* src = a.x + static_cast<int64_t>(t.rowBase + (r < t.rows ? r : t.rows - 1)) * a.K;
            union { v4i v; int8_t b[16]; } u;
            for (int j = 0; j < kChunk; ++j) {
                const int k = k0 + chunk * kChunk + j;
                u.b[j] = k < a.K ? src[k] : static_cast<int8_t>(0);
            }
            *reinterpret_cast<v4i*>(ldsA + LdsOffset(r, chunk)) = u.v;
        }
#pragma unroll
        for (int i = 0; i < kBLoads; ++i) {
            const int p = i * kThreads + tid;
            const int r = p % kTileN;
            const int chunk = p / kTileN;
            const int8_t* src = wGroup + WeightRowBase(a, ChannelOfRow<kOrderBlock, kSwiglu>(a, t, r / 128, r % 128));
            union { v4i v; int8_t b[16]; } u;
            for (int j = 0; j < kChunk; ++j) {
                const int k = k0 + chunk * kChunk + j;
                u.b[j] = k < a.K ? src[static_cast<int64_t>(k) * a.wStrideK] : static_cast<int8_t>(0);
            }
            *reinterpret_cast<v4i*>(ldsB + LdsOffset(r, chunk)) = u.v;
        }
        __syncthreads();
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            const int chunk = 4 * ks + quad;
            v4i b[4];
#pragma unroll
            for (int n = 0; n < 4; ++n) {
                b[n] = *reinterpret_cast<const v4i*>(ldsB + LdsOffset(128 * (n >> 1) + 32 * waveN + 16 * (n & 1) + l16, chunk));
            }
#pragma unroll
            for (int m = 0; m < Blocks::kAll; ++m) {
                const v4i av = *reinterpret_cast<const v4i*>(ldsA + LdsOffset(Blocks::RowOf(m, waveM) + l16, chunk));
#pragma unroll
                for (int n = 0; n < 4; ++n) acc[m][n] = __builtin_amdgcn_mfma_i32_16x16x64_i8(av, b[n], acc[m][n], 0, 0, 0);
            }
        }
        __syncthreads();
    }
    TileEpilogueWave<kRows, kEpi, kOrderBlock>(a, t, acc, waveM, waveN, l16, quad, nullptr, ldsRowScale, ldsRowMax);
    if constexpr (kSwiglu) {
        __syncthreads();
        TileEpilogueStoreMax<kRows>(a, t, t.tileN, 1, tid, ldsRowMax);
    }
}

// ---------------------------------------------------------------------------------------------- launchers
template <int kRows, Epilogue kEpi, bool kNz, bool kNMajor, bool kTail>
hipError_t LaunchStream(const KernelArgs& args, const int32_t* sched, int64_t maxTiles, hipStream_t stream) {
    using Cfg = StreamCfg<kRows, kEpi>;
    auto kernel = StreamGemmKernel<kRows, kEpi, kNz, kNMajor, kTail>;
    static std::atomic<uint64_t> optedIn{0};
    const hipError_t attr = opapi::EnsureDynamicLds(reinterpret_cast<const void*>(kernel), Cfg::kLdsBytes, optedIn);
    if (attr != hipSuccess) return attr;
    // persistent grid: one workgroup per CU (the LDS ring fills the CU), a multiple of the XCD count
    int64_t grid = DeviceCuCount();
    if (grid > maxTiles) grid = maxTiles;
    grid = grid / kXcds * kXcds;
    if (grid < kXcds) grid = kXcds;
    KernelArgs launchArgs = args;
    launchArgs.wgSpans = SpanBufferFor(kEpi, static_cast<int>(grid), kRows);
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(grid)), dim3(kThreads), Cfg::kLdsBytes, stream, launchArgs, sched);
    return hipGetLastError();
}

template <int kRows, Epilogue kEpi, bool kNz, bool kNMajor, bool kTail>
hipError_t LaunchMixed(const KernelArgs& args, const int32_t* sched, int64_t maxTiles, hipStream_t stream) {
    constexpr int kLdsBytes = std::max({StreamCfg<kRows, kEpi>::kLdsBytes, StreamCfg<kSmallRows, kEpi>::kLdsBytes, StreamCfg<kLowTileM, kEpi>::kLdsBytes,
                                        StreamCfg<kLowTileM, kEpi, 2>::kLdsBytes});
    auto kernel = MixedGemmKernel<kRows, kEpi, kNz, kNMajor, kTail>;
    static std::atomic<uint64_t> optedIn{0};
    const hipError_t attr = opapi::EnsureDynamicLds(reinterpret_cast<const void*>(kernel), kLdsBytes, optedIn);
    if (attr != hipSuccess) return attr;
    int64_t grid = DeviceCuCount();
    if (grid > maxTiles) grid = maxTiles;
    grid = grid / kXcds * kXcds;
    if (grid < kXcds) grid = kXcds;
    KernelArgs launchArgs = args;
    launchArgs.wgSpans = SpanBufferFor(kEpi, static_cast<int>(grid), kRows);
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(grid)), dim3(kThreads), kLdsBytes, stream, launchArgs, sched);
    return hipGetLastError();
}

template <Epilogue kEpi, bool kNz, bool kNMajor, bool kTail>
hipError_t LaunchStreamShapeOf(const Plan& plan, const KernelArgs& args, const int32_t* sched, hipStream_t stream) {
    switch (plan.tileM) {
        case 32: return LaunchStream<32, kEpi, kNz, kNMajor, kTail>(args, sched, plan.maxTiles, stream);
        case 64: return LaunchStream<64, kEpi, kNz, kNMajor, kTail>(args, sched, plan.maxTiles, stream);
        case 96: return LaunchStream<96, kEpi, kNz, kNMajor, kTail>(args, sched, plan.maxTiles, stream);
        case 128: return LaunchStream<128, kEpi, kNz, kNMajor, kTail>(args, sched, plan.maxTiles, stream);
        // (160-row tiles were measured in the two-geometry form as well: the down projection of the DeepSeek-V3 prefill
        // shape, whose few overflowing experts leave small second m-tiles, 0.834 against 0.820 ms -- sixteen k-steps
        // per tile do not repay a change of geometry)
        case 160: return LaunchStream<160, kEpi, kNz, kNMajor, kTail>(args, sched, plan.maxTiles, stream);
        // pulled tiles of 192 and 256 rows: the two runs of the table with a stage geometry each
        case 192:
            if (plan.pullTiles) return LaunchMixed<192, kEpi, kNz, kNMajor, kTail>(args, sched, plan.maxTiles, stream);
            return LaunchStream<192, kEpi, kNz, kNMajor, kTail>(args, sched, plan.maxTiles, stream);
        default:
            if (plan.pullTiles) return LaunchMixed<256, kEpi, kNz, kNMajor, kTail>(args, sched, plan.maxTiles, stream);
            return LaunchStream<256, kEpi, kNz, kNMajor, kTail>(args, sched, plan.maxTiles, stream);
    }
}

template <Epilogue kEpi, bool kTail>
hipError_t LaunchStreamShape(const Plan& plan, const KernelArgs& args, const int32_t* sched, hipStream_t stream) {
    if (args.wNz) return LaunchStreamShapeOf<kEpi, true, false, kTail>(plan, args, sched, stream);
    if (args.wStrideN == 1) return LaunchStreamShapeOf<kEpi, false, true, kTail>(plan, args, sched, stream);  // row-major [K, N]
    return LaunchStreamShapeOf<kEpi, false, false, kTail>(plan, args, sched, stream);
}

template <Epilogue kEpi>
hipError_t LaunchGenericShape(const Plan& plan, const KernelArgs& args, const int32_t* sched, hipStream_t stream) {
    const dim3 grid(static_cast<unsigned>(plan.maxTiles));
    if (plan.tileM <= 32) hipLaunchKernelGGL((GenericGemmKernel<32, kEpi>), grid, dim3(kThreads), 0, stream, args, sched);
    else hipLaunchKernelGGL((GenericGemmKernel<128, kEpi>), grid, dim3(kThreads), 0, stream, args, sched);
    return hipGetLastError();
}

}  // namespace
}  // namespace gemm

#pragma clang diagnostic pop
