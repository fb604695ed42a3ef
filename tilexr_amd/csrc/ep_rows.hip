// rows: destination row and assist tuple of every route in ONE launch (gfx950, wave64; memory route, one rank, keys =
// experts, up to kRowsTableRoutes routes).  Replaces the count launch's ticket and
// last-workgroup scan and the separate place launch.
//
// What such a kernel costs on this part, measured: a hand-over between launches or workgroups is a round trip through
// memory, 2 to 4 us while other traffic is about; LDS atomics run at about four lanes a clock (a histogram of 32 768
// ids is 4 to 5 us however the counters are laid out); and a wave that runs alone on its SIMD issues a dependent
// instruction only every 4 ns or so, so 1500 instructions per wave are 6 us whatever they do.  Hence: no hand-over, no
// histogram, few instructions per wave, many waves.
//
// The work is cut by KEY, not by route.  A workgroup of 16 waves takes key k and reads the WHOLE id table, wave w the
// w-th sixteenth of it in flat route order (16-byte loads, eight in flight per lane; L2 hits after an XCD's first
// workgroup).  Without a capacity limit
//   row of a route with id k = (valid ids below k in the whole table) + (earlier routes with id k)
// so pass 1 is two compares and two adds per id, all per lane, and one reduction per wave at its end; the waves'
// counts meet in LDS; pass 2 ranks the lanes that hold id k, slot by slot, and writes their rows and tuples.  Nobody
// waits for another workgroup; every rowOf entry and every tuple is written by exactly one workgroup (routes whose id
// names no expert get their -1 from one more workgroup behind those of the keys).  Workgroup k also knows
// sendCounts[k] (ids up to k) and expertTokenNums[k] without any scan.  Counting is cheap and ranking is not (a wave
// ranks its slots one after the other), so when the keys are few a key gets several workgroups: each counts the whole
// table and ranks one part of every wave's sixteenth.
//
// A token-prefix mask makes the table shorter: every workgroup adds the mask up first, one more round trip.  A capacity
// limit makes "valid ids below k" the sum of the smaller keys' counts, each cut at the limit, so those are counted in an
// LDS histogram after all (RouteRowsLimitPays: tables where that is cheaper than the hand-over), in eight counters a key
// taken by the lanes in turn: adds to one counter go one after the other, and a wave may hold one expert's ids only.  Routes
// beyond a key's limit get row -1 from the workgroup that ranks them.
//
// Same definitions as the count + place pair (reference: src/ep/kernels/tilexr_ep_dispatch_memory_kernel.h:791-818
// rank within expert, :820-1089 count exchange and inclusive cumulative sum, :1142-1168 count outputs, :1240-1258
// assist tuple).
#include <algorithm>

#include <hip/hip_runtime.h>

#include "ep_chunk_rank.hip.h"
#include "ep_kernel_common.hip.h"
#include "ep_launch.h"
#include "ep_numerics.hip.h"

namespace TileXREp {
namespace {

constexpr int kRowsThreads = 1024;
constexpr int kRowsWaves = kRowsThreads / kWave;
constexpr int kRowsSlotRoutes = 4 * kWave;             // routes a wave takes with one 16-byte load per lane
constexpr int kRowsWarmLoads = 4;
constexpr int kRowsBatch = 8;                          // 16-byte loads a lane has in flight
constexpr int kRowsPartSlots = 16;                     // slots a wave ranks at most: four bits per slot in one 64-bit word
constexpr int kRowsMaxParts = 16;
static_assert(kRowsTableRoutes <= kRowsMaxParts * kRowsPartSlots * kRowsWaves * kRowsSlotRoutes, "parts x slots cover the largest table");

struct RouteRowsArgs {
    const int32_t *ids;
    int n;
    int topK;
    int numKeys;
    int slots;                   // slots per wave: wave w owns routes [w, w + 1) * slots * 256 (its sixteenth of the table)
    int parts;                   // workgroups per key
    int partSlots;               // slots of its sixteenth that a wave of workgroup (key, part) ranks: [part, part + 1) * partSlots
    int32_t srcRank;
    int32_t expertIdBias;
    int32_t *rowOf;              // [n] out
    int32_t *assist;             // [rows, 4] out
    int assistAligned;           // the tuples can go out as one 16-byte store each
    int32_t *totalRowsOut;       // device word: rows the dispatch keeps
    int32_t *sendCountsOut;
    int32_t *firstOffsetOut;     // optional
    int64_t *expertTokenNumsOut;
    int tokenNumsType;
    const u32x4 *warmRows;
    int64_t warmVecs;
    const uint8_t *mask;         // kRowsPrefix: [bs]
    int bs;
    int capacity;                // kRowsCapped: rows a key keeps
};

// Which routes have rows: those whose id names a key; of these, those of the first sum(mask) tokens; or the first
// `capacity` of every key.
enum RowsLimit { kRowsAll, kRowsPrefix, kRowsCapped };

// Counters of a workgroup under a capacity limit: eight for each of half the most keys, four for more; a key's own are an odd
// multiple of four words apart, so in LDS banks of their own.
constexpr int kRowsFewKeys = kMaxKeys / 2;
constexpr int kRowsFewKeysStride = kRowsFewKeys + 4;
constexpr int kRowsManyKeysStride = kMaxKeys + 4;
constexpr int kRowsCounters = 8 * kRowsFewKeysStride;
static_assert(4 * kRowsManyKeysStride <= kRowsCounters, "both fit");

typedef int i32x4 __attribute__((ext_vector_type(4)));


// Slots s0 .. s0 + kRowsBatch - 1 of the wave's sixteenth (those below `slots`), all requested before any is looked
// at: slot s, lane l holds routes waveFirst + s * 256 + l * 4 ... + 3.  Elements beyond the table read as 0 (the buffer
// bound sees to that), which names an expert: the kernel corrects its counts by their number, which it knows, instead
// of patching the registers (they come last in route order, so they disturb no rank).
__device__ __forceinline__ void LoadSlots(const __amdgpu_buffer_rsrc_t &table, int waveFirst, int s0, int slots, int lane,
    i32x4 (&id)[kRowsBatch])
{
#pragma unroll
    for (int u = 0; u < kRowsBatch; ++u) {
        if (s0 + u < slots) {
            id[u] = __builtin_bit_cast(i32x4, __builtin_amdgcn_raw_buffer_load_b128(table, (waveFirst + (s0 + u) * kRowsSlotRoutes + lane * 4) * 4, 0, 0));
        }
    }
}

// Tokens that a prefix mask leaves active, four bytes of it in flight per lane.  All lanes of the workgroup call it.
__device__ __forceinline__ int TokensInPrefix(const uint8_t *mask, int tokens, int wave, int lane, int *s_part)
{
    constexpr int kBatch = 4;
    const __amdgpu_buffer_rsrc_t bytes = RowResource(mask, tokens);     // those beyond the end read as zero
    int live = 0;
    for (int first = 0; first < tokens; first += kBatch * kRowsThreads) {
        uint8_t m[kBatch];
#pragma unroll
        for (int u = 0; u < kBatch; ++u) {
            m[u] = __builtin_amdgcn_raw_buffer_load_b8(bytes, first + u * kRowsThreads + wave * kWave + lane, 0, 0);
        }
#pragma unroll
        for (int u = 0; u < kBatch; ++u) {
            live += __popcll(__ballot(m[u] != 0));
        }
    }
    if (lane == 0) {
        s_part[wave] = live;
    }
    __syncthreads();
    return WaveSum(lane < kRowsWaves ? s_part[lane] : 0);
}

// The kernel stays within 64 registers per lane whatever the table's size (ids are streamed, eight loads a lane at a
// time, and only one bit per id is kept), so that two workgroups of 1024 lanes fit a compute unit: the workgroups that
// read token rows start beside the routing ones instead of behind them (58.7 MB read in 15.6 us when they had to wait,
// the routing workgroups alone taking 9).
//
// SPLIT: a key has several workgroups (a.parts > 1).  The common case of one per key is compiled without the tests
// that tell a workgroup's own slots from the rest.
template <bool SPLIT, int LIMIT>
__global__ __launch_bounds__(kRowsThreads, 8) void ep_route_rows_kernel(RouteRowsArgs a)
{
    constexpr bool kPrefix = LIMIT == kRowsPrefix;
    constexpr bool kCapped = LIMIT == kRowsCapped;
    __shared__ int s_less[kRowsWaves];
    __shared__ int s_same[kRowsWaves];
    // routes of the keys below this workgroup's, counted apart by lane
    __shared__ int s_hist[kCapped ? kRowsCounters : 1];
    __shared__ int s_capped[kCapped ? kRowsWaves : 1];

    const int tid = threadIdx.x;
    const int wave = tid / kWave;
    const int lane = tid & (kWave - 1);
    const int keyBlocks = SPLIT ? a.numKeys * a.parts : a.numKeys;
    const int block = blockIdx.x;
    if (block > keyBlocks) {
        // not a routing workgroup.  A routing workgroup takes half a compute unit's wave slots, so only one of these
        // fits beside it: each carries four loads per lane to keep as much in flight as the smaller ones did
        WarmTokenRows<kRowsThreads, kRowsWarmLoads>(a.warmRows, a.warmVecs, block - keyBlocks - 1);
        return;
    }
    const int waveFirst = wave * a.slots * kRowsSlotRoutes;
    int n = a.n;                // routes that may have a row: the first n
    if (kPrefix) {
        n = TokensInPrefix(a.mask, a.bs, wave, lane, s_less) * a.topK;
        __syncthreads();        // s_less is used again below
    }
    const __amdgpu_buffer_rsrc_t table = RowResource(a.ids, (block == keyBlocks ? a.n : n) * 4);

    if (block == keyBlocks) {
        // ids outside [0, E) are skipped, not errors: their routes have no row, nor have those behind the mask's prefix, and
        // this workgroup says so
        const unsigned keys = static_cast<unsigned>(a.numKeys);
#pragma unroll 1
        for (int s0 = 0; s0 < a.slots; s0 += kRowsBatch) {
            i32x4 id[kRowsBatch];
            LoadSlots(table, waveFirst, s0, a.slots, lane, id);
#pragma unroll
            for (int u = 0; u < kRowsBatch; ++u) {
                if (s0 + u < a.slots) {
                    const int route = waveFirst + (s0 + u) * kRowsSlotRoutes + lane * 4;
                    const bool none = (kPrefix && route + 3 >= n) || static_cast<unsigned>(id[u][0]) >= keys || static_cast<unsigned>(id[u][1]) >= keys ||
                        static_cast<unsigned>(id[u][2]) >= keys || static_cast<unsigned>(id[u][3]) >= keys;
                    if (__ballot(none) != 0ull) {
#pragma unroll 1
                        for (int e = 0; e < 4; ++e) {
                            if (route + e < a.n && ((kPrefix && route + e >= n) || static_cast<unsigned>(id[u][e]) >= keys)) {
                                a.rowOf[route + e] = -1;
                            }
                        }
                    }
                }
            }
        }
        return;
    }
    const int key = SPLIT ? block / a.parts : block;
    const int part = SPLIT ? block - key * a.parts : 0;
    const int mineFirst = SPLIT ? part * a.partSlots : 0;           // the slots this workgroup's waves rank: [mineFirst, mineEnd)
    const int mineEnd = SPLIT ? (mineFirst + a.partSlots < a.slots ? mineFirst + a.partSlots : a.slots) : a.slots;

    // under a capacity limit: where a key's counters are, and the first of the lane's
    const bool fewKeys = a.numKeys <= kRowsFewKeys;
    const int stride = fewKeys ? kRowsFewKeysStride : kRowsManyKeysStride;
    const int counters = (lane & (fewKeys ? 7 : 3)) * stride;       // the lane's

    // pass 1, over the wave's whole sixteenth: per lane, ids below the key (unsigned compare: negative ids are above
    // every key) and ids equal to it, those ahead of the workgroup's own slots counted apart; which elements of its own
    // slots are equal is kept, four bits per slot, so that pass 2 needs no id any more
    if (kCapped) {
        for (int j = tid; j < key; j += kRowsThreads) {
#pragma unroll
            for (int c = 0; c < 8; ++c) {
                if (c < 4 || fewKeys) {
                    s_hist[c * stride + j] = 0;
                }
            }
        }
        __syncthreads();
    }
    int less = 0;
    int same = 0;
    int sameAhead = 0;
    uint64_t bits = 0;
#pragma unroll 1
    for (int s0 = 0; s0 < a.slots; s0 += kRowsBatch) {
        i32x4 id[kRowsBatch];
        LoadSlots(table, waveFirst, s0, a.slots, lane, id);
#pragma unroll
        for (int u = 0; u < kRowsBatch; ++u) {
            const int s = s0 + u;
            if (s < a.slots) {
                uint32_t mine = 0u;
                const int inTable = kCapped ? n - (waveFirst + s * kRowsSlotRoutes + lane * 4) : 4;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const bool below = static_cast<unsigned>(id[u][e]) < static_cast<unsigned>(key);
                    if (!kCapped) {
                        less += below ? 1 : 0;
                    } else if (below && e < inTable) {
                        atomicAdd(&s_hist[counters + id[u][e]], 1);
                    }
                    mine |= id[u][e] == key ? 1u << e : 0u;
                }
                const int hits = __popc(mine);
                same += hits;
                if (SPLIT) {
                    sameAhead += s < mineFirst ? hits : 0;
                }
                if (!SPLIT || (s >= mineFirst && s < mineEnd)) {
                    bits |= static_cast<uint64_t>(mine) << ((s - mineFirst) * 4);
                }
            }
        }
    }
    less = kCapped ? 0 : WaveSum(less);
    same = WaveSum(same);
    if (lane == 0) {
        s_less[wave] = less;
        s_same[wave] = same;
    }
    __syncthreads();
    int capped = 0;             // rows of the keys below
    if (kCapped) {
        for (int j = tid; j < key; j += kRowsThreads) {
            int count = 0;
#pragma unroll
            for (int c = 0; c < 8; ++c) {
                count += c < 4 || fewKeys ? s_hist[c * stride + j] : 0;
            }
            capped += min(count, a.capacity);
        }
        capped = WaveSum(capped);
        if (lane == 0) {
            s_capped[wave] = capped;
        }
        __syncthreads();
        capped = WaveSum(lane < kRowsWaves ? s_capped[lane] : 0);
    }
    // elements beyond the table read as id 0: below every other key, equal to key 0
    const int beyond = kRowsWaves * a.slots * kRowsSlotRoutes - n;
    // lane w of every wave takes wave w's two counts; sums over the lanes (few registers: this kernel has 64)
    const int lessOf = lane < kRowsWaves ? s_less[lane] : 0;
    const int sameOf = lane < kRowsWaves ? s_same[lane] : 0;
    const int lessTotal = kCapped ? capped : WaveSum(lessOf) - (key > 0 ? beyond : 0);
    const int total = WaveSum(sameOf) - (key == 0 ? beyond : 0);

    // pass 2: slot by slot, the lanes that hold the key are ranked (flat route order within a slot: lane, then element)
    if (__ballot(bits != 0ull) != 0ull) {
        // routes with this key earlier in route order: in earlier waves' sixteenths, and ahead of these slots in this one
        const int before = WaveSum((lane < wave ? sameOf : 0) + sameAhead);
        const unsigned long long lt = LaneMaskLt();
        int running = lessTotal + before;
        // (token, k) of the lane's first route, then 256 routes on per slot: one division per wave, none per route
        const int first = waveFirst + mineFirst * kRowsSlotRoutes + lane * 4;
        int token = first / a.topK;
        int k = first - token * a.topK;
        const int stepToken = kRowsSlotRoutes / a.topK;
        const int stepK = kRowsSlotRoutes - stepToken * a.topK;
#pragma unroll 1
        for (int s = 0; s < mineEnd - mineFirst; ++s) {
            const uint32_t mine = static_cast<uint32_t>(bits >> (s * 4)) & 15u;
            if (__ballot(mine != 0u) != 0ull) {
                const unsigned long long hit0 = __ballot((mine & 1u) != 0u);
                const unsigned long long hit1 = __ballot((mine & 2u) != 0u);
                const unsigned long long hit2 = __ballot((mine & 4u) != 0u);
                const unsigned long long hit3 = __ballot((mine & 8u) != 0u);
                int row = running + __popcll(hit0 & lt) + __popcll(hit1 & lt) + __popcll(hit2 & lt) + __popcll(hit3 & lt);
                running += __popcll(hit0) + __popcll(hit1) + __popcll(hit2) + __popcll(hit3);
                // a lane seldom holds more than one route of the key in a slot: a loop over its set bits, not its elements
                const int route = first + s * kRowsSlotRoutes;
                for (uint32_t left = mine; left != 0u; left &= left - 1u) {
                    const int e = __builtin_ctz(left);
                    if (route + e >= n) {
                        break;              // beyond the table (key 0 only): nothing real follows in this lane
                    }
                    if (kCapped && row - lessTotal >= a.capacity) {
                        a.rowOf[route + e] = -1;
                        continue;           // so are the key's routes that follow
                    }
                    int kOf = k + e;
                    int tokenOf = token;
                    while (kOf >= a.topK) {
                        kOf -= a.topK;
                        ++tokenOf;
                    }
                    const i32x4 tuple = {a.srcRank, tokenOf, kOf, key + a.expertIdBias};
                    int32_t *out = a.assist + static_cast<int64_t>(row) * 4;
                    if (a.assistAligned != 0) {
                        *reinterpret_cast<i32x4 *>(out) = tuple;
                    } else {
                        out[0] = tuple[0];
                        out[1] = tuple[1];
                        out[2] = tuple[2];
                        out[3] = tuple[3];
                    }
                    a.rowOf[route + e] = row;
                    ++row;
                }
            }
            token += stepToken;
            k += stepK;
            if (k >= a.topK) {
                k -= a.topK;
                ++token;
            }
        }
    }
    if (tid == 0 && part == 0) {
        // ids up to this key = the inclusive cumulative sum the counts output holds
        const int kept = kCapped ? min(total, a.capacity) : total;
        const int incl = lessTotal + kept;
        if (a.sendCountsOut != nullptr) {
            a.sendCountsOut[key] = incl;
        }
        if (a.expertTokenNumsOut != nullptr) {
            a.expertTokenNumsOut[key] = a.tokenNumsType == 0 ? incl : kept;
        }
        if (key == a.numKeys - 1) {
            *a.totalRowsOut = incl;
        }
        if (key == 0 && a.firstOffsetOut != nullptr) {
            *a.firstOffsetOut = 0;
        }
    }
}

// Routing of the MVP route on one rank without a mask in one launch: there is no key, a route's row is the number of live
// routes ahead of it.  No hand-over here either: a workgroup per kCompactRoutes routes counts the live ones ahead of
// its own by reading that part of the table itself and ranks its own, one per lane; a workgroup per expert counts the
// table for expertTokenNums; the rest read token rows ahead.  Bound by latency: three round trips (the table, LDS
// exchanges, the stores), where the count launch it replaces had the histograms written through, a ticket and the last
// workgroup's scan, and left the rows to be looked up through three dependent loads in the scatter.
// Reference: src/ep/kernels/tilexr_ep_dispatch_kernel.cpp:501-571 (compaction), src/ep/kernels/tilexr_ep_combine_helpers.h:49-80
// (routes per expert).
constexpr int kCompactRoutes = kRowsThreads;
constexpr int kCompactBatchRoutes = kRowsBatch * kRowsThreads * 4;      // ids a workgroup has in flight

struct RouteCompactArgs {
    const int32_t *ids;
    int n;
    int topK;
    int numExperts;
    int chunks;
    int32_t srcRank;
    int32_t expertIdBias;
    int32_t *rowOf;              // [n] out
    int32_t *assist;             // [rows, 4] out
    int assistAligned;
    int32_t *totalRowsOut;
    int32_t *recvCountOut;       // optional
    int64_t *expertTokenNumsOut; // optional: without it there are no expert workgroups
    int tokenNumsType;
    int expertBlocks;
    const u32x4 *warmRows;
    int64_t warmVecs;
};

// Ids of ids[0 .. count) in [lo, hi], summed over the workgroup (every lane gets the sum).  The table is asked for in
// batches of 16-byte loads; elements beyond `count` read as 0 and are taken off again where 0 is in the range.
__device__ __forceinline__ int CountIdsInRange(const int32_t *ids, int count, int lo, int hi, int *s_part)
{
    const int tid = threadIdx.x;
    const __amdgpu_buffer_rsrc_t table = RowResource(ids, count * 4);
    const unsigned span = static_cast<unsigned>(hi - lo);
    int hits = 0;
#pragma unroll 1
    for (int first = 0; first < count; first += kCompactBatchRoutes) {
        i32x4 id[kRowsBatch];
#pragma unroll
        for (int u = 0; u < kRowsBatch; ++u) {
            const int at = first + (u * kRowsThreads + tid) * 4;
            id[u] = i32x4{-1, -1, -1, -1};
            if (first + u * kRowsThreads * 4 < count) {
                id[u] = __builtin_bit_cast(i32x4, __builtin_amdgcn_raw_buffer_load_b128(table, at * 4, 0, 0));
            }
        }
#pragma unroll
        for (int u = 0; u < kRowsBatch; ++u) {
            if (first + u * kRowsThreads * 4 < count) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    hits += static_cast<unsigned>(id[u][e] - lo) <= span ? 1 : 0;
                }
            }
        }
    }
    hits = WaveSum(hits);
    if ((tid & (kWave - 1)) == 0) {
        s_part[tid / kWave] = hits;
    }
    __syncthreads();
    const int lane = tid & (kWave - 1);
    const int total = WaveSum(lane < kRowsWaves ? s_part[lane] : 0);
    const int step = kRowsThreads * 4;
    return total - (lo <= 0 ? (count + step - 1) / step * step - count : 0);
}

__global__ __launch_bounds__(kRowsThreads, 8) void ep_route_compact_kernel(RouteCompactArgs a)
{
    __shared__ int s_part[kRowsWaves];
    __shared__ int s_live[kRowsWaves];

    const int tid = threadIdx.x;
    const int wave = tid / kWave;
    const int lane = tid & (kWave - 1);
    const int block = blockIdx.x;
    if (block >= a.chunks + a.expertBlocks) {
        WarmTokenRows<kRowsThreads, kRowsWarmLoads>(a.warmRows, a.warmVecs, block - a.chunks - a.expertBlocks);
        return;
    }
    if (block >= a.chunks) {
        const int expert = block - a.chunks;
        // type 0: the inclusive prefix sum over the experts, otherwise the expert's own routes
        const int count = CountIdsInRange(a.ids, a.n, a.tokenNumsType == 0 ? 0 : expert, expert, s_part);
        if (tid == 0) {
            a.expertTokenNumsOut[expert] = count;
        }
        return;
    }
    const int first = block * kCompactRoutes;
    const int route = first + tid;
    const int id = route < a.n ? a.ids[route] : -1;         // in flight while the routes ahead are counted
    const int ahead = CountIdsInRange(a.ids, first, 0, a.numExperts - 1, s_part);
    const bool live = static_cast<unsigned>(id) < static_cast<unsigned>(a.numExperts);     // ids outside [0, E) are skipped, not errors
    const unsigned long long hit = __ballot(live);
    if (lane == 0) {
        s_live[wave] = __popcll(hit);
    }
    __syncthreads();
    const int ofWave = lane < kRowsWaves ? s_live[lane] : 0;
    const int row = ahead + WaveSum(lane < wave ? ofWave : 0) + __popcll(hit & LaneMaskLt());
    if (route < a.n) {
        a.rowOf[route] = live ? row : -1;
    }
    if (live) {
        const int token = route / a.topK;
        const i32x4 tuple = {a.srcRank, token, route - token * a.topK, id + a.expertIdBias};
        int32_t *out = a.assist + static_cast<int64_t>(row) * 4;
        if (a.assistAligned != 0) {
            *reinterpret_cast<i32x4 *>(out) = tuple;
        } else {
            out[0] = tuple[0];
            out[1] = tuple[1];
            out[2] = tuple[2];
            out[3] = tuple[3];
        }
    }
    if (block == a.chunks - 1) {
        const int total = ahead + WaveSum(ofWave);
        if (tid == 0) {
            *a.totalRowsOut = total;
            if (a.recvCountOut != nullptr) {
                *a.recvCountOut = total;
            }
        }
    }
}

} // namespace

bool RouteRowsFits(const int32_t *ids, int64_t routes, int64_t numKeys, int maskMode, int64_t capacity)
{
    return routes > 0 && routes <= kRowsTableRoutes && numKeys > 0 && numKeys <= kMaxKeys && Aligned16(ids) &&
        (maskMode == kMaskNone || (maskMode == kMaskTokenPrefix && capacity <= 0));
}

// Where the one-launch routing is the faster choice.  Every key's workgroups read and count the whole table, so the
// launch grows with routes x experts where the count launch does not.  Measured on dispatch + combine layers over
// 8192 .. 262 144 routes x 8 .. 2048 experts against count (+ place), both kernels forced in turn on the same buffers:
//   up to 16 384 routes              2-6 us faster throughout (level at 2048 experts without a place launch to save)
//   with workgroups that read token rows ahead in the same launch (14 KiB rows, bf16)
//     32 768 routes                  2-4 us faster up to 256 experts against count + place (rowsAhead: readiness flags
//                                    or the metadata event want the rows resolved before the scatter), level against a
//                                    count launch alone; 4-14 us slower from 1024 experts on
//     49 152 routes and more         level at best, 5-28 us slower from 512 experts on
//   without them (quantised payloads, 4 KiB rows)
//     32 768 routes                  1-4 us faster up to 512 experts
//     65 536 routes                  1-4 us faster up to 64 experts, level up to 256, slower beyond
//     131 072 routes and more        slower from 64 experts on (3-14 us at 128-256 experts, 200 us at 262 144 x 1024)
bool RouteRowsPays(int64_t routes, int64_t numKeys, bool rowsAhead, bool readsRowsAhead)
{
    if (routes <= 16384) {
        return rowsAhead || numKeys <= 1024;
    }
    if (readsRowsAhead) {
        return rowsAhead && routes <= 32768 && numKeys <= 256;
    }
    return routes <= 32768 ? numKeys <= 512 : (routes <= 65536 && numKeys <= 64);
}

// ... and of a call whose routes are limited, where the other would be.  Token-prefix masks, count and one launch: 400 x 2048 x
// top-8 of 64 20.0 -> 16.3 us, 1024 x 2048 of 256 24.2 -> 20.3, 2048 x 2048 34.6 -> 30.5, 8192 x 2048 x top-4 of 64 65.5 -> 60.0;
// up to kRowsMaskedTokens.  That line is where the first measurements ended, not where the gain does: 9000 x 2048 x top-2 of 64
// 50.7 and 39.9, 16384 x 1024 x top-4 72.7 and 65.4, 32768 x 1024 x top-1 82.7 and 54.6, 60000 x 512 122.6 and 68.9.
// Capacity limits, whose histogram grows with the routes: 518 x 2048 x top-8 of 64 18.4 -> 14.2, with flags (no place launch)
// 22.1 -> 17.2; 1729 x top-5 of 128 24.3 -> 20.8; 16 384 routes of 64 33.1 -> 30.0, of 512 35.0 -> 33.1, block fp8 23.0 and 22.9;
// where every token goes to the same experts (with one counter a key) 8192 x 1024 x top-2 of 512 18.9 -> 16.3 (38.7), 16384 x 512 x
// top-1 20.4 -> 18.3 (39.5), 4096 x 1024 x top-4 of 8 19.6 -> 17.5 (27.9);
// 32 768 routes of 128 55.1 and 54.9, block fp8 29.7 and 31.3, of 512 56.4 and 58.4; 65 536 routes 102.4 and 104.0, 53.2 and 58.0.
bool RouteRowsLimitPays(int64_t routes, int64_t numKeys, int64_t capacity)
{
    return capacity <= 0 || (routes <= 16384 && numKeys <= 512);
}

hipError_t LaunchRouteRows(const RouteRowsLaunch &l)
{
    const int64_t n = l.bs * l.topK;
    if (!RouteRowsFits(l.ids, n, l.numKeys, l.mask != nullptr ? kMaskTokenPrefix : kMaskNone, l.capacity)) {
        return hipErrorInvalidValue;
    }
    RouteRowsArgs a {};
    a.ids = l.ids;
    a.n = static_cast<int>(n);
    a.topK = static_cast<int>(l.topK);
    a.numKeys = static_cast<int>(l.numKeys);
    a.slots = static_cast<int>((n + kRowsWaves * kRowsSlotRoutes - 1) / (kRowsWaves * kRowsSlotRoutes));
    // Workgroups per key: more while the keys alone leave most compute units without a routing workgroup (each one
    // reads and counts the whole table, but ranks only its share of the key's routes, which is the longer part), and
    // as many as it takes to keep a wave's share within kRowsPartSlots slots.
    int parts = 1;
    while (parts < kRowsMaxParts && l.numKeys * parts < 256 && parts * 2 <= a.slots) {
        parts *= 2;
    }
    while ((a.slots + parts - 1) / parts > kRowsPartSlots) {
        parts *= 2;
    }
    a.partSlots = (a.slots + parts - 1) / parts;
    a.parts = (a.slots + a.partSlots - 1) / a.partSlots;
    a.srcRank = l.srcRank;
    a.expertIdBias = l.expertIdBias;
    a.rowOf = l.rowOf;
    a.assist = l.assist;
    a.assistAligned = Aligned16(l.assist) ? 1 : 0;
    a.totalRowsOut = l.totalRowsOut;
    a.sendCountsOut = l.sendCountsOut;
    a.firstOffsetOut = l.firstOffsetOut;
    a.expertTokenNumsOut = l.expertTokenNumsOut;
    a.tokenNumsType = l.tokenNumsType;
    a.mask = l.mask;
    a.bs = static_cast<int>(l.bs);
    a.capacity = static_cast<int>(std::min<int64_t>(l.capacity, n));
    // the keys' workgroups, one for the routes without an expert, then those that read token rows
    unsigned blocks = static_cast<unsigned>(l.numKeys) * static_cast<unsigned>(a.parts) + 1u;
    if (l.warmRows != nullptr && l.warmBytes >= 16 && Aligned16(l.warmRows)) {
        a.warmRows = static_cast<const u32x4 *>(l.warmRows);
        a.warmVecs = l.warmBytes / 16;
        blocks += WarmWorkgroups(a.warmVecs, kRowsThreads, kRowsWarmLoads);
    }
    auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3(blocks), dim3(kRowsThreads), 0, l.stream, a); };
    if (l.capacity > 0) {
        a.parts > 1 ? launch(ep_route_rows_kernel<true, kRowsCapped>) : launch(ep_route_rows_kernel<false, kRowsCapped>);
    } else if (l.mask != nullptr) {
        a.parts > 1 ? launch(ep_route_rows_kernel<true, kRowsPrefix>) : launch(ep_route_rows_kernel<false, kRowsPrefix>);
    } else {
        a.parts > 1 ? launch(ep_route_rows_kernel<true, kRowsAll>) : launch(ep_route_rows_kernel<false, kRowsAll>);
    }
    return hipGetLastError();
}

bool RouteCompactFits(const int32_t *ids, int64_t routes, int64_t numExperts, int maskMode)
{
    return routes > 0 && routes <= kCompactTableRoutes && numExperts > 0 && numExperts <= kMaxKeys && maskMode == kMaskNone && Aligned16(ids);
}

// Against the count launch, both forced in turn on the same buffers, us per dispatch + combine layer: up to 1024 experts no
// combination of 4 .. 131 072 routes, 1024 to 7168 columns, plain and int8 rows took longer (512 experts, 8 routes x 1024
// columns 11.8 -> 10.2; 1024 experts, 8 routes 12.0 -> 11.7, 131 072 routes 239 -> 132).  Beyond, each expert costs a
// workgroup, which few routes do not pay for (8 routes: 1280 experts 12.3 -> 12.5, 2048 experts 12.8 -> 14.8; 1024 routes x
// 2048 experts 15.5 -> 16.5) and 2048 or more do (2048 routes x 2048 experts 21.6 -> 17.7; 131 072 routes 355 -> 150).
bool RouteCompactPays(int64_t routes, int64_t numExperts)
{
    return numExperts <= 1024 || routes >= 2048;
}

hipError_t LaunchRouteCompact(const RouteCompactLaunch &l)
{
    const int64_t n = l.bs * l.topK;
    if (!RouteCompactFits(l.ids, n, l.numExperts, kMaskNone)) {
        return hipErrorInvalidValue;
    }
    RouteCompactArgs a {};
    a.ids = l.ids;
    a.n = static_cast<int>(n);
    a.topK = static_cast<int>(l.topK);
    a.numExperts = static_cast<int>(l.numExperts);
    a.chunks = static_cast<int>((n + kCompactRoutes - 1) / kCompactRoutes);
    a.srcRank = l.srcRank;
    a.expertIdBias = l.expertIdBias;
    a.rowOf = l.rowOf;
    a.assist = l.assist;
    a.assistAligned = Aligned16(l.assist) ? 1 : 0;
    a.totalRowsOut = l.totalRowsOut;
    a.recvCountOut = l.recvCountOut;
    a.expertTokenNumsOut = l.expertTokenNumsOut;
    a.tokenNumsType = l.tokenNumsType;
    a.expertBlocks = l.expertTokenNumsOut != nullptr ? static_cast<int>(l.numExperts) : 0;
    unsigned blocks = static_cast<unsigned>(a.chunks + a.expertBlocks);
    if (l.warmRows != nullptr && l.warmBytes >= 16 && Aligned16(l.warmRows)) {
        a.warmRows = static_cast<const u32x4 *>(l.warmRows);
        a.warmVecs = l.warmBytes / 16;
        blocks += WarmWorkgroups(a.warmVecs, kRowsThreads, kRowsWarmLoads);
    }
    hipLaunchKernelGGL(ep_route_compact_kernel, dim3(blocks), dim3(kRowsThreads), 0, l.stream, a);
    return hipGetLastError();
}

} // namespace TileXREp
