// Plan-driven (MoonEP) dispatch / combine kernels for ranks that share one MI355X (gfx950, wave64).
//
// HBM-bound row movement, no MFMA.  A plan names the destination row of every route directly, so there is nothing to
// count: dispatch is one read of each token row and one write per route; combine is one read per route and one write
// per token.  Rows are copied either per token, each row read once and stored once per route, or per route, where the
// workgroups of one token are given block indices that land on one XCD (block b runs on XCD b % 8) so that the token row is
// read from HBM once (LaunchMoonDispatch says which).
// Every kernel is launched once for the whole world: blockIdx.y is the rank whose share the workgroup works on.
//
//   what is computed  reference: src/moonep/dispatch/kernels/tilexr_moonep_dispatch_kernel.cpp:108-147, 268-461
//                                src/moonep/combine/kernels/tilexr_moonep_combine_kernel.cpp:117-177, 285-366, 449-541,
//                                568-606, 648-733
#include <atomic>
#include <initializer_list>
#include <type_traits>

#include <hip/hip_runtime.h>

#include "ep_kernel_common.hip.h"
#include "ep_numerics.hip.h"
#include "moonep_stage.h"

namespace TileXRMoon {
namespace {

using TileXREp::u32x4;
using TileXREp::kThreads;
using TileXREp::kWave;

constexpr int kXcds = 8;
constexpr int kComputeUnits = 256;
constexpr int kRowVecs = 2;     // 16-byte vectors per lane per row slice
constexpr int kTokenVecs = 4 * kThreads;    // 16-byte vectors of a row slice of the per-token scatter

constexpr int64_t kDefaultCachedRowBytes = int64_t{256} << 20;   // with this setting the library goes by rows and token rows
std::atomic<int64_t> gCachedRowBytes {kDefaultCachedRowBytes};  // TileXRMoonEpSetCachedRowBytes
// Workgroups per compute unit that the copying launches are held to.  Per route: eight keep more stores in flight than this
// memory system digests (4096 x 7168 x top-8, four stages, us at eight, seven, six, five, four, three, two: 420, 415, 401, 397,
// 410, 439, 512; 5800 x 4096, the forward two 170.3, 170.2, 170.1, 169.0, 169.2, 176.7, 200.5).
constexpr int kScatterCapWorkgroups = 5;
// Chunks of 256 rows per rank up to which the scatter launch builds a fresh plan.  Each of its workgroups looks at the totals of
// all chunks before its own, which wide rows' copies hide and narrow ones' do not.  Forward stages, top-8, us, launches
// behind the copies and one launch: 528 000 rows x 512 277.5 and 263.3, x 520 328 and 301; 786 000 x 64 221 and 213.5, x 256 305.7 and
// 298.8; 1 048 576 x 64 304 and 300, x 256 397 and 393.5, x 512 510 and 503.5, x 1024 908 and 892; 1 600 000 x 256 608 and 613; 2 097 152 x 256 777 and 793, x
// 512 1024 and 1019, x 1024 1835 and 1826.
constexpr int kFusedPlanChunks = 8192;
constexpr int kFusedNarrowPlanChunks = 4096;
constexpr int64_t kFusedWideRow = 512;      // elements
constexpr int64_t kMostCopyBlocks = 0x7fffffff - (1 << 26);     // a rank's share of a grid, less its other workgroups
constexpr int64_t kWarmRowBytes = int64_t{128} << 20;          // token rows of a world that are read ahead of the per-route scatter
                                                               // (with SetCachedRowBytes at its default there are 104 MiB at most)
constexpr int64_t kKeptRowBytes = int64_t{360} << 20;          // rows of a world up to which the per-token scatter is the faster one,
constexpr int64_t kPerRouteTokenBytes = int64_t{104} << 20;    // and token rows beyond which it is again (LaunchMoonDispatch)

const char *gScatterName = "";
const char *gReduceName = "";

__device__ __forceinline__ bool Tagged(uint64_t word, uint64_t epoch)
{
    return (word >> 32) == epoch;
}

__device__ __forceinline__ uint64_t Tag(uint64_t epoch, uint32_t value)
{
    return (epoch << 32) | value;
}

// Row tag bits.
constexpr uint32_t kRowWritten = 1u;    // a route wrote the row's hidden values
constexpr uint32_t kRowNamed = 2u;      // a route names the row: its weight is written
constexpr uint32_t kRowDirect = 4u;     // saved plan: a duplicate whose primary is a row of the same token, written by
                                        // the source like a fresh duplicate

// reference: dispatch kernel :268-279
struct Route {
    int peer;
    int row;
    bool duplicate;
    bool ok;
};

// Plans keep world * nvS within 31 bits, so a word is taken apart in 32: a 64-bit division is a hundred-odd dependent
// instructions, and where few waves run (prepare, walk, records) those were much of the launch.  With the group's words
// and the sibling record asked for a round trip earlier (WalkGroup, moon_finish_kernel): a layer of 128 tokens x 1024,
// top-8, 32.9 -> 31.8 us, 1024 x 7168 forward and backward 141.6 -> 139.9, 4096 x 7168 393.8 -> 391.9.
__device__ __forceinline__ Route Decode(int32_t encoded, int64_t nvS, int world)
{
    const uint32_t raw = static_cast<uint32_t>(encoded >= 0 ? encoded : ~encoded);
    const uint32_t rows = static_cast<uint32_t>(nvS);
    const uint32_t peer = raw / rows;
    Route r;
    r.ok = peer < static_cast<uint32_t>(world);
    r.peer = r.ok ? static_cast<int>(peer) : 0;
    r.row = static_cast<int>(raw - peer * rows);
    r.duplicate = encoded < 0;
    return r;
}

__device__ __forceinline__ void RecordFailure(const WorldTables &t, int rank, uint64_t epoch, int32_t code)
{
    __hip_atomic_store(&t.fail[rank], Tag(epoch, static_cast<uint32_t>(code)), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// ---------------------------------------------------------------------------------------------------------------
// dispatch: scatter
// ---------------------------------------------------------------------------------------------------------------

// Row of the first non-duplicate route of the token, before route k, that goes to `peer`; -1 when there is none.
// reference: dispatch kernel :281-301
__device__ __forceinline__ int OwnPrimaryRow(const DispatchWorld &a, const int32_t *words, int k, int peer)
{
    for (int j = 0; j < k; ++j) {
        const int32_t e = words[j];
        if (e < 0) {
            continue;
        }
        const Route o = Decode(e, a.nvS, a.world);
        if (o.ok && o.peer == peer) {
            return o.row;
        }
    }
    return -1;
}

// What the route's first workgroup records besides the row: the weight, the row tag and -- while the duplicate plan is
// being built -- which primary a duplicate belongs to and where it stands among that primary's duplicates.  Called by
// the first wave of the workgroup, all 64 lanes; s_dst holds the token's K route words.
//   primary of a duplicate = first earlier non-duplicate route of the token to the same rank (dispatch kernel :281-301)
//   the plan lists a primary's duplicates in ascending row order (dispatch kernel :393-419), so the rank of a
//   duplicate within its group is the number of the token's duplicates to that rank with a smaller row
template <bool FRESH>
__device__ __forceinline__ void RouteRecords(const DispatchWorld &a, int src, int token, int k, const Route &r, uint32_t tagBits,
    const int32_t *s_dst)
{
    const int lane = threadIdx.x;
    const int64_t at = static_cast<int64_t>(r.peer) * a.tables.stride + r.row;
    if (lane == 0) {
        if (a.weightsSk[src] != nullptr) {
            a.weightsNvs[r.peer][r.row] = a.weightsSk[src][static_cast<int64_t>(token) * a.k + k];
        }
        a.tables.rowTag[at] = Tag(a.epoch, tagBits);
    }
    if (!FRESH || !r.duplicate) {
        return;
    }
    Route other {0, 0, false, false};
    if (lane < a.k) {
        other = Decode(s_dst[lane], a.nvS, a.world);
    }
    const bool samePeer = lane < a.k && other.ok && other.peer == r.peer;
    const uint64_t primaries = __ballot(samePeer && !other.duplicate && lane < k);
    const uint64_t siblings = __ballot(samePeer && other.duplicate);
    const uint64_t before = __ballot(samePeer && other.duplicate && other.row < r.row);
    if (primaries == 0) {
        if (lane == 0) {
            RecordFailure(a.tables, src, a.epoch, kDispatchInvalidRoute);
        }
        return;
    }
    const int primaryLane = __ffsll(static_cast<unsigned long long>(primaries)) - 1;
    const int primaryRow = __shfl(other.row, primaryLane);
    if (lane == 0) {
        a.tables.parentTag[at] = Tag(a.epoch, static_cast<uint32_t>(primaryRow) + 1u);
        a.tables.sibling[at] = static_cast<uint32_t>(__popcll(before)) | (static_cast<uint32_t>(__popcll(siblings)) << 16);
    }
}

// Whether the row of this route holds its token's row before any copy is made from a primary, and the tag the row gets.
//   fresh plan   every route: the plan is being built from these very route words, so a duplicate row is by construction
//                a copy of this token's row
//   saved plan   non-duplicates; and a duplicate whose primary, according to the plan (parent records written by the walk
//                kernel), is the row this token's own non-duplicate route to that rank writes -- the copy that would be
//                made of its primary is a copy of this token's row (`direct`, worked out by the agree kernel).  Any other
//                duplicate is left to FinishRows.
template <bool FRESH>
__device__ __forceinline__ bool SourceWrites(const Route &r, uint8_t direct, uint32_t *tagBits)
{
    if (FRESH || !r.duplicate) {
        *tagBits = kRowNamed | kRowWritten;
        return true;
    }
    if (direct != 0) {
        *tagBits = kRowNamed | kRowWritten | kRowDirect;
        return true;
    }
    *tagBits = kRowNamed;
    return false;
}

// Reads 8 KiB of the token rows of source rank blockIdx.y (two 16-byte loads per lane) and drops them, ahead of the
// per-route scatter.  That kernel is the fastest copy only while the token rows are in the memory-side cache: when its
// one reading workgroup in K has to fetch a row from HBM between the writes of the others it runs at little more than
// half its speed.  After this read it finds the rows in that cache whatever their history.
constexpr int kWarmLoads = 2;
__device__ __forceinline__ void WarmRows(const DispatchWorld &a, int rank, int64_t block, int64_t vecs)
{
    const u32x4 *rows = static_cast<const u32x4 *>(a.hiddenSh[rank]);
    const int64_t base = block * (kThreads * kWarmLoads) + threadIdx.x;
    u32x4 v[kWarmLoads];
#pragma unroll
    for (int i = 0; i < kWarmLoads; ++i) {
        const int64_t at = base + static_cast<int64_t>(i) * kThreads;
        v[i] = rows[at < vecs ? at : vecs - 1];
    }
#pragma unroll
    for (int i = 0; i < kWarmLoads; ++i) {
        asm volatile("" ::"v"(v[i]));
    }
}

// Saved plans, one thread per route of source rank blockIdx.y: whether the source may write a duplicate's row itself
// (see SourceWrites).  Done ahead of the scatter so that its workgroups find the answer with the route word, in one
// round trip, instead of looking up the parent record after decoding it.  Ahead of a scatter that only copies (`records`) it
// also writes what a route records -- weight, row tag, the row's origin -- and reports a route that names no rank; `direct`
// then answers for every route, and is 0 too for a non-duplicate whose row the plan lists as a duplicate: FinishRows fills
// that row, in the scatter's own launch.  The workgroups from `routeBlocks` on read the token rows ahead (WarmRows) when
// warmVecs is not zero: this launch waits on a few small loads and leaves the memory system idle, so the read costs a
// saved-plan Dispatch no launch of its own.
__global__ __launch_bounds__(kThreads) void moon_agree_kernel(DispatchWorld a, unsigned routeBlocks, int64_t warmVecs, int records)
{
    if (blockIdx.x >= routeBlocks) {
        WarmRows(a, blockIdx.y, static_cast<int64_t>(blockIdx.x - routeBlocks), warmVecs);
        return;
    }
    const int src = blockIdx.y;
    const int64_t route = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
    if (route >= a.s * a.k) {
        return;
    }
    const int K = static_cast<int>(a.k);
    const int k = static_cast<int>(static_cast<uint32_t>(route) % static_cast<uint32_t>(K));
    const int32_t *words = a.dst[src] + route - k;
    const float weight = records != 0 && a.weightsSk[src] != nullptr ? a.weightsSk[src][route] : 0.0f;
    uint8_t direct = 0;
    const Route r = Decode(words[k], a.nvS, a.world);
    const int64_t at = static_cast<int64_t>(r.peer) * a.tables.stride + r.row;
    const uint64_t p = r.ok ? a.tables.parentTag[at] : 0ull;
    const bool listed = Tagged(p, a.epoch);
    if (r.ok && r.duplicate) {
        direct = listed && static_cast<int>(p & 0xffffffffu) - 1 == OwnPrimaryRow(a, words, k, r.peer) ? 1 : 0;
    }
    const int64_t at0 = static_cast<int64_t>(src) * a.tables.stride + route;
    if (records == 0) {
        a.tables.direct[at0] = direct;
        return;
    }
    a.tables.direct[at0] = r.ok && !r.duplicate && !listed ? 1 : direct;
    if (!r.ok) {
        RecordFailure(a.tables, src, a.epoch, kDispatchInvalidRoute);
        return;
    }
    uint32_t tagBits = 0;
    if (SourceWrites<false>(r, direct, &tagBits)) {
        a.tables.origin[at] = static_cast<uint32_t>(src * a.s * a.k + route);
    }
    if (a.weightsSk[src] != nullptr) {
        a.weightsNvs[r.peer][r.row] = weight;
    }
    a.tables.rowTag[at] = Tag(a.epoch, tagBits);
}

// Fresh plans, one thread per route of source rank blockIdx.y: everything a route records (RouteRecords) and the
// failure of a route that names no rank, ahead of the per-route scatter, whose workgroups then only copy: with the records
// in them they asked for route words, weights and the token's other routes between the copies of everybody else, and a
// scatter on tables that were not cached took 110 us instead of 76 (4096 x 7168 x top-8).  Nothing the plan is built from
// is written by the scatter launch, so extra workgroups of that launch build it (PlanChunk).
// The workgroups from `routeBlocks` on read the token rows ahead, as in moon_agree_kernel.
__global__ __launch_bounds__(kThreads) void moon_records_kernel(DispatchWorld a, unsigned routeBlocks, int64_t warmVecs)
{
    if (blockIdx.x >= routeBlocks) {
        WarmRows(a, blockIdx.y, static_cast<int64_t>(blockIdx.x - routeBlocks), warmVecs);
        return;
    }
    const int src = blockIdx.y;
    const int64_t route = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
    if (route >= a.s * a.k) {
        return;
    }
    const int K = static_cast<int>(a.k);
    const int k = static_cast<int>(static_cast<uint32_t>(route) % static_cast<uint32_t>(K));
    const int32_t *words = a.dst[src] + route - k;
    const float weight = a.weightsSk[src] != nullptr ? a.weightsSk[src][route] : 0.0f;
    const Route r = Decode(words[k], a.nvS, a.world);
    uint8_t *rankInGroup = a.tables.direct + static_cast<int64_t>(src) * a.tables.stride + route;
    if (!r.ok) {
        *rankInGroup = kNoRank;
        RecordFailure(a.tables, src, a.epoch, kDispatchInvalidRoute);
        return;
    }
    const int64_t at = static_cast<int64_t>(r.peer) * a.tables.stride + r.row;
    if (a.weightsSk[src] != nullptr) {
        a.weightsNvs[r.peer][r.row] = weight;
    }
    a.tables.rowTag[at] = Tag(a.epoch, kRowNamed | kRowWritten);
    if (!r.duplicate) {
        *rankInGroup = kNoRank;
        return;
    }
    // the token's other routes to the same rank: the first non-duplicate before this one is the primary, the duplicates
    // with a smaller row stand before this one in the primary's group (RouteRecords, one lane per route there)
    int primaryRow = -1;
    uint32_t siblings = 0;
    uint32_t before = 0;
    for (int j = 0; j < K; ++j) {
        const Route o = Decode(words[j], a.nvS, a.world);
        if (!o.ok || o.peer != r.peer) {
            continue;
        }
        if (!o.duplicate) {
            primaryRow = (primaryRow < 0 && j < k) ? o.row : primaryRow;
        } else {
            siblings += 1u;
            before += o.row < r.row ? 1u : 0u;
        }
    }
    if (primaryRow < 0) {
        *rankInGroup = kNoRank;
        RecordFailure(a.tables, src, a.epoch, kDispatchInvalidRoute);
        return;
    }
    *rankInGroup = static_cast<uint8_t>(before);
    a.tables.parentTag[at] = Tag(a.epoch, static_cast<uint32_t>(primaryRow) + 1u);
    a.tables.sibling[at] = before | (siblings << 16);
    if (before == 0) {
        a.tables.origin[at] = static_cast<uint32_t>(src * a.s * a.k + route);
    }
}

// Any hidden size and alignment: one workgroup per route, 2-byte elements.
template <bool FRESH>
__global__ __launch_bounds__(kThreads) void moon_scatter_generic_kernel(DispatchWorld a)
{
    __shared__ int32_t s_dst[kMaxTopK];
    const int src = blockIdx.y;
    const int K = static_cast<int>(a.k);
    const int token = blockIdx.x / K;
    const int k = blockIdx.x % K;
    const int lane = threadIdx.x;
    const int32_t *words = a.dst[src] + static_cast<int64_t>(token) * K;
    if (FRESH && lane < K) {
        s_dst[lane] = words[lane];
    }
    const Route r = Decode(words[k], a.nvS, a.world);
    if (!r.ok) {
        if (lane == 0) {
            RecordFailure(a.tables, src, a.epoch, kDispatchInvalidRoute);
        }
        return;
    }
    uint32_t tagBits = 0;
    const uint8_t direct = FRESH ? 0 : a.tables.direct[static_cast<int64_t>(src) * a.tables.stride + static_cast<int64_t>(token) * K + k];
    if (SourceWrites<FRESH>(r, direct, &tagBits)) {
        const uint16_t *srcRow = static_cast<const uint16_t *>(a.hiddenSh[src]) + static_cast<int64_t>(token) * a.h;
        uint16_t *dstRow = static_cast<uint16_t *>(a.hiddenNvsh[r.peer]) + static_cast<int64_t>(r.row) * a.h;
        for (int c = lane; c < a.h; c += kThreads) {
            dstRow[c] = srcRow[c];
        }
    }
    if (FRESH) {
        TileXREp::LdsBarrier();
    }
    if (lane < kWave) {
        RouteRecords<FRESH>(a, src, token, k, r, tagBits, s_dst);
    }
}

// ---------------------------------------------------------------------------------------------------------------
// dispatch: duplicate plan of every destination rank from the parent records (fresh plans)
// ---------------------------------------------------------------------------------------------------------------

// The reference scans the destination's rows in ascending order: a group is opened by the first duplicate row of its
// primary, groups take their dupLoffs slices in that order, and each slice lists its duplicates in ascending row order
// (dispatch kernel :330-424).  With the rank-within-group and group size recorded by the sources, both numberings are
// exclusive prefix sums over the rows: group index = number of earlier group-opening rows, slice start = sum of their
// group sizes.  PlanChunk does that within the scatter launch; the kernels here follow a scatter that does nothing else
// (moon_scatter_generic_kernel, plans beyond kFusedPlanChunks).  A workgroup scans one chunk of 2048 rows after adding
// up the chunks before its own -- from the rows themselves while the chunks are few, from the totals a first launch leaves
// otherwise.  The slices are filled by the finish kernel, which visits every row anyway.
constexpr int kBuildRows = kChunkRows;
constexpr int kBuildPer = kBuildRows / kThreads;
constexpr unsigned kSelfTotalChunks = 2;    // up to this many chunks a workgroup sums the earlier ones itself (one after
                                            // the other: measured 30 us for 17 chunks against 5 us for the extra launch)

struct ChunkRows {
    int opens[kBuildPer];
    int sizes[kBuildPer];
    int primaries[kBuildPer];
    int localOpen;
    int localSize;
};

__device__ __forceinline__ ChunkRows LoadChunkRows(const DispatchWorld &a, int rank, int64_t base)
{
    const uint64_t *parent = a.tables.parentTag + static_cast<int64_t>(rank) * a.tables.stride;
    const uint32_t *sibling = a.tables.sibling + static_cast<int64_t>(rank) * a.tables.stride;
    ChunkRows c;
    c.localOpen = 0;
    c.localSize = 0;
#pragma unroll
    for (int i = 0; i < kBuildPer; ++i) {
        const int64_t row = base + static_cast<int64_t>(threadIdx.x) * kBuildPer + i;
        c.opens[i] = 0;
        c.sizes[i] = 0;
        c.primaries[i] = -1;
        if (row < a.nvS) {
            const uint64_t p = parent[row];
            if (Tagged(p, a.epoch)) {
                const uint32_t sib = sibling[row];
                c.primaries[i] = static_cast<int>(p & 0xffffffffu) - 1;
                c.opens[i] = (sib & 0xffffu) == 0 ? 1 : 0;
                c.sizes[i] = c.opens[i] ? static_cast<int>(sib >> 16) : 0;
            }
        }
        c.localOpen += c.opens[i];
        c.localSize += c.sizes[i];
    }
    return c;
}

// Exclusive prefix of (open, size) over the threads of the workgroup, and the workgroup totals.
__device__ __forceinline__ void ScanPair(int localOpen, int localSize, int (*s_part)[kThreads / kWave], int *exclOpen,
    int *exclSize, int *totalOpen, int *totalSize)
{
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = threadIdx.x / kWave;
    const int inclOpen = TileXREp::WaveInclusiveSum(localOpen);
    const int inclSize = TileXREp::WaveInclusiveSum(localSize);
    if (lane == kWave - 1) {
        s_part[0][wave] = inclOpen;
        s_part[1][wave] = inclSize;
    }
    __syncthreads();
    *exclOpen = inclOpen - localOpen;
    *exclSize = inclSize - localSize;
    *totalOpen = 0;
    *totalSize = 0;
#pragma unroll
    for (int w = 0; w < kThreads / kWave; ++w) {
        *exclOpen += w < wave ? s_part[0][w] : 0;
        *exclSize += w < wave ? s_part[1][w] : 0;
        *totalOpen += s_part[0][w];
        *totalSize += s_part[1][w];
    }
}

__global__ __launch_bounds__(kThreads) void moon_dedup_totals_kernel(DispatchWorld a)
{
    __shared__ int s_part[2][kThreads / kWave];
    const int rank = blockIdx.y;
    const ChunkRows c = LoadChunkRows(a, rank, static_cast<int64_t>(blockIdx.x) * kBuildRows);
    int exclOpen, exclSize, totalOpen, totalSize;
    ScanPair(c.localOpen, c.localSize, s_part, &exclOpen, &exclSize, &totalOpen, &totalSize);
    if (threadIdx.x == 0) {
        int32_t *totals = a.tables.chunkTotals + (static_cast<int64_t>(rank) * a.tables.groupStride + blockIdx.x) * 2;
        totals[0] = totalOpen;
        totals[1] = totalSize;
    }
}

// What the thread's rows of the chunks before `chunks` add to their totals.  Both words of a row are asked for whatever
// the first one says: one trip to memory per chunk, not two.
__device__ __forceinline__ void AddEarlierChunks(const DispatchWorld &a, int rank, int chunks, int *open, int *size)
{
    const uint64_t *parent = a.tables.parentTag + static_cast<int64_t>(rank) * a.tables.stride;
    const uint32_t *sibling = a.tables.sibling + static_cast<int64_t>(rank) * a.tables.stride;
    for (int c = 0; c < chunks; ++c) {
        uint64_t p[kBuildPer];
        uint32_t sib[kBuildPer];
#pragma unroll
        for (int i = 0; i < kBuildPer; ++i) {
            const int64_t row = static_cast<int64_t>(c) * kBuildRows + static_cast<int64_t>(threadIdx.x) * kBuildPer + i;
            p[i] = row < a.nvS ? parent[row] : 0ull;            // the epoch is never zero: an untagged word
            sib[i] = row < a.nvS ? sibling[row] : 0u;
        }
#pragma unroll
        for (int i = 0; i < kBuildPer; ++i) {
            const bool opens = Tagged(p[i], a.epoch) && (sib[i] & 0xffffu) == 0;
            *open += opens ? 1 : 0;
            *size += opens ? static_cast<int>(sib[i] >> 16) : 0;
        }
    }
}

// Groups and slice starts of one chunk of destination rank `rank` (see above).
// SELF: the workgroup adds up the chunks before its own from the row records themselves, when the chunks are few; otherwise
// from the totals that a launch of moon_dedup_totals_kernel left.
template <bool SELF>
__device__ __forceinline__ void DedupGroupsOfChunk(const DispatchWorld &a, int rank, int chunk, bool lastChunk,
    int (*s_part)[kThreads / kWave], int *s_base)
{
    const int tid = threadIdx.x;
    // totals of the chunks before this one
    int beforeOpen = 0;
    int beforeSize = 0;
    if (SELF) {
        AddEarlierChunks(a, rank, chunk, &beforeOpen, &beforeSize);
    } else {
        const int32_t *totals = a.tables.chunkTotals + static_cast<int64_t>(rank) * a.tables.groupStride * 2;
        for (int c = tid; c < chunk; c += kThreads) {
            beforeOpen += totals[2 * c];
            beforeSize += totals[2 * c + 1];
        }
    }
    int exclOpen, exclSize, baseOpen, baseSize;
    ScanPair(beforeOpen, beforeSize, s_part, &exclOpen, &exclSize, &baseOpen, &baseSize);
    if (tid == 0) {
        s_base[0] = baseOpen;
        s_base[1] = baseSize;
    }
    __syncthreads();
    const ChunkRows c = LoadChunkRows(a, rank, static_cast<int64_t>(chunk) * kBuildRows);
    int totalOpen, totalSize;
    ScanPair(c.localOpen, c.localSize, s_part, &exclOpen, &exclSize, &totalOpen, &totalSize);
    int group = s_base[0] + exclOpen;
    int start = s_base[1] + exclSize;
    uint64_t *groupStart = a.tables.groupStart + static_cast<int64_t>(rank) * a.tables.stride;
#pragma unroll
    for (int i = 0; i < kBuildPer; ++i) {
        if (c.opens[i]) {
            // a plan in which duplicates of one token name the same row can claim more slots than there are rows
            if (group < a.nvS && static_cast<int64_t>(start) + c.sizes[i] <= a.nvS) {
                int32_t *g = a.dupGroups[rank] + static_cast<int64_t>(group) * 3;
                g[0] = c.primaries[i];
                g[1] = start;
                g[2] = c.sizes[i];
                groupStart[c.primaries[i]] = Tag(a.epoch, static_cast<uint32_t>(start));
            } else {
                RecordFailure(a.tables, rank, a.epoch, kDispatchInvalidRoute);
            }
            group += 1;
            start += c.sizes[i];
        }
    }
    if (lastChunk && tid == 0) {
        a.dupCounts[rank][0] = s_base[0] + totalOpen;
        a.dupCounts[rank][1] = s_base[1] + totalSize;
    }
}

template <bool SELF>
__global__ __launch_bounds__(kThreads) void moon_dedup_groups_kernel(DispatchWorld a)
{
    __shared__ int s_part[2][kThreads / kWave];
    __shared__ int s_base[2];
    DedupGroupsOfChunk<SELF>(a, blockIdx.y, blockIdx.x, blockIdx.x == gridDim.x - 1, s_part, s_base);
}

// ---------------------------------------------------------------------------------------------------------------
// saved duplicate plan -> records the later kernels follow (dispatch: parentTag per row; combine: per-slot tables)
// ---------------------------------------------------------------------------------------------------------------
struct WalkArgs {
    int64_t nvS;
    int rank;
    bool combine;
    const int32_t *dupGroups;
    const int32_t *dupLoffs;
    const int32_t *dupCounts;
    WorldTables t;
    uint64_t epoch;
    const int32_t *dstLocal;     // combine only
    int world;
    int64_t n;
};

// Slot (origin rank * stride + target) a receive row returns to, or -1 (reference: combine kernel :285-298).
__device__ __forceinline__ int64_t SlotOfRow(const WalkArgs &a, int32_t row)
{
    const int32_t encoded = a.dstLocal[row];
    if (encoded < 0) {
        return -1;
    }
    const Route r = Decode(encoded, a.nvS, a.world);
    return r.ok && r.row < a.n ? r.peer * a.t.stride + r.row : -1;
}

constexpr int kWalkBatch = 8;    // entries of a group a thread has in flight

__device__ __forceinline__ void LoadGroupEntries(const WalkArgs &a, int32_t start, int32_t count, int32_t i0, int32_t (&dup)[kWalkBatch])
{
#pragma unroll
    for (int j = 0; j < kWalkBatch; ++j) {
        dup[j] = i0 + j < count ? a.dupLoffs[start + i0 + j] : -1;
    }
}

// One thread per group.  Checks follow the reference (dispatch kernel :428-457, combine kernel :307-345).
__device__ __forceinline__ void WalkGroup(const WalkArgs &a, int64_t g)
{
    // the group's words are asked for with the counts that say whether there is such a group (the tensor holds nvS of them)
    const int32_t *words = a.dupGroups + (g < a.nvS ? g : 0) * 3;
    const int32_t primary = words[0];
    const int32_t start = words[1];
    const int32_t count = words[2];
    const int32_t groupCount = a.dupCounts[0];
    const int32_t duplicateCount = a.dupCounts[1];
    const int32_t invalid = a.combine ? kCombineInvalidRoute : kDispatchInvalidRoute;
    if (groupCount < 0 || groupCount > a.nvS || duplicateCount < 0 || duplicateCount > a.nvS) {
        if (g == 0) {
            RecordFailure(a.t, a.rank, a.epoch, invalid);
        }
        return;
    }
    if (g >= groupCount) {
        return;
    }
    if (primary < 0 || primary >= a.nvS || start < 0 || count <= 0 || static_cast<int64_t>(start) + count > duplicateCount) {
        RecordFailure(a.t, a.rank, a.epoch, invalid);
        return;
    }
    const int64_t base = static_cast<int64_t>(a.rank) * a.t.stride;
    // The group's entries are handled eight at a time with all loads of a batch issued together: a thread that took them
    // one by one would sit out two dependent round trips per duplicate (entry, then the entry's dstLocal word).
    // Nothing is recorded for a group with a bad entry: the kernels that follow these records do not check them again.
    bool bad = false;
    int32_t dup[kWalkBatch];
    for (int32_t i0 = 0; i0 < count; i0 += kWalkBatch) {
        LoadGroupEntries(a, start, count, i0, dup);
#pragma unroll
        for (int j = 0; j < kWalkBatch; ++j) {
            bad = bad || (i0 + j < count && (dup[j] < 0 || dup[j] >= a.nvS || (a.combine && dup[j] == primary)));
        }
    }
    if (bad) {
        RecordFailure(a.t, a.rank, a.epoch, invalid);
        return;
    }
    if (a.combine) {
        // the origin reads these per slot, next to the slot's row, so that one round trip tells it everything
        const int64_t slot = SlotOfRow(a, primary);
        if (slot >= 0) {
            a.t.slotCount[slot] = count;
            a.t.slotGroup[slot] = Tag(a.epoch, static_cast<uint32_t>(start));
        }
    }
    for (int32_t i0 = 0; i0 < count; i0 += kWalkBatch) {
        if (count > kWalkBatch) {
            LoadGroupEntries(a, start, count, i0, dup);     // a group of one batch still has it
        }
        if (a.combine) {
            int64_t slot[kWalkBatch];
#pragma unroll
            for (int j = 0; j < kWalkBatch; ++j) {
                slot[j] = dup[j] >= 0 ? SlotOfRow(a, dup[j]) : -1;
            }
#pragma unroll
            for (int j = 0; j < kWalkBatch; ++j) {
                if (slot[j] >= 0) {
                    a.t.slotDup[slot[j]] = Tag(a.epoch, 1u);
                }
            }
        } else {
#pragma unroll
            for (int j = 0; j < kWalkBatch; ++j) {
                if (dup[j] >= 0) {
                    a.t.parentTag[base + dup[j]] = Tag(a.epoch, static_cast<uint32_t>(primary) + 1u);
                }
            }
        }
    }
}

__global__ __launch_bounds__(kThreads) void moon_group_walk_kernel(DispatchWorld a)
{
    const int rank = blockIdx.y;
    WalkArgs w {a.nvS, rank, false, a.dupGroups[rank], a.dupLoffs[rank], a.dupCounts[rank], a.tables, a.epoch, nullptr, a.world, 0};
    WalkGroup(w, static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x);
}

// ---------------------------------------------------------------------------------------------------------------
// dispatch: rows nobody wrote, device status
// ---------------------------------------------------------------------------------------------------------------

constexpr int kFinishRows = kThreads;   // rows one workgroup looks after, one per thread
constexpr int kFinishRun = 16;          // ... so many neighbours at a time: their tags are a line of memory

// Own failure first, then the first failed peer walking upwards from this rank (dispatch kernel :559-574).
__device__ __forceinline__ void WriteDispatchStatus(const DispatchWorld &a, int rank)
{
    int32_t status = kDispatchOk;
    const uint64_t own = __hip_atomic_load(&a.tables.fail[rank], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (Tagged(own, a.epoch)) {
        status = static_cast<int32_t>(own & 0xffffffffu);
    } else {
        for (int o = 1; o < a.world; ++o) {
            const int peer = (rank + o) % a.world;
            const uint64_t f = __hip_atomic_load(&a.tables.fail[peer], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (Tagged(f, a.epoch)) {
                status = kDispatchRemoteFailureBase + peer;
                break;
            }
        }
    }
    a.status[rank][0] = status;
}

// Rows of `rank` that no route's own copy fills, workgroup `block` of `blocks`.  A wave looks at 64 rows, one per lane: nothing
// (a route writes the row), zeros (no route writes it: the reference clears the whole window first, dispatch kernel :206-230),
// or -- saved plans -- a copy of its primary row (dispatch kernel :426-461); the weight of a row no route names is zero for
// the same reason.  Then the wave writes the rows that need writing.  Such rows lie together, at the end of a rank's rows for
// instance: a workgroup's are 16 runs of neighbours from all over the rank, so that each has about as many to write.  (64
// neighbours to a workgroup, looked at by its first wave, us a pass before and now: four ranks x 1000 x 7168 x top-4 229 and 210, x
// 600 x top-2 all four stages 344 and 303, x 3000 x 4096 x top-8 434 and 422; 60000 x 1000 x top-8 498.6 and 488.8, 20000 167.0 and 165.0,
// 16000 x 2560 x top-6 all four 451.8 and 444.5.)
//
// AHEAD: the workgroup belongs to the scatter launch itself, after a launch that left what every route records.  A row is
// then either a copying workgroup's or this one's (moon_agree_kernel), and a primary row is not read where it is being
// written: its values are those of the token row its origin names.  A launch of its own for this took 4 us a Dispatch, and
// the two that built a fresh plan 10; together, us a pass before and now: forward 4096 x 1024 x top-5 50.3 and 41.9,
// 4096 x 2048 x top-8 76.3 and 68.9, 128 x 4096 x top-4 35 and 31; two ranks x 2048 x 2048 x top-8 137 and 126; all four stages 4096 x
// 7168 x top-8 400 and 382 (1.5 us of it are arguments asked for together, AskedTogether).
// Otherwise the rows are copied where they lie, once every source has scattered, and the duplicates of a fresh plan take
// their places in dupLoffs here.
template <bool VEC, bool AHEAD>
__device__ __forceinline__ void FinishRows(const DispatchWorld &a, int rank, int64_t block, int64_t blocks)
{
    const int tid = threadIdx.x;
    const int64_t base = static_cast<int64_t>(rank) * a.tables.stride;
    const int64_t row = (tid / kFinishRun * blocks + block) * kFinishRun + tid % kFinishRun;
    bool fill = false;
    uint32_t from = 0;          // 0: zeros; else what to copy, plus one
    if (row < a.nvS) {
        const uint64_t tag = a.tables.rowTag[base + row];
        const uint64_t p = a.tables.parentTag[base + row];
        const uint32_t sibling = !AHEAD && a.fresh ? a.tables.sibling[base + row] : 0u;
        const bool tagged = Tagged(tag, a.epoch);
        const bool named = tagged && (tag & kRowNamed) != 0;
        const bool written = tagged && (tag & kRowWritten) != 0;
        const bool direct = tagged && (tag & kRowDirect) != 0;
        const int64_t primary = static_cast<int64_t>(p & 0xffffffffu) - 1;
        if (!a.fresh && Tagged(p, a.epoch) && !direct) {
            // a primary no route wrote is all zeros in the reference too (the window was cleared)
            fill = true;
            const uint64_t ptag = a.tables.rowTag[base + primary];
            const uint32_t source = AHEAD ? a.tables.origin[base + primary] : static_cast<uint32_t>(primary);
            from = Tagged(ptag, a.epoch) && (ptag & kRowWritten) != 0 ? source + 1u : 0u;
        } else if (!written) {
            fill = true;
        }
        if (!named && a.weightsNvs[rank] != nullptr) {
            a.weightsNvs[rank][row] = 0.0f;
        }
        if (!AHEAD && a.fresh && Tagged(p, a.epoch)) {
            // slot of this duplicate in its group's slice (dispatch kernel :393-419)
            const uint64_t gs = a.tables.groupStart[base + primary];
            if (Tagged(gs, a.epoch)) {
                const int64_t at = static_cast<int64_t>(gs & 0xffffffffu) + (sibling & 0xffffu);
                if (at < a.nvS) {
                    a.dupLoffs[rank][at] = static_cast<int32_t>(row);
                } else {
                    RecordFailure(a.tables, rank, a.epoch, kDispatchInvalidRoute);
                }
            }
        }
    }
    const int h = static_cast<int>(a.h);
    const int lane = tid % kWave;
    char *tensor = static_cast<char *>(a.hiddenNvsh[rank]);
#pragma unroll 1
    for (uint64_t left = __ballot(fill); left != 0; left &= left - 1) {
        const int at = __builtin_ctzll(left);
        const uint32_t origin = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(from), at));
        // (rows are counted in 31 bits)
        char *dst = tensor + static_cast<int64_t>(__builtin_amdgcn_readlane(static_cast<int>(row), at)) * h * 2;
        const char *src = tensor;
        if (origin != 0 && AHEAD) {
            const uint32_t n = static_cast<uint32_t>(a.s * a.k);
            const uint32_t rankOf = (origin - 1u) / n;
            src = static_cast<const char *>(a.hiddenSh[rankOf]) +
                static_cast<int64_t>((origin - 1u - rankOf * n) / static_cast<uint32_t>(a.k)) * h * 2;
        } else if (origin != 0) {
            src = tensor + static_cast<int64_t>(origin - 1u) * h * 2;
        }
        if (VEC) {
            const int vecs = h / 8;
            u32x4 *dstRow = reinterpret_cast<u32x4 *>(dst);
            const u32x4 *srcRow = reinterpret_cast<const u32x4 *>(src);
            constexpr int kAtOnce = 4;
#pragma unroll 1
            for (int first = lane; first < vecs; first += kAtOnce * kWave) {
                u32x4 v[kAtOnce];
#pragma unroll
                for (int j = 0; j < kAtOnce; ++j) {
                    const int idx = first + j * kWave;
                    v[j] = origin != 0 && idx < vecs ? srcRow[idx] : u32x4{0u, 0u, 0u, 0u};
                }
#pragma unroll
                for (int j = 0; j < kAtOnce; ++j) {
                    const int idx = first + j * kWave;
                    if (idx < vecs) {
                        __builtin_nontemporal_store(v[j], dstRow + idx);
                    }
                }
            }
        } else {
            uint16_t *dstRow = reinterpret_cast<uint16_t *>(dst);
            const uint16_t *srcRow = reinterpret_cast<const uint16_t *>(src);
            for (int c = lane; c < h; c += kWave) {
                dstRow[c] = origin != 0 ? srcRow[c] : static_cast<uint16_t>(0);
            }
        }
    }
}

// What is left to do once every source has scattered, where no scatter launch does it.  Workgroup 0 of every rank writes
// the rank's device status.
template <bool VEC>
__global__ __launch_bounds__(kThreads) void moon_finish_kernel(DispatchWorld a)
{
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        WriteDispatchStatus(a, blockIdx.y);
    }
    FinishRows<VEC, false>(a, blockIdx.y, blockIdx.x, gridDim.x);
}

// ---------------------------------------------------------------------------------------------------------------
// dispatch: the plan as workgroups of the scatter launch
// ---------------------------------------------------------------------------------------------------------------

constexpr int kPlanRows = kThreads;     // rows of a plan workgroup, one per thread
static_assert(kTableAlign == kPlanRows, "a workgroup has a word, and all its rows are in the tables");
constexpr int kWordsAtOnce = 8;

// A chunk's totals in one word, so that whoever finds the word has both: group-opening rows and the sizes of their groups.
constexpr int kSizeShift = 12;
static_assert(kPlanRows < (1 << kSizeShift) && kPlanRows * kMaxTopK < (1 << (32 - kSizeShift)), "both totals fit a word");

__device__ __forceinline__ uint32_t PackTotals(int open, int size)
{
    return static_cast<uint32_t>(open) | (static_cast<uint32_t>(size) << kSizeShift);
}

// Totals of chunk c, which another workgroup of the launch leaves; the records they are made of were there before the
// launch, so a thread that has waited long enough adds them up and depends on nobody.
__device__ __forceinline__ uint32_t TotalsOfChunk(const DispatchWorld &a, int rank, int c)
{
    const uint64_t *word = a.tables.chunkTag + (static_cast<int64_t>(rank) * a.tables.stride / kPlanRows + c);
#pragma unroll 1
    for (int polls = 0; polls < a.totalsPolls; ++polls) {
        const uint64_t w = __hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (Tagged(w, a.epoch)) {
            return static_cast<uint32_t>(w);
        }
        __builtin_amdgcn_s_sleep(4);
    }
    const int64_t at = static_cast<int64_t>(rank) * a.tables.stride + static_cast<int64_t>(c) * kPlanRows;
    int open = 0;
    int size = 0;
#pragma unroll 1
    for (int i = 0; i < kPlanRows; ++i) {
        const uint32_t sibling = a.tables.sibling[at + i];
        const bool opens = Tagged(a.tables.parentTag[at + i], a.epoch) && (sibling & 0xffffu) == 0;
        open += opens ? 1 : 0;
        size += opens ? static_cast<int>(sibling >> 16) : 0;
    }
    return PackTotals(open, size);
}

// The duplicate plan of one chunk of 256 rows, by a workgroup of the scatter launch: groups are numbered and their slices
// start as in DedupGroupsOfChunk, and a thread whose row opens a group fills the group's slice too, so that nothing is left to
// a launch after the copies.  It needs only what the launch before left, besides the totals of the chunks before its own.
// Those the workgroups hand one another: they stand at the front of their rank's share of the launch, each waits for
// workgroups ahead of it alone, and none waits for ever (TotalsOfChunk).
//
// The workgroup of a rank's last chunk knows the plan's extent, hence whether it is one; the last of those among the ranks
// writes every rank's device status.  (One arrival per rank: atomics on one word complete at three per microsecond.)
//
// Beside the copies a trip to memory takes 3 to 5 us and a launch of narrow rows is over in 10, so there are two of them:
// the rows' records, then the route words of the tokens that open groups (their ranks beside them), which are on their way
// while the other chunks' totals are looked for.  A row per thread: in chunks of 2048 rows, eight per thread, the same steps
// took 8 us more, the loads of few compute units that each touch 64 lines at a time.
__device__ __forceinline__ void PlanChunk(const DispatchWorld &a, int rank, int chunk, int chunks, int (*s_part)[kThreads / kWave])
{
    const int tid = threadIdx.x;
    // rows from nvS up to the stride are never tagged with a running epoch
    const int64_t at = static_cast<int64_t>(rank) * a.tables.stride + static_cast<int64_t>(chunk) * kPlanRows + tid;
    const uint64_t parent = a.tables.parentTag[at];
    const uint32_t sibling = a.tables.sibling[at];
    const uint32_t origin = a.tables.origin[at];
    const bool opens = Tagged(parent, a.epoch) && (sibling & 0xffffu) == 0;
    const int size = opens ? static_cast<int>(sibling >> 16) : 0;
    int exclOpen, exclSize, totalOpen, totalSize;
    ScanPair(opens ? 1 : 0, size, s_part, &exclOpen, &exclSize, &totalOpen, &totalSize);
    if (tid == 0) {
        __hip_atomic_store(a.tables.chunkTag + (static_cast<int64_t>(rank) * a.tables.stride / kPlanRows + chunk),
            Tag(a.epoch, PackTotals(totalOpen, totalSize)), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    const int K = static_cast<int>(a.k);
    const uint32_t n = static_cast<uint32_t>(a.s * a.k);
    const uint32_t firstRow = static_cast<uint32_t>(rank) * static_cast<uint32_t>(a.nvS);
    const uint32_t src = opens ? origin / n : 0u;
    const int64_t route = opens ? static_cast<int64_t>((origin - src * n) / static_cast<uint32_t>(K)) * K : 0;
    const int32_t *words = a.dst[src] + route;
    const uint8_t *ranks = a.tables.direct + static_cast<int64_t>(src) * a.tables.stride + route;
    // rows of the group's members by route, and their ranks within it; other routes have no rank, or another rank's row
    uint32_t row[kWordsAtOnce];
    int place[kWordsAtOnce];
    auto load = [&](int k0) {
#pragma unroll
        for (int j = 0; j < kWordsAtOnce; ++j) {
            const int k = k0 + j < K ? k0 + j : K - 1;
            row[j] = opens ? static_cast<uint32_t>(~words[k]) - firstRow : 0u;
            place[j] = opens && k0 + j < K ? ranks[k] : kNoRank;
        }
    };
    load(0);
    int baseOpen = 0;
    int baseSize = 0;
    if (chunk != 0) {
        int beforeOpen = 0;
        int beforeSize = 0;
#pragma unroll 1
        for (int c = tid; c < chunk; c += kThreads) {
            const uint32_t totals = TotalsOfChunk(a, rank, c);
            beforeOpen += static_cast<int>(totals & ((1u << kSizeShift) - 1u));
            beforeSize += static_cast<int>(totals >> kSizeShift);
        }
        TileXREp::LdsBarrier();
        int dropOpen, dropSize;
        ScanPair(beforeOpen, beforeSize, s_part, &dropOpen, &dropSize, &baseOpen, &baseSize);
    }
    const int64_t group = static_cast<int64_t>(baseOpen) + exclOpen;
    const int64_t start = static_cast<int64_t>(baseSize) + exclSize;
    // a plan in which duplicates of one token name the same row can claim more slots than there are rows
    if (opens && group < a.nvS && start + size <= a.nvS) {
        int32_t *g = a.dupGroups[rank] + group * 3;
        g[0] = static_cast<int32_t>(parent & 0xffffffffu) - 1;
        g[1] = static_cast<int32_t>(start);
        g[2] = size;
        int32_t *slice = a.dupLoffs[rank] + start;
#pragma unroll 1
        for (int k0 = 0; k0 < K; k0 += kWordsAtOnce) {
            if (k0 != 0) {
                load(k0);
            }
#pragma unroll
            for (int j = 0; j < kWordsAtOnce; ++j) {
                if (place[j] < size && row[j] < static_cast<uint32_t>(a.nvS)) {
                    slice[place[j]] = static_cast<int32_t>(row[j]);
                }
            }
        }
    }
    if (chunk == chunks - 1 && tid == 0) {
        a.dupCounts[rank][0] = baseOpen + totalOpen;
        a.dupCounts[rank][1] = baseSize + totalSize;
        if (static_cast<int64_t>(baseSize) + totalSize > a.nvS) {
            RecordFailure(a.tables, rank, a.epoch, kDispatchInvalidRoute);
        }
        TileXREp::WaitOwnStores();
        bool last = true;
        if (a.world > 1) {
            last = __hip_atomic_fetch_add(a.tables.arrived, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1u ==
                static_cast<uint32_t>(a.world);
        }
        if (last) {
            if (a.world > 1) {
                __hip_atomic_store(a.tables.arrived, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            for (int r = 0; r < a.world; ++r) {
                WriteDispatchStatus(a, r);
            }
        }
    }
}

// ---------------------------------------------------------------------------------------------------------------
// dispatch: scatter
// ---------------------------------------------------------------------------------------------------------------

// What a scatter launch does besides its copies.  A rank's first workgroups build the plan of a fresh Dispatch
// (PlanChunk).  The last ones fill the rows nobody copies to (FinishRows); looking for such rows is a trip to memory, which at
// the front of the launch would hold the copies up.  Both are a multiple of eight, so that every rank's copies keep their XCDs.
struct ScatterExtras {
    unsigned planBlocks;
    int planChunks;
    unsigned copyBlocks;
    unsigned finishBlocks;
};

// A workgroup whose copy block, counted from the end of the plan's workgroups and so wrapped round for those, names no token.
// (Grids are within 2^31, so a wrapped block's token is beyond any.)  Copying workgroups come to it by the one test of
// their token that they make in any case: a test of the block number ahead of it, on arguments of its own, cost them a
// dependent scalar load each and the 4096 x 7168 x top-8 scatter 9 us on top of 73.
template <bool FRESH>
__device__ __forceinline__ void DoExtra(const DispatchWorld &a, const ScatterExtras &x, unsigned block)
{
    if constexpr (FRESH) {
        if (blockIdx.x < x.planBlocks) {
            if (static_cast<int>(blockIdx.x) < x.planChunks) {
                __shared__ int s_part[2][kThreads / kWave];
                PlanChunk(a, blockIdx.y, blockIdx.x, x.planChunks, s_part);
            }
            return;
        }
    }
    if (block < x.copyBlocks) {
        return;     // a token that only pads the grid
    }
    if (!FRESH && block == x.copyBlocks && threadIdx.x == 0) {
        WriteDispatchStatus(a, blockIdx.y);     // of a saved plan: nothing can fail any more
    }
    FinishRows<true, true>(a, blockIdx.y, block - x.copyBlocks, x.finishBlocks);
}

// Has the arguments asked for together, ahead of the first branch that needs one of them: a copying workgroup lives for some
// microseconds, and each further wait for a scalar load is a part of that (saved plan, 4096 x 7168 x top-8: 78.2 us with the
// plan's rows, the rank count and the `direct` table asked for behind the branch, 72.2 so).  Addresses go through as integers
// and are pointers again behind it (Global): what a pointer that comes out of an asm points to is not known, and an access
// through it is a flat one, by lanes, that is waited for with everything else.
template <typename... T>
__device__ __forceinline__ void AskedTogether(T &...v)
{
    (void)std::initializer_list<int>{([&v] { asm volatile("" : "+s"(v)); }(), 0)...};
}

template <typename T>
__device__ __forceinline__ T *Global(uintptr_t address)
{
    return (T *)(__attribute__((address_space(1))) T *)address;
}

// A value at an address that is the same for the whole workgroup, of memory that this launch does not write: through the scalar
// unit (the compiler finds the address uniform but sees the stores of DoExtra ahead of the load), or by every lane.
template <bool SCALAR, typename T>
__device__ __forceinline__ T UniformLoad(uintptr_t address, int64_t index)
{
    if (SCALAR) {
        return ((const __attribute__((address_space(4))) T *)address)[index];
    }
    int zero = 0;
    asm volatile("" : "+v"(zero));
    return Global<const T>(address)[index + zero];
}

// Whether the source's own workgroups copy the row of this route: every route's of a fresh plan; what moon_agree_kernel
// found for a saved one.
template <bool FRESH>
__device__ __forceinline__ bool SourceCopies(const Route &r, uint8_t direct)
{
    return r.ok && (FRESH || direct != 0);
}

// One workgroup per (token, route, slice of 512 vectors) of source rank blockIdx.y.  What the routes record was written
// ahead, by moon_records_kernel or moon_agree_kernel.
//
// SCALAR: the route word is taken apart by the scalar unit while the row is on its way, and with several ranks the receive
// tensor's address is there too before the row is (by lanes it is a further trip behind the row's).  Four stages, us, by lanes
// and so: two ranks x 2048 x 7168 x top-8 491 and 482, four x 1024 x 7168 591 and 575, one 3600 x 8192 x top-8 402 and 395, 5000 x
// 8192 x top-5 378 and 374, 5800 x 4096 x top-8 321 and 317; but where one rank's rows end within a slice 4096 x 7168 382 and
// 386, 4000 x 7168 x top-7 334 and 337, 4096 x 6144 341 and 346, 4096 x 5120 280 and 280: those keep the word by lanes.
template <bool FRESH, bool SCALAR>
__global__ __launch_bounds__(kThreads) void moon_scatter_kernel(DispatchWorld a, int colSlices, ScatterExtras extras)
{
    const int src = blockIdx.y;
    uintptr_t wordsAt = reinterpret_cast<uintptr_t>(a.dst[src]);
    uintptr_t rowsAt = reinterpret_cast<uintptr_t>(a.hiddenSh[src]);
    uintptr_t firstOutAt = reinterpret_cast<uintptr_t>(a.hiddenNvsh[0]);
    uintptr_t directsAt = reinterpret_cast<uintptr_t>(a.tables.direct + static_cast<int64_t>(src) * a.tables.stride);
    int64_t rowBytes = a.h * 2;
    int64_t nvS = a.nvS;
    int world = a.world;
    AskedTogether(wordsAt, rowsAt, firstOutAt, rowBytes, nvS, world);
    if (!FRESH) {
        AskedTogether(directsAt);
    }
    const char *rows = Global<const char>(rowsAt);
    char *firstOut = Global<char>(firstOutAt);
    const unsigned block = blockIdx.x - (FRESH ? extras.planBlocks : 0u);
    const unsigned j = block / kXcds;
    const unsigned K = static_cast<unsigned>(a.k);
    const unsigned perToken = K * static_cast<unsigned>(colSlices);
    const int64_t token = static_cast<int64_t>(j / perToken) * kXcds + block % kXcds;
    if (token >= a.s) {
        DoExtra<FRESH>(a, extras, block);
        return;
    }
    const unsigned k = (j % perToken) / static_cast<unsigned>(colSlices);
    const unsigned slice = (j % perToken) % static_cast<unsigned>(colSlices);
    const int lane = threadIdx.x;
    const int vecs = static_cast<int>(rowBytes / 16);
    const int colBase = static_cast<int>(slice) * (kRowVecs * kThreads);
    const int64_t route = token * K + k;
    const int32_t encoded = UniformLoad<SCALAR, int32_t>(wordsAt, route);
    // (a byte, out of the four that a scalar load takes; a rank's share of the table is a multiple of them)
    const uint32_t directWord = FRESH ? 0u : UniformLoad<SCALAR, uint32_t>(directsAt, route / 4);
    const u32x4 *srcRow = reinterpret_cast<const u32x4 *>(rows + token * rowBytes);
    u32x4 v[kRowVecs];
#pragma unroll
    for (int i = 0; i < kRowVecs; ++i) {
        const int idx = colBase + i * kThreads + lane;
        v[i] = idx < vecs ? srcRow[idx] : u32x4{0u, 0u, 0u, 0u};
    }
    const Route r = Decode(encoded, nvS, world);
    if (SourceCopies<FRESH>(r, static_cast<uint8_t>(directWord >> (route % 4 * 8)))) {
        char *out = !SCALAR || world == 1 ? firstOut : static_cast<char *>(a.hiddenNvsh[r.peer]);
        u32x4 *dstRow = reinterpret_cast<u32x4 *>(out + r.row * rowBytes);
#pragma unroll
        for (int i = 0; i < kRowVecs; ++i) {
            const int idx = colBase + i * kThreads + lane;
            if (idx < vecs) {
                __builtin_nontemporal_store(v[i], dstRow + idx);
            }
        }
    }
}

// G lanes per (token, slice of G x V vectors) of source rank blockIdx.y: the slice is loaded once and stored once per route.
// What the routes record was written ahead, as for moon_scatter_kernel.  Lane k of every wave works out the
// row of route k for itself, so nothing is handed round and no wave waits between its loads and its stores.  Workgroup b runs on
// XCD b % 8 and takes tokens t with t % 8 == b % 8, as the reduce of a small world does.
//
// AUX, the stores' cache policy.  Rows of whole 128-byte lines are written through and kept in the memory-side cache for Combine
// (kAuxAgentScopeKept; the per-route kernel's must stream, or they push the token rows that its workgroups share out of the L2s).
// Of other rows nearly every store of a wave begins and ends within a line, which written through are two trips for one line.
// They are ordinary stores (0), which come together in the L2, where a token has four and more of them, and stream below, where
// there is less for Combine to find.  Forward stages, us copied per route, kept and so: 2223 x 2008 x top-6 54.0, 56.8 and 56.1,
// 4000 x 2008 x top-2 48.2, 51.1 and 47.5, 2223 x 5000 x top-6 83.9, 89.6 and 86.4, 4000 x 5000 x top-2 72.0, 76.2 and 69.8, 7000 x
// 1000 x top-6 90.4, 71.6 and 68.6; all four 1501 x 7176 x top-8 205.7, 211.3 and 206.2, 4000 x 7176 x top-3 233.4, 244.7 and 242.3.
// (Ordinary stores for three of them 2223 x 7176 76.6, streaming ones 72.0.)
template <bool FRESH, int G, int V, int AUX>
__global__ __launch_bounds__(kThreads) void moon_scatter_token_kernel(DispatchWorld a, int colSlices, ScatterExtras extras)
{
    constexpr int kTokens = kThreads / G;
    const int src = blockIdx.y;
    uintptr_t wordsAt = reinterpret_cast<uintptr_t>(a.dst[src]);
    uintptr_t rowsAt = reinterpret_cast<uintptr_t>(a.hiddenSh[src]);
    uintptr_t firstOutAt = reinterpret_cast<uintptr_t>(a.hiddenNvsh[0]);
    uintptr_t directsAt = reinterpret_cast<uintptr_t>(a.tables.direct + static_cast<int64_t>(src) * a.tables.stride);
    int64_t rowBytes = a.h * 2;
    int64_t nvS = a.nvS;
    int world = a.world;
    AskedTogether(wordsAt, rowsAt, firstOutAt, rowBytes, nvS, world);
    if (!FRESH) {
        AskedTogether(directsAt);
    }
    const int32_t *words = Global<const int32_t>(wordsAt);
    const char *rows = Global<const char>(rowsAt);
    char *firstOut = Global<char>(firstOutAt);
    const uint8_t *directs = Global<const uint8_t>(directsAt);
    const unsigned block = blockIdx.x - (FRESH ? extras.planBlocks : 0u);
    const unsigned j = block / kXcds;
    const int slice = static_cast<int>(j % static_cast<unsigned>(colSlices));
    const int tg = threadIdx.x / G;
    const int64_t token = (static_cast<int64_t>(j / static_cast<unsigned>(colSlices)) * kTokens + tg) * kXcds + block % kXcds;
    if (token >= a.s) {
        DoExtra<FRESH>(a, extras, block);
        return;
    }
    const int lane = threadIdx.x % G;
    const int waveLane = threadIdx.x % kWave;
    const int K = static_cast<int>(a.k);
    const int vecs = static_cast<int>(rowBytes / 16);
    const int colBase = slice * (G * V);
    int32_t word = 0;
    uint8_t direct = 0;
    if (waveLane < K) {
        const int64_t route = token * K + waveLane;
        word = words[route];
        direct = FRESH ? 0 : directs[route];
    }
    const u32x4 *srcRow = reinterpret_cast<const u32x4 *>(rows + token * rowBytes);
    u32x4 v[V];
#pragma unroll
    for (int i = 0; i < V; ++i) {
        const int idx = colBase + i * G + lane;
        v[i] = idx < vecs ? srcRow[idx] : u32x4{0u, 0u, 0u, 0u};
    }
    const Route r = Decode(word, nvS, world);
    const int row = waveLane < K && SourceCopies<FRESH>(r, direct) ? r.row : -1;
    for (int k = 0; k < K; ++k) {
        const int rowOfK = __builtin_amdgcn_readlane(row, k);
        if (rowOfK < 0) {
            continue;
        }
        const int peer = __builtin_amdgcn_readlane(r.peer, k);
        const char *out = world == 1 ? firstOut : static_cast<const char *>(a.hiddenNvsh[peer]);
        const __amdgpu_buffer_rsrc_t dst = TileXREp::RowResource(out + rowOfK * rowBytes, vecs * 16);
#pragma unroll
        for (int i = 0; i < V; ++i) {
            const int idx = colBase + i * G + lane;
            if (idx < vecs) {
                __builtin_amdgcn_raw_buffer_store_b128(v[i], dst, idx * 16, 0, AUX);
            }
        }
    }
}

// ---------------------------------------------------------------------------------------------------------------
// combine: prepare
// ---------------------------------------------------------------------------------------------------------------

// Thread i of expert rank blockIdx.y walks duplicate group i (marks the slots of its duplicates, leaves the group's extent
// at the slot of its primary) and files receive row i under the slot of the origin it returns to.
// reference: combine kernel :285-298 (decode), :350-366 (validation), :568-606 (which rows travel)
__global__ __launch_bounds__(kThreads) void moon_combine_prepare_kernel(CombineWorld a)
{
    const int rank = blockIdx.y;
    const int64_t row = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
    WalkArgs w {a.nvS, rank, true, a.dupGroups[rank], a.dupLoffs[rank], a.dupCounts[rank], a.tables, a.epoch, a.dstLocal[rank],
        a.world, a.s * a.k};
    const int32_t encoded = row < a.nvS ? a.dstLocal[rank][row] : -1;      // in flight while the group is walked
    WalkGroup(w, row);
    if (encoded == -1) {
        return;
    }
    const Route r = Decode(encoded, a.nvS, a.world);
    if (r.duplicate || !r.ok || r.row >= a.s * a.k) {
        RecordFailure(a.tables, rank, a.epoch, kCombineInvalidRoute);
        return;
    }
    a.tables.slotSrc[r.peer * a.tables.stride + r.row] = Tag(a.epoch, static_cast<uint32_t>(rank * a.nvS + row));
}

// ---------------------------------------------------------------------------------------------------------------
// combine: reduce
// ---------------------------------------------------------------------------------------------------------------

// Device status of combine: own failure, else the first failed peer in rank order (combine kernel :391-411), else 0.
__device__ __forceinline__ void WriteCombineStatus(const CombineWorld &a, int rank)
{
    int32_t value = kCombineOk;
    const uint64_t own = __hip_atomic_load(&a.tables.fail[rank], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (Tagged(own, a.epoch)) {
        value = static_cast<int32_t>(own & 0xffffffffu);
    } else {
        for (int peer = 0; peer < a.world; ++peer) {
            const uint64_t f = __hip_atomic_load(&a.tables.fail[peer], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (Tagged(f, a.epoch)) {
                value = kCombineRemoteFailureBase + peer;
                break;
            }
        }
    }
    a.status[rank][0] = value;
}

// The lane's kRowVecs vectors of a row slice.  Lanes beyond the row's end read its last vector (and store nothing
// later): every lane issues every load, unconditionally.
__device__ __forceinline__ void LoadRowSlice(const void *tensor, int64_t row, int h, int vecs, int colBase, int lane, int lanes,
    u32x4 (&v)[kRowVecs])
{
    const u32x4 *p = reinterpret_cast<const u32x4 *>(static_cast<const char *>(tensor) + row * h * 2);
#pragma unroll
    for (int j = 0; j < kRowVecs; ++j) {
        const int idx = colBase + j * lanes + lane;
        v[j] = __builtin_nontemporal_load(p + (idx < vecs ? idx : vecs - 1));
    }
}

// What the reduce kernels need to know about the K slots of a token, gathered by K lanes at once so that the table
// lookups of all slots overlap (done slot after slot they would be K dependent round trips to memory).
struct TokenSlots {
    uint32_t where[kMaxTopK];   // expert rank * nvS + row of the slot's row; kNoRow when the slot contributes nothing
    int32_t start[kMaxTopK];    // first dupLoffs index of the row's duplicate group
    int32_t count[kMaxTopK];    // duplicates in the group; 0 for a row without duplicates
};
constexpr uint32_t kNoRow = 0xffffffffu;

// A slot contributes nothing when nothing was returned to it or when the row filed under it is a duplicate (a
// duplicate row does not travel: its values are part of its primary's slot, combine kernel :583-590).  Weights come
// back for every receive row, duplicates included (combine kernel :593-600).
__device__ __forceinline__ void LoadSlots(const CombineWorld &a, int rank, int token, bool writeWeights, TokenSlots *s)
{
    const int lane = threadIdx.x;
    const int K = static_cast<int>(a.k);
    if (lane >= K) {
        return;
    }
    const int64_t slot = static_cast<int64_t>(rank) * a.tables.stride + static_cast<int64_t>(token) * K + lane;
    const uint64_t w = a.tables.slotSrc[slot];
    const uint64_t dup = a.tables.slotDup[slot];
    const uint64_t group = a.tables.slotGroup[slot];
    const int32_t groupCount = a.tables.slotCount[slot];
    const bool present = Tagged(w, a.epoch);
    const uint32_t low = static_cast<uint32_t>(w);
    const uint32_t rows = static_cast<uint32_t>(a.nvS);
    if (writeWeights && a.weightsSk[rank] != nullptr) {
        a.weightsSk[rank][static_cast<int64_t>(token) * K + lane] = present ? a.weightsNvs[low / rows][low % rows] : 0.0f;
    }
    const bool travels = present && !Tagged(dup, a.epoch);
    const bool grouped = travels && Tagged(group, a.epoch);
    s->where[lane] = travels ? low : kNoRow;
    s->start[lane] = grouped ? static_cast<int32_t>(group & 0xffffffffu) : 0;
    s->count[lane] = grouped ? groupCount : 0;
}

// What a lane of the reduce kernel knows about one of the rows its token slice sums: bits.  A row without duplicates is
// a group of one (rounding a bf16 value to bf16 changes nothing).
constexpr int kItemOpens = 1;       // the group's sum starts as this row (otherwise the row is added to it)
constexpr int kItemCloses = 2;      // after this row the group's sum is rounded to bf16 and joins the token's sum
constexpr int kItemValid = 4;       // clear: no item (the tail of a batch of loads)

// sub = row (opens: a uniform condition) or sub + row.  -0.0 + x is x for every x, zeros of either sign included.
__device__ __forceinline__ void StartOrAddRow(float (&sub)[kRowVecs][8], const u32x4 (&v)[kRowVecs], bool opens)
{
#pragma unroll
    for (int j = 0; j < kRowVecs; ++j) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            sub[j][2 * e] = __fadd_rn(opens ? -0.0f : sub[j][2 * e], __uint_as_float(v[j][e] << 16));
            sub[j][2 * e + 1] = __fadd_rn(opens ? -0.0f : sub[j][2 * e + 1], __uint_as_float(v[j][e] & 0xffff0000u));
        }
    }
}

__device__ __forceinline__ void AddRounded(float (&acc)[kRowVecs][8], const float (&sub)[kRowVecs][8])
{
#pragma unroll
    for (int j = 0; j < kRowVecs; ++j) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const uint32_t packed = TileXREp::FloatPairToBf16Rne(sub[j][2 * e], sub[j][2 * e + 1]);
            acc[j][2 * e] = __fadd_rn(acc[j][2 * e], __uint_as_float(packed << 16));
            acc[j][2 * e + 1] = __fadd_rn(acc[j][2 * e + 1], __uint_as_float(packed & 0xffff0000u));
        }
    }
}

// Slot sum of one token slice of origin rank blockIdx.y.  Slots are taken in slot order from zero (combine kernel
// :664-699); a slot that holds a primary with duplicates contributes bf16(fp32(primary) + fp32(dup) + ...) in the plan's
// list order (combine kernel :489-530); slots that contribute nothing leave the sum as it is (their receive row stays
// zero in the reference).
//
// One wave per slice.  Every row the slice reads -- primaries and the duplicates of their groups, in the order in which
// they are summed -- becomes an item of one lane (which tensor, which row, what to do with it), so that all look-ups
// (slot tables, then the duplicates' row numbers) are two round trips for the whole token whatever its groups look like,
// and the rows themselves are read four at a time.  Items are dealt to the lanes 64 at a time.
//
// `placed`: units are dealt by XCD (workgroup b runs on XCD b % 8 and takes a slice of a token t with t % 8 == b % 8, the
// XCD on which the scatter kernels run the token's routes), for worlds whose rows can still be in the XCDs' L2s when
// Combine follows Dispatch: rows written on one XCD and read on another travel through memory.  The tokens are padded
// to a multiple of eight.
template <int G>
__global__ __launch_bounds__(G) void moon_reduce_kernel(CombineWorld a, int colSlices, int placed)
{
    static_assert(G == kWave, "the items of a token are spread over the lanes of one wave");
    constexpr int kRowsInFlight = 4;
    __shared__ TokenSlots s_slots;
    const int rank = blockIdx.y;
    const int unit = blockIdx.x;
    int token = unit / colSlices;
    int slice = unit % colSlices;
    if (placed != 0) {
        const int j = unit / kXcds;
        token = (j / colSlices) * kXcds + unit % kXcds;
        slice = j % colSlices;
    }
    const int lane = threadIdx.x;
    if (unit == 0 && lane == 0) {
        WriteCombineStatus(a, rank);
    }
    if (token >= a.s) {
        return;
    }
    const int colBase = slice * (G * kRowVecs);
    const int h = static_cast<int>(a.h);
    const int vecs = h / 8;
    LoadSlots(a, rank, token, colBase == 0, &s_slots);
    TileXREp::LdsBarrier();
    float acc[kRowVecs][8];
#pragma unroll
    for (int j = 0; j < kRowVecs; ++j) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            acc[j][e] = 0.0f;
        }
    }
    const int K = static_cast<int>(a.k);
    const uint32_t nvS = static_cast<uint32_t>(a.nvS);
    // lane k < K: slot k, the tensor and row of its primary, and how many items it makes
    uint32_t where = kNoRow;
    int slotStart = 0;
    int slotCount = 0;
    if (lane < K) {
        where = s_slots.where[lane];
        slotStart = s_slots.start[lane];
        slotCount = s_slots.count[lane];
    }
    const bool travels = where != kNoRow;
    const int slotQ = travels ? static_cast<int>(where / nvS) : 0;
    const int slotRow = travels ? static_cast<int>(where % nvS) : 0;
    const int slotItems = travels ? 1 + slotCount : 0;
    int slotFirst = TileXREp::WaveInclusiveSum(slotItems);     // over the K <= 32 slot lanes, then exclusive
    const int total = __builtin_amdgcn_readlane(slotFirst, kMaxTopK - 1);      // lanes from K on add nothing
    slotFirst -= slotItems;
    float sub[kRowVecs][8];                          // sum of the group that is open (groups may span windows)
#pragma unroll
    for (int j = 0; j < kRowVecs; ++j) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            sub[j][e] = 0.0f;
        }
    }
    // windows of 64 items (a token of a built plan has at most K; a saved plan may list any number of duplicates)
#pragma unroll 1
    for (int base = 0; base < total; base += kWave) {
        const int here = total - base < kWave ? total - base : kWave;
        // lane i < here: item base + i
        int itemQ = 0;
        int itemRow = 0;
        int itemKind = 0;
        const int32_t *listed = nullptr;             // where a duplicate's row number stands in its rank's dupLoffs
#pragma unroll 1
        for (int k = 0; k < K; ++k) {
            const int items = __builtin_amdgcn_readlane(slotItems, k);
            if (items == 0) {
                continue;
            }
            const int q = __builtin_amdgcn_readlane(slotQ, k);
            const int row = __builtin_amdgcn_readlane(slotRow, k);
            const int at = base + lane - __builtin_amdgcn_readlane(slotFirst, k);
            if (at >= 0 && at < items) {
                itemQ = q;
                itemRow = row;
                itemKind = kItemValid | (at == 0 ? kItemOpens : 0) | (at == items - 1 ? kItemCloses : 0);
            }
            if (items > 1) {
                const int32_t *list = a.dupLoffs[q] + __builtin_amdgcn_readlane(slotStart, k);
                if (at >= 1 && at < items) {
                    listed = list + (at - 1);
                }
            }
        }
        if (listed != nullptr) {
            itemRow = *listed;
        }
#pragma unroll 1
        for (int i0 = 0; i0 < here; i0 += kRowsInFlight) {
            u32x4 v[kRowsInFlight][kRowVecs];
            int kind[kRowsInFlight];
#pragma unroll
            for (int u = 0; u < kRowsInFlight; ++u) {
                // a batch that runs past the window reads its last row again and drops it: four loads are issued
                // whatever the count, so the sums below wait for exactly the load they need
                const int i = i0 + u < here ? i0 + u : here - 1;
                kind[u] = i0 + u < here ? __builtin_amdgcn_readlane(itemKind, i) : 0;
                const int q = __builtin_amdgcn_readlane(itemQ, i);
                const int row = __builtin_amdgcn_readlane(itemRow, i);
                LoadRowSlice(a.hiddenNvsh[q], row, h, vecs, colBase, lane, G, v[u]);
            }
#pragma unroll
            for (int u = 0; u < kRowsInFlight; ++u) {
                if ((kind[u] & kItemValid) != 0) {
                    StartOrAddRow(sub, v[u], (kind[u] & kItemOpens) != 0);
                    if ((kind[u] & kItemCloses) != 0) {
                        AddRounded(acc, sub);
                    }
                }
            }
        }
    }
    u32x4 *out = reinterpret_cast<u32x4 *>(static_cast<char *>(a.hiddenSh[rank]) + static_cast<int64_t>(token) * h * 2);
#pragma unroll
    for (int j = 0; j < kRowVecs; ++j) {
        const int idx = colBase + j * G + lane;
        if (idx < vecs) {
            u32x4 o;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                o[e] = TileXREp::FloatPairToBf16Rne(acc[j][2 * e], acc[j][2 * e + 1]);
            }
            __builtin_nontemporal_store(o, out + idx);
        }
    }
}

// Any hidden size and alignment: one workgroup per token, one element per thread step.
__global__ __launch_bounds__(kThreads) void moon_reduce_generic_kernel(CombineWorld a)
{
    __shared__ TokenSlots s_slots;
    const int rank = blockIdx.y;
    const int token = blockIdx.x;
    const int lane = threadIdx.x;
    if (token == 0 && lane == 0) {
        WriteCombineStatus(a, rank);
    }
    LoadSlots(a, rank, token, true, &s_slots);
    __syncthreads();
    const int K = static_cast<int>(a.k);
    const uint32_t nvS = static_cast<uint32_t>(a.nvS);
    for (int c = lane; c < a.h; c += kThreads) {
        float acc = 0.0f;
        for (int k = 0; k < K; ++k) {
            const uint32_t where = s_slots.where[k];
            if (where == kNoRow) {
                continue;
            }
            const int q = static_cast<int>(where / nvS);
            const int64_t row = where % nvS;
            const uint16_t *tensor = static_cast<const uint16_t *>(a.hiddenNvsh[q]);
            float value = __uint_as_float(static_cast<uint32_t>(tensor[row * a.h + c]) << 16);
            const int count = s_slots.count[k];
            if (count != 0) {
                const int start = s_slots.start[k];
                for (int i = 0; i < count; ++i) {
                    const int64_t dup = a.dupLoffs[q][start + i];
                    value = __fadd_rn(value, __uint_as_float(static_cast<uint32_t>(tensor[dup * a.h + c]) << 16));
                }
                value = __uint_as_float(TileXREp::FloatToBf16Rne(value) << 16);
            }
            acc = __fadd_rn(acc, value);
        }
        static_cast<uint16_t *>(a.hiddenSh[rank])[static_cast<int64_t>(token) * a.h + c] =
            static_cast<uint16_t>(TileXREp::FloatToBf16Rne(acc));
    }
}

hipError_t RecordIf(hipEvent_t e, hipStream_t stream)
{
    return e == nullptr ? hipSuccess : hipEventRecord(e, stream);
}

#define MOON_LAUNCH_CHECK()                \
    do {                                   \
        const hipError_t launchErr = hipGetLastError(); \
        if (launchErr != hipSuccess) {     \
            return launchErr;              \
        }                                  \
    } while (0)

} // namespace

// One device status word, written in stream order (a call that was dropped because a peer's call disagreed with it).
__global__ void moon_status_kernel(int32_t *status, int32_t value)
{
    if (threadIdx.x == 0 && blockIdx.x == 0) {
        status[0] = value;
    }
}

hipError_t LaunchMoonStatus(int32_t *status, int32_t value, hipStream_t stream)
{
    hipLaunchKernelGGL(moon_status_kernel, dim3(1), dim3(kWave), 0, stream, status, value);
    return hipGetLastError();
}

int64_t SetCachedRowBytes(int64_t bytes)
{
    return gCachedRowBytes.exchange(bytes < 0 ? 0 : bytes);
}

const char *MoonScatterKernelName()
{
    return gScatterName;
}

const char *MoonReduceKernelName()
{
    return gReduceName;
}

// What follows copies whose launch does nothing else: the duplicate plan of a fresh Dispatch, then the rows and weights no
// route wrote.
hipError_t LaunchPlanAndFinish(const DispatchWorld &w, hipStream_t stream, bool vec)
{
    const unsigned R = static_cast<unsigned>(w.world);
    if (w.fresh) {
        const unsigned chunks = static_cast<unsigned>((w.nvS + kBuildRows - 1) / kBuildRows);
        if (chunks <= kSelfTotalChunks) {
            hipLaunchKernelGGL(moon_dedup_groups_kernel<true>, dim3(chunks, R), dim3(kThreads), 0, stream, w);
        } else {
            hipLaunchKernelGGL(moon_dedup_totals_kernel, dim3(chunks, R), dim3(kThreads), 0, stream, w);
            MOON_LAUNCH_CHECK();
            hipLaunchKernelGGL(moon_dedup_groups_kernel<false>, dim3(chunks, R), dim3(kThreads), 0, stream, w);
        }
        MOON_LAUNCH_CHECK();
    }
    const unsigned groups = static_cast<unsigned>((w.nvS + kFinishRows - 1) / kFinishRows);
    if (vec) {
        hipLaunchKernelGGL(moon_finish_kernel<true>, dim3(groups, R), dim3(kThreads), 0, stream, w);
    } else {
        hipLaunchKernelGGL(moon_finish_kernel<false>, dim3(groups, R), dim3(kThreads), 0, stream, w);
    }
    return hipGetLastError();
}

hipError_t LaunchMoonDispatch(const DispatchWorld &w, hipStream_t stream, const LaunchTiming &timing)
{
    const unsigned R = static_cast<unsigned>(w.world);
    const unsigned rowBlocks = static_cast<unsigned>((w.nvS + kThreads - 1) / kThreads);
    bool vec = w.h % 8 == 0;
    for (int r = 0; r < w.world; ++r) {
        vec = vec && TileXREp::Aligned16(w.hiddenSh[r]) && TileXREp::Aligned16(w.hiddenNvsh[r]);
    }
    const int64_t vecs = w.h / 8;
    const int colSlices = static_cast<int>((vecs + kRowVecs * kThreads - 1) / (kRowVecs * kThreads));
    const int64_t blocks = (w.s + kXcds - 1) / kXcds * kXcds * w.k * colSlices;
    const int tokenSlices = static_cast<int>((vecs + kTokenVecs - 1) / kTokenVecs);
    // Which scatter: one workgroup per (token, route, slice) for wide rows that the memory-side cache cannot keep for Combine
    // but whose token rows can be read ahead, one per token slice everywhere else.  All four stages (fwd: the forward two),
    // top-8, us per route and per token, one rank: 128 x 7168 67 and 66, 1024 x 7168 139.5 and 129.5, 3000 x 7168 309 and 299,
    // 3500 x 7168 348 and 352, 4096 x 7168 398.2 and 405.7, 8192 x 4096 454 and 474, 8192 x 7168 778 and 772; narrow rows 3000
    // x 1024 125 and 95, 4096 x 2048 fwd 89 and 77, 16384 x 2048 fwd 255 and 246; four ranks, 4096 x 7168 2098 and 1785, two
    // ranks, top-6, fwd 386 and 374.
    const int64_t worldRowBytes = static_cast<int64_t>(w.world) * w.s * w.h * 2;
    const int64_t cachedRowBytes = gCachedRowBytes.load();
    const bool wantsPerToken = cachedRowBytes != kDefaultCachedRowBytes ? worldRowBytes > cachedRowBytes :
        vecs <= 4 * kWave || worldRowBytes * w.k <= kKeptRowBytes || worldRowBytes > kPerRouteTokenBytes;
    const int64_t rowVecs = w.s * vecs;
    const bool perToken = vec && wantsPerToken && (w.s + 4 * kXcds) * tokenSlices <= kMostCopyBlocks;
    const bool perRoute = vec && !perToken && blocks <= kMostCopyBlocks;
    const bool recordsAhead = perToken || perRoute;
    // per-route copies of up to half the memory-side cache of token rows: read them once so that the kernel finds them there
    // (one rank's share of 4096 x 7168: 257 -> about 210 us per layer on rows that were not cached, a few us more
    // on rows that were)
    const bool warm = perRoute && worldRowBytes <= kWarmRowBytes;
    const unsigned warmBlocks = warm ? static_cast<unsigned>((rowVecs + kThreads * kWarmLoads - 1) / (kThreads * kWarmLoads)) : 0u;
    const unsigned routeBlocks = static_cast<unsigned>((w.s * w.k + kThreads - 1) / kThreads);
    // What the routes record is written ahead of the scatter; the scatter launch then holds everything else a Dispatch does,
    // two launches for a fresh plan and three for a saved one.  A rank of more than kFusedPlanChunks chunks (narrow rows:
    // kFusedNarrowPlanChunks) keeps launches behind the copies.
    const int planChunks = static_cast<int>((w.nvS + kPlanRows - 1) / kPlanRows);
    const bool allInScatter = recordsAhead && (!w.fresh || planChunks <= (w.h >= kFusedWideRow ? kFusedPlanChunks : kFusedNarrowPlanChunks));
    ScatterExtras extras {};
    extras.planChunks = planChunks;
    extras.planBlocks = w.fresh && allInScatter ? static_cast<unsigned>((planChunks + kXcds - 1) / kXcds * kXcds) : 0u;
    // (a multiple of eight, as the others are: the next rank's share of the launch begins on the XCD that its tokens count from)
    extras.finishBlocks = allInScatter ? static_cast<unsigned>((w.nvS + kFinishRows - 1) / kFinishRows + kXcds - 1) / kXcds * kXcds : 0u;
    if (w.fresh && recordsAhead) {
        hipLaunchKernelGGL(moon_records_kernel, dim3(routeBlocks + warmBlocks, R), dim3(kThreads), 0, stream, w, routeBlocks,
            warm ? rowVecs : int64_t{0});
        MOON_LAUNCH_CHECK();
    } else if (!w.fresh) {
        hipLaunchKernelGGL(moon_group_walk_kernel, dim3(rowBlocks, R), dim3(kThreads), 0, stream, w);
        MOON_LAUNCH_CHECK();
        hipLaunchKernelGGL(moon_agree_kernel, dim3(routeBlocks + warmBlocks, R), dim3(kThreads), 0, stream, w, routeBlocks,
            warm ? rowVecs : int64_t{0}, recordsAhead ? 1 : 0);
        MOON_LAUNCH_CHECK();
    }
    hipError_t err = RecordIf(timing.start, stream);
    if (err != hipSuccess) {
        return err;
    }
    if (perToken) {
        gScatterName = "moon_scatter_token_kernel";
        // Two workgroups to a compute unit where each holds more than 512 vectors and stores them four times or more, four where it
        // does not (fewer have too little in flight), as many as fit where the rows come to a GiB and more.  us at eight, four,
        // three and two: 1024 x 7168 x top-8 132.7, 131.5, 130.1, 130.1; 1000 x 12288 205.8, 200.5, 199.5, 191.9; four ranks x 2000 x
        // 2048 438, 416, 412, 407; 2500 x 5120 x top-4, fwd, 66.5, 66.2, 64.9, 64.2.  Held 384 or 512: two ranks x 4000 x 3072 x
        // top-8 463, 455, 459, 470; 5064 x 3072 x top-4 155.8, 155.4, 160.5, 170.2; 8000 x 4096 x top-4 260.4, 257.5, 258.4, 268.4
        // (2000 x 4096 x top-6 129.9, 128.1, 127.3, 126.6).  Stored once or twice: two ranks x 16333 x 4096 798, 794, 810, 872; 11308
        // x 12288 x top-1, fwd, 263.3, 261.7, 268.2, 283.8; 3000 x 7168 x top-2 148.0, 147.2, 146.2, 149.8.  Four ranks x 4096 x 7168
        // x top-8 (1.9 GB) 1785, 1817, -, 1816, eight x 2500 x 7168, fwd, 1137, 1161, -, 1161.
        // Two for rows that end within a line, which are not written through; fwd, at eight, four and two: 4000 x 3000 x top-4 72.5,
        // 70.7 and 69.3, 4000 x 2008 x top-2 49.6, 49.9 and 47.3, 2223 x 5000 x top-2 53.0, 51.5 and 49.8, 2223 x 7176 x top-6 121.9,
        // 119.4 and 118.0.
        // No cap of two where the plan's workgroups are more than such a launch holds at once: they go ahead of the copies, and
        // it took them in rounds.  Fwd, top-8, two and as many as fit: 17000 x 1000 142.4 and 140.2, 20000 x 504 103.5 and 100.8, 40000
        // x 1000 323 and 315, 60000 x 1000 488 and 468, 66000 x 520 (launches behind the copies 328) 322 and 301, two ranks x 20000 x
        // 1000 368 and 366; but with fewer of them 4096 x 1000 51.1 and 53.0.  Four to a unit hold more than they lose: 60000 x 1024
        // 409.2 and 411.7.
        const int64_t heldVecs = vecs <= 4 * kWave ? vecs * (kThreads / kWave) : vecs;
        const bool wholeLines = vecs % 8 == 0;
        const int capWorkgroups = !wholeLines || (heldVecs > 2 * kThreads && w.k >= 4) ? 2 : 4;
        const bool capped = worldRowBytes * w.k <= (int64_t{1} << 30) && (capWorkgroups != 2 || extras.planBlocks <= 2 * kComputeUnits);
        const unsigned capLds = capped ? TileXREp::CapLdsBytes(capWorkgroups) : 0u;
        auto launch = [&](auto lanes, auto vecsPerLane, auto stores) {
            constexpr int G = decltype(lanes)::value;
            constexpr int V = decltype(vecsPerLane)::value;
            constexpr int kAux = decltype(stores)::value;
            constexpr int64_t kTokens = kThreads / G * kXcds;       // tokens of eight neighbouring workgroups
            extras.copyBlocks = static_cast<unsigned>((w.s + kTokens - 1) / kTokens * kXcds * tokenSlices);
            const dim3 grid(extras.planBlocks + extras.copyBlocks + extras.finishBlocks, R);
            if (w.fresh) {
                hipLaunchKernelGGL((moon_scatter_token_kernel<true, G, V, kAux>), grid, dim3(kThreads), capLds, stream, w, tokenSlices,
                    extras);
            } else {
                hipLaunchKernelGGL((moon_scatter_token_kernel<false, G, V, kAux>), grid, dim3(kThreads), capLds, stream, w, tokenSlices,
                    extras);
            }
        };
        auto pickStores = [&](auto lanes, auto vecsPerLane) {
            if (wholeLines) {
                launch(lanes, vecsPerLane, std::integral_constant<int, TileXREp::kAuxAgentScopeKept>{});
            } else if (w.k >= 4) {
                launch(lanes, vecsPerLane, std::integral_constant<int, 0>{});
            } else {
                launch(lanes, vecsPerLane, std::integral_constant<int, TileXREp::kAuxNonTemporal>{});
            }
        };
        // narrow rows: a wave per token (four tokens per workgroup); wide ones: the workgroup
        if (vecs <= 2 * kWave) {
            pickStores(std::integral_constant<int, kWave>{}, std::integral_constant<int, 2>{});
        } else if (vecs <= 4 * kWave) {
            pickStores(std::integral_constant<int, kWave>{}, std::integral_constant<int, 4>{});
        } else if (vecs <= 2 * kThreads) {
            pickStores(std::integral_constant<int, kThreads>{}, std::integral_constant<int, 2>{});
        } else {
            pickStores(std::integral_constant<int, kThreads>{}, std::integral_constant<int, kTokenVecs / kThreads>{});
        }
    } else if (perRoute) {
        gScatterName = "moon_scatter_kernel";
        // The cap takes workgroups with both of their lanes' loads to do (four stages, top-8, us without and with it: 4096 x
        // 4096 265 and 262, 4096 x 7168 436 and 415; up to 4096 x 2304 no difference beyond the runs' own).
        const unsigned capLds = vecs > kThreads ? TileXREp::CapLdsBytes(kScatterCapWorkgroups) : 0u;
        extras.copyBlocks = static_cast<unsigned>(blocks);
        const dim3 grid(extras.planBlocks + extras.copyBlocks + extras.finishBlocks, R);
        const bool scalar = w.world > 1 || vecs % (kRowVecs * kThreads) == 0;
        auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, dim3(kThreads), capLds, stream, w, colSlices, extras); };
        if (w.fresh) {
            scalar ? launch(moon_scatter_kernel<true, true>) : launch(moon_scatter_kernel<true, false>);
        } else {
            scalar ? launch(moon_scatter_kernel<false, true>) : launch(moon_scatter_kernel<false, false>);
        }
    } else {
        gScatterName = "moon_scatter_generic_kernel";
        const unsigned grid = static_cast<unsigned>(w.s * w.k);
        if (w.fresh) {
            hipLaunchKernelGGL(moon_scatter_generic_kernel<true>, dim3(grid, R), dim3(kThreads), 0, stream, w);
        } else {
            hipLaunchKernelGGL(moon_scatter_generic_kernel<false>, dim3(grid, R), dim3(kThreads), 0, stream, w);
        }
    }
    MOON_LAUNCH_CHECK();
    err = RecordIf(timing.stop, stream);
    if (err != hipSuccess) {
        return err;
    }
    return allInScatter ? hipSuccess : LaunchPlanAndFinish(w, stream, vec);
}

hipError_t LaunchMoonCombine(const CombineWorld &w, hipStream_t stream, const LaunchTiming &timing)
{
    const unsigned R = static_cast<unsigned>(w.world);
    const unsigned rowBlocks = static_cast<unsigned>((w.nvS + kThreads - 1) / kThreads);
    hipLaunchKernelGGL(moon_combine_prepare_kernel, dim3(rowBlocks, R), dim3(kThreads), 0, stream, w);
    MOON_LAUNCH_CHECK();
    bool vec = w.h % 8 == 0;
    for (int r = 0; r < w.world; ++r) {
        vec = vec && TileXREp::Aligned16(w.hiddenSh[r]) && TileXREp::Aligned16(w.hiddenNvsh[r]);
    }
    const int64_t vecs = w.h / 8;
    constexpr int G = kWave;
    const int colSlices = static_cast<int>((vecs + G * kRowVecs - 1) / (G * kRowVecs));
    // up to three times the L2s' 32 MB of receive rows in the world: the slices of a token go to the XCD that wrote its rows
    const bool placed = static_cast<int64_t>(w.world) * w.nvS * w.h * 2 <= (int64_t{96} << 20);
    const int64_t units = (placed ? (w.s + kXcds - 1) / kXcds * kXcds : w.s) * colSlices;
    hipError_t err = RecordIf(timing.start, stream);
    if (err != hipSuccess) {
        return err;
    }
    if (vec && units <= 0x7fffffff) {
        gReduceName = "moon_reduce_kernel";
        hipLaunchKernelGGL(moon_reduce_kernel<G>, dim3(static_cast<unsigned>(units), R), dim3(G), 0, stream, w, colSlices,
            placed ? 1 : 0);
    } else {
        gReduceName = "moon_reduce_generic_kernel";
        hipLaunchKernelGGL(moon_reduce_generic_kernel, dim3(static_cast<unsigned>(w.s), R), dim3(kThreads), 0, stream, w);
    }
    MOON_LAUNCH_CHECK();
    return RecordIf(timing.stop, stream);
}

} // namespace TileXRMoon
