// Small-batch dispatch in one launch (gfx950, wave64): decode-sized calls are bound by launch latency, not by HBM.
//
// Up to kSmallRoutes routes fit one workgroup's registers, so every workgroup counts the whole expert-id table for
// itself -- per-expert histogram in LDS, exclusive offsets, rank of its own token's routes among the earlier routes of
// the same expert -- while its token's row is already on its way from HBM, and then writes the row to its topK
// destination rows.  Workgroup 0 also writes the count outputs.  The results are the same as those of the count +
// scatter pair (same definitions, reference: src/ep/kernels/tilexr_ep_dispatch_memory_kernel.h:791-818, 1059-1074,
// 1159-1168, 1240-1258); only the number of launches differs.  With readiness flags the rows are written through to memory
// and reported landed as in the scatter kernels (ep_tile_publish.h); the rows the whole dispatch keeps, which the size of
// the last tile depends on, every workgroup has counted anyway or counts with four more ballots.
#include <algorithm>
#include <type_traits>

#include <hip/hip_runtime.h>

#include "ep_block_scan.hip.h"
#include "ep_kernel_common.hip.h"
#include "ep_launch.h"
#include "ep_numerics.hip.h"
#include "ep_tile_publish.h"

namespace TileXREp {
namespace {

constexpr int kIdsPerLane = kSmallRoutes / kThreads;

struct SmallArgs {
    const void *x;
    const int32_t *ids;
    int bs;
    int h;
    int topK;
    int numExperts;
    const uint8_t *mask;         // masked kernels: [bs] or [bs, topK]
    int maskPerRoute;            // 1: route live iff mask[token, k]; 0: iff token < sum(mask)
    int capacity;
    int32_t srcRank;
    int32_t expertIdBias;
    void *out;
    int32_t *assist;
    int32_t *rowOf;              // optional [bs, topK]
    int32_t *sendCountsOut;
    int32_t *firstOffsetOut;     // optional
    int64_t *expertTokenNumsOut;
    int tokenNumsType;
    TilePublishArgs tiles;       // flags == nullptr: none (totalRows is filled in by the kernels)
};

// The lane's vectors of a row.  AUX, the cache policy: published rows are written through to memory (kAuxAgentScope) and are
// complete for every XCD once the issuing wave's memory counter is zero.  Others stream (kAuxNonTemporal), or -- while token rows
// and rows of the call together are few (LeavesRowsToL2) -- are left to the L2 (0), where the combine that runs on the same XCD
// finds them.
template <int V, int AUX>
__device__ __forceinline__ void SmallRowStore(const SmallArgs &a, int row, const u32x4 (&v)[V])
{
    const int vecs = a.h / 8;
    u32x4 *dst = reinterpret_cast<u32x4 *>(static_cast<char *>(a.out) + static_cast<int64_t>(row) * a.h * 2);
    const __amdgpu_buffer_rsrc_t rsrc = RowResource(dst, vecs * 16);
#pragma unroll
    for (int j = 0; j < V; ++j) {
        const int idx = j * kThreads + static_cast<int>(threadIdx.x);
        if (idx >= vecs) {
            continue;
        }
        if constexpr (AUX == kAuxNonTemporal) {
            __builtin_nontemporal_store(v[j], dst + idx);
        } else {
            __builtin_amdgcn_raw_buffer_store_b128(v[j], rsrc, idx * 16, 0, AUX);
        }
    }
}

// us for eight layers in a graph, streaming and left to the L2: 4 x 7168 x top-8 53.5 -> 52.4, 17 x 7168 (2.2 MB with the token
// rows) 57.6 -> 56.6, 30 x 4096 56.5 -> 55.5, 60 x 4096 x top-2 (1.5 MB) 51.2 -> 49.8, top-4
// (2.5 MB) 54.2 -> 53.4; but 60 x 8192 x top-2 (2.9 MB) 55.5 and
// 57.6, 100 x 2048 (3.7 MB) 62.3 and 64.0, 100 x 7168 88.1 and 99.6.
inline bool LeavesRowsToL2(const SmallDispatchLaunch &l)
{
    return l.bs * (l.topK + 1) * l.h * 2 <= (int64_t{10} << 18);
}

// Masked calls: first route that a token-prefix mask leaves out (n for a mask per route).  The mask is read beside the id
// table, four bytes of it in flight per lane (1024 tokens), and one LDS exchange between the waves adds it up.  All lanes
// of the workgroup call it.
constexpr int kMaskBatch = 4;
__device__ __forceinline__ int SmallLiveLimit(const SmallArgs &a, int n, int *s_live)
{
    if (a.maskPerRoute != 0) {
        return n;
    }
    // bytes beyond the mask's end read as zero
    const __amdgpu_buffer_rsrc_t mask = RowResource(a.mask, a.bs);
    int live = 0;
    for (int first = 0; first < a.bs; first += kMaskBatch * kThreads) {
        uint8_t m[kMaskBatch];
#pragma unroll
        for (int u = 0; u < kMaskBatch; ++u) {
            m[u] = __builtin_amdgcn_raw_buffer_load_b8(mask, first + u * kThreads + static_cast<int>(threadIdx.x), 0, 0);
        }
#pragma unroll
        for (int u = 0; u < kMaskBatch; ++u) {
            live += __popcll(__ballot(m[u] != 0));
        }
    }
    if ((threadIdx.x & (kWave - 1)) == 0) {
        s_live[threadIdx.x / kWave] = live;
    }
    __syncthreads();
    return (s_live[0] + s_live[1] + s_live[2] + s_live[3]) * a.topK;
}

// Whether a route below `n` is dispatched.
__device__ __forceinline__ bool SmallRouteLive(const SmallArgs &a, int route, int limit)
{
    return a.maskPerRoute != 0 ? a.mask[route] != 0 : route < limit;
}

template <int V, bool WT, bool MASKED>
__global__ __launch_bounds__(kThreads) void ep_dispatch_small_kernel(SmallArgs a)
{
    __shared__ int s_live[kWavesPerBlock];
    __shared__ int s_hist[kMaxKeys];     // routes per expert, then exclusive row offsets
    __shared__ int s_kept[kMaxKeys];
    __shared__ int s_rank[kMaxTopK];
    __shared__ int s_key[kMaxTopK];
    __shared__ int s_pos[kMaxTopK];
    __shared__ int s_part[kThreads];

    const int tid = threadIdx.x;
    const int token = blockIdx.x;
    const int n = a.bs * a.topK;
    const int vecs = a.h / 8;

    // the token's row: in flight while the routing is worked out
    const u32x4 *src = reinterpret_cast<const u32x4 *>(static_cast<const char *>(a.x) + static_cast<int64_t>(token) * a.h * 2);
    u32x4 v[V];
#pragma unroll
    for (int j = 0; j < V; ++j) {
        const int idx = j * kThreads + tid;
        v[j] = idx < vecs ? src[idx] : u32x4{0u, 0u, 0u, 0u};
    }
    int e[kIdsPerLane];
#pragma unroll
    for (int j = 0; j < kIdsPerLane; ++j) {
        const int i = j * kThreads + tid;
        const int id = i < n ? a.ids[i] : -1;
        e[j] = (id >= 0 && id < a.numExperts) ? id : -1;      // ids outside [0, E) are skipped, not errors
    }
    for (int k = tid; k < a.numExperts; k += kThreads) {
        s_hist[k] = 0;
    }
    const int ownId = tid < a.topK ? a.ids[token * a.topK + tid] : -1;
    int limit = n;
    if (MASKED) {
        limit = SmallLiveLimit(a, n, s_live);
#pragma unroll
        for (int j = 0; j < kIdsPerLane; ++j) {
            const int i = j * kThreads + tid;
            e[j] = i < n && SmallRouteLive(a, i, limit) ? e[j] : -1;
        }
    }
    if (tid < a.topK) {
        const bool live = !MASKED || SmallRouteLive(a, token * a.topK + tid, limit);
        s_key[tid] = (live && ownId >= 0 && ownId < a.numExperts) ? ownId : -1;
        s_rank[tid] = 0;
    }
    __syncthreads();
    const int first = token * a.topK;
#pragma unroll
    for (int j = 0; j < kIdsPerLane; ++j) {
        const int i = j * kThreads + tid;
        if (e[j] < 0) {
            continue;
        }
        atomicAdd(&s_hist[e[j]], 1);
        // rank of the token's route k within its expert = earlier routes (flat order) with the same expert
        if (i < first + a.topK) {
            for (int k = 0; k < a.topK; ++k) {
                if (i < first + k && s_key[k] == e[j]) {
                    atomicAdd(&s_rank[k], 1);
                }
            }
        }
    }
    __syncthreads();
    for (int k = tid; k < a.numExperts; k += kThreads) {
        const int c = s_hist[k];
        const int kept = (a.capacity > 0 && c > a.capacity) ? a.capacity : c;
        s_kept[k] = kept;
        s_hist[k] = kept;
    }
    __syncthreads();
    const int totalRows = BlockExclusiveScan(s_hist, a.numExperts, s_part);
    if (tid < a.topK) {
        const int key = s_key[tid];
        int row = -1;
        if (key >= 0 && (a.capacity <= 0 || s_rank[tid] < a.capacity)) {
            row = s_hist[key] + s_rank[tid];
            int32_t *tuple = a.assist + static_cast<int64_t>(row) * 4;
            tuple[0] = a.srcRank;
            tuple[1] = token;
            tuple[2] = tid;
            tuple[3] = key + a.expertIdBias;
        }
        s_pos[tid] = row;
        if (a.rowOf != nullptr) {
            a.rowOf[first + tid] = row;
        }
    }
    if (token == 0) {
        if (tid == 0 && a.firstOffsetOut != nullptr) {
            *a.firstOffsetOut = 0;
        }
        for (int k = tid; k < a.numExperts; k += kThreads) {
            const int incl = s_hist[k] + s_kept[k];
            a.sendCountsOut[k] = incl;
            if (a.expertTokenNumsOut != nullptr) {
                a.expertTokenNumsOut[k] = a.tokenNumsType == 0 ? incl : s_kept[k];
            }
        }
    }
    __syncthreads();
    for (int k = 0; k < a.topK; ++k) {
        const int row = __builtin_amdgcn_readfirstlane(s_pos[k]);
        if (row < 0) {
            continue;
        }
        SmallRowStore<V, WT ? kAuxAgentScope : kAuxNonTemporal>(a, row, v);
    }
    if (WT) {
        // every wave waits for its own stores, the barrier collects the waves, then the rows are reported landed
        WaitOwnStores();
        __syncthreads();
        if (tid < a.topK && s_pos[tid] >= 0) {
            TilePublishArgs t = a.tiles;
            t.totalRows = totalRows;
            DeviceTileOps ops;
            PublishLanded(ops, t, s_pos[tid], 1);
        }
    }
}

// Without a capacity limit a route's row needs no histogram at all:
//   row = (valid routes with a smaller expert id) + (earlier routes with the same expert id)
// so one workgroup per route counts those two sets over the id table and writes its one row.  Workgroup b < E also
// counts expert b's routes for the count outputs.  Eight times as many workgroups as tokens spread a decode batch
// over the whole chip.
//
// The launch is two round trips to memory (id table and token row out, the row's stores back) with the counting in
// between, and at this size the counting is paid in instructions: a wave that runs alone on its SIMD issues a dependent
// instruction every 4 ns or so.  So every lane counts its own ids with compares and adds (no ballot and scalar count
// per id), the four sets share two registers (16 bits each: at most 2048 ids), one pair of reductions per wave and one
// LDS exchange between the four waves finish it.  IDS = ids per lane (4: up to 1024 routes, 8: up to 2048).
//
// MASKED: the routes a mask leaves out are dropped from the counts like ids outside [0, E) (token-prefix mask: one more
// LDS exchange, for the number of active tokens).  200 tokens x 7168 x top-8 of 256 with a token mask: 6.7 us, 13.3 us
// for the count and scatter launches such calls took before.
template <int V, int AUX, int IDS, bool MASKED>
__global__ __launch_bounds__(kThreads) void ep_dispatch_small_route_kernel(SmallArgs a)
{
    constexpr bool WT = AUX == kAuxAgentScope;
    __shared__ int s_live[kWavesPerBlock];
    __shared__ int s_sum[kWavesPerBlock][3];     // per wave: smaller | earlier equal << 16, equal to blockIdx | not above << 16, valid

    const int tid = threadIdx.x;
    const int lane = tid & (kWave - 1);
    const int wave = tid / kWave;
    // Workgroup b runs on XCD b % 8: the K routes of token t go to workgroups of XCD t % 8, where the decode-sized
    // combine places the token's slices as well, so that the rows it reads are still in the L2 that they were written
    // through (the tokens are padded to a multiple of eight: a workgroup of the padding has no route, only an expert to
    // count for).
    const int placed = static_cast<int>(blockIdx.x) / kXcdCount;
    const int token = (placed / a.topK) * kXcdCount + static_cast<int>(blockIdx.x) % kXcdCount;
    const bool hasRoute = token < a.bs;
    const int route = hasRoute ? token * a.topK + placed % a.topK : 0;
    const int n = a.bs * a.topK;
    const int vecs = a.h / 8;

    const u32x4 *src = reinterpret_cast<const u32x4 *>(static_cast<const char *>(a.x) + static_cast<int64_t>(hasRoute ? token : 0) * a.h * 2);
    u32x4 v[V];
#pragma unroll
    for (int j = 0; j < V; ++j) {
        const int idx = j * kThreads + tid;
        v[j] = idx < vecs ? src[idx] : u32x4{0u, 0u, 0u, 0u};
    }
    int e[IDS];
#pragma unroll
    for (int j = 0; j < IDS; ++j) {
        const int i = j * kThreads + tid;
        e[j] = i < n ? a.ids[i] : -1;
    }
    const int mine = a.ids[route];
    const unsigned experts = static_cast<unsigned>(a.numExperts);
    bool live = hasRoute;
    if (MASKED) {
        const int limit = SmallLiveLimit(a, n, s_live);
#pragma unroll
        for (int j = 0; j < IDS; ++j) {
            const int i = j * kThreads + tid;
            e[j] = i < n && SmallRouteLive(a, i, limit) ? e[j] : -1;
        }
        live = hasRoute && SmallRouteLive(a, route, limit);
    }
    const int key = live && static_cast<unsigned>(mine) < experts ? mine : -1;       // ids outside [0, E) are skipped, not errors
    const int expert = blockIdx.x;       // the expert this workgroup counts for the outputs (if there is one)
    int rowCounts = 0;      // valid ids below the key | earlier ids equal to it << 16
    int outCounts = 0;      // ids equal to `expert` | valid ids not above it << 16
    int valid = 0;
#pragma unroll
    for (int j = 0; j < IDS; ++j) {
        const int i = j * kThreads + tid;
        const unsigned id = static_cast<unsigned>(e[j]);
        const bool ok = id < experts;
        rowCounts += (ok && e[j] < key ? 1 : 0) + (e[j] == key && i < route ? 0x10000 : 0);
        outCounts += (e[j] == expert ? 1 : 0) + (ok && e[j] <= expert ? 0x10000 : 0);
        valid += ok ? 1 : 0;
    }
    rowCounts = WaveSum(rowCounts);
    outCounts = WaveSum(outCounts);
    if (WT) {
        valid = WaveSum(valid);
    }
    if (lane == 0) {
        s_sum[wave][0] = rowCounts;
        s_sum[wave][1] = outCounts;
        s_sum[wave][2] = valid;
    }
    __syncthreads();
    const int rowSum = s_sum[0][0] + s_sum[1][0] + s_sum[2][0] + s_sum[3][0];
    const int row = key >= 0 ? (rowSum & 0xffff) + (rowSum >> 16) : -1;
    if (tid == 0) {
        if (row >= 0) {
            int32_t *tuple = a.assist + static_cast<int64_t>(row) * 4;
            tuple[0] = a.srcRank;
            tuple[1] = token;
            tuple[2] = route % a.topK;
            tuple[3] = key + a.expertIdBias;
        }
        if (a.rowOf != nullptr && hasRoute) {
            a.rowOf[route] = row;
        }
        if (expert == 0 && a.firstOffsetOut != nullptr) {
            *a.firstOffsetOut = 0;
        }
        if (expert < a.numExperts) {
            const int outSum = s_sum[0][1] + s_sum[1][1] + s_sum[2][1] + s_sum[3][1];
            a.sendCountsOut[expert] = outSum >> 16;
            if (a.expertTokenNumsOut != nullptr) {
                a.expertTokenNumsOut[expert] = a.tokenNumsType == 0 ? outSum >> 16 : outSum & 0xffff;
            }
        }
    }
    if (row < 0) {
        return;
    }
    SmallRowStore<V, AUX>(a, row, v);
    if (WT) {
        WaitOwnStores();
        __syncthreads();        // uniform: a workgroup without a row has left as a whole
        if (tid == 0) {
            TilePublishArgs t = a.tiles;
            t.totalRows = s_sum[0][2] + s_sum[1][2] + s_sum[2][2] + s_sum[3][2];      // rows the whole dispatch keeps: the size of the last tile
            DeviceTileOps ops;
            PublishLanded(ops, t, row, 1);
        }
    }
}

} // namespace

bool SmallDispatchFits(const SmallDispatchLaunch &l)
{
    return l.bs * l.topK <= kSmallRoutes && l.numExperts <= kMaxKeys && l.topK <= kMaxTopK && l.h % 8 == 0 &&
        l.h / 8 <= 8 * kThreads && Aligned16(l.x) && Aligned16(l.out) &&
        (l.maskMode == kMaskNone || (l.mask != nullptr && (l.maskMode == kMaskPerRoute || l.maskMode == kMaskTokenPrefix)));
}

hipError_t LaunchSmallDispatch(const SmallDispatchLaunch &l)
{
    SmallArgs a {};
    a.x = l.x;
    a.ids = l.ids;
    a.bs = static_cast<int>(l.bs);
    a.h = static_cast<int>(l.h);
    a.topK = static_cast<int>(l.topK);
    a.numExperts = static_cast<int>(l.numExperts);
    a.mask = l.mask;
    a.maskPerRoute = l.maskMode == kMaskPerRoute ? 1 : 0;
    a.capacity = static_cast<int>(l.capacity);
    a.srcRank = l.srcRank;
    a.expertIdBias = l.expertIdBias;
    a.out = l.out;
    a.assist = l.assist;
    a.rowOf = l.rowOf;
    a.sendCountsOut = l.sendCountsOut;
    a.firstOffsetOut = l.firstOffsetOut;
    a.expertTokenNumsOut = l.expertTokenNumsOut;
    a.tokenNumsType = l.tokenNumsType;
    const bool flags = l.tileFlags != nullptr;
    if (flags) {
        a.tiles.flags = l.tileFlags;
        a.tiles.counters = l.tileCounters;
        a.tiles.tileRows = static_cast<int>(l.tileRows);
        a.tiles.maxTiles = static_cast<int>((l.bs * l.topK + l.tileRows - 1) / l.tileRows);
        a.tiles.epoch = l.epoch;
    }
    const int64_t vecs = l.h / 8;
    const int v = vecs <= 2 * kThreads ? 2 : (vecs <= 4 * kThreads ? 4 : 8);
    auto launch = [&](auto kernel, dim3 grid) { hipLaunchKernelGGL(kernel, grid, dim3(kThreads), 0, l.stream, a); };
    if (l.capacity <= 0) {
        // one workgroup per route, and further ones until every expert's count outputs have theirs (those cost less than
        // one workgroup per token that builds the whole histogram, as calls with fewer routes than experts used to get:
        // dispatch + combine from a graph, 7168 columns, top-8 of 256: 1 token 8.2 -> 6.8 us, 8 tokens 9.1 -> 7.4, 31
        // tokens 9.9 -> 8.3)
        if (l.kernelNameOut != nullptr) {
            *l.kernelNameOut = "ep_dispatch_small_route_kernel";
        }
        const dim3 routes(static_cast<unsigned>(std::max<int64_t>(XcdPlacedUnits(static_cast<int>(l.bs), static_cast<int>(l.topK)), l.numExperts)));
        const bool few = l.bs * l.topK <= 4 * kThreads;
        const bool plain = LeavesRowsToL2(l);
        auto pickStores = [&](auto vecsPerLane, auto masked, auto ids) {
            constexpr int kV = decltype(vecsPerLane)::value;
            constexpr int kIds = decltype(ids)::value;
            constexpr bool kMasked = decltype(masked)::value;
            if (flags) {
                launch(ep_dispatch_small_route_kernel<kV, kAuxAgentScope, kIds, kMasked>, routes);
            } else if (plain) {
                launch(ep_dispatch_small_route_kernel<kV, 0, kIds, kMasked>, routes);
            } else {
                launch(ep_dispatch_small_route_kernel<kV, kAuxNonTemporal, kIds, kMasked>, routes);
            }
        };
        auto pickMasked = [&](auto vecsPerLane, auto masked) {
            if (few) {
                pickStores(vecsPerLane, masked, std::integral_constant<int, 4> {});
            } else {
                pickStores(vecsPerLane, masked, std::integral_constant<int, kIdsPerLane> {});
            }
        };
        auto pick = [&](auto vecsPerLane) {
            if (l.maskMode != kMaskNone) {
                pickMasked(vecsPerLane, std::true_type {});
            } else {
                pickMasked(vecsPerLane, std::false_type {});
            }
        };
        if (v == 2) {
            pick(std::integral_constant<int, 2>{});
        } else if (v == 4) {
            pick(std::integral_constant<int, 4>{});
        } else {
            pick(std::integral_constant<int, 8>{});
        }
        return hipGetLastError();
    }
    const dim3 grid(static_cast<unsigned>(l.bs));
    if (l.kernelNameOut != nullptr) {
        *l.kernelNameOut = "ep_dispatch_small_kernel";
    }
    auto pick = [&](auto vecsPerLane) {
        constexpr int kV = decltype(vecsPerLane)::value;
        if (l.maskMode != kMaskNone) {
            flags ? launch(ep_dispatch_small_kernel<kV, true, true>, grid) : launch(ep_dispatch_small_kernel<kV, false, true>, grid);
        } else {
            flags ? launch(ep_dispatch_small_kernel<kV, true, false>, grid) : launch(ep_dispatch_small_kernel<kV, false, false>, grid);
        }
    };
    if (v == 2) {
        pick(std::integral_constant<int, 2>{});
    } else if (v == 4) {
        pick(std::integral_constant<int, 4>{});
    } else {
        pick(std::integral_constant<int, 8>{});
    }
    return hipGetLastError();
}

} // namespace TileXREp
