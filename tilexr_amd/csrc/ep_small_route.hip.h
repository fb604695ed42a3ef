// The decode-sized dispatch without a capacity limit, one workgroup per route (ep_small.hip): the kernel, for plain rows
// (instantiated there) and for quantised ones (ep_small_quant.hip).
#ifndef TILEXR_AMD_EP_SMALL_ROUTE_HIP_H
#define TILEXR_AMD_EP_SMALL_ROUTE_HIP_H

#include <hip/hip_runtime.h>

#include "ep_kernel_common.hip.h"
#include "ep_launch.h"
#include "ep_numerics.hip.h"
#include "ep_row_quant.hip.h"
#include "ep_tile_publish.h"

namespace TileXREp {

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
    int32_t *sendCountsOut;      // MVP route: one count of all rows, optional
    int32_t *firstOffsetOut;     // optional
    int64_t *expertTokenNumsOut;
    int tokenNumsType;
    TilePublishArgs tiles;       // flags == nullptr: none (totalRows is filled in by the kernels)
    void *scalesOut;             // quantised payloads
};

// ep_small_quant.hip: the launch for quantised rows of at most 4 * kThreads vectors.
hipError_t LaunchSmallQuantRoutes(const SmallDispatchLaunch &l, const SmallArgs &a, unsigned workgroups);

namespace {

constexpr int kIdsPerLane = kSmallRoutes / kThreads;

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
//
// QMODE: quantised payloads.  Every route's workgroup quantises the token's row for itself, K times the arithmetic of the scatter
// kernel, which at this size costs less than the launch it saves.
//
// MVP: rows in route order, whatever the expert: row = (earlier valid routes), and one count of all rows.
template <int V, int AUX, int IDS, bool MASKED, int QMODE = TILEXR_EP_QUANT_NONE, bool BF16 = true, bool E5M2 = false, bool MVP = false>
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
        rowCounts += MVP ? (ok && i < route ? 1 : 0) : (ok && e[j] < key ? 1 : 0) + (e[j] == key && i < route ? 0x10000 : 0);
        outCounts += (e[j] == expert ? 1 : 0) + (ok && e[j] <= expert ? 0x10000 : 0);
        valid += ok ? 1 : 0;
    }
    rowCounts = WaveSum(rowCounts);
    outCounts = WaveSum(outCounts);
    if (WT || MVP) {
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
            if (!MVP) {
                a.sendCountsOut[expert] = outSum >> 16;
            } else if (expert == 0 && a.sendCountsOut != nullptr) {
                *a.sendCountsOut = s_sum[0][2] + s_sum[1][2] + s_sum[2][2] + s_sum[3][2];
            }
            if (a.expertTokenNumsOut != nullptr) {
                a.expertTokenNumsOut[expert] = a.tokenNumsType == 0 ? outSum >> 16 : outSum & 0xffff;
            }
        }
    }
    if (row < 0) {
        return;
    }
    if constexpr (QMODE == TILEXR_EP_QUANT_NONE) {
        SmallRowStore<V, AUX>(a, row, v);
    } else {
        __shared__ float s_red[kWavesPerBlock];
        QuantisedRow<V> out;
        QuantiseRow<kThreads, V, QMODE, BF16, E5M2>(a, v, s_red, tid, out);
        StoreRow<kThreads, V, QMODE, RowStores::kKeep, WT>(a, row, v, out, tid);
    }
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
} // namespace TileXREp

#endif // TILEXR_AMD_EP_SMALL_ROUTE_HIP_H
