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
#include "ep_small_route.hip.h"

namespace TileXREp {
namespace {

// us for eight layers in a graph, streaming and left to the L2: 4 x 7168 x top-8 53.5 -> 52.4, 17 x 7168 (2.2 MB with the token
// rows) 57.6 -> 56.6, 30 x 4096 56.5 -> 55.5, 60 x 4096 x top-2 (1.5 MB) 51.2 -> 49.8, top-4
// (2.5 MB) 54.2 -> 53.4; but 60 x 8192 x top-2 (2.9 MB) 55.5 and
// 57.6, 100 x 2048 (3.7 MB) 62.3 and 64.0, 100 x 7168 88.1 and 99.6.
inline bool LeavesRowsToL2(const SmallDispatchLaunch &l)
{
    return l.bs * (l.topK + 1) * l.h * 2 <= (int64_t{10} << 18);
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

} // namespace

constexpr int64_t kSmallMvpExperts = 512;

// Quantised rows: no capacity limit, and at most four vectors to a lane.  Dispatch + combine, routing and scatter launch before
// and the one launch now, us: int8 512 x 2048 x top-4 12.4 -> 10.2, 2048 x 4096 x top-1 16.5 -> 15.4, 1000 x 7168 x top-2 16.9
// and 16.8, 512 x 8192 x top-4 15.6 and 16.0 (each route's workgroup quantises the token's row again), block fp8 12.4 -> 10.7,
// 16.4 -> 15.2, 17.4 and 17.3, 16.3 and 16.3; with flags, which cost the others a place launch as well, block fp8 17.6 -> 13.4,
// 22.1 -> 18.5, 22.5 -> 19.3, 21.5 -> 18.5.  MXFP8, its combine without the invert launch as well, 1 x 7168 x top-8 15.2 -> 10.0,
// 128 x 7168 16.9 -> 13.0, 250 x 8192 20.2 -> 16.8, 1000 x 7168 x top-2 21.7 -> 20.6.
static bool SmallQuantFits(const SmallDispatchLaunch &l)
{
    const bool copesWithAny = l.tileFlags != nullptr || l.quantMode == TILEXR_EP_QUANT_MXFP8;
    return (l.quantMode == TILEXR_EP_QUANT_TOKEN_INT8 || l.quantMode == TILEXR_EP_QUANT_MXFP8 ||
            l.quantMode == TILEXR_EP_QUANT_FP8_BLOCK128) &&
        l.capacity <= 0 && l.h / 8 <= 4 * kThreads && Aligned8(l.out) && l.scalesOut != nullptr &&
        (copesWithAny || l.bs * l.topK * l.h <= (int64_t{12} << 20));
}

// MVP route: no mask, no capacity limit, no flags.  Every expert wants a workgroup for its count, and kSmallMvpExperts is where
// the first measurements ended; the gain goes on (64 x 1024 x top-2 of 768 experts 11.8 and 8.4, of 2048 14.4 and 8.5; 200 x 7168 x
// top-5 of 1024 14.9 and 10.8; 2000 x 1024 x top-1 of 2048 23.0 and 11.7).  Dispatch + combine, us, routing
// and scatter launch before and the one launch now: 64 x 1024 x top-2 12.0 -> 8.1, 200 x 7168 x top-5 12.7 -> 10.4, 256 x 4096 x
// top-8 13.6 -> 11.6, 2000 x 1024 x top-1 14.9 -> 11.7, 300 x 7168 x top-6 18.3 -> 16.7; int8 68 x 2048 x top-8 12.3 -> 8.8, 2000 x
// 1024 x top-1 15.2 -> 12.6, 400 x 2048 x top-5 (4.1 M elements) 12.4 and 12.4, 256 x 4096 x top-8 (8.4 M) 12.9 and 13.8.
static bool SmallMvpFits(const SmallDispatchLaunch &l)
{
    return l.numExperts <= kSmallMvpExperts && l.maskMode == kMaskNone && l.capacity <= 0 && l.tileFlags == nullptr &&
        (l.quantMode == TILEXR_EP_QUANT_NONE || (l.quantMode == TILEXR_EP_QUANT_TOKEN_INT8 && !l.inputBf16 && l.bs * l.topK * l.h <= (int64_t{3} << 20)));
}

// Many rows of whole lines are written through and stay in the memory-side cache, where Combine finds them.  Streamed, wide ones had
// become slower than with the routing and scatter launches, us with those, streamed and kept: fp16 1000 x 16384 x top-1 of 64 32.1,
// 34.2 and 29.6, 700 x top-2 30.0, 31.4 and 28.0, 512 x top-4 32.7, 33.4 and 30.2, 2048 x top-1 49.8, 50.2 and 48.0.  Level at
// the line (256 x 6144 x top-8 17.4, 14.9 and 14.8, 240 x 7168 17.9, 15.5 and 15.5); rows that end within a line stream (2048 x
// 16376 x top-1 56.4 and 51.2).
static bool KeepsMvpRows(const SmallDispatchLaunch &l)
{
    return l.h % 64 == 0 && l.bs * l.topK * l.h * 2 >= (int64_t{24} << 20);
}

bool SmallDispatchFits(const SmallDispatchLaunch &l)
{
    return (!l.mvp || SmallMvpFits(l)) && l.bs * l.topK <= kSmallRoutes && l.numExperts <= kMaxKeys && l.topK <= kMaxTopK && l.h % 8 == 0 &&
        l.h / 8 <= 8 * kThreads && Aligned16(l.x) &&
        (l.quantMode == TILEXR_EP_QUANT_NONE ? Aligned16(l.out) : SmallQuantFits(l)) &&
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
    a.scalesOut = l.scalesOut;
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
        if (l.quantMode != TILEXR_EP_QUANT_NONE) {
            return LaunchSmallQuantRoutes(l, a, routes.x);
        }
        if (l.mvp) {
            auto pickMvp = [&](auto vecsPerLane) {
                constexpr int kV = decltype(vecsPerLane)::value;
                if (LeavesRowsToL2(l)) {
                    launch(ep_dispatch_small_route_kernel<kV, 0, kIdsPerLane, false, TILEXR_EP_QUANT_NONE, true, false, true>, routes);
                } else if (KeepsMvpRows(l)) {
                    launch(ep_dispatch_small_route_kernel<kV, kAuxAgentScopeKept, kIdsPerLane, false, TILEXR_EP_QUANT_NONE, true, false, true>, routes);
                } else {
                    launch(ep_dispatch_small_route_kernel<kV, kAuxNonTemporal, kIdsPerLane, false, TILEXR_EP_QUANT_NONE, true, false, true>, routes);
                }
            };
            v == 2 ? pickMvp(std::integral_constant<int, 2> {}) : v == 4 ? pickMvp(std::integral_constant<int, 4> {}) :
                pickMvp(std::integral_constant<int, 8> {});
            return hipGetLastError();
        }
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
