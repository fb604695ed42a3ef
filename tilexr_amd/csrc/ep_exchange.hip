// Exchange kernels for logical ranks that share one device (gfx950): drain (dispatch) and return (combine).
//
// They stand where the reference moves rows between peer windows:
//   MVP route      per-source slots drained in source-rank order, recvCounts[src], expertTokenNums
//                  (reference: src/ep/kernels/tilexr_ep_combine_helpers.h:81-145, tilexr_ep_dispatch_kernel.cpp:783-817)
//   memory route   segments ordered local expert -> source rank, sendCounts = inclusive sum, expertTokenNums from it
//                  (reference: src/ep/kernels/tilexr_ep_dispatch_memory_kernel.h:1017-1089, 1142-1168, 1208-1317)
//   combine        rows go back to the slot (token, k) of their source rank
//                  (reference: tilexr_ep_combine_memory_kernel.h:329-386, tilexr_ep_combine_kernel.cpp:28-52)
// On one device the "window" is ordinary HBM owned by the world, and readiness is stream order, not flags.
#include <hip/hip_runtime.h>

#include "ep_block_scan.hip.h"
#include "ep_exchange.h"
#include "ep_kernel_common.hip.h"
#include "ep_launch.h"
#include "ep_numerics.hip.h"

namespace TileXREp {
namespace {

// Segment idx of destination rank dstRank: which source's staging area it comes from and under which key.
//   memory route             local expert major, source minor
//   MVP route                one segment per source
//   MVP route, tp lanes      the sources of the rank's own lane first (in expert-rank order), then those of the other
//                            lanes of its group in lane order; the key is the expert rank
//                            (reference: src/ep/kernels/tilexr_ep_dispatch_kernel.cpp:809-827, 662-697)
__device__ __forceinline__ void SegmentOf(int idx, int rankSize, int dstRank, int localExperts, bool memoryRoute, int tp,
    int *src, int *key)
{
    if (memoryRoute) {
        *src = idx % rankSize;
        *key = dstRank * localExperts + idx / rankSize;
    } else if (tp <= 1) {
        *src = idx;
        *key = dstRank;
    } else {
        const int expertRanks = rankSize / tp;
        const int myLane = dstRank % tp;
        const int block = idx / expertRanks;
        const int lane = block == 0 ? myLane : (block - 1 < myLane ? block - 1 : block);
        *src = (idx % expertRanks) * tp + lane;
        *key = dstRank / tp;
    }
}

// Shared experts: route table of one source rank in the world's key space.
//   shared route s   -> rank srcRank % per + s * per (per = sharedRanks / sharedNum), tuple expert id s
//   routed id e      -> rank sharedRanks + e / localExperts, local index e % localExperts, tuple expert id sharedNum + e
// (reference: src/ep/kernels/tilexr_ep_dispatch_helpers.h:78-103, tilexr_ep_dispatch_memory_kernel.h:635-643,686-688,
//  tests/ep/demo/tilexr_ep_dispatch_demo.cpp:647-673)
struct AugmentArgs {
    const int32_t *ids;
    int n;                   // bs * (sharedNum + topK)
    int topK;
    int moeExpertNum;
    int srcRank;
    int sharedNum;
    int sharedRanks;
    int localExperts;
    int keysPerRank;
    int sharedAtExpertId;
    int32_t *keyIdsOut;
    int32_t *tupleExpertsOut;
    const uint8_t *routeMask;
    uint8_t *routeMaskOut;
};

__global__ __launch_bounds__(kThreads) void ep_augment_kernel(AugmentArgs a)
{
    const int i = blockIdx.x * kThreads + threadIdx.x;
    if (i >= a.n) {
        return;
    }
    const int perToken = a.sharedNum + a.topK;
    const int token = i / perToken;
    const int pos = i % perToken;
    int keyId = -1;
    int tupleExpert = -1;
    if (pos < a.sharedNum) {
        const int per = a.sharedRanks / a.sharedNum;
        const int dst = a.srcRank % per + pos * per;
        keyId = dst * a.keysPerRank + (a.sharedAtExpertId ? pos : 0);
        tupleExpert = pos;
    } else {
        const int e = a.ids[token * a.topK + (pos - a.sharedNum)];
        if (e >= 0 && e < a.moeExpertNum) {
            keyId = (a.sharedRanks + e / a.localExperts) * a.keysPerRank + e % a.localExperts;
            tupleExpert = a.sharedNum + e;
        }
    }
    a.keyIdsOut[i] = keyId;
    a.tupleExpertsOut[i] = tupleExpert;
    if (a.routeMaskOut != nullptr) {
        // (reference: src/ep/kernels/tilexr_ep_dispatch_memory_kernel.h:1412-1441 keeps the tokens whose mask row
        // has a set byte and walks the shared routes over those, :641-647)
        uint8_t live = 0;
        if (pos < a.sharedNum) {
            for (int k = 0; k < a.topK; ++k) {
                live |= a.routeMask[token * a.topK + k];
            }
        } else {
            live = a.routeMask[token * a.topK + (pos - a.sharedNum)];
        }
        a.routeMaskOut[i] = live != 0 ? 1 : 0;
    }
}

struct DrainArgs {
    StageLayout stage;
    int rankSize;
    int localExperts;
    int tp;
    int memoryRoute;
    int64_t rowBytes;
    int64_t scaleBytesPerRow;
    DrainTarget target[kDrainTargets];
};

__device__ __forceinline__ int SegmentsOf(const DrainArgs &a, const DrainTarget &d)
{
    return a.memoryRoute ? d.outLocalExperts * a.rankSize : a.rankSize;
}

// Rows of every segment of destination `d` and their exclusive offsets (s_off[numSeg] = all of them), in LDS.  s_base,
// where given, receives each segment's first row within its source's staging area.  Ends with a barrier.
__device__ __forceinline__ int SegmentOffsets(const DrainArgs &a, const DrainTarget &d, int numSeg, int *s_cnt, int *s_off, int *s_base,
    int *s_part)
{
    const int tid = threadIdx.x;
    for (int idx = tid; idx < numSeg; idx += kThreads) {
        int src, key;
        SegmentOf(idx, a.rankSize, d.dstRank, a.localExperts, a.memoryRoute != 0, a.tp, &src, &key);
        const int32_t *ko = a.stage.counts + static_cast<int64_t>(src) * a.stage.countsStride;
        const int first = ko[key];
        const int c = ko[key + 1] - first;
        s_cnt[idx] = c;
        s_off[idx] = c;
        if (s_base != nullptr) {
            s_base[idx] = first;
        }
    }
    LdsBarrier();
    return BlockExclusiveScan(s_off, numSeg, s_part);
}

// The count outputs of destination `d`, by one workgroup that has its segments in LDS.
__device__ __forceinline__ void DrainCounts(const DrainArgs &a, const DrainTarget &d, int numSeg, int *s_cnt, const int *s_off, int *s_tok,
    int *s_part)
{
    const int tid = threadIdx.x;
    const int expertRanks = a.tp > 1 ? a.rankSize / a.tp : a.rankSize;
    for (int idx = tid; idx < numSeg; idx += kThreads) {
        if (a.memoryRoute) {
            d.countsOut[idx] = s_off[idx] + s_cnt[idx];
        } else if (idx < expertRanks) {
            // plain per-source counts, indexed by the source's rank; with tp lanes only the rank's own lane is
            // counted here and the other entries are left alone (reference: tilexr_ep_combine_helpers.h:92-95)
            int src, key;
            SegmentOf(idx, a.rankSize, d.dstRank, a.localExperts, false, a.tp, &src, &key);
            d.countsOut[src] = s_cnt[idx];
            if (d.tpCountsOut != nullptr) {
                d.tpCountsOut[src] = s_cnt[idx];
            }
        }
    }
    if (a.tp > 1 && d.tpCountsOut != nullptr) {
        // afterwards the first tp entries become rows per lane (reference: tilexr_ep_dispatch_kernel.cpp:818-827)
        __syncthreads();
        if (tid < a.tp) {
            int rows = 0;
            for (int es = 0; es < expertRanks; ++es) {
                rows += s_cnt[tid * expertRanks + es];
            }
            const int myLane = d.dstRank % a.tp;
            const int lane = tid == 0 ? myLane : (tid - 1 < myLane ? tid - 1 : tid);
            d.tpCountsOut[lane] = rows;
        }
    }
    // rows per local expert
    for (int le = tid; le < d.tokenNumsCount; le += kThreads) {
        int n = 0;
        if (a.memoryRoute) {
            for (int s = 0; s < a.rankSize; ++s) {
                n += s_cnt[le * a.rankSize + s];
            }
        } else {
            for (int s = 0; s < a.rankSize; ++s) {
                const int32_t *et = a.stage.counts + static_cast<int64_t>(s) * a.stage.countsStride +
                    a.stage.expertTotalOffset;
                n += et[(a.tp > 1 ? d.dstRank / a.tp : d.dstRank) * a.localExperts + le];
            }
        }
        s_tok[le] = n;
    }
    __syncthreads();
    if (d.tokenNumsType == 0) {
        for (int le = tid; le < d.tokenNumsCount; le += kThreads) {
            s_cnt[le] = s_tok[le];
        }
        __syncthreads();
        BlockExclusiveScan(s_cnt, d.tokenNumsCount, s_part);
        for (int le = tid; le < d.tokenNumsCount; le += kThreads) {
            d.expertTokenNumsOut[le] = static_cast<int64_t>(s_cnt[le]) + s_tok[le];
        }
    } else {
        for (int le = tid; le < d.tokenNumsCount; le += kThreads) {
            d.expertTokenNumsOut[le] = s_tok[le];
        }
    }
}

// One workgroup per destination rank, for worlds whose segments do not fit the copying workgroups' LDS.
__global__ __launch_bounds__(kThreads) void ep_drain_plan_kernel(DrainArgs a)
{
    __shared__ int s_cnt[kMaxKeys];
    __shared__ int s_off[kMaxKeys];
    __shared__ int s_tok[kMaxKeys];
    __shared__ int s_part[kThreads];
    const DrainTarget &d = a.target[blockIdx.x];
    const int numSeg = SegmentsOf(a, d);
    const int total = SegmentOffsets(a, d, numSeg, s_cnt, s_off, nullptr, s_part);
    for (int idx = threadIdx.x; idx < numSeg; idx += kThreads) {
        d.planOffsets[idx] = s_off[idx];
    }
    if (threadIdx.x == 0) {
        d.planOffsets[numSeg] = total;
    }
    DrainCounts(a, d, numSeg, s_cnt, s_off, s_tok, s_part);
}

// Said of an address that is the same for all lanes of a wave, which the compiler cannot see of a row that it gets from the
// lane's index: without a word it wraps every store in a loop over the resources that the lanes might have.  (Drain and return
// launches, us, with the loops and without: 4 x 128 x 1024 x top-2 6.2 and 4.2, 6.1 and 4.3; 4 x 512 x 4096 x top-8 46.4 and 13.3,
// 45.7 and 13.1: they wait for memory either way.  The row's index made uniform instead, at its root, turns the tuple's loads
// into scalar ones that the copy waits for: return 20.2.)
__device__ __forceinline__ char *UniformPointer(char *p)
{
    const uint64_t at = reinterpret_cast<uintptr_t>(p);
    const uint32_t low = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(at)));
    const uint32_t high = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(at >> 32)));
    return reinterpret_cast<char *>(static_cast<uintptr_t>(uint64_t{high} << 32 | low));
}

// A row is read here for the last time and read next by whoever it was copied for: it is loaded past the caches and left in the
// memory-side cache.  dispatch + combine with ordinary loads and stores, and so, us: 4 ranks x 512 x 4096 x top-8 232 -> 217, 8
// x 500 438 -> 417, 4 x 1000 x 7168 x top-4 355 -> 317, top-8 620 -> 587.  (Ordinary loads, kept stores 235; streaming loads,
// ordinary stores 219; streaming both 234.)
// Rows that end within a 128-byte line are copied by ordinary loads and stores (KEPT = false): written through, the parts of a
// line are trips of their own.  Before the rows were kept, kept and now: 4 x 1500 x 7176 x top-6 715, 797 and 723, 8 x 700 x 7176 x
// top-8 945, 1038 and 938, 4 x 1500 x 5000 x top-6 525, 557 and 533, 2 x 4000 x 3000 x top-4 283, 308 and 287 (streaming loads,
// ordinary stores 319).
template <bool KEPT>
__device__ __forceinline__ void CopyVectors(char *dst, const char *src, int vecs, int tid, int threads)
{
    const u32x4 *s = reinterpret_cast<const u32x4 *>(src);
    constexpr int kAhead = 4;       // vectors a lane has in flight
    const __amdgpu_buffer_rsrc_t rows = RowResource(UniformPointer(dst), vecs * 16);
    for (int i = tid; i < vecs; i += kAhead * threads) {
        u32x4 v[kAhead];
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
            const int at = i + u * threads;
            const u32x4 *from = s + (at < vecs ? at : i);
            v[u] = KEPT ? __builtin_nontemporal_load(from) : *from;
        }
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
            const int at = i + u * threads;
            if (at < vecs) {
                __builtin_amdgcn_raw_buffer_store_b128(v[u], rows, at * 16, 0, KEPT ? kAuxAgentScopeKept : 0);
            }
        }
    }
}

__device__ __forceinline__ void CopyBytes(char *dst, const char *src, int64_t bytes, int tid, int threads)
{
    if (((reinterpret_cast<uintptr_t>(dst) | reinterpret_cast<uintptr_t>(src) | static_cast<uintptr_t>(bytes)) & 15u) != 0) {
        for (int64_t i = tid; i < bytes; i += threads) {
            dst[i] = src[i];
        }
    } else if (bytes % 128 == 0) {
        CopyVectors<true>(dst, src, static_cast<int>(bytes / 16), tid, threads);
    } else {
        CopyVectors<false>(dst, src, static_cast<int>(bytes / 16), tid, threads);
    }
}

// Lanes that share a row: a wave for rows of up to 4 KiB, the workgroup for wider ones (a wave would take a 14 KiB row in
// four trips to memory).
constexpr int64_t kWaveRowBytes = 4096;

inline int LanesPerRow(int64_t rowBytes)
{
    return rowBytes <= kWaveRowBytes ? kWave : kThreads;
}

// The rows of destination rank blockIdx.y, G lanes per row: rows group, group + groups of the rank's workgroups, ...  What a
// logical world moves is small, and a launch costs as much as the rows: hence one launch for all ranks, and (PLANNED =
// false) no launch ahead that adds up the segments -- every workgroup does so for itself, two loads and a scan in LDS,
// in less time than a launch takes to begin.  With the sends, the returns and the reduces put together the same way a
// dispatch and a combine of 4 ranks with 128 x 1024 and 2 routes take 143 to 156 us (a plan and a copy launch per rank with a
// workgroup per row: 203 us), of 8 ranks with 1000 x 4096 and 8 routes 760 us (898 us).
template <bool PLANNED, int G>
__global__ __launch_bounds__(kThreads) void ep_drain_rows_kernel(DrainArgs a)
{
    constexpr int kSeg = PLANNED ? 1 : kThreads;
    constexpr int kRows = kThreads / G;
    __shared__ int s_cnt[kSeg];
    __shared__ int s_off[kSeg];
    __shared__ int s_base[kSeg];
    __shared__ int s_tok[kSeg];
    __shared__ int s_part[kThreads];
    const DrainTarget &d = a.target[blockIdx.y];
    const int numSeg = SegmentsOf(a, d);
    const int waveLane = threadIdx.x % kWave;
    const int lane = threadIdx.x % G;
    const int total = PLANNED ? d.planOffsets[numSeg] : SegmentOffsets(a, d, numSeg, s_cnt, s_off, s_base, s_part);
    for (int row = static_cast<int>(blockIdx.x) * kRows + static_cast<int>(threadIdx.x) / G; row < total;
         row += static_cast<int>(gridDim.x) * kRows) {
        // last segment whose exclusive offset is <= row (empty segments share an offset with their successor)
        int seg;
        if (PLANNED) {
            int lo = 0;
            int hi = numSeg - 1;
            while (lo < hi) {
                const int mid = (lo + hi + 1) / 2;
                if (d.planOffsets[mid] <= row) {
                    lo = mid;
                } else {
                    hi = mid - 1;
                }
            }
            seg = lo;
        } else {
            seg = -1;
            for (int first = 0; first < numSeg; first += kWave) {
                seg += __popcll(__ballot(first + waveLane < numSeg && s_off[first + waveLane] <= row));
            }
        }
        int src, key;
        SegmentOf(seg, a.rankSize, d.dstRank, a.localExperts, a.memoryRoute != 0, a.tp, &src, &key);
        int64_t srcRow;
        if (PLANNED) {
            srcRow = a.stage.counts[static_cast<int64_t>(src) * a.stage.countsStride + key] + (row - d.planOffsets[seg]);
        } else {
            srcRow = s_base[seg] + (row - s_off[seg]);
        }
        const char *rows = a.stage.rows + static_cast<int64_t>(src) * a.stage.rowsStride;
        const char *aux = a.stage.aux + static_cast<int64_t>(src) * a.stage.auxStride;
        int32_t word = 0;
        if (lane < 4) {
            word = reinterpret_cast<const int32_t *>(aux)[srcRow * 4 + lane];
        }
        CopyBytes(d.expandXOut + static_cast<int64_t>(row) * a.rowBytes, rows + srcRow * a.rowBytes, a.rowBytes, lane, G);
        if (lane < 4) {
            d.assistOut[static_cast<int64_t>(row) * 4 + lane] = word;
        }
        if (a.scaleBytesPerRow > 0) {
            CopyBytes(d.scalesOut + static_cast<int64_t>(row) * a.scaleBytesPerRow,
                aux + a.stage.scalesOffset + srcRow * a.scaleBytesPerRow, a.scaleBytesPerRow, lane, G);
        }
    }
    if (!PLANNED && blockIdx.x == gridDim.x - 1) {
        // the last workgroup has the fewest rows
        __syncthreads();
        DrainCounts(a, d, numSeg, s_cnt, s_off, s_tok, s_part);
    }
}

struct ReturnRowsArgs {
    const char *expertOut;
    const int32_t *assist;
    const int32_t *counts;
    int numCounts;
    int memoryRoute;
    int maxCountPerEntry;
    int maxRows;
    int64_t rowBytes;
    int rankSize;
    int expertRank;
    int bs;
    int topK;
    uint64_t epoch;
    char *slots;
    int64_t slotsStride;
    uint64_t *meta;
    uint64_t *orderKeys;
    int64_t metaStride;
};

// G lanes per row of the expert rank, for as many rows at once as it holds on average: rows group, group + groups, ...
template <int G>
__global__ __launch_bounds__(kThreads) void ep_return_rows_kernel(ReturnRowsArgs a)
{
    __shared__ int s_first[kThreads];       // MVP route: first row of every source's rows (at most 128 sources)
    __shared__ int s_part[kThreads];
    constexpr int kRows = kThreads / G;
    const int waveLane = threadIdx.x % kWave;
    const int lane = threadIdx.x % G;
    int total;
    if (a.memoryRoute) {
        total = a.counts[a.numCounts - 1];
    } else {
        // rows are grouped by the per-source counts; entries outside [0, max] read as 0
        for (int s = threadIdx.x; s < a.numCounts; s += kThreads) {
            const int c = a.counts[s];
            s_first[s] = (c < 0 || c > a.maxCountPerEntry) ? 0 : c;
        }
        LdsBarrier();
        total = BlockExclusiveScan(s_first, a.numCounts, s_part);
    }
    total = total < 0 ? 0 : (total > a.maxRows ? a.maxRows : total);
    for (int row = static_cast<int>(blockIdx.x) * kRows + static_cast<int>(threadIdx.x) / G; row < total;
         row += static_cast<int>(gridDim.x) * kRows) {
        const int32_t *t = a.assist + static_cast<int64_t>(row) * 4;
        int src = t[0];
        const int token = t[1];
        const int k = t[2];
        if (!a.memoryRoute) {
            src = -1;
            for (int first = 0; first < a.numCounts; first += kWave) {
                src += __popcll(__ballot(first + waveLane < a.numCounts && s_first[first + waveLane] <= row));
            }
        }
        if (src < 0 || src >= a.rankSize || token < 0 || token >= a.bs || k < 0 || k >= a.topK) {
            continue;
        }
        const int64_t slot = static_cast<int64_t>(token) * a.topK + k;
        CopyBytes(a.slots + static_cast<int64_t>(src) * a.slotsStride + slot * a.rowBytes,
            a.expertOut + static_cast<int64_t>(row) * a.rowBytes, a.rowBytes, lane, G);
        if (lane == 0) {
            const int64_t at = static_cast<int64_t>(src) * a.metaStride + slot;
            a.meta[at] = (a.epoch << 32) | static_cast<uint32_t>(slot);
            if (a.orderKeys != nullptr) {
                a.orderKeys[at] = (static_cast<uint64_t>(static_cast<uint32_t>(a.expertRank)) << 32) | static_cast<uint32_t>(row);
            }
        }
    }
}

} // namespace

hipError_t LaunchAugment(const AugmentLaunch &l)
{
    AugmentArgs a {};
    a.ids = l.ids;
    a.n = static_cast<int>(l.bs * (l.sharedNum + l.topK));
    a.topK = static_cast<int>(l.topK);
    a.moeExpertNum = static_cast<int>(l.moeExpertNum);
    a.srcRank = l.srcRank;
    a.sharedNum = l.sharedNum;
    a.sharedRanks = l.sharedRanks;
    a.localExperts = l.localExperts;
    a.keysPerRank = l.keysPerRank;
    a.sharedAtExpertId = l.sharedAtExpertId ? 1 : 0;
    a.keyIdsOut = l.keyIdsOut;
    a.tupleExpertsOut = l.tupleExpertsOut;
    a.routeMask = l.routeMask;
    a.routeMaskOut = l.routeMaskOut;
    const int grid = (a.n + kThreads - 1) / kThreads;
    hipLaunchKernelGGL(ep_augment_kernel, dim3(grid > 0 ? grid : 1), dim3(kThreads), 0, l.stream, a);
    return hipGetLastError();
}

bool DrainPlansItself(int64_t segmentsPerRank, int64_t tokenNumsCount)
{
    return segmentsPerRank <= kThreads && tokenNumsCount <= kThreads;       // their tables in a workgroup's LDS
}

hipError_t LaunchDrain(const DrainLaunch &l)
{
    DrainArgs a {};
    a.stage = l.stage;
    a.rankSize = l.rankSize;
    a.localExperts = l.localExperts;
    a.tp = l.tp;
    a.memoryRoute = l.memoryRoute ? 1 : 0;
    a.rowBytes = l.rowBytes;
    a.scaleBytesPerRow = l.scaleBytesPerRow;
    bool planned = false;
    for (int t = 0; t < l.targets; ++t) {
        a.target[t] = l.target[t];
        const int64_t segments = l.memoryRoute ? static_cast<int64_t>(l.target[t].outLocalExperts) * l.rankSize : l.rankSize;
        planned = planned || !DrainPlansItself(segments, l.target[t].tokenNumsCount);
    }
    // room for the rows a rank receives on average; one that receives more has its workgroups go round again
    const int lanes = LanesPerRow(l.rowBytes);
    const int perGroup = kThreads / lanes;
    const unsigned groups = static_cast<unsigned>((l.routesPerRank + perGroup - 1) / perGroup);
    const dim3 grid(groups > 0 ? groups : 1, static_cast<unsigned>(l.targets));
    if (planned) {
        hipLaunchKernelGGL(ep_drain_plan_kernel, dim3(static_cast<unsigned>(l.targets)), dim3(kThreads), 0, l.stream, a);
        const hipError_t err = hipGetLastError();
        if (err != hipSuccess) {
            return err;
        }
        if (lanes == kWave) {
            hipLaunchKernelGGL((ep_drain_rows_kernel<true, kWave>), grid, dim3(kThreads), 0, l.stream, a);
        } else {
            hipLaunchKernelGGL((ep_drain_rows_kernel<true, kThreads>), grid, dim3(kThreads), 0, l.stream, a);
        }
    } else if (lanes == kWave) {
        hipLaunchKernelGGL((ep_drain_rows_kernel<false, kWave>), grid, dim3(kThreads), 0, l.stream, a);
    } else {
        hipLaunchKernelGGL((ep_drain_rows_kernel<false, kThreads>), grid, dim3(kThreads), 0, l.stream, a);
    }
    return hipGetLastError();
}

hipError_t LaunchReturnRows(const ReturnRowsLaunch &l)
{
    ReturnRowsArgs a {};
    a.expertOut = static_cast<const char *>(l.expertOut);
    a.assist = l.assist;
    a.counts = l.counts;
    a.numCounts = static_cast<int>(l.numCounts);
    a.memoryRoute = l.memoryRoute ? 1 : 0;
    a.maxCountPerEntry = static_cast<int>(l.maxCountPerEntry);
    a.maxRows = static_cast<int>(l.maxRows);
    a.rowBytes = l.rowBytes;
    a.rankSize = l.rankSize;
    a.expertRank = l.expertRank;
    a.bs = static_cast<int>(l.bs);
    a.topK = static_cast<int>(l.topK);
    a.epoch = l.epoch;
    a.slots = l.slots;
    a.slotsStride = l.slotsStride;
    a.meta = l.meta;
    a.orderKeys = l.orderKeys;
    a.metaStride = l.metaStride;
    const int lanes = LanesPerRow(l.rowBytes);
    const int perGroup = kThreads / lanes;
    const unsigned groups = static_cast<unsigned>((l.routesPerRank + perGroup - 1) / perGroup);
    if (lanes == kWave) {
        hipLaunchKernelGGL(ep_return_rows_kernel<kWave>, dim3(groups > 0 ? groups : 1), dim3(kThreads), 0, l.stream, a);
    } else {
        hipLaunchKernelGGL(ep_return_rows_kernel<kThreads>, dim3(groups > 0 ? groups : 1), dim3(kThreads), 0, l.stream, a);
    }
    return hipGetLastError();
}

} // namespace TileXREp
