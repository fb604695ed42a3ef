// scatter: each token row is read once and written to the rows its routes were placed at (gfx950, wave64).
//
// HBM-bound byte movement, no MFMA.  Three kernels share the work:
//   ep_scatter_route_kernel    plain copies of wide rows, 1024 tokens and more, that the memory-side cache cannot hold or that
//                              a consumer beside the launch waits for (ScatterCopiesPerRoute): one workgroup per (token, k,
//                              slice of 512 vectors; 1024 when readiness flags are published for this stream), two 16-byte
//                              loads and two 16-byte stores per lane
//   ep_scatter_vec_kernel      everything else that is 16-byte aligned (quantised payloads, narrow rows, small
//                              batches): G lanes cooperate on one token (a wave for narrow rows, the whole workgroup
//                              for wide ones); a lane keeps V 16-byte vectors of the row in registers, so every load of
//                              the row is in flight before the first store, then writes them to each destination row
//   ep_scatter_generic_kernel  any width and alignment, element by element
// How rows are stored decides where the next kernel finds them: see RowStores (ep_row_quant.hip.h, with the quantisers).
//
#include <hip/hip_runtime.h>

#include "ep_kernel_common.hip.h"
#include "ep_launch.h"
#include "ep_numerics.hip.h"
#include "ep_place.hip.h"
#include "ep_row_quant.hip.h"
#include "ep_tile_publish.h"
#include "tilexr_ep.h"

namespace TileXREp {
namespace {

struct ScatterArgs {
    const void *x;
    const int32_t *rowOf;
    PlaceArgs place;             // place.ids != nullptr: resolve the rows here instead of reading rowOf
    int bs;
    int h;
    int topK;
    const float *staticScale;
    void *out;
    void *scalesOut;
    uint64_t *tileFlags;
    uint32_t *tileCounters;
    int maxTiles;                // tiles of the largest possible row count: the group counters start there
    int tileRows;
    uint64_t epoch;
    const int32_t *totalRowsPtr;
    int colSlices;               // route kernel: workgroups a row is cut into
};

__device__ __forceinline__ int RowOfRoute(const ScatterArgs &a, int route)
{
    return a.place.ids != nullptr ? PlaceRoute(a.place, route) : a.rowOf[route];
}

__device__ __forceinline__ void PublishRow(const ScatterArgs &a, int row, int parts)
{
    TilePublishArgs t;
    t.flags = a.tileFlags;
    t.counters = a.tileCounters;
    t.tileRows = a.tileRows;
    t.maxTiles = a.maxTiles;
    t.totalRows = (a.tileRows > 1 || parts > 1) ? *a.totalRowsPtr : 0;
    t.epoch = a.epoch;
    DeviceTileOps ops;
    PublishLanded(ops, t, row, parts);
}

// Publishes the rows of one token.  Each wave waits for its own stores and the barrier collects the waves.
// WT = true: the rows were written through (kKeep, kPublish) and are then complete for every XCD, with no L2 write-back.
// WT = false: the rows may still sit dirty in this XCD's L2 and one release fence per publishing wave writes them back (slow
// under load; element-granular fallback only).
template <bool WT>
__device__ __forceinline__ void PublishRows(const ScatterArgs &a, const int *pos, int lane, int G)
{
    WaitOwnStores();
    if (G > kWave) {
        __syncthreads();
    }
    if (lane < a.topK) {
        if (!WT) {
            ReleaseRowsToAgent();
        }
        for (int k = lane; k < a.topK; k += G) {
            const int row = pos[k];
            if (row >= 0) {
                PublishRow(a, row, 1);
            }
        }
    }
}

// Plain copy of wide rows, one workgroup per (route, slice of 512 vectors): the workgroup loads its part of the token's
// row and writes it to the destination row of route (token, k).  The workgroups of a token are given block indices that
// the dispatcher places on the same XCD (block b runs on XCD b % 8), so the row comes from HBM once and from that
// XCD's L2 the other topK - 1 times.  Two 16-byte loads then two 16-byte stores per lane is what this memory system
// rewards, whatever the workgroup size: measured on 4096 x 7168 x top-8, 83-85 us with two vectors per lane (128 to
// 448 lanes per workgroup), 92-95 us with three to fourteen, 105-130 us with one; 93 us for "one workgroup writes all
// topK rows", and 132 us when the workgroups of a token are spread over the XCDs.  The rows must stream: kept ones push the
// token rows out of the L2s (dispatch + combine 182 us, 234 us with kKeep).
constexpr int kRouteVecs = 2;
constexpr int kRouteCapWorkgroups = 5;
template <int THREADS, int V, bool WT>
__global__ __launch_bounds__(THREADS) void ep_scatter_route_kernel(ScatterArgs a)
{
    constexpr int kXcds = 8;
    __shared__ int s_row;
    // grid = (8 * slices, topK, groups of eight tokens): the hardware hands out the three indices, so no workgroup
    // starts with a division (this kernel runs at the rate its resident workgroups allow: a prologue of sixty scalar
    // instructions ahead of the first load was a tenth of a workgroup's life).  Workgroups are dealt to the XCDs in
    // linear order, x fastest, and gridDim.x is a multiple of eight: the XCD is blockIdx.x % 8.
    const int token = static_cast<int>(blockIdx.z) * kXcds + static_cast<int>(blockIdx.x % kXcds);
    const int k = blockIdx.y;
    const int colBase = static_cast<int>(blockIdx.x / kXcds) * (V * THREADS);
    if (token >= a.bs) {
        return;
    }
    const int lane = threadIdx.x;
    const int vecs = a.h / 8;
    if (lane == 0) {
        s_row = RowOfRoute(a, token * a.topK + k);
    }
    const u32x4 *src = reinterpret_cast<const u32x4 *>(static_cast<const char *>(a.x) + static_cast<int64_t>(token) * a.h * 2);
    u32x4 v[V];
#pragma unroll
    for (int i = 0; i < V; ++i) {
        const int idx = colBase + i * THREADS + lane;
        v[i] = idx < vecs ? src[idx] : u32x4{0u, 0u, 0u, 0u};
    }
    __syncthreads();
    const int row = __builtin_amdgcn_readfirstlane(s_row);
    if (row < 0) {
        return;
    }
    char *dst = static_cast<char *>(a.out) + static_cast<int64_t>(row) * a.h * 2;
    const __amdgpu_buffer_rsrc_t rsrc = RowResource(dst, vecs * 16);
#pragma unroll
    for (int i = 0; i < V; ++i) {
        const int idx = colBase + i * THREADS + lane;
        if (idx < vecs) {
            RowStore<WT ? RowStores::kPublish : RowStores::kStream>(v[i], dst, rsrc, idx * 16);
        }
    }
    if (WT && a.tileFlags != nullptr) {
        WaitOwnStores();
        __syncthreads();
        if (lane == 0) {
            PublishRow(a, row, a.colSlices);
        }
    }
}

// Publishing launches: one token per group, because a group stays until its own stores have landed.
template <int G, int V, int QMODE, bool BF16, bool E5M2, RowStores S>
__device__ __forceinline__ void ScatterAndPublish(const ScatterArgs &a)
{
    constexpr int kTokens = kThreads / G;
    __shared__ int s_pos[kTokens][kMaxTopK];
    __shared__ float s_red[kTokens][kWavesPerBlock];

    const int tg = threadIdx.x / G;
    const int lane = threadIdx.x % G;
    const int token = blockIdx.x * kTokens + tg;
    const bool tokOk = token < a.bs;
    const int vecs = a.h / 8;

    for (int k = lane; k < a.topK; k += G) {
        s_pos[tg][k] = tokOk ? RowOfRoute(a, token * a.topK + k) : -1;
    }
    const u32x4 *src = reinterpret_cast<const u32x4 *>(static_cast<const char *>(a.x) +
        static_cast<int64_t>(tokOk ? token : 0) * a.h * 2);
    u32x4 v[V];
#pragma unroll
    for (int j = 0; j < V; ++j) {
        const int idx = j * G + lane;
        v[j] = (tokOk && idx < vecs) ? src[idx] : u32x4{0u, 0u, 0u, 0u};
    }
    __syncthreads();
    QuantisedRow<V> out;
    if (QMODE != TILEXR_EP_QUANT_NONE) {
        QuantiseRow<G, V, QMODE, BF16, E5M2>(a, v, s_red[tg], lane, out);
    }
    for (int k = 0; k < a.topK; ++k) {
        // the lanes of a wave share one token, so the row is wave-uniform
        const int row = __builtin_amdgcn_readfirstlane(s_pos[tg][k]);
        if (row >= 0) {
            StoreRow<G, V, QMODE, S, true>(a, row, v, out, lane);
        }
    }
    if (a.tileFlags != nullptr) {
        PublishRows<true>(a, s_pos[tg], lane, G);
    }
}

// Everything else.  Nothing is shared between the waves of a group but the int8 maximum: lane k of every wave works out the
// row of route (token, k) for itself, so no wave waits at a barrier between its loads and its stores (16384 x 7168 bf16
// x top-8 from HBM: 400 us = 5.3 TB/s, 426 us with the rows handed round through LDS).  Bound by memory: with token rows
// that come from HBM the reads and the writes share it.  (One to four tokens in flight per group, a token read ahead of the
// stores, and quantised rows stored sixteen bytes a lane instead of eight made no difference; the token rows read once by
// the routing launch, as for the per-route kernel, cost int8 8192 x 4096 as much as they saved while rows streamed, 108.4
// and 109.0 us, and more since they are kept, 99.8 and 106.9: the read-ahead and the routing want the same memory.)
template <int G, int V, int QMODE, bool BF16, bool E5M2, RowStores S>
__device__ __forceinline__ void ScatterOnly(const ScatterArgs &a)
{
    constexpr int kTokens = kThreads / G;
    __shared__ float s_red[kTokens][kWavesPerBlock];

    const int tg = threadIdx.x / G;
    const int lane = threadIdx.x % G;
    const int waveLane = threadIdx.x % kWave;
    const int token = static_cast<int>(blockIdx.x) * kTokens + tg;
    if (token >= a.bs) {
        return;                     // a group of several waves has the workgroup to itself: nobody is left at a barrier
    }
    const int vecs = a.h / 8;
    int row = -1;
    if (waveLane < a.topK) {
        const int route = token * a.topK + waveLane;
        row = a.place.ids != nullptr ? PlaceRoute(a.place, route, lane < kWave) : a.rowOf[route];
    }
    const u32x4 *src = reinterpret_cast<const u32x4 *>(static_cast<const char *>(a.x) + static_cast<int64_t>(token) * a.h * 2);
    u32x4 v[V];
#pragma unroll
    for (int j = 0; j < V; ++j) {
        const int idx = j * G + lane;
        v[j] = idx < vecs ? src[idx] : u32x4{0u, 0u, 0u, 0u};
    }
    QuantisedRow<V> out;
    if (QMODE != TILEXR_EP_QUANT_NONE) {
        QuantiseRow<G, V, QMODE, BF16, E5M2>(a, v, s_red[tg], lane, out);
    }
    for (int k = 0; k < a.topK; ++k) {
        const int rowOfK = __builtin_amdgcn_readlane(row, k);
        if (rowOfK >= 0) {
            StoreRow<G, V, QMODE, S, false>(a, rowOfK, v, out, lane);
        }
    }
}

template <int G, int V, int QMODE, bool BF16, bool E5M2, bool WT, RowStores S>
__global__ __launch_bounds__(kThreads) void ep_scatter_vec_kernel(ScatterArgs a)
{
    if constexpr (WT) {
        ScatterAndPublish<G, V, QMODE, BF16, E5M2, S>(a);
    } else {
        ScatterOnly<G, V, QMODE, BF16, E5M2, S>(a);
    }
}

// Any row width / alignment: one workgroup per token, element-granular.  Used when h is not a multiple of 8, a
// base pointer is not 16-byte aligned or the row does not fit the register-resident kernel.
template <bool BF16, bool E5M2>
__global__ __launch_bounds__(kThreads) void ep_scatter_generic_kernel(ScatterArgs a, int qmode)
{
    __shared__ int s_pos[kMaxTopK];
    __shared__ float s_red[kWavesPerBlock];
    const int token = blockIdx.x;
    const int tid = threadIdx.x;
    for (int k = tid; k < a.topK; k += kThreads) {
        s_pos[k] = RowOfRoute(a, token * a.topK + k);
    }
    const uint16_t *src = static_cast<const uint16_t *>(a.x) + static_cast<int64_t>(token) * a.h;
    float rowScale = 1.0f;
    float rowScaleInv = qmode == TILEXR_EP_QUANT_STATIC_INT8 ? a.staticScale[0] : 1.0f;
    if (qmode == TILEXR_EP_QUANT_TOKEN_INT8) {
        float amax = 0.0f;
        for (int i = tid; i < a.h; i += kThreads) {
            amax = fmaxf(amax, fabsf(Decode16<BF16>(src[i])));
        }
        amax = GroupMax<kThreads>(amax, s_red, tid);
        rowScale = amax > 0.0f ? __fdiv_rn(amax, 127.0f) : 1.0f;
        rowScaleInv = rowScale > 0.0f ? __fdiv_rn(1.0f, rowScale) : 1.0f;
    }
    __syncthreads();
    const int mxBlocks = (a.h + 31) / 32;
    const int mxScales = (mxBlocks + 1) / 2 * 2;
    const int b128 = (a.h + 127) / 128;
    for (int k = 0; k < a.topK; ++k) {
        const int row = s_pos[k];
        if (row < 0) {
            continue;
        }
        if (qmode == TILEXR_EP_QUANT_NONE) {
            uint16_t *dst = static_cast<uint16_t *>(a.out) + static_cast<int64_t>(row) * a.h;
            for (int i = tid; i < a.h; i += kThreads) {
                dst[i] = src[i];
            }
        } else if (qmode == TILEXR_EP_QUANT_STATIC_INT8 || qmode == TILEXR_EP_QUANT_TOKEN_INT8) {
            int8_t *dst = static_cast<int8_t *>(a.out) + static_cast<int64_t>(row) * a.h;
            for (int i = tid; i < a.h; i += kThreads) {
                dst[i] = static_cast<int8_t>(ClampInt8(__fmul_rn(Decode16<BF16>(src[i]), rowScaleInv)));
            }
            if (qmode == TILEXR_EP_QUANT_TOKEN_INT8 && tid == 0) {
                static_cast<float *>(a.scalesOut)[row] = rowScale;
            }
        } else if (qmode == TILEXR_EP_QUANT_MXFP8) {
            uint8_t *dst = static_cast<uint8_t *>(a.out) + static_cast<int64_t>(row) * a.h;
            uint8_t *sc = static_cast<uint8_t *>(a.scalesOut) + static_cast<int64_t>(row) * mxScales;
            for (int b = tid; b < mxScales; b += kThreads) {
                if (b >= mxBlocks) {
                    sc[b] = 0;
                    continue;
                }
                const int begin = b * 32;
                const int end = min(begin + 32, a.h);
                float amax = 0.0f;
                for (int i = begin; i < end; ++i) {
                    amax = fmaxf(amax, fabsf(Decode16<BF16>(src[i])));
                }
                const int se = MxSharedExponent<E5M2>(amax);
                sc[b] = static_cast<uint8_t>(se + 127);
                for (int i = begin; i < end; ++i) {
                    dst[i] = static_cast<uint8_t>(Fp8Encode<E5M2>(ldexpf(Decode16<BF16>(src[i]), -se)));
                }
            }
        } else {
            uint8_t *dst = static_cast<uint8_t *>(a.out) + static_cast<int64_t>(row) * a.h;
            float *sc = static_cast<float *>(a.scalesOut) + static_cast<int64_t>(row) * b128;
            for (int b = tid; b < b128; b += kThreads) {
                const int begin = b * 128;
                const int end = min(begin + 128, a.h);
                float amax = 0.0f;
                for (int i = begin; i < end; ++i) {
                    amax = fmaxf(amax, fabsf(Decode16<BF16>(src[i])));
                }
                const float scale = amax > 0.0f ? __fdiv_rn(amax, 448.0f) : 1.0f;
                sc[b] = scale;
                for (int i = begin; i < end; ++i) {
                    dst[i] = static_cast<uint8_t>(Fp8Encode<false>(__fdiv_rn(Decode16<BF16>(src[i]), scale)));
                }
            }
        }
    }
    if (a.tileFlags != nullptr) {
        PublishRows<false>(a, s_pos, tid, kThreads);
    }
}

// Whether readiness flags are published: rows are then written through, streaming or kept, and reported once they have landed.
inline bool Publishes(const ScatterArgs &a)
{
    return a.tileFlags != nullptr;
}

// Workgroups per compute unit that the launch without flags is held to, 0 for as many as fit.  Eight workgroups that each
// store a wide row topK times oversubscribe the memory system like those of the per-route kernel.
//   quantised: five.  (Dispatch + combine, us at eight, seven, six, five, four, three, two: 2048 x 7168 x top-8 block fp8 61.5,
//     60.6, 59.9, 59.4, 60.1, 59.8, 61.2, MXFP8 83.4, 83.2, 82.7, 82.0, 81.5, 81.3, 81.5; 8192 x 4096 int8 x top-6 97.2, 96.9,
//     97.3, 97.4, 97.3, 96.5, 104.8.)  That takes rows that store enough: at eight and at five, int8 or block fp8, 2048 x 7168
//     top-8 65.7 -> 62.3, 4096 x 7168 top-4 69.3 -> 67.1, 2048 x 8192 top-4 43.4 -> 42.1, 8192 x 4096 top-6 107.9 -> 105.5; but
//     2048 x 4096 top-2 20.4 and 21.4, 8192 x 2304 top-2 42.3 and 44.6, 16384 x 2304 top-8 181 and 201, 16384 x 3072 top-8 205
//     and 213, 16384 x 4096 top-5 181 and 187, 2048 x 12288 top-2 46.8 and 48.6.  (Rows a wave holds: no difference.)
//   copies, dispatch + combine at eight, four, three and two: 2200 x 7168 x top-8 95.9, 93.4, 92.7, 91.2; 3000 x 5120 93.9, 92.2,
//     90.6, 89.6; 16384 x 7168 768.5, 763.5, 768.9, 760.2; up to 512 vectors 16384 x 4096 x top-8 441.6, 431.4, 437.0, 466.7; 6000
//     x 2560 95.0, 91.5, 91.0, -; 10000 x 2056 160, 167, -, 188.  1000 tokens and fewer: no difference.
//     Where the rows are known and the token rows come from memory, fewer workgroups have too few of those under way: MVP route
//     30000 x 3072 x top-5 404, 438, 467, 503; 16384 x 7168 x top-8 740, 745, 752, 764; 24000 x 5120 x top-6 617, 607, 603, 639;
//     10000 x 7168 x top-8 444, 446, 450, 454; memory route 16384 x 7168 x top-4 411, 413, 414, 413.
//     Workgroups that resolve their rows themselves (three dependent loads ahead of the first store) have to store enough to be
//     worth fewer beside them.  Vectors stored, us at eight and four: 16384 x 2560 x top-3 960, 113.7 and 143.4; 24000 x 2560 x
//     top-2 640, 135.8 and 179.0; 12000 x 3072 x top-4 1536, 127.6 and 137.2; 24000 x 3072 x top-5 1920, 318.7 and 344.2; 16384
//     x 4096 x top-4 2048, 242.8 and 246.5; 6000 x 2560 x top-8 2560, 103.9 and 106.2; 24000 x 3072 x top-8 3072, 492.7 and
//     499.4; 4500 x 3584 x top-8 3584, 110.3 and 106.5; 5000 x 4096 x top-8 4096, 137.1 and 132.3.  Wider rows at eight, four
//     and two: 5558 x 5120 x top-3 1920, 79.4, 81.6, 94.8; 9000 x 4608 x top-4 2304, 148.2, 148.6, 162.7; 19884 x 5120 x top-5
//     3200, 437.6, 431.4, 465.9; 24000 x 5120 x top-6 3840, 613.8, 606.6, 632.9; 4200 x 4608 x top-8 4608, 127.5, 123.4, 126.5;
//     11304 x 5120 x top-8 5120, 387.2, 380.1, 384.9; 3000 x 7168 x top-6 5376, 110.6, 105.9, 105.4.
template <int G, int QMODE>
int CapWorkgroups(const ScatterArgs &a)
{
    const int vecs = a.h / 8;
    if (QMODE != TILEXR_EP_QUANT_NONE) {
        return vecs >= 2 * kThreads && a.topK >= 4 && vecs * a.topK >= 12 * kThreads ? 5 : 0;
    }
    if (G < kThreads || vecs < 320) {
        return 0;
    }
    const int stored = vecs * a.topK;
    const bool resolves = a.place.ids != nullptr;
    const bool cachedTokens = static_cast<int64_t>(a.bs) * a.h * 2 <= kMemorySideCacheBytes / 2;
    if (resolves ? stored < 14 * kThreads : !cachedTokens) {
        return 0;
    }
    return vecs > 2 * kThreads && (!resolves || (stored >= 18 * kThreads && (cachedTokens || a.topK > 4))) ? 2 : 4;
}

template <int QMODE>
int64_t RowBytes(const ScatterArgs &a)
{
    return QMODE == TILEXR_EP_QUANT_NONE ? int64_t{2} * a.h : a.h;
}

// Whether the rows are left in the memory-side cache.  They are where this library's combine can take them as they are.  A
// payload that only an expert stage decodes streams (dispatch + combine of other rows with nothing in between, streaming and
// kept: MXFP8 2048 x 7168 88.9 and 91.2 us, 4096 x 7168 155 and 168, int8 on the MVP route 4000 x 2048 49.0 and 51.4).
//   With an expert stage in between, dispatch + stage + combine in us, rows streamed (by the launches that suit that) and kept.
// Two matrix products through 2048 columns into another buffer: 1000 x 7168 x top-8 437 -> 426, 1500 x 7168 689 -> 684, 2200
// x 7168 1050 -> 1046, 16384 x 7168 6813 -> 6792, 4000 x 4096 950 -> 944, 16384 x 2048 2002 -> 1976; int8 1000 x 7168 533 ->
// 492, 8192 x 4096 x top-6 1816 -> 1802, block fp8 16384 x 2048 2501 -> 2498.  One elementwise pass over the rows where they
// are: 87.4 -> 78.2, 119.6 -> 114.1, 173.6 -> 163.9, 1392 and 1392, 179 -> 173, 398 -> 390.  A stage that is bound by memory
// and writes elsewhere pays for the write-back of the kept rows itself: the same pass into another buffer 88.5 and 88.6,
// 122.1 and 129.1, 182.2 and 189.0, 1379 and 1384, 187.6 and 196.6, 402 and 408; products through 256 columns 185.4 and
// 184.2, 244 and 251, 312 and 323, 1984 and 1990, 294 and 305, 633 and 648.  Rows are kept all the same: what stands between
// dispatch and combine at these sizes are products.
//   Block fp8 rows beyond twice that cache stream too (16384 x 7168 x top-6 378 and 388, 8192 x 8192 x top-8 274 -> 269), int8
// and plain ones are kept at any size (16384 x 7168 x top-8 int8 468.5 -> 466.2, plain 775.5 -> 770.3).  Rows that end within
// a 128-byte line (ordinary stores unless they are published) want a launch worth it: 1000 columns, streaming and written through,
// 1501 tokens x top-6 19.1 and 19.6, 4000 x top-6 31.2 and 31.4, 4000 x top-8 39.4 -> 37.1.
template <int QMODE>
bool KeepsRows(const ScatterArgs &a)
{
    const int64_t rowBytes = RowBytes<QMODE>(a);
    const int64_t bytes = static_cast<int64_t>(a.bs) * a.topK * rowBytes;
    if (QMODE == TILEXR_EP_QUANT_FP8_BLOCK128 && bytes > 2 * kMemorySideCacheBytes) {
        return false;
    }
    return Publishes(a) || rowBytes % 128 == 0 || bytes >= (int64_t{32} << 20);
}

template <int G, int V, int QMODE, bool BF16, bool E5M2, RowStores S>
void LaunchVecStoring(const ScatterArgs &a, hipStream_t stream)
{
    constexpr int kTokens = kThreads / G;
    const dim3 groups((a.bs + kTokens - 1) / kTokens);
    if constexpr (S == RowStores::kKeep || S == RowStores::kPublish) {
        if (Publishes(a)) {
            hipLaunchKernelGGL((ep_scatter_vec_kernel<G, V, QMODE, BF16, E5M2, true, S>), groups, dim3(kThreads), 0, stream, a);
            return;
        }
    }
    if constexpr (S != RowStores::kPublish) {
        hipLaunchKernelGGL((ep_scatter_vec_kernel<G, V, QMODE, BF16, E5M2, false, S>), groups, dim3(kThreads),
            CapLdsBytes(CapWorkgroups<G, QMODE>(a)), stream, a);
    }
}

template <int G, int V, int QMODE, bool BF16, bool E5M2>
void LaunchVec(const ScatterLaunch &l, const ScatterArgs &a)
{
    constexpr bool kCombineTakes = QMODE == TILEXR_EP_QUANT_NONE || QMODE == TILEXR_EP_QUANT_TOKEN_INT8 ||
        QMODE == TILEXR_EP_QUANT_FP8_BLOCK128;
    if constexpr (kCombineTakes) {
        if (l.combineTakesRows && KeepsRows<QMODE>(a)) {
            if (Publishes(a) || RowBytes<QMODE>(a) % 128 == 0) {
                LaunchVecStoring<G, V, QMODE, BF16, E5M2, RowStores::kKeep>(a, l.stream);
            } else {
                LaunchVecStoring<G, V, QMODE, BF16, E5M2, RowStores::kOrdinary>(a, l.stream);
            }
            return;
        }
    }
    if (Publishes(a)) {
        LaunchVecStoring<G, V, QMODE, BF16, E5M2, RowStores::kPublish>(a, l.stream);
    } else {
        LaunchVecStoring<G, V, QMODE, BF16, E5M2, RowStores::kStream>(a, l.stream);
    }
}

template <int G, int V>
void LaunchByMode(const ScatterLaunch &l, const ScatterArgs &a)
{
    switch (l.quantMode) {
        case TILEXR_EP_QUANT_NONE:
            if (G == kThreads && ScatterCopiesPerRoute(l)) {
                const dim3 blocks(static_cast<unsigned>(8 * a.colSlices), static_cast<unsigned>(a.topK),
                    static_cast<unsigned>((a.bs + 7) / 8));
                if (l.kernelNameOut != nullptr) {
                    *l.kernelNameOut = "ep_scatter_route_kernel";
                }
                if (Publishes(a) && a.colSlices > 1 && !l.consumerBeside) {
                    // A publishing workgroup stays until its stores have landed and then counts its part of the row
                    // towards the tile: worth doing once per row rather than once per half row, so rows wider than 512
                    // vectors get workgroups of 512 lanes (4096 x 7168 x top-8: 82.2 instead of 84.7 us; without
                    // flags the narrower workgroups are the faster ones, 81.9 against 82.5 us).  Not when a consumer
                    // is expected beside this launch: its waiting workgroups leave room for the narrower ones only
                    // (dispatch + combine on two streams: 272 us with the wide ones, 244 us with the narrow ones).
                    constexpr int kWide = 2 * kThreads;
                    ScatterArgs wide = a;
                    wide.colSlices = (a.h / 8 + kRouteVecs * kWide - 1) / (kRouteVecs * kWide);
                    const dim3 wideBlocks(static_cast<unsigned>(8 * wide.colSlices), static_cast<unsigned>(a.topK),
                        static_cast<unsigned>((a.bs + 7) / 8));
                    hipLaunchKernelGGL((ep_scatter_route_kernel<kWide, kRouteVecs, true>), wideBlocks, dim3(kWide), 0,
                        l.stream, wide);
                } else if (Publishes(a)) {
                    hipLaunchKernelGGL((ep_scatter_route_kernel<kThreads, kRouteVecs, true>), blocks, dim3(kThreads), 0,
                        l.stream, a);
                } else {
                    // Workgroups that only look their row up in the row map are short-lived, and eight of them per
                    // compute unit keep more stores in flight than this memory system digests (dispatch + combine, us at
                    // eight, seven, six, five, four, three, two: 1500 x 14336 x top-8 137.5, 136.0, 134.3, 132.9, 134.3,
                    // 144.3, 168.6; 2000 x 12288 158.5, 157.8, 157.5, 156.4, 148.6, 153.4, 171.8).
                    // Workgroups that resolve their row themselves (three dependent loads) are slow enough as they are.
                    const unsigned capLds = a.place.ids == nullptr ? CapLdsBytes(kRouteCapWorkgroups) : 0u;
                    hipLaunchKernelGGL((ep_scatter_route_kernel<kThreads, kRouteVecs, false>), blocks, dim3(kThreads), capLds,
                        l.stream, a);
                }
            } else {
                LaunchVec<G, V, TILEXR_EP_QUANT_NONE, true, false>(l, a);
            }
            break;
        case TILEXR_EP_QUANT_STATIC_INT8:
            LaunchVec<G, V, TILEXR_EP_QUANT_STATIC_INT8, false, false>(l, a);
            break;
        case TILEXR_EP_QUANT_TOKEN_INT8:
            if (l.inputBf16) {
                LaunchVec<G, V, TILEXR_EP_QUANT_TOKEN_INT8, true, false>(l, a);
            } else {
                LaunchVec<G, V, TILEXR_EP_QUANT_TOKEN_INT8, false, false>(l, a);
            }
            break;
        case TILEXR_EP_QUANT_MXFP8:
            if (l.inputBf16) {
                if (l.fp8E5m2) {
                    LaunchVec<G, V, TILEXR_EP_QUANT_MXFP8, true, true>(l, a);
                } else {
                    LaunchVec<G, V, TILEXR_EP_QUANT_MXFP8, true, false>(l, a);
                }
            } else {
                if (l.fp8E5m2) {
                    LaunchVec<G, V, TILEXR_EP_QUANT_MXFP8, false, true>(l, a);
                } else {
                    LaunchVec<G, V, TILEXR_EP_QUANT_MXFP8, false, false>(l, a);
                }
            }
            break;
        default:
            if (l.inputBf16) {
                LaunchVec<G, V, TILEXR_EP_QUANT_FP8_BLOCK128, true, false>(l, a);
            } else {
                LaunchVec<G, V, TILEXR_EP_QUANT_FP8_BLOCK128, false, false>(l, a);
            }
            break;
    }
}

} // namespace

// The per-route kernel's rows have to stream, the per-token kernel's are kept: dispatch + combine, per route and per token
// (two or four workgroups to a compute unit), us: 235 MB of rows (2048 x 7168 x top-8) 93.9 and 85.0, 315 MB 128.1 and
// 122.8, 367 MB 144.8 and 145.4, 470 MB 182.2 and 187.8, 688 MB 273.0 and 274.4; 4096 columns, 328 MB 132.1 and 128.3, 393 MB
// 155.8 and 157.1, 786 MB 310.7 and 316.2.  So it takes what the memory-side cache cannot hold, and of that what has token
// rows it can: beyond 104 MiB of them reading them ahead no longer pays (117 MB 379.8 and 375.6, 123 MB 405.6 and 392.4, 134
// MB 470 and 428); publishing, where the per-token kernel waits for its stores topK at a time, beyond 128 MiB (117 MB 378.4
// and 379.9, 123 MB 395.3 and 398.0).  Rows wider than one of its publishing workgroups (1024 vectors) are no exception (published
// on one stream, 1024 x 12288 x top-4 52.5 and 45.2, 1024 x 16384 x top-8 107.6 and 94.9, 4096 x 16384 x top-2 150.5 and 133.4).  A
// consumer that runs beside the launch gets its rows one by one as they land, not a token's topK at a time.
bool ScatterCopiesPerRoute(const ScatterLaunch &l)
{
    const int64_t vecs = l.h / 8;
    const int64_t tokenBytes = l.bs * l.h * 2;
    const bool publishes = l.tileFlags != nullptr;
    return l.quantMode == TILEXR_EP_QUANT_NONE && l.h % 8 == 0 && Aligned16(l.x) && Aligned16(l.out) && vecs > 4 * kWave &&
        vecs <= 8 * kThreads && l.topK > 1 && l.bs >= 1024 && tokenBytes <= (publishes ? int64_t{128} << 20 : int64_t{104} << 20) &&
        (l.consumerBeside || tokenBytes * l.topK > (int64_t{320} << 20)) && (l.bs + 7) / 8 <= 65535 && l.topK <= 65535;
}

bool ScatterCopiesPerRoute(const void *x, const void *out, int64_t bs, int64_t h, int64_t topK, int quantMode)
{
    ScatterLaunch l {};
    l.x = x;
    l.out = const_cast<void *>(out);       // only its alignment is looked at
    l.bs = bs;
    l.h = h;
    l.topK = topK;
    l.quantMode = quantMode;
    return ScatterCopiesPerRoute(l);
}

hipError_t LaunchScatter(const ScatterLaunch &l)
{
    ScatterArgs a {};
    a.x = l.x;
    a.rowOf = l.rowOf;
    if (l.fusedPlace != nullptr) {
        a.place = MakePlaceArgs(*l.fusedPlace);
    }
    a.bs = static_cast<int>(l.bs);
    a.h = static_cast<int>(l.h);
    a.topK = static_cast<int>(l.topK);
    a.staticScale = l.staticScale;
    a.out = l.out;
    a.scalesOut = l.scalesOut;
    a.tileFlags = l.tileFlags;
    a.tileCounters = l.tileCounters;
    a.tileRows = static_cast<int>(l.tileRows);
    a.maxTiles = l.tileRows > 0 ? static_cast<int>((l.bs * l.topK + l.tileRows - 1) / l.tileRows) : 0;
    a.epoch = l.epoch;
    a.totalRowsPtr = l.totalRowsPtr;
    a.colSlices = static_cast<int>((l.h / 8 + kRouteVecs * kThreads - 1) / (kRouteVecs * kThreads));
    const int64_t vecs = l.h / 8;
    const bool vecOk = l.h % 8 == 0 && Aligned16(l.x) && vecs <= 8 * kThreads &&
        (l.quantMode == TILEXR_EP_QUANT_NONE ? Aligned16(l.out) : Aligned8(l.out));
    if (l.kernelNameOut != nullptr) {
        *l.kernelNameOut = vecOk ? "ep_scatter_vec_kernel" : "ep_scatter_generic_kernel";
    }
    if (vecOk) {
        // narrow rows: a wave per token (four tokens per workgroup); wide rows: the workgroup per token
        if (vecs <= 2 * kWave) {
            LaunchByMode<kWave, 2>(l, a);
        } else if (vecs <= 4 * kWave) {
            LaunchByMode<kWave, 4>(l, a);
        } else if (vecs <= 2 * kThreads) {
            LaunchByMode<kThreads, 2>(l, a);
        } else if (vecs <= 4 * kThreads) {
            LaunchByMode<kThreads, 4>(l, a);
        } else {
            LaunchByMode<kThreads, 8>(l, a);
        }
    } else {
        const dim3 grid(static_cast<unsigned>(l.bs));
        if (l.inputBf16) {
            if (l.fp8E5m2) {
                hipLaunchKernelGGL((ep_scatter_generic_kernel<true, true>), grid, dim3(kThreads), 0, l.stream, a, l.quantMode);
            } else {
                hipLaunchKernelGGL((ep_scatter_generic_kernel<true, false>), grid, dim3(kThreads), 0, l.stream, a, l.quantMode);
            }
        } else {
            if (l.fp8E5m2) {
                hipLaunchKernelGGL((ep_scatter_generic_kernel<false, true>), grid, dim3(kThreads), 0, l.stream, a, l.quantMode);
            } else {
                hipLaunchKernelGGL((ep_scatter_generic_kernel<false, false>), grid, dim3(kThreads), 0, l.stream, a, l.quantMode);
            }
        }
    }
    return hipGetLastError();
}

} // namespace TileXREp
