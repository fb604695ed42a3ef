// Launch geometry shared by the EP kernels (gfx950: 64-lane wavefronts, 256-thread workgroups).
#ifndef TILEXR_AMD_EP_KERNEL_COMMON_HIP_H
#define TILEXR_AMD_EP_KERNEL_COMMON_HIP_H

#include <cstdint>

#if defined(__HIPCC__)
#include <hip/hip_runtime.h>

#include "tilexr_ep_publish.hip.h"
#endif

namespace TileXREp {

constexpr int kThreads = 256;
constexpr int kWave = 64;
constexpr int kWavesPerBlock = kThreads / kWave;

inline bool Aligned16(const void *p)
{
    return (reinterpret_cast<uintptr_t>(p) & 15u) == 0;
}

inline bool Aligned8(const void *p)
{
    return (reinterpret_cast<uintptr_t>(p) & 7u) == 0;
}

#if defined(__HIPCC__)
// Workgroup barrier that orders LDS traffic only: global stores still in flight are not waited for (a plain
// __syncthreads() drains them first, which costs a full store round trip when nobody in the workgroup reads them).
__device__ __forceinline__ void LdsBarrier()
{
#if defined(__HIP_DEVICE_COMPILE__)
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
#endif
}

// Cache-policy operand of raw buffer loads and stores on gfx950.  Each XCD has its own L2 and the L2s are not coherent
// with one another: an ordinary store may sit dirty in the writer's L2 until a release fence writes the whole L2 back
// (measured: a scatter of 32 768 rows with one such fence per row takes 965 us instead of 90 us), and an ordinary load
// may hit a stale line until an acquire fence invalidates the reader's L2 (measured: 240 us instead of 90 us for the
// reduce with one fence per token).  An agent-scope (sc1) store is written through to memory and is complete, for
// every XCD, when the wave's vmcnt reaches zero; an agent-scope load is served from memory.  Rows published through
// readiness flags therefore move with sc1 accesses and need no cache maintenance at all.  The streaming hint (nt) is
// for rows whose token row several workgroups share: without it the written-through rows are also allocated in L2 and push
// out the input rows those workgroups find there (measured: 132 us instead of 93 us for the per-route scatter).
constexpr int kAuxAgentScope = 16 | 2;      // sc1 nt
constexpr int kAuxNonTemporal = 2;          // nt
constexpr int kAuxAgentScopeKept = 16;      // sc1 alone: for rows one workgroup copies to all their places (RowStores in
                                            // ep_scatter.hip) and for small tables a later kernel reads again (with nt on
                                            // the loads of the count kernel's histograms the scatter that resolves rows
                                            // from the same table afterwards ran 10 us slower: 92 instead of 82 us)
constexpr unsigned kRawBufferWord3 = 0x00020000u;

// Unused dynamic LDS that holds a kernel to so many workgroups per compute unit, 0 for as many as fit.  A compute unit hands its
// 160 KiB out in blocks of 1280 bytes (workgroups of a fixed wait, counted by the rounds a launch takes: 53 760 bytes three, one
// block more two; 40 960 four, 40 bytes more three), so a size takes what the kernel's own tables come to into account.
constexpr unsigned kLdsBlockBytes = 1280;
constexpr unsigned kLdsBlocks = 128;
constexpr unsigned kOwnLdsBytes = 1024;         // of the kernels that are capped, at most

constexpr unsigned CapLdsBytes(int workgroups)
{
    return workgroups == 2 ? 56u * 1024u : workgroups == 4 ? 39u * 1024u : workgroups == 5 ? 27u * 1024u : 0u;
}

constexpr bool CapHolds(int workgroups)
{
    const unsigned least = (CapLdsBytes(workgroups) + kLdsBlockBytes - 1) / kLdsBlockBytes;
    const unsigned most = (CapLdsBytes(workgroups) + kOwnLdsBytes + kLdsBlockBytes - 1) / kLdsBlockBytes;
    return kLdsBlocks / least == static_cast<unsigned>(workgroups) && kLdsBlocks / most == static_cast<unsigned>(workgroups);
}
static_assert(CapHolds(2) && CapHolds(4) && CapHolds(5), "as many workgroups fit as the cap says");

// The cache between the L2s and memory, one for the device.
constexpr int64_t kMemorySideCacheBytes = int64_t{256} << 20;

// Workgroup b of a launch runs on XCD b % kXcdCount.  Units (token x part) placed by XCD: unit u belongs to token
// (u / 8 / parts) * 8 + u % 8, part (u / 8) % parts, so that all parts of a token run on XCD token % 8; the tokens are
// padded to a multiple of eight.
constexpr int kXcdCount = 8;
__host__ __device__ inline int XcdPlacedUnits(int tokens, int parts)
{
    return (tokens + kXcdCount - 1) / kXcdCount * kXcdCount * parts;
}

// Sums, maxima and scans of a wave, all 64 lanes active, in the registers' own cross-lane moves: four moves within rows of
// sixteen lanes, then four scalar reads, where shuffles are six dependent trips through LDS of about a hundred clocks each.
constexpr int kDppQuadSwap1 = 0xb1;         // lanes 1 0 3 2 of a quad
constexpr int kDppQuadSwap2 = 0x4e;         // lanes 2 3 0 1
constexpr int kDppHalfRowMirror = 0x141;    // lane i of eight takes lane 7 - i
constexpr int kDppRowMirror = 0x140;        // lane i of sixteen takes lane 15 - i
constexpr int kDppRowShift = 0x110;         // + n: lane i of sixteen takes lane i - n, zero below
constexpr int kDppRowBroadcast15 = 0x142;   // rows one and three take the last lane of the row before them
constexpr int kDppRowBroadcast31 = 0x143;   // rows two and three take lane 31

template <int CTRL, int ROWS = 0xf>
__device__ __forceinline__ int DppMove(int v)
{
    return __builtin_amdgcn_update_dpp(0, v, CTRL, ROWS, 0xf, true);
}

__device__ __forceinline__ int WaveSum(int v)
{
    v += DppMove<kDppQuadSwap1>(v);
    v += DppMove<kDppQuadSwap2>(v);
    v += DppMove<kDppHalfRowMirror>(v);
    v += DppMove<kDppRowMirror>(v);
    return __builtin_amdgcn_readlane(v, 0) + __builtin_amdgcn_readlane(v, 16) + __builtin_amdgcn_readlane(v, 32) +
        __builtin_amdgcn_readlane(v, 48);
}

// Largest of the lane's row of sixteen.
__device__ __forceinline__ float RowMax(float v)
{
    v = fmaxf(v, __int_as_float(DppMove<kDppQuadSwap1>(__float_as_int(v))));
    v = fmaxf(v, __int_as_float(DppMove<kDppQuadSwap2>(__float_as_int(v))));
    v = fmaxf(v, __int_as_float(DppMove<kDppHalfRowMirror>(__float_as_int(v))));
    return fmaxf(v, __int_as_float(DppMove<kDppRowMirror>(__float_as_int(v))));
}

__device__ __forceinline__ float WaveMax(float v)
{
    const int m = __float_as_int(RowMax(v));
    return fmaxf(fmaxf(__int_as_float(__builtin_amdgcn_readlane(m, 0)), __int_as_float(__builtin_amdgcn_readlane(m, 16))),
        fmaxf(__int_as_float(__builtin_amdgcn_readlane(m, 32)), __int_as_float(__builtin_amdgcn_readlane(m, 48))));
}

__device__ __forceinline__ int WaveInclusiveSum(int v)
{
    v += DppMove<kDppRowShift + 1>(v);
    v += DppMove<kDppRowShift + 2>(v);
    v += DppMove<kDppRowShift + 4>(v);
    v += DppMove<kDppRowShift + 8>(v);
    v += DppMove<kDppRowBroadcast15, 0xa>(v);
    v += DppMove<kDppRowBroadcast31, 0xc>(v);
    return v;
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t RowResource(const void *row, int bytes)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(row), 0, bytes, kRawBufferWord3);
}

// Waits until every store this wave has issued is complete (vmcnt, expcnt and lgkmcnt all zero).
__device__ __forceinline__ void WaitOwnStores()
{
    TileXREpWaitOwnStores();
}

// Release / acquire at agent scope for rows that move with ordinary stores and loads: the installed header
// tilexr_ep_publish.hip.h holds the one implementation (and the ordering rule), so that a producer or consumer outside
// the library runs the same instructions as the kernels here.  Both spell out the wait that follows the cache
// operation: in the code hipcc 7.2 generates for the fence alone, the L2 write-back of a release is followed directly
// by the next store (the wait the fence asks for does not survive the compiler's wait-count pass), and a readiness word
// then reaches memory ahead of the rows now and then: one row in a few thousand was read before it was there.  The
// acquire side gets the same treatment, and every wave that reads rows with ordinary loads issues its own.
__device__ __forceinline__ void ReleaseRowsToAgent()
{
    TileXREpReleaseRowsToAgent();
}

__device__ __forceinline__ void AcquireRowsFromAgent()
{
    TileXREpAcquireRowsFromAgent();
}

// Device side of ep_tile_publish.h: relaxed agent-scope atomics.  The caller has made the row complete in memory
// first, so has every earlier counter of the tile, and the atomics on one counter are totally ordered: when the last
// one returns, all rows of the tile are in memory.
struct DeviceTileOps {
    __device__ __forceinline__ uint32_t FetchAdd(uint32_t *p)
    {
        return __hip_atomic_fetch_add(p, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __device__ __forceinline__ void Store(uint32_t *p, uint32_t v)
    {
        __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __device__ __forceinline__ void Store(uint64_t *p, uint64_t v)
    {
        __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
};
#endif

} // namespace TileXREp

#endif // TILEXR_AMD_EP_KERNEL_COMMON_HIP_H
