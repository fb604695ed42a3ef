// Quantisers of token rows and the stores of rows, for the kernels that hold a row in registers (gfx950, wave64): the scatter
// and the decode-sized dispatch.  `Args` names the row's width (h), the outputs (out, scalesOut) and the static scale.
//
//   QMODE 0  byte copy             (reference: src/ep/kernels/tilexr_ep_dispatch_helpers.h:104-112)
//   QMODE 1  static int8           (reference: tilexr_ep_dispatch_helpers.h:114-136)
//   QMODE 2  per-token int8        (reference: tilexr_ep_dispatch_helpers.h:153-191; BF16 decode has no counterpart)
//   QMODE 4  MXFP8, 32-wide blocks (reference: tests/ep/demo/mxfp8_golden.h:116-152)
//   QMODE 5  fp8 e4m3, fp32 scale per 128 columns (no reference counterpart)
#ifndef TILEXR_AMD_EP_ROW_QUANT_HIP_H
#define TILEXR_AMD_EP_ROW_QUANT_HIP_H

#include <hip/hip_runtime.h>

#include "ep_kernel_common.hip.h"
#include "ep_numerics.hip.h"
#include "tilexr_ep.h"

namespace TileXREp {
namespace {

template <int G>
__device__ __forceinline__ float GroupMax(float v, float *red, int lane)
{
    v = WaveMax(v);
    if (G > kWave) {
        if ((lane & (kWave - 1)) == 0) {
            red[lane / kWave] = v;
        }
        LdsBarrier();
        v = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    }
    return v;
}

// Row stores of the register-resident kernels.  A streaming store goes past the L2 and past the 256 MiB memory-side cache:
// whoever reads the row next fetches it from memory, row by row at unrelated places.  One that is written through without the
// streaming hint leaves the row in that cache, and it is the cheaper store as well, since what the cache takes need not reach
// memory within the launch.  Dispatch + combine of the rows as they are, us, streaming and kept, six sets of
// buffers in turn: 1000 x 7168 x top-8 52.4 -> 45.3, 600 tokens 34.9 -> 31.1, 3000 x 2048 48.3 -> 41.3; int8 8192 x 4096 x
// top-6 108.4 -> 100.2 (its scatter 49.9 -> 42.5), 4096 x 7168 x top-8 127.0 -> 109.0; block fp8 16384 x 2048 under a
// capacity 98.4 -> 92.0 (scatter 48.9 -> 39.0, reduce 40.7 -> 44.4: it waits for rows that leave the cache).  Ordinary
// stores (dirty in the L2 until the launch ends) come in between: 46.0, 101.8, 93.1 for three of those.
// Rows that end within a 128-byte line are the exception: nearly every store of a wave begins and ends within a line, and written
// through each half is a trip of its own, where the L2 puts ordinary ones together.  Streaming (by the launches that suit that),
// kept and ordinary: 9000 x 7176 x top-6 369, 382 and 354, under a capacity 366, 389 and 341, on the MVP route 332, 370 and 334;
// 1200 x 7176 x top-8 67.6, 68.0 and 65.6; 4000 x 6408 x top-6 156.9, 146.4 and 141.3; 4500 x 2008 x top-8 79.2, 75.0 and 70.7; int8
// 9000 x 2064 x top-6 91.9, 79.0 and 77.0; but 2500 x 7176 x top-4 73.7, 75.9 and 75.3.
enum class RowStores {
    kStream,        // non-temporal
    kKeep,          // written through (sc1) and kept
    kPublish,       // written through and streaming (sc1 nt)
    kOrdinary,      // dirty in the L2 until the launch ends
};

template <RowStores S>
constexpr int kRowAux = S == RowStores::kKeep ? kAuxAgentScopeKept : S == RowStores::kPublish ? kAuxAgentScope : 0;

template <RowStores S>
__device__ __forceinline__ void RowStore(const u32x4 &v, char *rowBase, __amdgpu_buffer_rsrc_t rsrc, int byteOffset)
{
    if (S == RowStores::kStream) {
        __builtin_nontemporal_store(v, reinterpret_cast<u32x4 *>(rowBase + byteOffset));
    } else {
        __builtin_amdgcn_raw_buffer_store_b128(v, rsrc, byteOffset, 0, kRowAux<S>);
    }
}

template <RowStores S>
__device__ __forceinline__ void RowStore(const u32x2 &v, char *rowBase, __amdgpu_buffer_rsrc_t rsrc, int byteOffset)
{
    if (S == RowStores::kStream) {
        __builtin_nontemporal_store(v, reinterpret_cast<u32x2 *>(rowBase + byteOffset));
    } else {
        __builtin_amdgcn_raw_buffer_store_b64(v, rsrc, byteOffset, 0, kRowAux<S>);
    }
}

template <bool WT, typename T>
__device__ __forceinline__ void ScalarStore(T *p, T v)
{
    if (WT) {
        __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    } else {
        *p = v;
    }
}

// The low bytes of four words, first one lowest.
__device__ __forceinline__ uint32_t PackBytes(uint32_t a, uint32_t b, uint32_t c, uint32_t d)
{
    constexpr uint32_t kLowBytes = 0x0c0c0400u;         // bytes 0 of the second and of the first operand, zeros
    constexpr uint32_t kLowHalves = 0x05040100u;
    return __builtin_amdgcn_perm(__builtin_amdgcn_perm(d, c, kLowBytes), __builtin_amdgcn_perm(b, a, kLowBytes), kLowHalves);
}

// A row's payload and scales, as the lanes of its group hold them: eight bytes per 16-byte vector.
template <int V>
struct QuantisedRow {
    u32x2 q[V];
    float blockScale[V];        // fp8: scale of the vector's 128 columns
    int sharedExp[V];           // MXFP8: exponent of the vector's 32 columns
    float rowScale;             // int8
};

template <int G, int V, int QMODE, bool BF16, bool E5M2, typename Args>
__device__ __forceinline__ void QuantiseRow(const Args &a, const u32x4 (&v)[V], float *red, int lane, QuantisedRow<V> &out)
{
    out.rowScale = 1.0f;
    // per-row / per-block scale, then 8 output bytes per input vector
    float rowScaleInv = 1.0f;
    if constexpr (QMODE == TILEXR_EP_QUANT_STATIC_INT8) {
        rowScaleInv = a.staticScale[0];
    }
    if (QMODE == TILEXR_EP_QUANT_TOKEN_INT8) {
        float amax = 0.0f;
#pragma unroll
        for (int j = 0; j < V; ++j) {
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                amax = fmaxf(amax, fabsf(Decode16<BF16>(v[j][w] & 0xffffu)));
                amax = fmaxf(amax, fabsf(Decode16<BF16>(v[j][w] >> 16)));
            }
        }
        amax = GroupMax<G>(amax, red, lane);
        out.rowScale = amax > 0.0f ? __fdiv_rn(amax, 127.0f) : 1.0f;
        rowScaleInv = out.rowScale > 0.0f ? __fdiv_rn(1.0f, out.rowScale) : 1.0f;
    }
#pragma unroll
    for (int j = 0; j < V; ++j) {
        float f[8];
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            f[2 * w] = Decode16<BF16>(v[j][w] & 0xffffu);
            f[2 * w + 1] = Decode16<BF16>(v[j][w] >> 16);
        }
        uint32_t bytes[8];
        uint32_t fp8Words[2] = {0u, 0u};
        if (QMODE == TILEXR_EP_QUANT_MXFP8) {
            const MxScaling mx = MxScalingOf<BF16, E5M2>(MxBlockMaxBits(v[j]));
            out.sharedExp[j] = mx.exponent;
            if (__all(mx.plain ? 1 : 0)) {
                fp8Words[0] = MxEncodePair<BF16, E5M2, true>(MxEncodePair<BF16, E5M2, false>(0u, v[j][0], mx), v[j][1], mx);
                fp8Words[1] = MxEncodePair<BF16, E5M2, true>(MxEncodePair<BF16, E5M2, false>(0u, v[j][2], mx), v[j][3], mx);
            } else {
                // infinities and NaNs: the codec that defines what becomes of them
                float amax = 0.0f;
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    amax = fmaxf(amax, fabsf(f[e]));
                }
                amax = fmaxf(amax, __shfl_xor(amax, 1));
                amax = fmaxf(amax, __shfl_xor(amax, 2));
                const int se = MxSharedExponent<E5M2>(amax);
                out.sharedExp[j] = se;
#pragma unroll 1
                for (int e = 0; e < 8; ++e) {
                    const uint32_t pair = e < 4 ? (e < 2 ? v[j][0] : v[j][1]) : (e < 6 ? v[j][2] : v[j][3]);
                    const float one = Decode16<BF16>((e & 1) != 0 ? pair >> 16 : pair & 0xffffu);
                    const uint32_t code = Fp8Encode<E5M2>(ldexpf(one, -se)) << (8 * (e % 4));
                    fp8Words[0] |= e < 4 ? code : 0u;
                    fp8Words[1] |= e < 4 ? 0u : code;
                }
            }
        } else if (QMODE == TILEXR_EP_QUANT_FP8_BLOCK128) {
            float amax = 0.0f;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                amax = fmaxf(amax, fabsf(f[e]));
            }
            amax = RowMax(amax);        // 128 columns = 16 neighbouring lanes
            const float sc = amax > 0.0f ? __fdiv_rn(amax, 448.0f) : 1.0f;
            out.blockScale[j] = sc;
            // eight quotients by one divisor: what depends on the divisor alone is done once (ep_numerics.hip.h)
            float quot[8];
            const bool shortForm = __all(SharedReciprocalHolds(sc) ? 1 : 0) != 0;
            if (shortForm) {
                const float y = SharedReciprocal(sc);
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    quot[e] = DivideByShared(f[e], sc, y);
                }
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    quot[e] = __fdiv_rn(f[e], sc);
                }
            }
            bool anyNan = false;
#pragma unroll
            for (int e = 0; e < 8; e += 2) {
                anyNan |= __builtin_isunordered(quot[e], quot[e + 1]);
            }
            if (!anyNan) {
                // four codes per word straight from the converts: the second one fills the word's upper half
                fp8Words[0] = Fp8E4m3EncodeFourSat(quot[0], quot[1], quot[2], quot[3]);
                fp8Words[1] = Fp8E4m3EncodeFourSat(quot[4], quot[5], quot[6], quot[7]);
            } else {
#pragma unroll
                for (int e = 0; e < 8; e += 4) {
                    fp8Words[e / 4] = Fp8E4m3EncodePairSat(quot[e], quot[e + 1]) |
                        (Fp8E4m3EncodePairSat(quot[e + 2], quot[e + 3]) << 16);
                }
            }
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                bytes[e] = static_cast<uint32_t>(ClampInt8(__fmul_rn(f[e], rowScaleInv)));
            }
        }
        if (QMODE == TILEXR_EP_QUANT_MXFP8 || QMODE == TILEXR_EP_QUANT_FP8_BLOCK128) {
            out.q[j][0] = fp8Words[0];
            out.q[j][1] = fp8Words[1];
        } else {
            out.q[j][0] = PackBytes(bytes[0], bytes[1], bytes[2], bytes[3]);
            out.q[j][1] = PackBytes(bytes[4], bytes[5], bytes[6], bytes[7]);
        }
    }
}

// Writes the row (or its payload and scales) held by the group's lanes to row `row` of the outputs.
template <int G, int V, int QMODE, RowStores S, bool WT, typename Args>
__device__ __forceinline__ void StoreRow(const Args &a, int row, const u32x4 (&v)[V], const QuantisedRow<V> &out, int lane)
{
    const int vecs = a.h / 8;
    if (QMODE == TILEXR_EP_QUANT_NONE) {
        char *dst = static_cast<char *>(a.out) + static_cast<int64_t>(row) * a.h * 2;
        const __amdgpu_buffer_rsrc_t rsrc = RowResource(dst, vecs * 16);
#pragma unroll
        for (int j = 0; j < V; ++j) {
            const int idx = j * G + lane;
            if (idx < vecs) {
                RowStore<S>(v[j], dst, rsrc, idx * 16);
            }
        }
        return;
    }
    const int mxBlocks = (a.h + 31) / 32;
    const int mxScales = (mxBlocks + 1) / 2 * 2;
    const int b128 = (a.h + 127) / 128;
    char *dst = static_cast<char *>(a.out) + static_cast<int64_t>(row) * a.h;
    const __amdgpu_buffer_rsrc_t rsrc = RowResource(dst, vecs * 8);
#pragma unroll
    for (int j = 0; j < V; ++j) {
        const int idx = j * G + lane;
        if (idx < vecs) {
            RowStore<S>(out.q[j], dst, rsrc, idx * 8);
            if (QMODE == TILEXR_EP_QUANT_MXFP8 && (idx & 3) == 0) {
                uint8_t *sc = static_cast<uint8_t *>(a.scalesOut) + static_cast<int64_t>(row) * mxScales;
                ScalarStore<WT>(sc + (idx >> 2), static_cast<uint8_t>(out.sharedExp[j] + 127));
                if ((idx >> 2) + 1 == mxBlocks && mxBlocks < mxScales) {
                    ScalarStore<WT>(sc + mxBlocks, static_cast<uint8_t>(0));    // padding byte of an odd block count
                }
            }
            if (QMODE == TILEXR_EP_QUANT_FP8_BLOCK128 && (idx & 15) == 0) {
                ScalarStore<WT>(static_cast<float *>(a.scalesOut) + static_cast<int64_t>(row) * b128 + (idx >> 4),
                    out.blockScale[j]);
            }
        }
    }
    if (QMODE == TILEXR_EP_QUANT_TOKEN_INT8 && lane == 0) {
        ScalarStore<WT>(static_cast<float *>(a.scalesOut) + row, out.rowScale);
    }
}

} // namespace
} // namespace TileXREp

#endif // TILEXR_AMD_EP_ROW_QUANT_HIP_H
