// reduce: y[token] = sum over the token's rows, gathered through the inverse map (gfx950, wave64).
//
// HBM-bound: topK row reads per output row, < 0.5 FLOP per byte, no MFMA.  G lanes cooperate on one token and keep
// V x 8 fp32 accumulators in registers; for each route in k order a lane issues all V of its 128-bit non-temporal
// loads of that row before touching the accumulators, so 64-128 bytes per lane are in flight while the previous
// row is being summed.  Measured on MI355X this moves 4096 x 7168 bf16 x top-8 (529 MB) at about 6 TB/s.
//
//   KIND fp32     sum = 0; for k = 0..K-1: sum = sum + (w_k * row_k) in fp32 (separate multiply and add), then the
//                 shared-expert row, then one round-to-nearest-even (saturating for fp16) to the output type;
//                 an inactive token (mask) gives zeros
//                 (reference: src/ep/kernels/tilexr_ep_combine_memory_kernel.h:505-553, 555-571, 573-601, 632-662)
//   KIND per-add  rows in ascending row index; y = T(float(y) + float(row)) after every add
//                 (reference: src/ep/kernels/tilexr_ep_combine_kernel.cpp:15-26, 54-101)
//   COMMQ 3/4     every row first takes the MXFP8 e5m2 / e4m3 round trip and is accumulated as
//                 ((fp8 * 2^(s-127)) * w) (reference: src/ep/kernels/tilexr_ep_mxfp8_quant.h:286-352)
//   INQ 2/5       rows hold int8 / fp8 payloads that are dequantised with their scales and rounded to the element
//                 type first (no reference counterpart)
//
// This file: the element-granular kernel for any width and alignment, and the choice of kernel and geometry.  The
// register-resident kernels are in ep_reduce_vec.hip.h and ep_reduce_quant.hip.h.
#include "ep_reduce_common.hip.h"

namespace TileXREp {
namespace {

// Element-granular reduce for any h / alignment.  One workgroup per token; a thread owns whole 32-column blocks so
// that the MXFP8 round trip needs no cross-lane traffic.
template <bool BF16>
__global__ __launch_bounds__(kThreads) void ep_reduce_generic_kernel(ReduceArgs a, int kind, int inq, int commq)
{
    __shared__ int s_row[kMaxTopK];
    __shared__ float s_w[kMaxTopK];
    const int tid = threadIdx.x;
    const int b128 = (a.h + 127) / 128;
    for (int token = blockIdx.x; token < a.bs; token += gridDim.x) {
        __syncthreads();
        LoadRoutes<true>(a, token, true, tid, kThreads, s_row, s_w, kRouteCheck);
        __syncthreads();
        if (a.tileFlags != nullptr) {
            // pairs with the producer's release.  Every wave reads rows with ordinary loads below, so every wave
            // invalidates for itself, after the barrier behind which all the token's waits have succeeded and before
            // its first row load: an invalidate issued by one wave says nothing about when a sibling's load may issue
            AcquireRowsFromAgent();
        }
        if (kind == kReducePerAdd) {
            if (tid == 0) {
                SortRows(s_row, a.slots, a.orderKeys);
            }
            __syncthreads();
        }
        const bool active = (a.tokenMask == nullptr || a.tokenMask[token] != 0) &&
            !(a.tileFlags != nullptr && AnyExpired(s_row, a.slots));
        uint16_t *dst = static_cast<uint16_t *>(a.y) + static_cast<int64_t>(token) * a.h;
        const int blocks = (a.h + 31) / 32;
        for (int b = tid; b < blocks; b += kThreads) {
            const int begin = b * 32;
            const int end = min(begin + 32, a.h);
            float acc[32];
            for (int i = 0; i < 32; ++i) {
                acc[i] = 0.0f;
            }
            if (active) {
                for (int k = 0; k < a.slots; ++k) {
                    const int row = s_row[k];
                    if (row < 0) {
                        continue;
                    }
                    const float w = s_w[k];
                    const char *base = static_cast<const char *>(a.expertOut) + static_cast<int64_t>(row) * a.rowBytes;
                    float f[32];
                    float amax = 0.0f;
                    for (int i = begin; i < end; ++i) {
                        float v;
                        if (inq == 0) {
                            v = Decode16<BF16>(reinterpret_cast<const uint16_t *>(base)[i]);
                        } else {
                            const uint32_t byte = reinterpret_cast<const uint8_t *>(base)[i];
                            const float d = inq == TILEXR_EP_QUANT_TOKEN_INT8 ?
                                __fmul_rn(static_cast<float>(static_cast<int>(static_cast<int8_t>(byte))), a.inScales[row]) :
                                __fmul_rn(Fp8Decode<false>(byte), a.inScales[static_cast<int64_t>(row) * b128 + i / 128]);
                            v = BF16 ? __uint_as_float(FloatToBf16Rne(d) << 16) :
                                       __half2float(__ushort_as_half(static_cast<unsigned short>(FloatToHalfRneSat(d))));
                        }
                        f[i - begin] = v;
                        amax = fmaxf(amax, fabsf(v));
                    }
                    if (commq != 0) {
                        const bool e5 = commq == TILEXR_EP_QUANT_COMM_MXFP8_E5M2;
                        const int se = e5 ? MxSharedExponent<true>(amax) : MxSharedExponent<false>(amax);
                        const float up = Exp2Int(se);
                        for (int i = 0; i < end - begin; ++i) {
                            const float s = ldexpf(f[i], -se);
                            const float back = e5 ? Fp8Decode<true>(Fp8Encode<true>(s)) : Fp8Decode<false>(Fp8Encode<false>(s));
                            f[i] = __fmul_rn(back, up);
                        }
                    }
                    for (int i = 0; i < end - begin; ++i) {
                        if (kind == kReducePerAdd) {
                            acc[i] = RoundTo16<BF16>(__fadd_rn(acc[i], f[i]));
                        } else {
                            acc[i] = __fadd_rn(acc[i], __fmul_rn(f[i], w));
                        }
                    }
                }
                if (a.sharedExpertX != nullptr) {
                    const uint16_t *sx = static_cast<const uint16_t *>(a.sharedExpertX) + static_cast<int64_t>(token) * a.h;
                    for (int i = begin; i < end; ++i) {
                        acc[i - begin] = __fadd_rn(acc[i - begin], Decode16<BF16>(sx[i]));
                    }
                }
            }
            for (int i = begin; i < end; ++i) {
                dst[i] = active ? static_cast<uint16_t>(Encode16Sat<BF16>(acc[i - begin])) : static_cast<uint16_t>(0);
            }
        }
    }
}


void LaunchVecKernels(int g, int v, const ReduceLaunch &l, const ReduceArgs &a, int gridLimit, const WorldReduceArgs *world, int ranks)
{
    // one workgroup per token is a geometry of the units with flags only
    const bool flags = a.tileFlags != nullptr || g == kThreads;
    if (l.bf16) {
        (flags ? LaunchReduceVecBf16Flags : LaunchReduceVecBf16)(g, v, l, a, gridLimit, world, ranks);
    } else {
        (flags ? LaunchReduceVecFp16Flags : LaunchReduceVecFp16)(g, v, l, a, gridLimit, world, ranks);
    }
}

void LaunchQuantKernels(int g, int v, const ReduceLaunch &l, const ReduceArgs &a, int gridLimit)
{
    // flags that were all published before this launch began take the kernels without the waiting code
    const bool flags = a.tileFlags != nullptr;
    const bool settled = flags && a.flagsSettled != 0;
    if (l.bf16) {
        (settled ? LaunchReduceQuantBf16Settled : flags ? LaunchReduceQuantBf16Flags : LaunchReduceQuantBf16)(g, v, l, a, gridLimit);
    } else {
        (settled ? LaunchReduceQuantFp16Settled : flags ? LaunchReduceQuantFp16Flags : LaunchReduceQuantFp16)(g, v, l, a, gridLimit);
    }
}

ReduceArgs ArgsOf(const ReduceLaunch &l)
{
    ReduceArgs a {};
    a.expertOut = l.expertOut;
    a.rowBytes = l.rowBytes;
    a.inverseTagged = l.inverseTagged;
    a.epoch = l.epoch;
    a.rowIndexMap = l.rowIndexMap;
    a.orderKeys = l.orderKeys;
    a.expertScales = l.expertScales;
    a.tokenMask = l.tokenMask;
    a.sharedExpertX = l.sharedExpertX;
    a.inScales = l.inScales;
    a.bs = static_cast<int>(l.bs);
    a.h = static_cast<int>(l.h);
    a.topK = static_cast<int>(l.topK);
    a.slots = static_cast<int>(l.topK + l.sharedSlots);
    a.maxRows = l.maxRows > 0 ? static_cast<int>(l.maxRows) : 0x7fffffff;
    a.y = l.y;
    a.tileFlags = l.tileFlags;
    a.tileRows = static_cast<int>(l.tileRows);
    a.tileShift = -1;
    if (l.tileRows > 0 && (l.tileRows & (l.tileRows - 1)) == 0) {
        a.tileShift = __builtin_ctzll(static_cast<unsigned long long>(l.tileRows));
    }
    a.flagEpoch = l.flagEpoch;
    a.waitTimeoutTicks = l.waitTimeoutTicks;
    a.deviceStatus = l.deviceStatus;
    a.flagsSettled = (l.tileFlags != nullptr && l.producerOrdered) ? 1 : 0;
    a.claim = l.claimWord;
    a.colSlices = 1;
    return a;
}

// 16-bit rows the register-resident kernel takes.
bool IsPlain(const ReduceLaunch &l)
{
    return l.inQuant == 0 && l.h % 8 == 0 && Aligned16(l.y) && l.h / 8 <= 8 * kThreads &&
        Aligned16(l.expertOut) && l.rowBytes % 16 == 0 &&
        (l.sharedExpertX == nullptr || Aligned16(l.sharedExpertX)) && (l.commQuant == 0 || l.h % 32 == 0);
}

// Slices that a token's row is cut into by the plain kernels, a wave each; `ranks` reduces of this shape in the launch.
// Narrow rows: a wave per token.  Wide ones: slices of 128 vectors (many small independent waves with four rows in flight
// each reach the highest gather bandwidth here).  Rows of 129 to 256 vectors: a wave that has a token to itself keeps two
// rows in flight; a launch of at most kWideReduceUnits waves with half a row each keeps eight.  Eight layers in a graph, us
// with one slice and with two, 2048 columns, top-8: 16 tokens 92 -> 56, 512 tokens 150 -> 134, 1024 tokens 186 -> 171, 2048
// tokens 280 and 278.  One or two rows arrive in one trip either way, and a second wave pays only while the waves are few:
// top-2, 512 tokens 76.6 -> 72.6, 640 tokens 82.2 -> 79.6, 768 tokens 85.1 and 84.1 (1032 columns 80.7 and 81.7), 1024
// tokens 95.5 and 96.1 (1032 columns 88.2 and 90.5).  The reduce of a logical world, us of its launch: 4 ranks x 128 tokens,
// top-8 7.9 -> 5.7, 2 x 512 8.5 and 8.4, top-2 2 x 64 4.6 -> 4.4, 2 x 300 4.8 and 5.0.
int SlicesOf(const ReduceLaunch &l, int ranks)
{
    constexpr int64_t kPairTokens = 640;
    const int64_t vecs = l.h / 8;
    const int slices = static_cast<int>((vecs + 2 * kWave - 1) / (2 * kWave));
    if (vecs > 4 * kWave) {
        return slices;
    }
    const int64_t tokens = l.bs * ranks;
    const bool few = l.tileFlags == nullptr && l.reduceKind == kReduceFp32 && l.commQuant == 0 &&
        tokens * slices <= kWideReduceUnits && (l.topK + l.sharedSlots > 2 || tokens <= kPairTokens);
    return few ? slices : 1;
}

// Whether a workgroup is one wave with one unit.  Sliced rows: many small workgroups reach the highest gather bandwidth here.
// Narrow rows that a single-launch dispatch wrote, too: their tokens can then run on the XCD that wrote them (PlacesByXcd;
// eight layers in a graph, 1024 columns, top-8, us: 4 tokens 54.5 -> 50.9, 100 tokens 64.3 -> 58.8, 250 tokens 81.1 -> 75.1).
// Beyond, four neighbouring tokens to a workgroup follow the per-token scatter, which has them so (600 x 1024 11.2 us, 13.3
// with a wave each).
bool WaveUnits(const ReduceLaunch &l, int slices, int ranks)
{
    return slices > 1 || (l.tileFlags == nullptr && ranks == 1 && l.bs * (l.topK + l.sharedSlots) <= kSmallRoutes);
}

// Quantised rows, one or two to a token: several tokens to a wave (ep_reduce_quant_few_kernel) where the launch is long enough
// to be bound by what its waves have under way, up to the largest outputs that both payloads were measured to gain at; at the
// next sizes int8 loses and block fp8 gains or loses.  Dispatch + combine, us, a token to a wave and several, int8 and block fp8:
//   top-1, outputs of 33 MB 16384 x 1024 25.1 and 25.6, 26.2 and 27.0; 49 MB 12000 x 2048 35.7 -> 34.6, 36.3 -> 35.6; 67 MB
//     16384 x 2048 48.6 -> 44.3, 50.2 -> 46.2; 86 MB 6000 x 7168 59.8 -> 55.7, 63.2 -> 56.9; 164 MB 10000 x 8192 103.3 ->
//     96.8, 108.9 -> 98.1; 235 MB 16384 x 7168 163.8 -> 160.7, 169.0 -> 159.7; 268 MB 16384 x 8192 174.3 and 175.9, 178.6 ->
//     174.9
//   top-2, 41 MB 5000 x 4096 36.3 and 36.8, 36.9 and 37.6; 67 MB 16384 x 2048 59.7 -> 56.1, 61.1 -> 58.4; 98 MB 6000 x 8192
//     75.5 -> 74.0, 80.4 -> 75.7; 134 MB 16384 x 4096 103.6 -> 100.3, 104.4 -> 100.9; 164 MB 10000 x 8192 121.5 and 123.4,
//     127.9 -> 125.8; 221 MB 13500 x 8192 179.1 and 181.7, 178.8 and 183.6
// Rows that end within a 128-byte line gain less, since most slices' ends are within one too, and lose from 449 to 495 vectors,
// where the last of eight slices is short and the other kernel's 512 are not, and beyond 832, where its 1024 are nearly full:
// 5000 x 7184 x top-2 67.4 and 70.1, 69.3 and 71.9; 9000 x 7184 top-1 89.1 and 92.1, 90.0 and 91.9; 5000 x 7696 top-2 72.4 and
// 74.2, 73.9 and 75.7; 16368 columns top-1 112.4 and 118.5, 113.5 and 118.3.  But 9000 x 4112 top-1 62.1 -> 58.0, 66.4 -> 60.6; 8000 x 6160 top-2 90.2 and 91.0, 92.8 and 92.4; 6000 x 8016 top-1 70.1 and 70.9, 71.8 and
// 71.6; 5000 x 9232 top-2 83.7 and 83.7, 92.8 -> 87.5; 5000 x 12304 top-1 83.2 and 84.5, 90.2 -> 85.9.
bool QuantTakesFew(const ReduceLaunch &l)
{
    const int64_t outBytes = l.bs * l.h * 2;
    const int64_t vecs = l.h / 16;
    if (l.h % 128 != 0 && ((vecs > 7 * kWave && vecs < 8 * kWave - kWave / 4) || vecs > 13 * kWave)) {
        return false;
    }
    return l.tileFlags == nullptr && l.topK <= 2 && l.sharedSlots == 0 && outBytes >= (int64_t{45} << 20) &&
        outBytes <= (l.topK == 1 ? int64_t{224} << 20 : int64_t{128} << 20);
}

// 16-byte vectors per lane of a wave that takes one of `slices` slices.
int VecsPerLane(int64_t vecs, int slices)
{
    return slices == 1 && vecs > 2 * kWave ? 4 : 2;
}

} // namespace

bool ReduceWorldFits(const ReduceLaunch *ls, int ranks)
{
    for (int r = 0; r < ranks; ++r) {
        if (!IsPlain(ls[r]) || ls[r].tileFlags != nullptr || ls[r].bf16 != ls[0].bf16) {
            return false;
        }
    }
    return ranks > 0 && ranks <= kReduceRanks;
}

hipError_t LaunchReduceWorld(const ReduceLaunch *ls, int ranks)
{
    if (!ReduceWorldFits(ls, ranks)) {
        return hipErrorInvalidValue;
    }
    const int slices = SlicesOf(ls[0], ranks);
    WorldReduceArgs w {};
    for (int r = 0; r < ranks; ++r) {
        w.rank[r] = ArgsOf(ls[r]);
        w.rank[r].colSlices = slices;
        w.rank[r].waveUnits = WaveUnits(ls[0], slices, ranks) ? 1 : 0;
        if (ls[r].kernelNameOut != nullptr) {
            *ls[r].kernelNameOut = "ep_reduce_vec_world_kernel";
        }
    }
    LaunchVecKernels(kWave, VecsPerLane(ls[0].h / 8, slices), ls[0], w.rank[0], 0, &w, ranks);
    return hipGetLastError();
}

hipError_t LaunchReduce(const ReduceLaunch &l)
{
    ReduceArgs a = ArgsOf(l);
    // A kernel that waits on flags must never crowd out the producer it waits for: its waiting waves keep their
    // registers, and with three or more of these workgroups per compute unit a producer workgroup no longer fits
    // beside them (measured: flag waits expire at six).  Two workgroups per compute unit walk the tokens.
    // A launch whose flags were published earlier on its own stream never waits and gets the ordinary geometry.
    const bool mayWait = l.tileFlags != nullptr && !l.producerOrdered;
    const int gridLimit = mayWait ? 2 * (l.numComputeUnits > 0 ? l.numComputeUnits : 256) : 0;
    const int64_t vecs = l.h / 8;
    const bool plain = IsPlain(l);
    const int64_t qvecs = l.h / 16;
    const bool quant = l.inQuant != 0 && l.commQuant == 0 && l.reduceKind == kReduceFp32 && l.h % 16 == 0 &&
        qvecs <= 4 * kThreads && Aligned16(l.y) && Aligned16(l.expertOut) && l.rowBytes % 16 == 0 &&
        (l.sharedExpertX == nullptr || Aligned16(l.sharedExpertX));
    if (l.kernelNameOut != nullptr) {
        *l.kernelNameOut = quant ? "ep_reduce_quant_kernel" : (plain ? "ep_reduce_vec_kernel" : "ep_reduce_generic_kernel");
    }
    if (quant) {
        if (QuantTakesFew(l)) {
            a.colSlices = static_cast<int>((qvecs + kWave - 1) / kWave);
            if (l.kernelNameOut != nullptr) {
                *l.kernelNameOut = "ep_reduce_quant_few_kernel";
            }
            LaunchQuantKernels(kWave, kQuantFewSlots, l, a, 0);
        } else if (qvecs <= kWave) {
            LaunchQuantKernels(kWave, 1, l, a, gridLimit);
        } else if (qvecs <= 2 * kWave) {
            LaunchQuantKernels(2 * kWave, 1, l, a, gridLimit);
        } else if (qvecs <= kThreads) {
            LaunchQuantKernels(kThreads, 1, l, a, gridLimit);
        } else if (qvecs <= 2 * kThreads) {
            LaunchQuantKernels(kThreads, 2, l, a, gridLimit);
        } else {
            LaunchQuantKernels(kThreads, 4, l, a, gridLimit);
        }
    } else if (plain) {
        if (vecs > 4 * kWave && mayWait) {
            // readiness flags that may still be pending: one workgroup per token, so that one wave polls the token's
            // tiles instead of one per slice, and few enough workgroups that the producer fits beside them
            if (vecs <= 2 * kThreads) {
                LaunchVecKernels(kThreads, 2, l, a, gridLimit, nullptr, 1);
            } else if (vecs <= 4 * kThreads) {
                LaunchVecKernels(kThreads, 4, l, a, gridLimit, nullptr, 1);
            } else {
                LaunchVecKernels(kThreads, 8, l, a, gridLimit, nullptr, 1);
            }
        } else {
            a.colSlices = SlicesOf(l, 1);
            a.waveUnits = WaveUnits(l, a.colSlices, 1) ? 1 : 0;
            LaunchVecKernels(kWave, VecsPerLane(vecs, a.colSlices), l, a, gridLimit, nullptr, 1);
        }
    } else {
        int grid = static_cast<int>(l.bs);
        if (gridLimit > 0 && grid > gridLimit) {
            grid = gridLimit;
        }
        if (l.bf16) {
            hipLaunchKernelGGL((ep_reduce_generic_kernel<true>), dim3(grid), dim3(kThreads), 0, l.stream, a,
                l.reduceKind, l.inQuant, l.commQuant);
        } else {
            hipLaunchKernelGGL((ep_reduce_generic_kernel<false>), dim3(grid), dim3(kThreads), 0, l.stream, a,
                l.reduceKind, l.inQuant, l.commQuant);
        }
    }
    return hipGetLastError();
}

} // namespace TileXREp

