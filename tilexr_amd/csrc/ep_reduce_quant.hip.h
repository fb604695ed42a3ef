// reduce of quantised rows (int8 with a scale per row, fp8 e4m3 with a scale per 128 columns): ep_reduce.hip says what
// is computed.  Compiled once per (element type, readiness flags): the including file sets TILEXR_REDUCE_BF16,
// TILEXR_REDUCE_FLAGS and TILEXR_REDUCE_ENTRY.  TILEXR_REDUCE_FLAGS: 0 no flags; 1 flags that may still be pending
// (the launch can wait: tokens are claimed, rows and scales are read past the L2); 2 flags that were all published
// before the launch began (a dispatch earlier on the same stream): nothing waits, every wave only looks at the words
// of its token's tiles, and the kernel carries none of the waiting code -- with it in the same kernel the registers
// of the claim loop cost the fp8 kernel a wave per SIMD and the settled case ran 4 us behind the kernel without flags.
#if !defined(TILEXR_REDUCE_BF16) || !defined(TILEXR_REDUCE_FLAGS) || !defined(TILEXR_REDUCE_ENTRY)
#error "include from ep_reduce_quant_*.hip"
#endif

#include "ep_reduce_common.hip.h"

namespace TileXREp {
namespace {

// A row's largest magnitude is 128 (448) times its scale: below this scale none reaches the 65520 from which rounding to fp16
// has to saturate.
template <int INQ>
constexpr float kScaleSaturates = INQ == TILEXR_EP_QUANT_TOKEN_INT8 ? 511.875f : 146.25f;

// Sixteen columns of a row: dequantised, rounded to the element type, weighted, added.  EXACT: the reference decode of NaN
// codes and, for fp16, the saturating rounding.  For ep_reduce_quant_few_kernel.  The K loop of ep_reduce_quant_kernel has
// the same steps in place and has to change with them: called there, this costs it up to 26 vector registers (block fp8, four
// rows 60 and 70; int8 to fp16, six rows 66 and 92), and eight of the twelve narrower instances that may wait for flags spill two to
// eleven; those without flags take the same time either way (int8 8192 x 4096 x top-6 96.6 us, block fp8 16384 x 2048 x top-8 133.5).
template <int INQ, bool BF16, bool EXACT>
__device__ __forceinline__ void AddQuantRow(const u32x4 &q, float scale, float w, float (&acc)[16])
{
#pragma unroll
    for (int d = 0; d < 4; ++d) {
        const uint32_t word = q[d];
        float f[4];
        if (INQ == TILEXR_EP_QUANT_TOKEN_INT8) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                f[e] = static_cast<float>(static_cast<int>(static_cast<int8_t>((word >> (8 * e)) & 0xffu)));
            }
        } else if (EXACT) {
            Fp8E4m3DecodeWord(word, f);
        } else {
            Fp8E4m3DecodeWordFast(word, f);
        }
#pragma unroll
        for (int e = 0; e < 4; e += 2) {
            const float d0 = __fmul_rn(f[e], scale);
            const float d1 = __fmul_rn(f[e + 1], scale);
            float r0;
            float r1;
            if (BF16) {
                r0 = FloatRoundedToBf16(d0);
                r1 = FloatRoundedToBf16(d1);
            } else if (!EXACT) {
                FloatPairRoundedToHalf(d0, d1, &r0, &r1);
            } else {
                r0 = __half2float(__ushort_as_half(static_cast<unsigned short>(FloatToHalfRneSat(d0))));
                r1 = __half2float(__ushort_as_half(static_cast<unsigned short>(FloatToHalfRneSat(d1))));
            }
            acc[4 * d + e] = __fadd_rn(acc[4 * d + e], __fmul_rn(r0, w));
            acc[4 * d + e + 1] = __fadd_rn(acc[4 * d + e + 1], __fmul_rn(r1, w));
        }
    }
}

constexpr int kFlagsNone = 0;
constexpr int kFlagsMayWait = 1;
constexpr int kFlagsSettled = 2;

// Quantised expert output: int8 rows with one fp32 scale per row, or fp8 e4m3 rows with one fp32 scale per 128
// columns.  Each value is dequantised, rounded to the output element type, then accumulated exactly like an ordinary
// row (fp32, k order, separate multiply and add).  Rows are a quarter the bytes of bf16 rows, so a lane owns 16
// consecutive columns per vector (one 16-byte load) and KB rows are kept in flight at once.
//
// KB rows in flight per lane: four, or two of the widest rows.  Five or six slots to a token take six at once instead of four
// and then the rest, at five waves per SIMD instead of seven (8192 x 4096 x top-6 int8, dispatch + combine 99.4 -> 97.5 us;
// eight for eight slots is no such bargain: 16384 x 2048 int8 130.6 -> 129.8, but block fp8 that lost rows to a capacity, four
// left of eight, 91.0 -> 93.0, and 8192 x 4096 x top-2 57.0 -> 59.4).
template <int G, int V, int INQ, bool BF16, int FL, int KB>
__global__ __launch_bounds__(kThreads, V == 1 ? (KB > 4 ? 5 : (FL == kFlagsMayWait && (!BF16 || INQ == TILEXR_EP_QUANT_FP8_BLOCK128)) ? 6 : 7) : 1) void ep_reduce_quant_kernel(ReduceArgs a)
{
    constexpr int kTokens = kThreads / G;
    constexpr bool kWaits = FL == kFlagsMayWait;
    // route tables of launches that may wait
    __shared__ int s_row[kWaits ? kTokens : 1][kMaxTopK];
    __shared__ float s_w[kWaits ? kTokens : 1][kMaxTopK];

    const int tg = threadIdx.x / G;
    const int lane = threadIdx.x % G;
    const int vecs = a.h / 16;
    const int groups = (a.bs + kTokens - 1) / kTokens;
    const int b128 = (a.h + 127) / 128;

    auto tokenAt = [&](int group, int t) {
        const int token = group * kTokens + t;
        return token < a.bs ? token : -1;
    };
    auto load = [&](int group, int mode) {
        const int token = group * kTokens + tg;
        return LoadRoutes<false>(a, token, token < a.bs, lane, G, s_row[tg], s_w[tg], mode);
    };
    auto reduceUnit = [&](int group) {
        const int token = group * kTokens + tg;
        const bool tokOk = token < a.bs;
        // Lane k of every wave keeps slot k's row and weight; the K loop takes the slots that have a row, in k order,
        // KB at a time.  Where tokens lose rows to an expert's capacity that is often one trip to memory, not two
        // (absent rows are skipped by the sum anyway, so the order of the additions is the same).
        static_assert(G % kWave == 0, "a wave works on one token");
        const int waveLane = threadIdx.x % kWave;
        int slotRow = -1;
        float myWeight = 0.0f;
        if (!kWaits) {
            slotRow = RouteOfLane(a, token, tokOk, waveLane, &myWeight);
        } else if (waveLane < a.slots) {
            slotRow = s_row[tg][waveLane];
            myWeight = s_w[tg][waveLane];
        }
        constexpr bool checkWords = FL == kFlagsSettled;
        const bool expired = FL == kFlagsMayWait && __ballot(slotRow == kRowExpired) != 0;
        const bool active = tokOk && (a.tokenMask == nullptr || a.tokenMask[token] != 0) && !expired;
        const int myRow = active ? slotRow : -1;
        // (an inactive token's output is zeros whatever its words say: only the rows that are read are asked about)
        const uint32_t tileWord = checkWords ? SettledWordLoad(a, myRow) : 0u;
        const uint64_t live = __ballot(myRow >= 0);

        bool saturates = false;
        float acc[V][16];
        // The K loop.  fp8 rows are decoded by the hardware convert alone, which differs from the reference decode in
        // one respect only (the sign of the NaN it returns for code 0x7f); a NaN code always surfaces as a NaN in the
        // sum, so a wave that finds a NaN among its sums runs the loop once more with the exact decode.  That keeps a
        // test of every word (four instructions and a branch per four values) out of the loop that everything else
        // shares.  Rounding to fp16 likewise: the loop takes the plain converts and looks at the scales, once per row
        // and lane; a wave that meets a scale whose row could saturate, or a NaN, runs the loop once more with the
        // saturating ones (2756 x 8192 x top-8, dispatch + combine, fp16 before and now, and bf16: int8 106.4, 84.7 and 81.5
        // us, block fp8 108.8, 87.9 and 84.1; 8192 x 2048 x top-6 int8 69.2 -> 58.4).
        // throughMemory: rows and scales are read past this XCD's L2, as they must be while their producer may still
        // be writing neighbours of theirs.  Once the producer has finished (flagsSettled) the L2 is as good as memory,
        // and the scales, which the lanes of a token share, are worth keeping there (4096 x int8 rows: 58 -> 49 us).
        auto accumulate = [&](auto exactDecode, auto throughMemory) {
            constexpr bool kExactDecode = decltype(exactDecode)::value;
            constexpr bool kThroughMemory = decltype(throughMemory)::value;
#pragma unroll
            for (int j = 0; j < V; ++j) {
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    acc[j][e] = 0.0f;
                }
            }
            uint64_t todo = live;
            while (todo != 0) {
                u32x4 q[KB][V];
                float sc[KB][V];
                int rowOfK[KB];
                float weightOfK[KB];
#pragma unroll
                for (int u = 0; u < KB; ++u) {
                    const bool any = todo != 0;
                    const int k = any ? __builtin_ctzll(todo) : 0;
                    todo &= todo - 1;
                    const int row = any ? __builtin_amdgcn_readlane(myRow, k) : -1;
                    rowOfK[u] = row;
                    weightOfK[u] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(myWeight), k));
                    // Bounds are the buffer resources' business: an absent row gets resources of zero bytes, so its loads, like
                    // those of the lanes past the end of a row, return zeros without a branch (and without the register
                    // clears a branch would need).
                    const int64_t rowAt = row < 0 ? 0 : row;
                    const char *base = static_cast<const char *>(a.expertOut) + rowAt * a.rowBytes;
                    const __amdgpu_buffer_rsrc_t rsrc = RowResource(base, row < 0 ? 0 : vecs * 16);
                    const bool perRow = INQ == TILEXR_EP_QUANT_TOKEN_INT8;
                    const float *scaleBase = a.inScales + (perRow ? rowAt : rowAt * b128);
                    const __amdgpu_buffer_rsrc_t scaleRsrc = RowResource(scaleBase, row < 0 ? 0 : (perRow ? 4 : b128 * 4));
#pragma unroll
                    for (int j = 0; j < V; ++j) {
                        const int idx = j * G + lane;
                        q[u][j] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, idx * 16, 0,
                            kThroughMemory ? kAuxAgentScope : kAuxNonTemporal);
                        sc[u][j] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(scaleRsrc, perRow ? 0 : (idx >> 3) * 4, 0,
                            kThroughMemory ? kAuxAgentScope : 0));
                    }
                }
#pragma unroll
                for (int u = 0; u < KB; ++u) {
                    if (rowOfK[u] < 0) {
                        continue;                       // uniform across the lanes of a token
                    }
                    const float w = weightOfK[u];
#pragma unroll
                    for (int j = 0; j < V; ++j) {
                        if (!BF16 && !kExactDecode) {
                            saturates |= !(fabsf(sc[u][j]) < kScaleSaturates<INQ>);
                        }
                        // AddQuantRow's steps
#pragma unroll
                        for (int d = 0; d < 4; ++d) {
                            const uint32_t word = q[u][j][d];
                            float f[4];
                            if (INQ == TILEXR_EP_QUANT_TOKEN_INT8) {
#pragma unroll
                                for (int e = 0; e < 4; ++e) {
                                    f[e] = static_cast<float>(static_cast<int>(static_cast<int8_t>((word >> (8 * e)) & 0xffu)));
                                }
                            } else if (kExactDecode) {
                                Fp8E4m3DecodeWord(word, f);
                            } else {
                                Fp8E4m3DecodeWordFast(word, f);
                            }
#pragma unroll
                            for (int e = 0; e < 4; e += 2) {
                                const float d0 = __fmul_rn(f[e], sc[u][j]);
                                const float d1 = __fmul_rn(f[e + 1], sc[u][j]);
                                float r0;
                                float r1;
                                if (BF16) {
                                    r0 = FloatRoundedToBf16(d0);
                                    r1 = FloatRoundedToBf16(d1);
                                } else if (!kExactDecode) {
                                    FloatPairRoundedToHalf(d0, d1, &r0, &r1);
                                } else {
                                    r0 = __half2float(__ushort_as_half(static_cast<unsigned short>(FloatToHalfRneSat(d0))));
                                    r1 = __half2float(__ushort_as_half(static_cast<unsigned short>(FloatToHalfRneSat(d1))));
                                }
                                acc[j][4 * d + e] = __fadd_rn(acc[j][4 * d + e], __fmul_rn(r0, w));
                                acc[j][4 * d + e + 1] = __fadd_rn(acc[j][4 * d + e + 1], __fmul_rn(r1, w));
                            }
                        }
                    }
                }
            }
        };
        constexpr bool throughMemory = FL == kFlagsMayWait;
        if (throughMemory) {
            accumulate(std::false_type {}, std::true_type {});
        } else {
            accumulate(std::false_type {}, std::false_type {});
        }
        if (INQ == TILEXR_EP_QUANT_FP8_BLOCK128 || !BF16) {
            bool again = saturates;
            if (INQ == TILEXR_EP_QUANT_FP8_BLOCK128) {
#pragma unroll
                for (int j = 0; j < V; ++j) {
#pragma unroll
                    for (int e = 0; e < 16; ++e) {
                        again |= acc[j][e] != acc[j][e];
                    }
                }
            }
            if (__any(again ? 1 : 0)) {
                if (throughMemory) {
                    accumulate(std::true_type {}, std::true_type {});
                } else {
                    accumulate(std::true_type {}, std::false_type {});
                }
            }
        }
        if (a.sharedExpertX != nullptr && active) {
            const u32x4 *sx = reinterpret_cast<const u32x4 *>(static_cast<const char *>(a.sharedExpertX) +
                static_cast<int64_t>(token) * a.h * 2);
#pragma unroll
            for (int j = 0; j < V; ++j) {
                const int idx = j * G + lane;
                if (idx < vecs) {
#pragma unroll
                    for (int half = 0; half < 2; ++half) {
                        const u32x4 v = sx[idx * 2 + half];
#pragma unroll
                        for (int q2 = 0; q2 < 4; ++q2) {
                            float &lo = acc[j][half * 8 + 2 * q2];
                            float &hi = acc[j][half * 8 + 2 * q2 + 1];
                            lo = __fadd_rn(lo, Decode16<BF16>(v[q2] & 0xffffu));
                            hi = __fadd_rn(hi, Decode16<BF16>(v[q2] >> 16));
                        }
                    }
                }
            }
        }
        const bool keep = active && !(checkWords && SettledWordMissing(a, myRow, tileWord, waveLane));
        if (tokOk) {
            u32x4 *dst = reinterpret_cast<u32x4 *>(static_cast<char *>(a.y) + static_cast<int64_t>(token) * a.h * 2);
            // the lane index once more, from the thread index and out of the optimiser's sight: values derived from it
            // for these stores are then computed here instead of being kept (or spilled) across the K loop, where every
            // register counts towards the seventh wave per SIMD
            int storeThread = threadIdx.x;
            asm volatile("" : "+v"(storeThread));
            const int storeLane = storeThread % G;
#pragma unroll
            for (int j = 0; j < V; ++j) {
                const int idx = j * G + storeLane;
                if (idx < vecs) {
#pragma unroll
                    for (int half = 0; half < 2; ++half) {
                        u32x4 o;
#pragma unroll
                        for (int q2 = 0; q2 < 4; ++q2) {
                            o[q2] = keep ? EncodePair16Sat<BF16>(acc[j][half * 8 + 2 * q2], acc[j][half * 8 + 2 * q2 + 1]) : 0u;
                        }
                        // An ordinary store, not a streaming one: a lane's 32 bytes go out as two 16-byte stores, each
                        // of which fills every other 16 bytes of the lines it touches; the L2 puts the halves together
                        // before they go to memory (4096-column int8 rows: 46.3 us, 48.4 us with streaming stores;
                        // trading halves between lanes so that each store covers whole lines: 46.8 us).
                        dst[idx * 2 + half] = o;
                    }
                }
            }
        }
    };
    if constexpr (kWaits) {
        ForEachGroup(a, groups, kTokens, tokenAt, load, reduceUnit);
    } else {
        reduceUnit(blockIdx.x);         // a workgroup for every group
    }
}

// Tokens of one or two slots, launches without flags (QuantTakesFew).  A wave of the kernel above has one row or two in flight
// then and is done with them before its look-up, its rows and its stores, one after the other, have cost it three trips to
// memory: the waves a compute unit holds are too few for that.  Here a wave takes a slice of 64 vectors of ROWS / SLOTS
// neighbouring tokens: their look-ups together, their ROWS rows together, then token by token the sum and the store.
// Groups of tokens are dealt to the XCDs in turn (workgroup b runs on XCD b % 8) and all slices of a group go to the same one, so
// that a line in which a slice ends is fetched and put together in one L2: 5000 x 7184 x top-2 int8 71.6 -> 70.1 us, 5000 x 8176
// 77.7 -> 75.6, 9000 x 6160 top-1 80.7 -> 78.4, rows of whole lines unchanged (16384 x 4096 x top-2 100.1 and 100.2).  XCDs with a
// range of tokens each are no choice (100 -> 117.8).
constexpr int kQuantFewRows = 4;

template <int SLOTS, int INQ, bool BF16>
__global__ __launch_bounds__(kThreads) void ep_reduce_quant_few_kernel(ReduceArgs a)
{
    constexpr int ROWS = kQuantFewRows;
    constexpr int kTokens = ROWS / SLOTS;
    constexpr bool perRow = INQ == TILEXR_EP_QUANT_TOKEN_INT8;
    const int lane = threadIdx.x % kWave;
    const int vecs = a.h / 16;
    const int b128 = (a.h + 127) / 128;
    const int unit = static_cast<int>(blockIdx.x / kXcdCount) * kWavesPerBlock + static_cast<int>(threadIdx.x) / kWave;
    const int round = unit / a.colSlices;
    const int group = round * kXcdCount + static_cast<int>(blockIdx.x % kXcdCount);
    const int idx = (unit - round * a.colSlices) * kWave + lane;
    const int firstToken = __builtin_amdgcn_readfirstlane(group * kTokens);

    // lane l < ROWS: slot l % SLOTS of token firstToken + l / SLOTS
    int myRow = -1;
    float myWeight = 1.0f;
    bool myActive = false;
    const int myToken = firstToken + lane / SLOTS;
    if (lane < ROWS && myToken < a.bs) {
        const int64_t route = static_cast<int64_t>(firstToken) * SLOTS + lane;
        if (a.expertScales != nullptr) {
            myWeight = a.expertScales[route];
        }
        myActive = a.tokenMask == nullptr || a.tokenMask[myToken] != 0;
        myRow = LookupRow(a, route);
        myRow = myActive ? myRow : -1;
    }
    const uint64_t active = __ballot(myActive);
    u32x4 q[ROWS];
    float sc[ROWS];
#pragma unroll
    for (int u = 0; u < ROWS; ++u) {
        const int row = __builtin_amdgcn_readlane(myRow, u);
        const int64_t rowAt = row < 0 ? 0 : row;
        // an absent row gets resources of zero bytes (as above)
        const __amdgpu_buffer_rsrc_t rsrc = RowResource(static_cast<const char *>(a.expertOut) + rowAt * a.rowBytes, row < 0 ? 0 : vecs * 16);
        const __amdgpu_buffer_rsrc_t scales = RowResource(a.inScales + (perRow ? rowAt : rowAt * b128), row < 0 ? 0 : (perRow ? 4 : b128 * 4));
        q[u] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, idx * 16, 0, kAuxNonTemporal);
        sc[u] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(scales, perRow ? 0 : (idx >> 3) * 4, 0, 0));
    }
#pragma unroll
    for (int t = 0; t < kTokens; ++t) {
        const int token = firstToken + t;
        if (token >= a.bs) {
            return;
        }
        float acc[16];
        auto accumulate = [&](auto exact) {
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                acc[e] = 0.0f;
            }
#pragma unroll
            for (int s = 0; s < SLOTS; ++s) {
                const int u = t * SLOTS + s;
                if (__builtin_amdgcn_readlane(myRow, u) >= 0) {
                    AddQuantRow<INQ, BF16, decltype(exact)::value>(q[u], sc[u], __int_as_float(__builtin_amdgcn_readlane(__float_as_int(myWeight), u)), acc);
                }
            }
        };
        accumulate(std::false_type {});
        if (INQ == TILEXR_EP_QUANT_FP8_BLOCK128 || !BF16) {
            bool again = false;
#pragma unroll
            for (int s = 0; s < SLOTS; ++s) {
                again |= !BF16 && !(fabsf(sc[t * SLOTS + s]) < kScaleSaturates<INQ>);
            }
            if (INQ == TILEXR_EP_QUANT_FP8_BLOCK128) {
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    again |= acc[e] != acc[e];
                }
            }
            if (__any(again ? 1 : 0)) {
                accumulate(std::true_type {});
            }
        }
        if (idx >= vecs) {
            continue;
        }
        if (a.sharedExpertX != nullptr && ((active >> (t * SLOTS)) & 1ull) != 0ull) {
            const u32x4 *sx = reinterpret_cast<const u32x4 *>(static_cast<const char *>(a.sharedExpertX) + static_cast<int64_t>(token) * a.h * 2);
#pragma unroll
            for (int half = 0; half < 2; ++half) {
                const u32x4 v = sx[idx * 2 + half];
#pragma unroll
                for (int q2 = 0; q2 < 4; ++q2) {
                    acc[half * 8 + 2 * q2] = __fadd_rn(acc[half * 8 + 2 * q2], Decode16<BF16>(v[q2] & 0xffffu));
                    acc[half * 8 + 2 * q2 + 1] = __fadd_rn(acc[half * 8 + 2 * q2 + 1], Decode16<BF16>(v[q2] >> 16));
                }
            }
        }
        // (a token without active rows has sums of zero)
        u32x4 *dst = reinterpret_cast<u32x4 *>(static_cast<char *>(a.y) + static_cast<int64_t>(token) * a.h * 2);
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            u32x4 o;
#pragma unroll
            for (int q2 = 0; q2 < 4; ++q2) {
                o[q2] = EncodePair16Sat<BF16>(acc[half * 8 + 2 * q2], acc[half * 8 + 2 * q2 + 1]);
            }
            dst[idx * 2 + half] = o;
        }
    }
}

template <int SLOTS, bool BF16>
void LaunchQuantFew(const ReduceLaunch &l, const ReduceArgs &a)
{
    constexpr int kTokens = kQuantFewRows / SLOTS;
    const int rounds = ((a.bs + kTokens - 1) / kTokens + kXcdCount - 1) / kXcdCount;
    const dim3 g(static_cast<unsigned>((rounds * a.colSlices + kWavesPerBlock - 1) / kWavesPerBlock * kXcdCount));
    if (l.inQuant == TILEXR_EP_QUANT_TOKEN_INT8) {
        hipLaunchKernelGGL((ep_reduce_quant_few_kernel<SLOTS, TILEXR_EP_QUANT_TOKEN_INT8, BF16>), g, dim3(kThreads), 0, l.stream, a);
    } else {
        hipLaunchKernelGGL((ep_reduce_quant_few_kernel<SLOTS, TILEXR_EP_QUANT_FP8_BLOCK128, BF16>), g, dim3(kThreads), 0, l.stream, a);
    }
}

template <int G, int V, bool BF16, int FL, int KB>
void LaunchQuantRows(const ReduceLaunch &l, const ReduceArgs &a, int gridLimit)
{
    constexpr int kTokens = kThreads / G;
    int grid = (a.bs + kTokens - 1) / kTokens;
    if (gridLimit > 0 && grid > gridLimit) {
        grid = gridLimit;
    }
    const dim3 g(grid);
    const dim3 b(kThreads);
    if (l.inQuant == TILEXR_EP_QUANT_TOKEN_INT8) {
        hipLaunchKernelGGL((ep_reduce_quant_kernel<G, V, TILEXR_EP_QUANT_TOKEN_INT8, BF16, FL, KB>), g, b, 0, l.stream, a);
    } else {
        hipLaunchKernelGGL((ep_reduce_quant_kernel<G, V, TILEXR_EP_QUANT_FP8_BLOCK128, BF16, FL, KB>), g, b, 0, l.stream, a);
    }
}

template <int G, int V, bool BF16, int FL>
void LaunchQuant(const ReduceLaunch &l, const ReduceArgs &a, int gridLimit)
{
    if constexpr (V == 1 && FL != kFlagsMayWait) {
        if (a.slots == 5 || a.slots == 6) {
            LaunchQuantRows<G, V, BF16, FL, 6>(l, a, gridLimit);
            return;
        }
    }
    LaunchQuantRows<G, V, BF16, FL, V >= 4 ? 2 : 4>(l, a, gridLimit);
}

} // namespace

void TILEXR_REDUCE_ENTRY(int g, int v, const ReduceLaunch &l, const ReduceArgs &a, int gridLimit)
{
    constexpr bool kBf16 = TILEXR_REDUCE_BF16;
    constexpr int kFlags = TILEXR_REDUCE_FLAGS;
    if constexpr (kFlags == kFlagsNone) {
        if (v == kQuantFewSlots) {
            a.slots == 1 ? LaunchQuantFew<1, kBf16>(l, a) : LaunchQuantFew<2, kBf16>(l, a);
            return;
        }
    }
    if (g == kWave && v == 1) {
        LaunchQuant<kWave, 1, kBf16, kFlags>(l, a, gridLimit);
    } else if (g == 2 * kWave && v == 1) {
        LaunchQuant<2 * kWave, 1, kBf16, kFlags>(l, a, gridLimit);
    } else if (g == kThreads && v == 1) {
        LaunchQuant<kThreads, 1, kBf16, kFlags>(l, a, gridLimit);
    } else if (g == kThreads && v == 2) {
        LaunchQuant<kThreads, 2, kBf16, kFlags>(l, a, gridLimit);
    } else if (g == kThreads && v == 4) {
        LaunchQuant<kThreads, 4, kBf16, kFlags>(l, a, gridLimit);
    }
}

} // namespace TileXREp
