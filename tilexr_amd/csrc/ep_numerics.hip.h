// Device-side element conversions shared by the scatter and reduce kernels (gfx950, wave64).
//
// Every routine is written so that its result is a pure function of the input bits: separate multiplies and adds
// (the build uses -ffp-contract=off and the explicit *_rn intrinsics) and saturation made explicit.  That is what
// lets the parity tests demand bit equality.  Hardware converts are used only where an exhaustive comparison on
// gfx950 showed them equal to the software codec: v_cvt_pk_bf16_f32 (all 2^32 inputs, NaNs included),
// v_cvt_pk_f32_fp8 (all codes except the sign of NaN code 0x7f) and v_cvt_pk_fp8_f32 (all finite |x| < 464; beyond
// that the hardware returns NaN where this codec saturates, so inputs are clamped first and NaNs patched).
//   int8 rounding      reference: src/ep/kernels/tilexr_ep_dispatch_kernel.cpp:183-193
//   MXFP8 / fp8 codec  reference: tests/ep/demo/mxfp8_golden.h:45-152
//   output casts       reference: src/ep/kernels/tilexr_ep_combine_memory_kernel.h:595 (CAST_RINT, saturating)
#ifndef TILEXR_AMD_EP_NUMERICS_HIP_H
#define TILEXR_AMD_EP_NUMERICS_HIP_H

#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

namespace TileXREp {

// exponent fields of the divisors for which DivideByShared is used (see there)
constexpr uint32_t kSharedDivisionMinExponent = 16;
constexpr uint32_t kSharedDivisionMaxExponent = 254;

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

template <bool BF16>
__device__ __forceinline__ float Decode16(uint32_t bits16)
{
    if (BF16) {
        return __uint_as_float(bits16 << 16);
    }
    return __half2float(__ushort_as_half(static_cast<unsigned short>(bits16)));
}

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

// Two fp32 -> two bf16 (round to nearest even, NaN -> (bits >> 16) | 0x40), packed lo | hi << 16.
__device__ __forceinline__ uint32_t FloatPairToBf16Rne(float lo, float hi)
{
    const f32x2 f = {lo, hi};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, bf16x2));
}

__device__ __forceinline__ uint32_t FloatToBf16Rne(float v)
{
    return FloatPairToBf16Rne(v, 0.0f) & 0xffffu;
}

// An fp32 value rounded to bf16 (same rounding), returned as fp32: the pair convert with 0.0 in the low half leaves the
// rounded value's own fp32 bit pattern, so one instruction does the rounding and no unpacking follows.
__device__ __forceinline__ float FloatRoundedToBf16(float v)
{
    return __uint_as_float(FloatPairToBf16Rne(0.0f, v));
}

// IEEE round-to-nearest-even; overflow becomes infinity.
__device__ __forceinline__ uint32_t FloatToHalfRne(float v)
{
    return __half_as_ushort(__float2half_rn(v));
}

// Same rounding, but magnitudes that would round past 65504 stay at +-65504.
__device__ __forceinline__ uint32_t FloatToHalfRneSat(float v)
{
    const uint32_t u = __float_as_uint(v);
    const uint32_t a = u & 0x7fffffffu;
    if (a >= 0x477ff000u && a <= 0x7f800000u) {
        return ((u >> 16) & 0x8000u) | 0x7bffu;
    }
    return FloatToHalfRne(v);
}

// Two fp32 values that do not saturate (finite, below 65520) rounded to fp16 (same rounding), returned as fp32.  Three
// instructions for the two, where FloatToHalfRneSat and a decode take eight each: one pair convert, two converts back.
__device__ __forceinline__ void FloatPairRoundedToHalf(float lo, float hi, float *rlo, float *rhi)
{
    typedef _Float16 half2 __attribute__((ext_vector_type(2)));
    const f32x2 f = {lo, hi};
    const half2 h = __builtin_convertvector(f, half2);
    *rlo = static_cast<float>(h[0]);
    *rhi = static_cast<float>(h[1]);
}

template <bool BF16>
__device__ __forceinline__ uint32_t Encode16Sat(float v)
{
    return BF16 ? FloatToBf16Rne(v) : FloatToHalfRneSat(v);
}

// Two values -> packed 16-bit elements (lo | hi << 16), fp16 saturating as above.
template <bool BF16>
__device__ __forceinline__ uint32_t EncodePair16Sat(float lo, float hi)
{
    return BF16 ? FloatPairToBf16Rne(lo, hi) : (FloatToHalfRneSat(lo) | (FloatToHalfRneSat(hi) << 16));
}

// Round an fp32 value to the 16-bit element type and return it as fp32 again (IEEE, non-saturating).
template <bool BF16>
__device__ __forceinline__ float RoundTo16(float v)
{
    return BF16 ? __uint_as_float(FloatToBf16Rne(v) << 16) : __half2float(__float2half_rn(v));
}

// add +-0.5, truncate toward zero, clamp to [-128, 127] (ahead of the truncation, which comes to the same); NaN -> -128, which
// is what the median of three makes of it
__device__ __forceinline__ int ClampInt8(float v)
{
    const float r = __fadd_rn(v, __builtin_copysignf(0.5f, v));
    return static_cast<int>(__builtin_amdgcn_fmed3f(r, -128.0f, 127.0f));
}

// Saturating round-to-nearest-even fp32 -> fp8 code (OCP e4m3fn / e5m2), by bit manipulation.
template <bool E5M2>
__device__ __forceinline__ uint32_t Fp8Encode(float v)
{
    constexpr int kMantBits = E5M2 ? 2 : 3;
    constexpr int kBias = E5M2 ? 15 : 7;
    constexpr int kMinNormalExp = 1 - kBias;
    constexpr uint32_t kMaxCode = E5M2 ? 0x7bu : 0x7eu;
    const uint32_t u = __float_as_uint(v);
    const uint32_t sign = (u >> 24) & 0x80u;
    const uint32_t a = u & 0x7fffffffu;
    if (a > 0x7f800000u) {
        return sign | 0x7fu;
    }
    const int e = static_cast<int>(a >> 23) - 127;
    const uint32_t mant = a & 0x7fffffu;
    uint32_t code;
    if (e < kMinNormalExp) {
        const int shift = 23 - e + kMinNormalExp - kMantBits;   // value / subnormal step = full >> shift
        if (shift > 24) {
            code = 0;
        } else {
            const uint32_t full = mant | 0x800000u;
            const uint32_t kept = full >> shift;
            const uint32_t rem = full & ((1u << shift) - 1u);
            const uint32_t half = 1u << (shift - 1);
            code = kept + ((rem > half || (rem == half && (kept & 1u))) ? 1u : 0u);
        }
    } else if (e > 20) {
        code = kMaxCode;
    } else {
        const uint32_t kept = mant >> (23 - kMantBits);
        const uint32_t rem = mant & ((1u << (23 - kMantBits)) - 1u);
        const uint32_t half = 1u << (22 - kMantBits);
        code = (static_cast<uint32_t>(e + kBias) << kMantBits) + kept +
            ((rem > half || (rem == half && (kept & 1u))) ? 1u : 0u);
        code = code > kMaxCode ? kMaxCode : code;
    }
    return sign | code;
}

template <bool E5M2>
__device__ __forceinline__ float Fp8Decode(uint32_t code)
{
    constexpr int kMantBits = E5M2 ? 2 : 3;
    constexpr int kBias = E5M2 ? 15 : 7;
    constexpr uint32_t kExpMask = E5M2 ? 31u : 15u;
    constexpr uint32_t kMantMask = (1u << kMantBits) - 1u;
    const uint32_t sign = (code & 0x80u) << 24;
    const uint32_t exp = (code >> kMantBits) & kExpMask;
    const uint32_t man = code & kMantMask;
    if (exp == 0) {
        const float mag = static_cast<float>(man) * __uint_as_float(static_cast<uint32_t>(127 + 1 - kBias - kMantBits) << 23);
        return __uint_as_float(__float_as_uint(mag) | sign);
    }
    if (E5M2 && exp == kExpMask) {
        return __uint_as_float(sign | 0x7f800000u | (man << 21));
    }
    if (!E5M2 && exp == kExpMask && man == kMantMask) {
        return __uint_as_float(sign | 0x7fc00000u);
    }
    return __uint_as_float(sign | ((exp + 127u - kBias) << 23) | (man << (23 - kMantBits)));
}

// e4m3 code of x with round-to-nearest-even and saturation to +-448; NaN -> sign | 0x7f.  Same function as
// Fp8Encode<false>, through the hardware convert.
__device__ __forceinline__ uint32_t Fp8E4m3EncodePairSat(float lo, float hi)
{
    const float clo = __builtin_amdgcn_fmed3f(lo, -448.0f, 448.0f);
    const float chi = __builtin_amdgcn_fmed3f(hi, -448.0f, 448.0f);
    uint32_t code = static_cast<uint32_t>(__builtin_amdgcn_cvt_pk_fp8_f32(clo, chi, 0, false)) & 0xffffu;
    if (lo != lo) {
        code = (code & 0xff00u) | ((__float_as_uint(lo) >> 24) & 0x80u) | 0x7fu;
    }
    if (hi != hi) {
        code = (code & 0x00ffu) | ((((__float_as_uint(hi) >> 24) & 0x80u) | 0x7fu) << 8);
    }
    return code;
}

// Four values that are not NaNs -> four e4m3 codes in one word (a | b << 8 | c << 16 | d << 24), same codes as
// Fp8E4m3EncodePairSat: the second convert writes the upper half of the word the first one started.
__device__ __forceinline__ uint32_t Fp8E4m3EncodeFourSat(float a, float b, float c, float d)
{
    const int lower = __builtin_amdgcn_cvt_pk_fp8_f32(__builtin_amdgcn_fmed3f(a, -448.0f, 448.0f),
        __builtin_amdgcn_fmed3f(b, -448.0f, 448.0f), 0, false);
    return static_cast<uint32_t>(__builtin_amdgcn_cvt_pk_fp8_f32(__builtin_amdgcn_fmed3f(c, -448.0f, 448.0f),
        __builtin_amdgcn_fmed3f(d, -448.0f, 448.0f), lower, true));
}

// x / b for many x and one b > 0, for a caller that encodes the quotient as e4m3: the code is the one the correctly
// rounded quotient __fdiv_rn(x, b) gives, on every pair a block quantiser can meet.
// The correctly rounded quotient costs about eleven instructions per element when the compiler expands the division
// (range scaling, reciprocal, two refinements of the reciprocal, quotient, two remainders, fix-up).  Everything that
// depends on b alone is done once here (SharedReciprocal): the reciprocal refined to within a rounding of 1 / b.  An
// element then takes a product, an exact remainder and one correction, plus the sign (b > 0, so the quotient has the
// sign of x; a zero remainder would otherwise turn -0 into +0).  The long form corrects the quotient twice and scales
// the operands' ranges; without that the quotient can be off in its last place (about one pair in five hundred) or,
// for very small divisors, by more.  An exhaustive run over all pairs of 16-bit element patterns and block maxima, bf16
// and fp16 (tests/cxx/shared_division_check.hip), found no pair whose e4m3 code differs for divisors with the exponent
// fields that SharedReciprocalHolds accepts; other divisors (block maxima below 2^-102, or infinite) take the long form.
__device__ __forceinline__ bool SharedReciprocalHolds(float b)
{
    const uint32_t exponent = (__float_as_uint(b) >> 23) & 0xffu;
    return exponent >= kSharedDivisionMinExponent && exponent <= kSharedDivisionMaxExponent;
}

__device__ __forceinline__ float SharedReciprocal(float b)
{
    const float y0 = __builtin_amdgcn_rcpf(b);
    const float e = __builtin_fmaf(-b, y0, 1.0f);
    return __builtin_fmaf(e, y0, y0);
}

__device__ __forceinline__ float DivideByShared(float x, float b, float y)
{
    const float q0 = __fmul_rn(x, y);
    const float r = __builtin_fmaf(-b, q0, x);
    return __builtin_copysignf(__builtin_fmaf(r, y, q0), x);
}

// True when one of the four e4m3 codes in `word` is a NaN code (0x7f / 0xff).
__device__ __forceinline__ bool Fp8E4m3WordHasNan(uint32_t word)
{
    return (((word & 0x7f7f7f7fu) + 0x01010101u) & 0x80808080u) != 0u;
}

// Four e4m3 codes -> four fp32 through the hardware convert alone: the values of Fp8Decode<false> for every code but
// the NaN code 0x7f, whose NaN comes back with the other sign.  For callers that notice a NaN in their result and then
// redo the work with Fp8E4m3DecodeWord.
__device__ __forceinline__ void Fp8E4m3DecodeWordFast(uint32_t word, float *out)
{
    const f32x2 lo = __builtin_amdgcn_cvt_pk_f32_fp8(static_cast<int>(word), false);
    const f32x2 hi = __builtin_amdgcn_cvt_pk_f32_fp8(static_cast<int>(word), true);
    out[0] = lo[0];
    out[1] = lo[1];
    out[2] = hi[0];
    out[3] = hi[1];
}

// Four e4m3 codes -> four fp32, same values as Fp8Decode<false> (NaN codes take the software path).
__device__ __forceinline__ void Fp8E4m3DecodeWord(uint32_t word, float *out)
{
    if (Fp8E4m3WordHasNan(word)) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            out[i] = Fp8Decode<false>((word >> (8 * i)) & 0xffu);
        }
        return;
    }
    const f32x2 lo = __builtin_amdgcn_cvt_pk_f32_fp8(static_cast<int>(word), false);
    const f32x2 hi = __builtin_amdgcn_cvt_pk_f32_fp8(static_cast<int>(word), true);
    out[0] = lo[0];
    out[1] = lo[1];
    out[2] = hi[0];
    out[3] = hi[1];
}

// Shared exponent of an MXFP8 block: clamp(floor(log2 amax) - emax, -127, 127); all-zero block -> -127.
template <bool E5M2>
__device__ __forceinline__ int MxSharedExponent(float amax)
{
    constexpr int kEmax = E5M2 ? 15 : 8;
    const uint32_t a = __float_as_uint(amax) & 0x7fffffffu;
    if (a == 0) {
        return -127;
    }
    int se = static_cast<int>(a >> 23) - 127 - kEmax;    // denormal amax gives < -127 and is clamped below
    se = se < -127 ? -127 : se;
    se = se > 127 ? 127 : se;
    return se;
}

// 2^e for e in [-127, 127] (2^-127 is a denormal fp32 and is produced exactly)
__device__ __forceinline__ float Exp2Int(int e)
{
    return e >= -126 ? __uint_as_float(static_cast<uint32_t>(e + 127) << 23) : __uint_as_float(0x00400000u);
}

// ---- MXFP8 through the scaled converts -------------------------------------------------------------------------------
//
// A block is 32 columns: the four words (eight elements) of a lane and those of the three other lanes of its quad.  The
// scaled converts take packed 16-bit elements as they are, divide by 2^e exactly and round once, two elements per
// instruction; an exhaustive comparison on gfx950 (tests/cxx/mx_convert_check.hip: every block maximum x every element
// under it, bf16 and fp16, e4m3 and e5m2) finds the functions below equal to Fp8Encode(ldexpf(x, -e)) and, back,
// code x scale, to Fp8Decode(code) * 2^e, subnormal results and the scale 2^-127 included.  The software codec costs about
// forty instructions per element, this about three.  What the converts do not do is saturate: elements beyond 1.75 * 2^emax times the scale are brought down to
// that value, which has the largest finite code, beforehand, as 16-bit magnitudes.
// Blocks that hold an infinity or a NaN take the software codec (MxScaling::plain is false).
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
typedef short s16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

constexpr uint32_t kPackedMagnitude = 0x7fff7fffu;

__device__ __forceinline__ uint32_t PackedMaxU16(uint32_t a, uint32_t b)
{
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(u16x2, a), __builtin_bit_cast(u16x2, b)));
}

__device__ __forceinline__ uint32_t PackedMinU16(uint32_t a, uint32_t b)
{
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_min(__builtin_bit_cast(u16x2, a), __builtin_bit_cast(u16x2, b)));
}

// Largest magnitude of the lane's block, as its 16-bit pattern (magnitudes of one format order like their patterns; a
// NaN is above the infinity).  All four lanes of the quad have to be active.
__device__ __forceinline__ uint32_t MxBlockMaxBits(const u32x4 &v)
{
    uint32_t m = PackedMaxU16(PackedMaxU16(v[0] & kPackedMagnitude, v[1] & kPackedMagnitude),
        PackedMaxU16(v[2] & kPackedMagnitude, v[3] & kPackedMagnitude));
    constexpr int kQuadSwap1 = 0xb1;        // lanes 1 0 3 2
    constexpr int kQuadSwap2 = 0x4e;        // lanes 2 3 0 1
    m = PackedMaxU16(m, static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(m), kQuadSwap1, 0xf, 0xf, true)));
    m = PackedMaxU16(m, static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(m), kQuadSwap2, 0xf, 0xf, true)));
    const uint32_t lo = m & 0xffffu;
    const uint32_t hi = m >> 16;
    return lo > hi ? lo : hi;
}

struct MxScaling {
    int exponent;           // MxSharedExponent of the block
    float scale;            // 2^exponent, the operand of the scaled converts
    uint32_t limit;         // magnitude that has the largest finite code, in both halves
    bool plain;             // every element is finite
};

template <bool BF16, bool E5M2>
__device__ __forceinline__ MxScaling MxScalingOf(uint32_t maxBits)
{
    constexpr int kEmax = E5M2 ? 15 : 8;
    MxScaling s;
    int biased;             // exponent field of the scale
    if (BF16) {
        // an exponent field below emax means a shared exponent clamped at -127, where nothing can saturate
        int e = static_cast<int>(maxBits >> 7);
        e = e < kEmax ? kEmax : e;
        biased = e - kEmax;
        const uint32_t one = (static_cast<uint32_t>(e) << 7) | 0x60u;
        s.limit = one | (one << 16);
        s.plain = maxBits < 0x7f80u;
    } else {
        const uint32_t bits = __float_as_uint(Decode16<false>(maxBits));
        biased = static_cast<int>(bits >> 23) - kEmax;          // at least 127 - 24 - emax, or below zero for a block of zeros
        biased = biased < 0 ? 0 : biased;
        // rounded down where it is a subnormal fp16: no magnitude lies between the two
        const float one = __uint_as_float((bits & 0x7f800000u) | 0x00600000u);
        s.limit = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(one, one));
        s.plain = maxBits < 0x7c00u;
    }
    s.exponent = biased - 127;
    // 2^-127 is a subnormal fp32
    const uint32_t bits = static_cast<uint32_t>(biased) << 23;
    s.scale = __uint_as_float(bits < 0x00400000u ? 0x00400000u : bits);
    return s;
}

// Two elements of a plain block -> two codes in the upper or lower half of `old`.
template <bool BF16, bool E5M2, bool UPPER>
__device__ __forceinline__ uint32_t MxEncodePair(uint32_t old, uint32_t pair, const MxScaling &s)
{
    const uint32_t clamped = PackedMinU16(pair & kPackedMagnitude, s.limit) | (pair & ~kPackedMagnitude);
    const s16x2 to = __builtin_bit_cast(s16x2, old);
    s16x2 r;
    if constexpr (BF16 && E5M2) {
        r = __builtin_amdgcn_cvt_scalef32_pk_bf8_bf16(to, __builtin_bit_cast(bf16x2, clamped), s.scale, UPPER);
    } else if constexpr (BF16) {
        r = __builtin_amdgcn_cvt_scalef32_pk_fp8_bf16(to, __builtin_bit_cast(bf16x2, clamped), s.scale, UPPER);
    } else if constexpr (E5M2) {
        r = __builtin_amdgcn_cvt_scalef32_pk_bf8_f16(to, __builtin_bit_cast(f16x2, clamped), s.scale, UPPER);
    } else {
        r = __builtin_amdgcn_cvt_scalef32_pk_fp8_f16(to, __builtin_bit_cast(f16x2, clamped), s.scale, UPPER);
    }
    return __builtin_bit_cast(uint32_t, r);
}

// The two codes in the lower half of `codes`, each times the block's scale.
template <bool E5M2>
__device__ __forceinline__ f32x2 MxDecodePair(uint32_t codes, const MxScaling &s)
{
    if constexpr (E5M2) {
        return __builtin_amdgcn_cvt_scalef32_pk_f32_bf8(codes, s.scale, false);
    } else {
        return __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(codes, s.scale, false);
    }
}

} // namespace TileXREp

#endif // TILEXR_AMD_EP_NUMERICS_HIP_H
