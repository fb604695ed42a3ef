// Exhaustive check of the MXFP8 codec through the scaled converts (MxScalingOf, MxEncodePair and MxDecodePair of
// tilexr_amd/csrc/ep_numerics.hip.h) against the software codec, on everything a block can hold: every non-negative 16-bit
// block maximum of the type (bf16 or fp16) with every element of no larger magnitude, both signs, e4m3 and e5m2.  Test
// infrastructure: built by tilexr_amd/csrc/Makefile into tests/cxx/bin/mx_convert_check and run by
// tests/test_gpu_mx_blocks.py.
//
//   mx_convert_check <bf16|fp16> <e4m3|e5m2>
//
// Passes when for every finite maximum the shared exponent is MxSharedExponent's, every element's code (in the lower and in
// the upper half of a word, beside a neighbour of another value) is Fp8Encode's of the element divided by the scale, and
// every such code times the scale is Fp8Decode's value times it, bit for bit; and when the maxima that are infinities or
// NaNs, and no others, ask for the software codec.
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>

#include <hip/hip_runtime.h>

#include "ep_numerics.hip.h"

namespace {

using namespace TileXREp;

struct Tally {
    unsigned long long pairs;
    unsigned long long exponent;
    unsigned long long code;
    unsigned long long value;
    unsigned long long plain;
    unsigned int haveFirst;
    unsigned int firstX;
    unsigned int firstMax;
};

// One workgroup per block maximum.
template <bool BF16, bool E5M2>
__global__ __launch_bounds__(256) void check_kernel(Tally *tally)
{
    constexpr uint32_t kInfinity = BF16 ? 0x7f80u : 0x7c00u;
    const uint32_t maxBits = blockIdx.x;                 // 0 .. 0x7fff: sign bit clear
    const MxScaling s = MxScalingOf<BF16, E5M2>(maxBits);
    const bool finite = maxBits < kInfinity;
    if (threadIdx.x == 0 && s.plain != finite) {
        atomicAdd(&tally->plain, 1ull);
    }
    if (!finite) {
        return;
    }
    const int exponent = MxSharedExponent<E5M2>(Decode16<BF16>(maxBits));
    const float up = Exp2Int(exponent);
    if (threadIdx.x == 0 && (s.exponent != exponent || __float_as_uint(s.scale) != __float_as_uint(up))) {
        atomicAdd(&tally->exponent, 1ull);
    }
    unsigned long long pairs = 0, badCode = 0, badValue = 0;
    for (uint32_t i = threadIdx.x; i < 2u * (maxBits + 1u); i += blockDim.x) {
        const uint32_t x = (i >> 1) | ((i & 1u) << 15);
        const uint32_t other = maxBits - (i >> 1);
        const uint32_t wantX = Fp8Encode<E5M2>(ldexpf(Decode16<BF16>(x), -exponent));
        const uint32_t wantOther = Fp8Encode<E5M2>(ldexpf(Decode16<BF16>(other), -exponent));
        const uint32_t low = MxEncodePair<BF16, E5M2, false>(0u, x | (other << 16), s);
        const uint32_t word = MxEncodePair<BF16, E5M2, true>(low, other | (x << 16), s);
        const uint32_t want = wantX | (wantOther << 8) | (wantOther << 16) | (wantX << 24);
        const f32x2 back = MxDecodePair<E5M2>(low, s);
        ++pairs;
        const bool sameCode = word == want && low == (want & 0xffffu);
        const bool sameValue = __float_as_uint(back[0]) == __float_as_uint(__fmul_rn(Fp8Decode<E5M2>(wantX), up)) &&
            __float_as_uint(back[1]) == __float_as_uint(__fmul_rn(Fp8Decode<E5M2>(wantOther), up));
        badCode += sameCode ? 0 : 1;
        badValue += sameValue ? 0 : 1;
        if (!(sameCode && sameValue) && atomicExch(&tally->haveFirst, 1u) == 0u) {
            tally->firstX = x;
            tally->firstMax = maxBits;
        }
    }
    atomicAdd(&tally->pairs, pairs);
    atomicAdd(&tally->code, badCode);
    atomicAdd(&tally->value, badValue);
}

#define HIP_OK(call)                                                                                  \
    do {                                                                                              \
        hipError_t e_ = (call);                                                                       \
        if (e_ != hipSuccess) {                                                                       \
            std::fprintf(stderr, "%s failed: %s\n", #call, hipGetErrorString(e_));                    \
            std::exit(2);                                                                             \
        }                                                                                             \
    } while (0)

} // namespace

int main(int argc, char **argv)
{
    const bool bf16 = argc > 1 && std::strcmp(argv[1], "bf16") == 0;
    const bool e5m2 = argc > 2 && std::strcmp(argv[2], "e5m2") == 0;
    if (argc != 3 || (!bf16 && std::strcmp(argv[1], "fp16") != 0) || (!e5m2 && std::strcmp(argv[2], "e4m3") != 0)) {
        std::fprintf(stderr, "usage: mx_convert_check <bf16|fp16> <e4m3|e5m2>\n");
        return 2;
    }
    HIP_OK(hipSetDevice(0));
    Tally *dev = nullptr;
    HIP_OK(hipMalloc(&dev, sizeof(Tally)));
    HIP_OK(hipMemset(dev, 0, sizeof(Tally)));
    const auto kernel = bf16 ? (e5m2 ? check_kernel<true, true> : check_kernel<true, false>) :
                               (e5m2 ? check_kernel<false, true> : check_kernel<false, false>);
    hipLaunchKernelGGL(kernel, dim3(0x8000), dim3(256), 0, nullptr, dev);
    HIP_OK(hipGetLastError());
    HIP_OK(hipDeviceSynchronize());
    Tally host;
    HIP_OK(hipMemcpy(&host, dev, sizeof(Tally), hipMemcpyDeviceToHost));
    HIP_OK(hipFree(dev));
    if (host.haveFirst != 0) {
        std::printf("first difference: element 0x%04x in a block of maximum 0x%04x\n", host.firstX, host.firstMax);
    }
    const bool ok = host.exponent == 0 && host.code == 0 && host.value == 0 && host.plain == 0;
    std::printf("%s %s %s: %llu pairs, %llu exponents, %llu codes, %llu values, %llu choices of the codec differ\n",
        ok ? "OK" : "DIFF", argv[1], argv[2], host.pairs, host.exponent, host.code, host.value, host.plain);
    return ok ? 0 : 1;
}
