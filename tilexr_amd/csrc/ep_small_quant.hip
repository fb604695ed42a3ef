// The decode-sized dispatch of quantised rows (gfx950, wave64): ep_small.hip, ep_small_route.hip.h.
#include <type_traits>

#include "ep_small_route.hip.h"

namespace TileXREp {
namespace {

template <int QMODE, bool BF16, bool E5M2>
void LaunchMode(const SmallDispatchLaunch &l, const SmallArgs &a, unsigned workgroups)
{
    auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3(workgroups), dim3(kThreads), 0, l.stream, a); };
    auto pick = [&](auto vecsPerLane, auto masked) {
        constexpr int kV = decltype(vecsPerLane)::value;
        constexpr bool kMasked = decltype(masked)::value;
        if (l.tileFlags != nullptr) {
            launch(ep_dispatch_small_route_kernel<kV, kAuxAgentScope, kIdsPerLane, kMasked, QMODE, BF16, E5M2>);
        } else {
            launch(ep_dispatch_small_route_kernel<kV, kAuxAgentScopeKept, kIdsPerLane, kMasked, QMODE, BF16, E5M2>);
        }
    };
    auto pickMasked = [&](auto vecsPerLane) {
        if (l.maskMode != kMaskNone) {
            pick(vecsPerLane, std::true_type {});
        } else {
            pick(vecsPerLane, std::false_type {});
        }
    };
    if (l.h / 8 <= 2 * kThreads) {
        pickMasked(std::integral_constant<int, 2> {});
    } else {
        pickMasked(std::integral_constant<int, 4> {});
    }
}

template <bool BF16>
void LaunchByMode(const SmallDispatchLaunch &l, const SmallArgs &a, unsigned workgroups)
{
    if (l.quantMode == TILEXR_EP_QUANT_TOKEN_INT8) {
        LaunchMode<TILEXR_EP_QUANT_TOKEN_INT8, BF16, false>(l, a, workgroups);
    } else if (l.quantMode == TILEXR_EP_QUANT_FP8_BLOCK128) {
        LaunchMode<TILEXR_EP_QUANT_FP8_BLOCK128, BF16, false>(l, a, workgroups);
    } else if (l.fp8E5m2) {
        LaunchMode<TILEXR_EP_QUANT_MXFP8, BF16, true>(l, a, workgroups);
    } else {
        LaunchMode<TILEXR_EP_QUANT_MXFP8, BF16, false>(l, a, workgroups);
    }
}

} // namespace

hipError_t LaunchSmallQuantRoutes(const SmallDispatchLaunch &l, const SmallArgs &a, unsigned workgroups)
{
    if (l.mvp) {
        // MVP route: int8 rows, decoded as fp16, no flags, no mask
        auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3(workgroups), dim3(kThreads), 0, l.stream, a); };
        if (l.h / 8 <= 2 * kThreads) {
            launch(ep_dispatch_small_route_kernel<2, kAuxAgentScopeKept, kIdsPerLane, false, TILEXR_EP_QUANT_TOKEN_INT8, false, false, true>);
        } else {
            launch(ep_dispatch_small_route_kernel<4, kAuxAgentScopeKept, kIdsPerLane, false, TILEXR_EP_QUANT_TOKEN_INT8, false, false, true>);
        }
    } else if (l.inputBf16) {
        LaunchByMode<true>(l, a, workgroups);
    } else {
        LaunchByMode<false>(l, a, workgroups);
    }
    return hipGetLastError();
}

} // namespace TileXREp
