// The launches of a plan-driven Dispatch: tilexr_amd/csrc/moonep_stage.hip's host side, linked against a runtime that only
// notes what is launched.  Built and run by tests/test_plan_launches.py on the CPU.
//
//   plan_launches_check <ranks> <tokens> <top-k> <hidden> <rows per rank> <fresh>      a line per launch: kernel, grid x and y, dynamic LDS
#include <cstdio>
#include <cstdlib>
#include <map>
#include <string>

#include <hip/hip_runtime_api.h>

#include "moonep_stage.h"

namespace {

std::map<const void *, std::string> gKernels;
dim3 gGrid, gBlock;
size_t gLds;

} // namespace

extern "C" {

void **__hipRegisterFatBinary(const void *)
{
    static void *module;
    return &module;
}

void __hipUnregisterFatBinary(void **) {}

void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, void *, void *, int *)
{
    gKernels[host] = name;
}

hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t)
{
    gLds = lds;
    gGrid = grid;
    gBlock = block;
    return hipSuccess;
}

hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *lds, hipStream_t *stream)
{
    *grid = gGrid;
    *block = gBlock;
    *lds = gLds;
    *stream = nullptr;
    return hipSuccess;
}

hipError_t hipLaunchKernel(const void *host, dim3 grid, dim3, void **, size_t lds, hipStream_t)
{
    std::printf("%s %u %u %zu\n", gKernels[host].c_str(), grid.x, grid.y, lds);
    return hipSuccess;
}

hipError_t hipGetLastError()
{
    return hipSuccess;
}

hipError_t hipEventRecord(hipEvent_t, hipStream_t)
{
    return hipSuccess;
}

} // extern "C"

int main(int argc, char **argv)
{
    if (argc != 7) {
        return 2;
    }
    TileXRMoon::DispatchWorld w {};
    w.world = std::atoi(argv[1]);
    w.s = std::atoll(argv[2]);
    w.k = std::atoll(argv[3]);
    w.h = std::atoll(argv[4]);
    w.nvS = std::atoll(argv[5]);
    w.fresh = std::atoi(argv[6]) != 0;
    return TileXRMoon::LaunchMoonDispatch(w, nullptr, {}) == hipSuccess ? 0 : 1;
}
