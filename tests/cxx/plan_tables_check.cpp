// Where the plan-driven stages (tilexr_amd/csrc/moonep_api.cpp) put a world's tables for calls of several sizes: words that
// carry the number of their exchange are never cleared, so a place where one size keeps anything else may not be one where
// another size looks for such words.  The launches only note the tables; no device, no runtime.  Built and run by
// tests/test_plan_tables.py on the CPU.
//
//   plan_tables_check <ranks>        exit status 0 = every expectation held
#include <cstdio>
#include <cstdlib>
#include <map>
#include <vector>

#include "ep_context.h"
#include "moonep_stage.h"
#include "tilexr_moonep.h"

namespace {

struct Range {
    const char *first, *end;
};
std::vector<Range> gTagged;      // looked through for words of the running exchange
std::vector<Range> gOther;       // everything else
std::vector<TileXREp::EpComm> gComms;
int gFailures = 0;

template <typename T>
Range RangeOf(T *first, int64_t count)
{
    return {reinterpret_cast<const char *>(first), reinterpret_cast<const char *>(first + count)};
}

constexpr size_t kTagged = 8, kOther = 6;     // tables of a call

bool Overlap(const Range &a, const Range &b)
{
    return a.first < b.end && b.first < a.end;
}

void Expect(bool ok, const char *what)
{
    if (!ok) {
        std::printf("FAIL: %s\n", what);
        ++gFailures;
    }
}

void NoteTables(int world, const TileXRMoon::WorldTables &t)
{
    const int64_t n = world * t.stride;
    for (uint64_t *words : {t.rowTag, t.parentTag, t.groupStart, t.slotSrc, t.slotDup, t.slotGroup}) {
        gTagged.push_back(RangeOf(words, n));
    }
    gTagged.push_back(RangeOf(t.fail, world));
    gTagged.push_back(RangeOf(t.chunkTag, n / TileXRMoon::kTableAlign));
    gOther.push_back(RangeOf(t.sibling, n));
    gOther.push_back(RangeOf(t.slotCount, n));
    gOther.push_back(RangeOf(t.chunkTotals, world * t.groupStride * 2));
    gOther.push_back(RangeOf(t.direct, n));
    gOther.push_back(RangeOf(t.origin, n));
    // (zero between dispatches, of whatever sizes: neither another table's place nor one that moves with the sizes)
    gOther.push_back(RangeOf(t.arrived, 1));
    static const uint32_t *const arrived = t.arrived;
    Expect(t.arrived == arrived, "the count of built plans is at another place");
}

TileXRMoonEpTensorV1 Tensor(uint32_t dtype, int64_t rows, int64_t columns)
{
    static char memory[64];
    TileXRMoonEpTensorV1 t {};
    t.structSize = sizeof(t);
    t.abiVersion = TILEXR_MOONEP_ABI_VERSION_V1;
    t.data = memory;
    t.dtype = dtype;
    t.rank = 2;
    t.shape[0] = rows;
    t.shape[1] = columns;
    t.elementCount = static_cast<uint64_t>(rows * columns);
    return t;
}

// One Dispatch that builds its plan, one Combine and one Dispatch along the plan, by every rank.
void Exchange(int ranks, int64_t tokens, int64_t k, int64_t nvS)
{
    static int32_t words[64];
    TileXRMoonEpPlanV1 plan {};
    plan.structSize = sizeof(plan);
    plan.abiVersion = TILEXR_MOONEP_ABI_VERSION_V1;
    plan.n = tokens * k;
    plan.r = ranks;
    plan.e = ranks;
    plan.b = 1;
    plan.nvS = nvS;
    plan.k = k;
    plan.dst = plan.expertsToCopy = plan.zeroFillRanges = plan.remoteStats = plan.dupGroups = plan.dupLoffs = plan.dupCounts =
        plan.status = words;
    TileXRMoonEpTensorV1 sh = Tensor(TILEXR_MOONEP_DTYPE_BFLOAT16, tokens, 64);
    TileXRMoonEpTensorV1 nvsh = Tensor(TILEXR_MOONEP_DTYPE_BFLOAT16, nvS, 64);
    for (int stage = 0; stage < 3; ++stage) {
        for (int r = 0; r < ranks; ++r) {
            aclrtStream stream = reinterpret_cast<aclrtStream>(static_cast<uintptr_t>(0x1000 + r));
            int status = 0;
            if (stage == 1) {
                TileXRMoonEpCombineArgsV1 a {};
                a.structSize = sizeof(a);
                a.abiVersion = TILEXR_MOONEP_ABI_VERSION_V1;
                a.comm = &gComms[static_cast<size_t>(r)];
                a.plan = &plan;
                a.dstLocal = words;
                a.hiddenNvsh = &nvsh;
                a.hiddenSh = &sh;
                status = TileXRMoonEpCombineV1(&a, stream);
            } else {
                TileXRMoonEpDispatchArgsV1 a {};
                a.structSize = sizeof(a);
                a.abiVersion = TILEXR_MOONEP_ABI_VERSION_V1;
                a.comm = &gComms[static_cast<size_t>(r)];
                a.plan = &plan;
                a.hiddenSh = &sh;
                a.hiddenNvsh = &nvsh;
                a.flags = stage == 0 ? TILEXR_MOONEP_FLAG_BUILD_DEDUP : 0;
                status = TileXRMoonEpDispatchV1(&a, stream);
            }
            Expect(status == 0, "a call was refused");
        }
    }
}

} // namespace

namespace TileXREp {

bool DeviceBuffer::Reserve(size_t want, bool)
{
    // every buffer has addresses of its own, and room for whatever is asked of it
    static std::map<DeviceBuffer *, uintptr_t> places;
    ptr = reinterpret_cast<void *>(places.emplace(this, (places.size() + 1) << 40).first->second);
    bytes = want;
    return true;
}
void DeviceBuffer::Release() {}
hipError_t LaunchClearTagged(uint64_t *, int64_t, hipStream_t) { return hipErrorUnknown; }
EpComm *LookupComm(TileXRCommPtr comm) { return static_cast<EpComm *>(comm); }

} // namespace TileXREp

namespace TileXRMoon {

hipError_t LaunchMoonDispatch(const DispatchWorld &w, hipStream_t, const LaunchTiming &)
{
    NoteTables(w.world, w.tables);
    return hipSuccess;
}
hipError_t LaunchMoonCombine(const CombineWorld &w, hipStream_t, const LaunchTiming &)
{
    NoteTables(w.world, w.tables);
    return hipSuccess;
}
hipError_t LaunchMoonStatus(int32_t *, int32_t, hipStream_t) { return hipSuccess; }
int64_t SetCachedRowBytes(int64_t) { return 0; }
const char *MoonScatterKernelName() { return ""; }
const char *MoonReduceKernelName() { return ""; }

} // namespace TileXRMoon

extern "C" {

hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned)
{
    *e = reinterpret_cast<hipEvent_t>(static_cast<uintptr_t>(0x10));
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned)
{
    *s = reinterpret_cast<hipStream_t>(static_cast<uintptr_t>(0x20));
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *status)
{
    *status = hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipMemset(void *, int, size_t) { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "failure"; }

}

int main(int argc, char **argv)
{
    const int ranks = argc > 1 ? std::atoi(argv[1]) : 1;
    TileXREp::EpWorld world;
    world.rankSize = ranks;
    world.deviceReady = true;
    gComms = std::vector<TileXREp::EpComm>(static_cast<size_t>(ranks));
    for (int r = 0; r < ranks; ++r) {
        TileXREp::EpComm &c = gComms[static_cast<size_t>(r)];
        c.world = &world;
        c.rank = r;
        c.host.rank = r;
        c.host.rankSize = ranks;
        c.host.localRank = r;
        c.host.localRankSize = ranks;
        world.comms.push_back(&c);
    }
    Exchange(ranks, 2048, 8, 16384);
    Exchange(ranks, 16, 8, 128);
    Exchange(ranks, 300, 2, 5000);
    Exchange(ranks, 1, 1, 1);
    Expect(gTagged.size() == 4 * 3 * kTagged, "tables of every exchange");
    bool apart = true;
    for (const Range &t : gTagged) {
        for (const Range &o : gOther) {
            apart = apart && !Overlap(t, o);
        }
    }
    Expect(apart, "one size's untagged words lie where another looks for tagged ones");
    // within a call no two tables share a word
    for (size_t call = 0; call < gTagged.size() / kTagged; ++call) {
        std::vector<Range> all(gTagged.begin() + static_cast<long>(call * kTagged), gTagged.begin() + static_cast<long>((call + 1) * kTagged));
        all.insert(all.end(), gOther.begin() + static_cast<long>(call * kOther), gOther.begin() + static_cast<long>((call + 1) * kOther));
        for (size_t i = 0; i < all.size(); ++i) {
            for (size_t j = 0; j < i; ++j) {
                Expect(!Overlap(all[i], all[j]), "two tables of a call overlap");
            }
        }
    }
    std::printf("%zu tables, %d failures\n", gTagged.size() + gOther.size(), gFailures);
    return gFailures == 0 ? 0 : 1;
}
