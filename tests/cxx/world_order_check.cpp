// Order of the launches of logical worlds (tilexr_amd/csrc/multi_rank.cpp) on a model of HIP's streams and events: an
// enqueued operation knows every operation it is ordered behind.  The launches do nothing but enqueue; no device, no
// runtime.  Built and run by tests/test_world_order.py on the CPU.
//
//   world_order_check <scenario>        exit status 0 = every expectation held
#include <cstdio>
#include <cstring>
#include <map>
#include <set>
#include <string>
#include <utility>
#include <vector>

#include "ep_context.h"
#include "ep_exchange.h"
#include "ep_host.h"
#include "ep_launch.h"

namespace TileXREp {
int RunDispatchMulti(EpComm *comm, const EpDispatchParams &p, bool memoryRoute, int64_t magic);
int RunCombineMulti(EpComm *comm, const EpCombineParams &p, bool memoryRoute, int64_t magic);
} // namespace TileXREp

using namespace TileXREp;

namespace {

struct Op {
    std::string name;
    std::set<int> behind;
};
std::vector<Op> gOps;
std::map<std::pair<void *, int>, std::set<int>> gTails;      // what the next operation of a stream is ordered behind
std::vector<std::set<int>> gEvents;
int gThread = 0;                                             // the calling host thread
int gLaunchesUntilFailure = -1;                              // of drains and reduces
int gFailures = 0;

std::set<int> &Tail(hipStream_t s)
{
    return gTails[{s, s == hipStreamPerThread ? gThread : 0}];
}

int Enqueue(hipStream_t s, const std::string &name)
{
    gOps.push_back({name, Tail(s)});
    Tail(s).insert(static_cast<int>(gOps.size()) - 1);
    return static_cast<int>(gOps.size()) - 1;
}

// Every operation `first` is ahead of every operation `then` that was enqueued at or after `from`.
void ExpectOrder(const std::string &first, const std::string &then, int from = 0)
{
    int pairs = 0;
    for (int b = from; b < static_cast<int>(gOps.size()); ++b) {
        if (gOps[static_cast<size_t>(b)].name != then) {
            continue;
        }
        for (int a = 0; a < b; ++a) {
            if (gOps[static_cast<size_t>(a)].name != first) {
                continue;
            }
            ++pairs;
            if (gOps[static_cast<size_t>(b)].behind.count(a) == 0) {
                std::printf("FAIL: '%s' (operation %d) is not ordered behind '%s' (%d)\n", then.c_str(), b, first.c_str(), a);
                ++gFailures;
            }
        }
    }
    if (pairs == 0) {
        std::printf("FAIL: no '%s' ahead of a '%s'\n", first.c_str(), then.c_str());
        ++gFailures;
    }
}

// Where the reduces of the calls so far found their tagged slot tables and their order keys.
struct Range {
    const char *first, *end;
};
std::vector<Range> gTagWords;
std::vector<Range> gKeyWords;

void NoteTables(const ReduceLaunch &l)
{
    const int64_t bytes = l.bs * (l.topK + l.sharedSlots) * 8;
    const char *tags = reinterpret_cast<const char *>(l.inverseTagged);
    gTagWords.push_back({tags, tags + bytes});
    if (l.orderKeys != nullptr) {
        const char *keys = reinterpret_cast<const char *>(l.orderKeys);
        gKeyWords.push_back({keys, keys + bytes});
    }
}

// A word that one call uses as an order key (a rank in its upper half) may not be one that another call takes for a slot's
// tag (an epoch in its upper half).
void ExpectTagsApartFromKeys()
{
    if (gTagWords.empty() || gKeyWords.empty()) {
        std::printf("FAIL: no tables were seen\n");
        ++gFailures;
    }
    for (const Range &t : gTagWords) {
        for (const Range &k : gKeyWords) {
            if (t.first < k.end && k.first < t.end) {
                std::printf("FAIL: order keys of one call lie where another looks for tags\n");
                ++gFailures;
                return;
            }
        }
    }
}

hipError_t SecondHalf(hipStream_t s, const char *name)
{
    if (gLaunchesUntilFailure == 0) {
        return hipErrorUnknown;
    }
    gLaunchesUntilFailure -= gLaunchesUntilFailure > 0 ? 1 : 0;
    Enqueue(s, name);
    return hipSuccess;
}

std::string Named(const char *what, int rank)
{
    return std::string(what) + " " + std::to_string(rank);
}

struct World {
    explicit World(int ranks) : comms(static_cast<size_t>(ranks))
    {
        world.rankSize = ranks;
        world.pendingDispatch.resize(comms.size());
        world.pendingCombine.resize(comms.size());
        world.dispatchOrder.reached.assign(comms.size(), nullptr);
        world.combineOrder.reached.assign(comms.size(), nullptr);
        for (int r = 0; r < ranks; ++r) {
            EpComm &c = comms[static_cast<size_t>(r)];
            c.world = &world;
            c.rank = r;
            world.comms.push_back(&c);
        }
    }
    int Call(bool combine, int r, hipStream_t stream, int64_t tokens = 4, bool memoryRoute = true)
    {
        static int32_t words[64] = {};
        EpComm *c = &comms[static_cast<size_t>(r)];
        if (combine) {
            EpCombineParams p {};
            p.bs = tokens, p.h = 64, p.topK = 2, p.moeExpertNum = world.rankSize;
            p.stream = stream;
            p.epRecvCounts = words;
            return RunCombineMulti(c, p, memoryRoute, 1);
        }
        EpDispatchParams p {};
        p.x = words;
        p.bs = 4, p.h = 64, p.topK = 2, p.moeExpertNum = world.rankSize;
        p.stream = stream;
        return RunDispatchMulti(c, p, true, 1);
    }
    EpWorld world;
    std::vector<EpComm> comms;
};

hipStream_t StreamNo(int i)
{
    return reinterpret_cast<hipStream_t>(static_cast<uintptr_t>(0x1000 + i));
}

// Work that ranks give their streams between their own call and the last one's stays ahead of the second half, and what
// they give them afterwards is behind it.
void LateWork(bool combine)
{
    const char *second = combine ? "reduce" : "drain";
    for (int last = 0; last < 3; ++last) {
        World w(3);
        for (int i = 1; i <= 3; ++i) {
            const int r = (last + i) % 3;
            if (w.Call(combine, r, StreamNo(r)) != 0) {
                ++gFailures;
            }
            if (r != last) {
                Enqueue(StreamNo(r), "meanwhile");
            }
        }
        for (int r = 0; r < 3; ++r) {
            Enqueue(StreamNo(r), "afterwards");
        }
    }
    for (int r = 0; r < 3; ++r) {
        ExpectOrder(Named(combine ? "return" : "send", r), second);
    }
    ExpectOrder("meanwhile", second);
    ExpectOrder(second, "afterwards");
}

// A second exchange, every rank on a stream of its own that no call has used yet.
void NextExchange(World &w, bool combine)
{
    const int from = static_cast<int>(gOps.size());
    for (int r = 0; r < w.world.rankSize; ++r) {
        if (w.Call(combine, r, StreamNo(100 + r)) != 0) {
            ++gFailures;
        }
    }
    for (int r = 0; r < w.world.rankSize; ++r) {
        ExpectOrder(combine ? "reduce" : "drain", Named(combine ? "return" : "send", r), from);
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
bool SmallDispatchFits(const SmallDispatchLaunch &) { return true; }
hipError_t LaunchSmallDispatch(const SmallDispatchLaunch &l)
{
    Enqueue(l.stream, Named("send", l.srcRank));
    return hipSuccess;
}
bool DrainPlansItself(int64_t, int64_t) { return true; }
hipError_t LaunchDrain(const DrainLaunch &l) { return SecondHalf(l.stream, "drain"); }
hipError_t LaunchReturnRows(const ReturnRowsLaunch &l)
{
    Enqueue(l.stream, Named("return", l.expertRank));
    return hipSuccess;
}
bool ReduceWorldFits(const ReduceLaunch *, int) { return true; }
hipError_t LaunchReduceWorld(const ReduceLaunch *ls, int ranks)
{
    for (int r = 0; r < ranks; ++r) {
        NoteTables(ls[r]);
    }
    return SecondHalf(ls[0].stream, "reduce");
}
hipError_t LaunchClearTagged(uint64_t *, int64_t, hipStream_t) { return hipErrorUnknown; }
// launches these calls do not make
hipError_t LaunchReduce(const ReduceLaunch &) { return hipErrorUnknown; }
hipError_t LaunchAugment(const AugmentLaunch &) { return hipErrorUnknown; }
hipError_t LaunchScatter(const ScatterLaunch &) { return hipErrorUnknown; }
hipError_t LaunchRouteRows(const RouteRowsLaunch &) { return hipErrorUnknown; }
hipError_t LaunchRouteCount(const RouteCountLaunch &) { return hipErrorUnknown; }
hipError_t LaunchDebugStamp(uint64_t *, uint64_t, int, int, hipStream_t) { return hipErrorUnknown; }
bool RouteRowsFits(const int32_t *, int64_t, int64_t, int, int64_t) { return false; }
bool RouteRowsPays(int64_t, int64_t, bool, bool) { return false; }
bool ScatterCopiesPerRoute(const void *, const void *, int64_t, int64_t, int64_t, int) { return false; }
CountScratchLayout PlanCountScratch(int64_t, int64_t, int64_t, bool) { return {}; }

} // namespace TileXREp

extern "C" {

hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned)
{
    gEvents.emplace_back();
    *e = reinterpret_cast<hipEvent_t>(gEvents.size());
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s)
{
    gEvents[reinterpret_cast<size_t>(e) - 1] = Tail(s);
    return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned)
{
    const std::set<int> &reached = gEvents[reinterpret_cast<size_t>(e) - 1];
    Tail(s).insert(reached.begin(), reached.end());
    return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *status)
{
    *status = hipStreamCaptureStatusNone;
    return hipSuccess;
}
const char *hipGetErrorString(hipError_t) { return "failure asked for"; }

}

int main(int argc, char **argv)
{
    const std::string scenario = argc > 1 ? argv[1] : "";
    const bool combine = argc > 2 && std::strcmp(argv[2], "combine") == 0;
    if (scenario == "late-work") {
        LateWork(combine);
    } else if (scenario == "next-exchange") {
        World w(3);
        for (int r = 0; r < 3; ++r) {
            gFailures += w.Call(combine, r, StreamNo(r)) != 0 ? 1 : 0;
        }
        NextExchange(w, combine);
    } else if (scenario == "per-thread-streams") {
        // every rank on hipStreamPerThread of a thread of its own
        World w(3);
        for (gThread = 0; gThread < 3; ++gThread) {
            gFailures += w.Call(combine, gThread, hipStreamPerThread) != 0 ? 1 : 0;
        }
        for (int r = 0; r < 3; ++r) {
            ExpectOrder(Named(combine ? "return" : "send", r), combine ? "reduce" : "drain");
        }
    } else if (scenario == "failed-launch") {
        // the second half takes two launches, of which the second fails
        World w(20);
        int status = 0;
        for (int r = 0; r < 20; ++r) {
            gLaunchesUntilFailure = r == 19 ? 1 : -1;
            status = w.Call(combine, r, StreamNo(r));
        }
        gLaunchesUntilFailure = -1;
        if (status == 0) {
            std::printf("FAIL: the failed launch was not reported\n");
            ++gFailures;
        }
        NextExchange(w, combine);
    } else if (scenario == "shapes") {
        // combines of several sizes, on both routes, through one world's tables
        World w(3);
        for (const bool memoryRoute : {false, true}) {
            for (const int64_t tokens : {4, 40, 7, 23}) {
                for (int r = 0; r < 3; ++r) {
                    gFailures += w.Call(true, r, StreamNo(r), tokens, memoryRoute) != 0 ? 1 : 0;
                }
            }
        }
        ExpectTagsApartFromKeys();
    } else {
        std::printf("unknown scenario\n");
        return 2;
    }
    std::printf("%d operations, %d failures\n", static_cast<int>(gOps.size()), gFailures);
    return gFailures == 0 ? 0 : 1;
}
