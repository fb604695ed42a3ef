// Dispatch / combine across several logical ranks that share the device (rankSize > 1).
//
// The reference runs one process per rank and lets kernels spin on flags in each other's peer windows
// (src/ep/kernels/tilexr_ep_dispatch_kernel.cpp:700-836, tilexr_ep_dispatch_memory_kernel.h:1549-1562).  With every
// rank in one process and on one device, spinning kernels could starve each other, so the exchange is ordered by
// the host instead: a call enqueues its rank's SEND half on the caller's stream immediately; when the last rank of
// the world has called, the second half of all ranks (dispatch: one drain launch; combine: the reduces) is enqueued on
// that last caller's stream, behind everything the other ranks' streams have been given by then and ahead of what they
// are given afterwards.
// A rank's outputs are therefore complete once every rank has made the call and the rank's stream has been synchronised
// -- the same moment the reference's kernels would pass their barriers.
#include <algorithm>

#include "ep_context.h"
#include "ep_exchange.h"
#include "ep_host.h"
#include "ep_launch.h"
#include "ep_run_common.h"

namespace TileXREp {
namespace {

constexpr int kOk = TileXR::TILEXR_SUCCESS;

constexpr int kReduceBatch = 16;

// Timed for one launch that works for `ranks` ranks from `first` on: every one of them records its events and stamps.
template <typename Launch>
int TimedForRanks(EpWorld *world, int first, int ranks, int kernel, hipStream_t stream, const char *what, Launch launch)
{
    if (ranks == 0) {
        return LaunchStatus(launch(), what);
    }
    int inner = kOk;
    const int outer = Timed(world->comms[static_cast<size_t>(first)], kernel, stream, what, [&] {
        inner = TimedForRanks(world, first + 1, ranks - 1, kernel, stream, what, launch);
        return hipSuccess;
    });
    return inner != kOk ? inner : outer;
}

int64_t Align256(int64_t v)
{
    return (v + 255) / 256 * 256;
}

int64_t MxScaleBytes(int64_t h)
{
    return ((h + 31) / 32 + 1) / 2 * 2;
}

// What a call of a logical world mostly consists of is the runtime's price for ordering streams: a kernel launch costs
// the calling thread 2.5 us, a wait for an event that another stream has just recorded 4 to 8 us, one for an event recorded
// a little earlier much less.  Hence one launch per half and one wait per other rank's stream at either end of the second
// half.
bool EnsureEvent(hipEvent_t *e)
{
    return *e != nullptr || hipEventCreateWithFlags(e, hipEventDisableTiming) == hipSuccess;
}

// The first half of a call waits for the world's previous exchange, whose second half reads the staging it overwrites.
bool AwaitPrevious(const ExchangeOrder &order, hipStream_t stream)
{
    return !order.doneArmed || hipStreamWaitEvent(stream, order.done, 0) == hipSuccess;
}

// hipStreamPerThread names another stream in every thread.  What such a rank's own thread has not recorded, the last
// caller's cannot.
bool NamesOneStream(hipStream_t stream)
{
    return stream != hipStreamPerThread;
}

// Behind the first half of rank r's call, for a stream that JoinStreams cannot name.
bool MarkSent(ExchangeOrder *order, int r, hipStream_t stream)
{
    hipEvent_t *e = &order->reached[static_cast<size_t>(r)];
    return EnsureEvent(e) && (NamesOneStream(stream) || hipEventRecord(*e, stream) == hipSuccess);
}

// `stream` waits for the other ranks' streams as they stand: their first halves, and whatever their callers have given
// them since, which may fill or read an output or write an input that only the second half reads.  All events are recorded
// before the first is waited for: 4 ranks x 128 x 1024, 2 routes, 156 us a layer, 192 us with each wait right behind its
// record.  (Recorded behind the first halves they cost 15 us less and leave out what follows those.)
template <typename Pending>
bool JoinStreams(const ExchangeOrder &order, const std::vector<Pending> &calls, hipStream_t stream)
{
    auto isOther = [&](hipStream_t s) { return s != stream || !NamesOneStream(s); };
    for (size_t r = 0; r < calls.size(); ++r) {
        hipStream_t s = StreamOf(calls[r].params.stream);
        if (isOther(s) && NamesOneStream(s) && hipEventRecord(order.reached[r], s) != hipSuccess) {
            return false;
        }
    }
    for (size_t r = 0; r < calls.size(); ++r) {
        if (isOther(StreamOf(calls[r].params.stream)) && hipStreamWaitEvent(stream, order.reached[r], 0) != hipSuccess) {
            return false;
        }
    }
    return true;
}

// Marks the end of the exchange on `stream` and makes the other ranks' streams wait for it.  Also where a launch failed:
// the ones ahead of it still read the staging that the next exchange overwrites.
template <typename Pending>
bool ReleaseStreams(ExchangeOrder *order, const std::vector<Pending> &calls, hipStream_t stream)
{
    if (!EnsureEvent(&order->done) || hipEventRecord(order->done, stream) != hipSuccess) {
        return false;
    }
    order->doneArmed = true;
    for (const Pending &c : calls) {
        hipStream_t other = StreamOf(c.params.stream);
        if (other != stream && hipStreamWaitEvent(other, order->done, 0) != hipSuccess) {
            return false;
        }
    }
    return true;
}

// Key space of a world: position = rank * keysPerRank + local index on that rank.  Without shared experts this is
// the expert id itself (keysPerRank = experts per rank).  With shared experts (reference: expert placement in
// src/ep/kernels/tilexr_ep_dispatch_helpers.h:63-103) ranks [0, sharedRanks) host them, the routed experts are spread
// over the other ranks, and a shared route takes local index 0 on its rank (memory route: a shared rank presents one
// local expert, tilexr_ep_dispatch_memory_kernel.h:1153) or its own expert id (MVP route: the drain files a shared row
// under index expertId, tilexr_ep_combine_helpers.h:124-128), hence keysPerRank = max(localExperts, sharedNum) there.
struct StagePlan {
    StageLayout layout {};
    int64_t rowBytes = 0;
    int64_t scaleBytesPerRow = 0;
    int64_t numKeys = 0;
    int64_t keyDiv = 1;
    int64_t localExperts = 0;    // routed experts per non-shared rank
    int64_t keysPerRank = 0;
    int64_t keySpace = 0;        // rankSize * keysPerRank
    int64_t perToken = 0;        // routes per token: shared + topK
    bool expertHist = false;
};

// Sizes the world's staging for one dispatch shape and points `layout` at it.
bool PlanStage(EpWorld *world, const ExchangeShape &shape, bool reserve, StagePlan *plan)
{
    const int64_t R = world->rankSize;
    plan->perToken = shape.topK + shape.sharedNum;
    const int64_t n = shape.bs * plan->perToken;
    // with tensor-parallel groups (MVP route) experts are placed on the R / tp expert ranks and a key names an
    // expert rank; the lane a row travels on is the source's own (reference: tilexr_ep_dispatch_kernel.cpp:382-392)
    const int64_t expertRanks = R / shape.tp;
    plan->localExperts = shape.experts / (expertRanks - shape.sharedRanks);
    plan->keysPerRank = shape.memoryRoute ? plan->localExperts : std::max(plan->localExperts, shape.sharedNum);
    plan->keySpace = expertRanks * plan->keysPerRank;
    plan->rowBytes = shape.quantMode == TILEXR_EP_QUANT_NONE ? shape.h * 2 : shape.h;
    plan->scaleBytesPerRow = shape.quantMode == TILEXR_EP_QUANT_TOKEN_INT8 ? 4 :
        (shape.quantMode == TILEXR_EP_QUANT_MXFP8 ? MxScaleBytes(shape.h) : 0);
    plan->numKeys = shape.memoryRoute ? plan->keySpace : expertRanks;
    plan->keyDiv = shape.memoryRoute ? 1 : plan->keysPerRank;
    plan->expertHist = !shape.memoryRoute;
    StageLayout &l = plan->layout;
    l.rowsStride = Align256(n * plan->rowBytes);
    l.scalesOffset = Align256(n * 16);
    l.auxStride = l.scalesOffset + Align256(n * plan->scaleBytesPerRow);
    l.expertTotalOffset = plan->numKeys + 1;
    l.countsStride = (plan->numKeys + 1 + plan->keySpace + 63) / 64 * 64;
    if (reserve) {
        if (!world->stageRows.Reserve(static_cast<size_t>(R * l.rowsStride), false) ||
            !world->stageAux.Reserve(static_cast<size_t>(R * l.auxStride), false) ||
            !world->stageCounts.Reserve(static_cast<size_t>(R * l.countsStride * 4), true)) {
            return false;
        }
    }
    l.rows = static_cast<char *>(world->stageRows.ptr);
    l.aux = static_cast<char *>(world->stageAux.ptr);
    l.counts = static_cast<int32_t *>(world->stageCounts.ptr);
    return true;
}

// The send half of a call of any size and kind: this rank's rows grouped by destination key in its staging area, in two
// launches (three with shared experts).
int SendRoutes(EpComm *comm, const EpDispatchParams &p, bool memoryRoute, const ExchangeShape &shape, const StagePlan &plan)
{
    const int R = comm->world->rankSize;
    const int r = comm->rank;
    const int64_t shared = shape.sharedNum;
    const int64_t tp = shape.tp;
    const int64_t n = p.bs * plan.perToken;
    hipStream_t stream = StreamOf(p.stream);
    const CountScratchLayout cs = PlanCountScratch(n, plan.numKeys, plan.keySpace, plan.expertHist);
    const int64_t tableBytes = shared > 0 ? Align256(n * 4) : 0;      // key ids, tuple expert ids, widened mask
    if (!comm->dispatchScratch.Reserve(static_cast<size_t>(cs.totalBytes + 3 * tableBytes), true)) {
        return TileXR::TILEXR_ERROR_INTERNAL;
    }
    const uint8_t *routeMask = reinterpret_cast<const uint8_t *>(p.xActiveMask);
    CountScratch scratch = CarveCountScratch(comm->dispatchScratch.ptr, cs, plan.expertHist);
    const int32_t *routeIds = p.expertIds;
    const int32_t *tupleExperts = nullptr;
    if (shared > 0) {
        int32_t *keyIds = reinterpret_cast<int32_t *>(static_cast<char *>(comm->dispatchScratch.ptr) + cs.totalBytes);
        int32_t *tuples = reinterpret_cast<int32_t *>(static_cast<char *>(comm->dispatchScratch.ptr) + cs.totalBytes +
            tableBytes);
        AugmentLaunch aug {};
        aug.ids = p.expertIds;
        aug.bs = p.bs;
        aug.topK = p.topK;
        aug.moeExpertNum = p.moeExpertNum;
        aug.rankSize = R;
        aug.srcRank = static_cast<int>(r / tp);      // the placement rules see the source's expert rank
        aug.sharedNum = static_cast<int>(shared);
        aug.sharedRanks = static_cast<int>(p.sharedExpertRankNum);
        aug.localExperts = static_cast<int>(plan.localExperts);
        aug.keysPerRank = static_cast<int>(plan.keysPerRank);
        aug.sharedAtExpertId = !memoryRoute;
        aug.keyIdsOut = keyIds;
        aug.tupleExpertsOut = tuples;
        if (memoryRoute && p.xActiveMask != nullptr && p.activeMaskType == TILEXR_EP_ACTIVE_MASK_EXPERT) {
            uint8_t *wide = reinterpret_cast<uint8_t *>(static_cast<char *>(comm->dispatchScratch.ptr) + cs.totalBytes +
                2 * tableBytes);
            aug.routeMask = routeMask;
            aug.routeMaskOut = wide;
            routeMask = wide;
        }
        aug.stream = stream;
        const int ar = LaunchStatus(LaunchAugment(aug), "route tables");
        if (ar != kOk) {
            return ar;
        }
        routeIds = keyIds;
        tupleExperts = tuples;
    }
    int32_t *myCounts = plan.layout.counts + static_cast<int64_t>(r) * plan.layout.countsStride;
    scratch.keyOffset = myCounts;
    scratch.expertTotal = myCounts + plan.layout.expertTotalOffset;
    int32_t *rowOf = reinterpret_cast<int32_t *>(static_cast<char *>(comm->dispatchScratch.ptr) + cs.rowOfOff);
    char *myRows = plan.layout.rows + static_cast<int64_t>(r) * plan.layout.rowsStride;
    char *myAux = plan.layout.aux + static_cast<int64_t>(r) * plan.layout.auxStride;

    int maskMode = kMaskNone;
    if (p.xActiveMask != nullptr) {
        maskMode = !memoryRoute ? kMaskPerToken :
            (p.activeMaskType == TILEXR_EP_ACTIVE_MASK_EXPERT ? kMaskPerRoute : kMaskTokenPrefix);
    }
    // as on a single rank (api.cpp): the rows resolved in one launch where that pays, else count and place, the latter
    // folded into the scatter; the launch ahead of a scatter that copies per route reads the token rows ahead
    const bool warm = ScatterCopiesPerRoute(p.x, myRows, p.bs, p.h, plan.perToken, static_cast<int>(p.quantMode));
    const bool oneLaunch = memoryRoute && shared == 0 && comm->routing != EpComm::Routing::kLegacy &&
        RouteRowsFits(routeIds, n, plan.numKeys, maskMode, 0) &&
        (comm->routing == EpComm::Routing::kOneLaunch || (RouteRowsPays(n, plan.numKeys, false, warm) &&
            (maskMode == kMaskNone || p.bs <= kRowsMaskedTokens)));
    int ret = kOk;
    RoutePlaceLaunch place {};
    if (oneLaunch) {
        RouteRowsLaunch rows {};
        rows.ids = routeIds;
        rows.bs = p.bs;
        rows.topK = plan.perToken;
        rows.numKeys = plan.numKeys;
        rows.srcRank = r;
        rows.rowOf = rowOf;
        rows.assist = reinterpret_cast<int32_t *>(myAux);
        // exclusive offsets of the keys: a zero, then the inclusive sums, the last of which is the total
        rows.firstOffsetOut = myCounts;
        rows.sendCountsOut = myCounts + 1;
        rows.totalRowsOut = myCounts + plan.numKeys;
        rows.tokenNumsType = static_cast<int>(p.expertTokenNumsType);
        rows.warmRows = warm ? p.x : nullptr;
        rows.warmBytes = p.bs * p.h * 2;
        rows.mask = routeMask;
        rows.stream = stream;
        comm->lastKernel[kKernelCount] = "ep_route_rows_kernel";
        ret = Timed(comm, kKernelCount, stream, "route rows", [&] { return LaunchRouteRows(rows); });
    } else {
        RouteCountLaunch count {};
        count.ids = routeIds;
        count.mask = routeMask;
        count.maskMode = maskMode;
        count.bs = p.bs;
        count.topK = plan.perToken;
        count.numExperts = plan.keySpace;
        count.keyDiv = plan.keyDiv;
        count.numKeys = plan.numKeys;
        count.capacity = 0;
        count.scratch = scratch;
        count.tokenNumsType = static_cast<int>(p.expertTokenNumsType);
        count.stream = stream;
        count.warmRows = warm ? p.x : nullptr;
        count.warmBytes = p.bs * p.h * 2;
        comm->lastKernel[kKernelCount] = "ep_route_count_kernel";
        ret = Timed(comm, kKernelCount, stream, "route count", [&] { return LaunchRouteCount(count); });
        place.ids = routeIds;
        place.bs = p.bs;
        place.topK = plan.perToken;
        place.keyDiv = plan.keyDiv;
        place.numKeys = plan.numKeys;
        place.scratch = scratch;
        place.srcRank = r;
        place.expertIdBias = 0;
        place.sharedNum = static_cast<int32_t>(shared);
        place.tupleExperts = tupleExperts;
        place.rowOf = nullptr;          // the scatter resolves its own rows
        place.assist = reinterpret_cast<int32_t *>(myAux);
        place.stream = stream;
    }
    if (ret != kOk) {
        return ret;
    }
    ScatterLaunch scatter {};
    scatter.x = p.x;
    scatter.rowOf = rowOf;
    scatter.fusedPlace = oneLaunch ? nullptr : &place;
    scatter.bs = p.bs;
    scatter.h = p.h;
    scatter.topK = plan.perToken;
    scatter.quantMode = static_cast<int>(p.quantMode);
    scatter.inputBf16 = memoryRoute && p.dtype == TileXR::TILEXR_DATA_TYPE_BFP16;
    scatter.fp8E5m2 = p.expandXOutDtype == TileXR::TILEXR_DATA_TYPE_FP8E5M2;
    scatter.staticScale = static_cast<const float *>(p.scales);
    scatter.out = myRows;
    scatter.combineTakesRows = true;        // the drain does (MXFP8 and static int8 rows stream all the same)
    scatter.scalesOut = myAux + plan.layout.scalesOffset;
    scatter.stream = stream;
    return Timed(comm, kKernelScatter, stream, "scatter", [&] { return LaunchScatter(scatter); });
}

// The drain of every rank of the world, on the stream of the last rank to call.
int DrainWorld(EpWorld *world, const ExchangeShape &shape, const StagePlan &plan, hipStream_t stream)
{
    const int R = world->rankSize;
    if (!JoinStreams(world->dispatchOrder, world->pendingDispatch, stream)) {
        return TileXR::TILEXR_ERROR_INTERNAL;
    }
    const int64_t maxSegments = shape.memoryRoute ? std::max<int64_t>(plan.localExperts, 1) * R : R;
    if (!DrainPlansItself(maxSegments, plan.localExperts) &&
        !world->drainPlans.Reserve(static_cast<size_t>(R * (maxSegments + 1)) * 4, false)) {
        return TileXR::TILEXR_ERROR_INTERNAL;
    }
    DrainLaunch drain {};
    drain.stage = plan.layout;
    drain.rankSize = R;
    drain.localExperts = static_cast<int>(plan.keysPerRank);
    drain.tp = static_cast<int>(shape.tp);
    drain.memoryRoute = shape.memoryRoute;
    drain.rowBytes = plan.rowBytes;
    drain.scaleBytesPerRow = plan.scaleBytesPerRow;
    drain.routesPerRank = shape.bs * plan.perToken;
    drain.stream = stream;
    int ret = kOk;
    for (int q = 0; q < R && ret == kOk; ++q) {
        const EpDispatchParams &p = world->pendingDispatch[static_cast<size_t>(q)].params;
        DrainTarget &d = drain.target[drain.targets++];
        d = DrainTarget {};
        d.dstRank = q;
        // a shared-expert rank presents one local expert on the memory route
        // (reference: src/ep/kernels/tilexr_ep_dispatch_memory_kernel.h:1153, tests/ep/demo/tilexr_ep_dispatch_demo.cpp:632-635)
        d.outLocalExperts = q < shape.sharedRanks ? 1 : static_cast<int>(plan.localExperts);
        d.tokenNumsCount = shape.memoryRoute ? d.outLocalExperts : static_cast<int>(plan.localExperts);
        d.tokenNumsType = static_cast<int>(p.expertTokenNumsType);
        d.planOffsets = world->drainPlans.ptr == nullptr ? nullptr :
            static_cast<int32_t *>(world->drainPlans.ptr) + q * (maxSegments + 1);
        d.countsOut = p.epRecvCountsOut;
        d.tpCountsOut = shape.memoryRoute ? nullptr : p.tpRecvCountsOut;
        d.expertTokenNumsOut = p.expertTokenNumsOut;
        d.expandXOut = static_cast<char *>(p.expandXOut);
        d.assistOut = p.assistInfoForCombineOut;
        d.scalesOut = static_cast<char *>(p.dynamicScalesOut);
        if (drain.targets == kDrainTargets || q == R - 1) {
            ret = LaunchStatus(LaunchDrain(drain), "drain");
            drain.targets = 0;
        }
    }
    if (!ReleaseStreams(&world->dispatchOrder, world->pendingDispatch, stream) && ret == kOk) {
        ret = TileXR::TILEXR_ERROR_INTERNAL;
    }
    return ret;
}

} // namespace

int RunDispatchMulti(EpComm *comm, const EpDispatchParams &p, bool memoryRoute, int64_t magic)
{
    EpWorld *world = comm->world;
    const int R = world->rankSize;
    const int r = comm->rank;
    const int64_t shared = p.sharedExpertNum;
    const int64_t tp = (!memoryRoute && p.tpWorldSize > 1) ? p.tpWorldSize : 1;
    const int64_t keySpaceBound = static_cast<int64_t>(R / tp) *
        std::max(p.moeExpertNum / (R / tp - p.sharedExpertRankNum), shared);
    if (!WithinKernelLimits(p.bs, p.h, p.topK + shared, std::max(p.moeExpertNum, keySpaceBound), R) || p.extended) {
        return TileXR::TILEXR_ERROR_NOT_SUPPORT;
    }
    hipStream_t stream = StreamOf(p.stream);
    ExchangeShape shape {};
    shape.bs = p.bs;
    shape.h = p.h;
    shape.topK = p.topK;
    shape.experts = p.moeExpertNum;
    shape.quantMode = p.quantMode;
    shape.sharedNum = shared;
    shape.sharedRanks = p.sharedExpertRankNum;
    shape.tp = tp;
    shape.dtype = static_cast<int>(p.dtype);
    shape.outDtype = static_cast<int>(p.expandXOutDtype);
    shape.memoryRoute = memoryRoute;

    std::lock_guard<std::mutex> lock(world->mu);
    comm->debug.magic = magic;
    for (int s = 0; s < R; ++s) {
        if (world->comms[static_cast<size_t>(s)] == nullptr) {
            return TileXR::TILEXR_ERROR_NOT_INITIALIZED;     // the world is not complete yet
        }
    }
    if (world->pendingDispatch[static_cast<size_t>(r)].present) {
        return TileXR::TILEXR_ERROR_INTERNAL;                // this rank already sent in the exchange in flight
    }
    bool first = true;
    for (const PendingDispatch &pd : world->pendingDispatch) {
        first = first && !pd.present;
    }
    if (first) {
        world->dispatchShape = shape;
    } else if (!(shape == world->dispatchShape)) {
        return TileXR::TILEXR_ERROR_PARA_CHECK_FAIL;         // all ranks of one exchange use the same shape
    }
    StagePlan plan {};
    if (!PlanStage(world, shape, first, &plan)) {
        return TileXR::TILEXR_ERROR_INTERNAL;
    }
    if (!AwaitPrevious(world->dispatchOrder, stream)) {
        return TileXR::TILEXR_ERROR_INTERNAL;
    }

    // ---- send half: group this rank's rows by destination in its staging area ----
    int ret = kOk;
    SmallDispatchLaunch small {};
    if (memoryRoute && p.quantMode == TILEXR_EP_QUANT_NONE && shared == 0) {
        // decode-sized: the same one launch that serves such a call on a single rank, into the staging area
        small.x = p.x;
        small.ids = p.expertIds;
        small.bs = p.bs;
        small.h = p.h;
        small.topK = p.topK;
        small.numExperts = plan.keySpace;
        small.mask = reinterpret_cast<const uint8_t *>(p.xActiveMask);
        small.maskMode = p.xActiveMask == nullptr ? kMaskNone :
            (p.activeMaskType == TILEXR_EP_ACTIVE_MASK_EXPERT ? kMaskPerRoute : kMaskTokenPrefix);
        small.srcRank = r;
        small.out = plan.layout.rows + static_cast<int64_t>(r) * plan.layout.rowsStride;
        small.assist = reinterpret_cast<int32_t *>(plan.layout.aux + static_cast<int64_t>(r) * plan.layout.auxStride);
        // exclusive offsets of the keys: a zero, then the inclusive sums
        small.firstOffsetOut = plan.layout.counts + static_cast<int64_t>(r) * plan.layout.countsStride;
        small.sendCountsOut = small.firstOffsetOut + 1;
        small.kernelNameOut = &comm->lastKernel[kKernelScatter];
        small.stream = stream;
    }
    if (small.x != nullptr && SmallDispatchFits(small)) {
        ret = Timed(comm, kKernelScatter, stream, "small dispatch", [&] { return LaunchSmallDispatch(small); });
    } else {
        ret = SendRoutes(comm, p, memoryRoute, shape, plan);
    }
    if (ret == kOk && !MarkSent(&world->dispatchOrder, r, stream)) {
        ret = TileXR::TILEXR_ERROR_INTERNAL;
    }
    if (ret != kOk) {
        return ret;
    }
    world->pendingDispatch[static_cast<size_t>(r)].present = true;
    world->pendingDispatch[static_cast<size_t>(r)].params = p;

    // ---- drain halves, once the last rank has sent ----
    for (const PendingDispatch &pd : world->pendingDispatch) {
        if (!pd.present) {
            return kOk;
        }
    }
    ret = DrainWorld(world, shape, plan, stream);
    for (PendingDispatch &pd : world->pendingDispatch) {
        pd.present = false;
    }
    return ret;
}

int RunCombineMulti(EpComm *comm, const EpCombineParams &p, bool memoryRoute, int64_t magic)
{
    (void)magic;
    EpWorld *world = comm->world;
    const int R = world->rankSize;
    const int er = comm->rank;
    // shared-expert rows come back to the slots after the routed ones on the memory route; the MVP route's combine
    // drops them (reference: src/ep/kernels/tilexr_ep_combine_kernel.cpp:94-97)
    const int64_t shared = memoryRoute ? p.sharedExpertNum : 0;
    const int64_t perToken = p.topK + shared;
    if (!WithinKernelLimits(p.bs, p.h, perToken, p.moeExpertNum, R) || p.extended) {
        return TileXR::TILEXR_ERROR_NOT_SUPPORT;
    }
    hipStream_t stream = StreamOf(p.stream);
    ExchangeShape shape {};
    shape.bs = p.bs;
    shape.h = p.h;
    shape.topK = p.topK;
    shape.experts = p.moeExpertNum;
    shape.quantMode = p.quantMode;
    shape.sharedNum = shared;
    shape.sharedRanks = memoryRoute ? p.sharedExpertRankNum : 0;
    shape.dtype = static_cast<int>(p.dtype);
    shape.memoryRoute = memoryRoute;

    std::lock_guard<std::mutex> lock(world->mu);
    comm->debug.magic = magic;
    for (int s = 0; s < R; ++s) {
        if (world->comms[static_cast<size_t>(s)] == nullptr) {
            return TileXR::TILEXR_ERROR_NOT_INITIALIZED;
        }
    }
    if (world->pendingCombine[static_cast<size_t>(er)].present) {
        return TileXR::TILEXR_ERROR_INTERNAL;
    }
    bool first = true;
    for (const PendingCombine &pc : world->pendingCombine) {
        first = first && !pc.present;
    }
    const int64_t n = p.bs * perToken;
    const int64_t rowBytes = p.h * 2;
    const int64_t slotsStride = Align256(n * rowBytes);
    const int64_t metaStride = (n + 31) / 32 * 32;
    if (first) {
        world->combineShape = shape;
        ++world->combineEpoch;
        if (!world->combineSlots.Reserve(static_cast<size_t>(R * slotsStride), false) ||
            !world->combineMeta.Reserve(static_cast<size_t>(R * metaStride * 8), true) ||
            (!memoryRoute && !world->combineKeys.Reserve(static_cast<size_t>(R * metaStride * 8), false))) {
            return TileXR::TILEXR_ERROR_INTERNAL;
        }
    } else if (!(shape == world->combineShape)) {
        return TileXR::TILEXR_ERROR_PARA_CHECK_FAIL;
    }
    if (!AwaitPrevious(world->combineOrder, stream)) {
        return TileXR::TILEXR_ERROR_INTERNAL;
    }
    const uint64_t epoch = world->combineEpoch & 0xffffffffull;

    // ---- send half: every row of this expert rank goes back to the slot (token, k) of its source rank ----
    ReturnRowsLaunch back {};
    back.expertOut = p.expertOut;
    back.assist = p.assistInfoForCombine;
    back.counts = p.epRecvCounts;
    // memory route: the rows of this expert rank = last entry of its sendCounts, which has one block of R entries per
    // local expert (a single block on a shared-expert rank)
    const int64_t localExperts = p.moeExpertNum / (R - shape.sharedRanks);
    back.numCounts = memoryRoute ? (er < shape.sharedRanks ? 1 : localExperts) * R : R;
    back.memoryRoute = memoryRoute;
    back.maxCountPerEntry = n;
    back.maxRows = static_cast<int64_t>(R) * n;
    back.routesPerRank = n;
    back.rowBytes = rowBytes;
    back.rankSize = R;
    back.expertRank = er;
    back.bs = p.bs;
    back.topK = perToken;
    back.epoch = epoch;
    back.slots = static_cast<char *>(world->combineSlots.ptr);
    back.slotsStride = slotsStride;
    back.meta = static_cast<uint64_t *>(world->combineMeta.ptr);
    back.orderKeys = memoryRoute ? nullptr : static_cast<uint64_t *>(world->combineKeys.ptr);
    back.metaStride = metaStride;
    back.stream = stream;
    int ret = LaunchStatus(LaunchReturnRows(back), "return rows");
    if (ret == kOk && !MarkSent(&world->combineOrder, er, stream)) {
        ret = TileXR::TILEXR_ERROR_INTERNAL;
    }
    if (ret != kOk) {
        return ret;
    }
    world->pendingCombine[static_cast<size_t>(er)].present = true;
    world->pendingCombine[static_cast<size_t>(er)].params = p;
    for (const PendingCombine &pc : world->pendingCombine) {
        if (!pc.present) {
            return kOk;
        }
    }

    // ---- reduce halves ----
    int status = JoinStreams(world->combineOrder, world->pendingCombine, stream) ? kOk : TileXR::TILEXR_ERROR_INTERNAL;
    std::vector<ReduceLaunch> reduces(static_cast<size_t>(R));
    for (int r = 0; r < R; ++r) {
        const EpCombineParams &rp = world->pendingCombine[static_cast<size_t>(r)].params;
        ReduceLaunch &red = reduces[static_cast<size_t>(r)];
        red.expertOut = static_cast<char *>(world->combineSlots.ptr) + static_cast<int64_t>(r) * slotsStride;
        red.rowBytes = rowBytes;
        red.inverseTagged = back.meta + static_cast<int64_t>(r) * metaStride;
        red.epoch = epoch;
        red.orderKeys = memoryRoute ? nullptr : back.orderKeys + static_cast<int64_t>(r) * metaStride;
        red.expertScales = memoryRoute ? rp.expertScales : nullptr;
        red.tokenMask = memoryRoute ? reinterpret_cast<const uint8_t *>(rp.xActiveMask) : nullptr;
        red.sharedExpertX = memoryRoute ? rp.sharedExpertX : nullptr;
        red.reduceKind = memoryRoute ? kReduceFp32 : kReducePerAdd;
        red.commQuant = memoryRoute ? static_cast<int>(rp.quantMode) : 0;
        red.bf16 = rp.dtype == TileXR::TILEXR_DATA_TYPE_BFP16;
        red.bs = rp.bs;
        red.h = rp.h;
        red.topK = rp.topK;
        red.sharedSlots = shared;
        red.y = rp.yOut;
        red.numComputeUnits = world->numComputeUnits;
        red.stream = stream;
        red.kernelNameOut = &world->comms[static_cast<size_t>(r)]->lastKernel[kKernelReduce];
    }
    // batches of ranks in one launch each, or a launch per rank for rows that take another kernel
    for (int first = 0; first < R && status == kOk; first += kReduceBatch) {
        const int ranks = std::min(kReduceBatch, R - first);
        const ReduceLaunch *batch = reduces.data() + first;
        if (ReduceWorldFits(batch, ranks)) {
            status = TimedForRanks(world, first, ranks, kKernelReduce, stream, "reduce", [&] { return LaunchReduceWorld(batch, ranks); });
        } else {
            for (int r = 0; r < ranks && status == kOk; ++r) {
                status = Timed(world->comms[static_cast<size_t>(first + r)], kKernelReduce, stream, "reduce",
                    [&] { return LaunchReduce(batch[r]); });
            }
        }
    }
    if (status == kOk && IsCapturing(stream)) {
        // replays share this exchange's epoch: each finds the tables empty
        status = LaunchStatus(LaunchClearTagged(back.meta, R * metaStride, stream), "clear of the slot tables");
    }
    if (!ReleaseStreams(&world->combineOrder, world->pendingCombine, stream) && status == kOk) {
        status = TileXR::TILEXR_ERROR_INTERNAL;
    }
    for (PendingCombine &pc : world->pendingCombine) {
        pc.present = false;
    }
    return status;
}

} // namespace TileXREp
