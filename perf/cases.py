"""The work this library is used for, as cases that a timing harness can run: one MoE layer's dispatch and combine
(with the identity as expert stage), through the entry points a program calls.

`listed()` names the cases, `draw(rng)` gives further ones of the same ranges, `prepare(case, seed)` makes what a program
holds before the call, `run(state)` is one pass, `work(case)` the bytes a pass cannot do without and `tolerance(case)` how
closely outputs have to agree.

Kinds of case:
  ref    TileXRMoeEpDispatchMemoryV2 + TileXRMoeEpCombineMemoryV2: plain or MXFP8 rows, optionally a token mask and a
         shared-expert row per token
  ex     TileXRMoeEpDispatchMemoryEx + TileXRMoeEpCombineMemoryEx with the row map: plain, int8 or block fp8 rows, a
         capacity per expert, readiness flags on one stream
  graph  eight layers of `ex` calls, each on its predecessor's output, captured once in a HIP graph and replayed
  layer  tilexr_amd.layer.MoeEpLayer, the torch-facing wrapper that allocates the outputs
  mvp    TileXRMoeEpDispatchV2 + TileXRMoeEpCombineV2: plain or int8 rows
  world  the memory route across several logical ranks of the device, one stream per rank
  plan   the plan-driven stages: forward (the duplicate plan is built), optionally backward too (dispatch along the
         saved plan is the adjoint of combine, combine that of dispatch)
"""
import math

import torch

from tilexr_amd import ep, layer, workloads
from tilexr_amd import moonep as mp

DEV = "cuda:0"
GRAPH_LAYERS = 8
TORCH_TYPE = {"bf16": torch.bfloat16, "fp16": torch.float16}
EP_TYPE = {"bf16": ep.DT_BF16, "fp16": ep.DT_FP16}
QUANT = {"none": ep.Q_NONE, "int8": ep.Q_TOKEN_INT8, "mxfp8": ep.Q_MXFP8, "fp8": ep.Q_FP8_BLOCK128}


def case_of(kind, tokens, hidden, top_k, experts, routing="gating", **more):
    c = dict(kind=kind, tokens=tokens, hidden=hidden, top_k=top_k, experts=experts, routing=routing, dtype="bf16",
             payload="none", capacity_factor=0.0, flags=False, masked=False, shared=False, ranks=1, backward=False)
    c.update(more)
    return c


def listed():
    return [
        # the smallest decode step: a handful of sequences, called eagerly
        case_of("ref", 8, 7168, 8, 256, name="decode_8_eager"),
        # a full decode batch of a serving loop that replays a captured graph
        case_of("graph", 128, 7168, 8, 256, name="decode_128_graph"),
        # a decode batch padded to a fixed size, the padding masked out, with the shared expert's row added in combine
        case_of("ref", 200, 7168, 8, 256, masked=True, shared=True, name="decode_200_masked_shared"),
        # a chunk of a prompt beside decode, from a torch program
        case_of("layer", 1000, 7168, 8, 256, "zipf", name="chunk_1000_torch"),
        # the target configuration: prefill with tile readiness flags
        case_of("ex", 4096, 7168, 8, 256, "zipf", flags=True, name="prefill_4096_flags"),
        # the largest prefill: token rows and receive rows far beyond every cache
        case_of("ex", 16384, 7168, 8, 256, "zipf", name="prefill_16384"),
        # quantised dispatch, per-token int8, dequantised in combine
        case_of("ex", 8192, 4096, 6, 64, "uniform", payload="int8", name="int8_8192"),
        # heavily skewed routing under a capacity limit, block fp8
        case_of("ex", 16384, 2048, 8, 128, "zipf12", payload="fp8", capacity_factor=1.25, name="fp8_16384_capacity"),
        # MXFP8 rows out of dispatch, MXFP8 exchange in combine
        case_of("ref", 2048, 7168, 8, 256, payload="mxfp8", name="mxfp8_2048"),
        # the route ordered by source rank, in fp16, with a ragged number of tokens
        case_of("mvp", 1501, 4096, 6, 64, "uniform", dtype="fp16", name="mvp_1501_fp16"),
        # several logical ranks on one device
        case_of("world", 128, 1024, 2, 16, "uniform", ranks=4, name="world_4x128"),
        # a training step's four stages along a plan
        case_of("plan", 4096, 7168, 8, 8, "uniform", backward=True, name="plan_4096_train"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


# bytes of routed 16-bit rows of the largest listed case: a drawn one has no more
_MOST_ROW_BYTES = 16384 * 8 * 7168 * 2


def draw(rng):
    kind = rng.choice(["ref", "ref", "ex", "ex", "ex", "graph", "layer", "layer", "mvp", "world", "plan"])
    payload = "none"
    if kind == "ex":
        payload = rng.choice(["none", "int8", "fp8"])
    elif kind == "ref":
        payload = rng.choice(["none", "none", "mxfp8"])
    elif kind == "layer":
        payload = rng.choice(["none", "none", "int8", "fp8"])
    elif kind == "mvp":
        payload = rng.choice(["none", "int8"])
    hidden = rng.choice([1024, 2048, 4096, 7168, 8192])
    if kind in ("layer", "mvp", "world", "plan") and payload == "none":
        hidden = rng.choice([1000, 1024, 2048, 4096, 7168])
    experts = rng.choice([16, 32, 64, 128, 256])
    top_k = rng.choice([1, 2, 4, 5, 6, 8, 8])
    most = {"ref": 8192, "ex": 16384, "graph": 256, "layer": 8192, "mvp": 4096, "world": 1024, "plan": 4096}[kind]
    least = {"ex": 512, "layer": 64, "mvp": 64, "world": 16, "plan": 128}.get(kind, 1)
    ranks = rng.choice([2, 4, 8]) if kind == "world" else rng.choice([1, 1, 2, 4]) if kind == "plan" else 1
    tokens = min(_log_int(rng, least, most), _MOST_ROW_BYTES // (ranks * top_k * hidden * 2))
    more = dict(payload=payload, ranks=ranks)
    if kind in ("ref", "ex", "layer"):
        more["dtype"] = rng.choice(["bf16", "bf16", "fp16"])
    elif kind == "mvp":
        more["dtype"] = "fp16" if payload == "int8" else rng.choice(["bf16", "fp16"])
    if kind == "ref":
        more["masked"] = rng.random() < 0.4
        more["shared"] = rng.random() < 0.4
    if kind == "ex":
        more["flags"] = rng.random() < 0.4
        more["capacity_factor"] = rng.choice([0.0, 0.0, 1.25])
    if kind == "plan":
        more["backward"] = rng.random() < 0.5
        experts = max(ranks, rng.choice([8, 16, 32]))
    routing = rng.choice(["gating", "uniform", "zipf", "zipf12"])
    return case_of(kind, tokens, hidden, min(top_k, experts), experts, routing, **more)


# ---- inputs --------------------------------------------------------------------------------------------------------
def _popularity(case, dev, gen):
    """Logits of the experts' popularity: Zipf over a seeded permutation, or level."""
    e = case["experts"]
    s = {"zipf": 1.0, "zipf12": 1.2}.get(case["routing"], 0.0)
    logp = -s * torch.log(torch.arange(1, e + 1, dtype=torch.float32, device=dev))
    return logp[torch.randperm(e, device=dev, generator=gen)]


def _routing(case, tokens, dev, gen):
    """(ids int32 [tokens, K] of distinct experts, weights fp32): the K best of random gating logits, or Gumbel keys, which
    samples without replacement in proportion to the popularity."""
    e, k = case["experts"], case["top_k"]
    if case["routing"] == "gating":
        top, ids = torch.topk(torch.randn(tokens, e, device=dev, generator=gen), k, dim=1)
        weights = torch.softmax(top, dim=1)
    else:
        logp = _popularity(case, dev, gen)
        u = torch.rand(tokens, e, device=dev, generator=gen).clamp_(1e-12, 1.0 - 1e-7)
        ids = torch.topk(logp - torch.log(-torch.log(u)), k, dim=1).indices
        weights = torch.softmax(torch.randn(tokens, k, device=dev, generator=gen), dim=1)
    return ids.to(torch.int32).contiguous(), weights.float().contiguous()


def _rows(case, tokens, gen):
    """Token rows: N(0, 1), and for block fp8 the heavy-tailed ones that payload is for (Student-t, 3 degrees)."""
    x = torch.randn(tokens, case["hidden"], device=DEV, generator=gen)
    if case["payload"] == "fp8":
        chi = sum(torch.randn(tokens, case["hidden"], device=DEV, generator=gen).square_() for _ in range(3))
        x = x / torch.sqrt(chi / 3.0)
    return x.to(TORCH_TYPE[case["dtype"]])


def _capacity(case):
    if case["capacity_factor"] <= 0:
        return 0
    return int(math.ceil(case["capacity_factor"] * case["tokens"] * case["top_k"] / case["experts"]))


def _active(case):
    """Tokens that the mask leaves active: a prefix, as in a batch padded to a fixed size."""
    return max(1, case["tokens"] * 4 // 5) if case["masked"] else case["tokens"]


def _scale_shape(payload, rows, hidden):
    if payload == "int8":
        return (rows, 1), torch.float32
    if payload == "mxfp8":
        return (rows, ((hidden + 31) // 32 + 1) // 2 * 2), torch.uint8
    return (rows, (hidden + 127) // 128), torch.float32


_comms = {}


def _handles(ranks):
    """The communicators and streams a program keeps for its lifetime."""
    if ranks not in _comms:
        torch.cuda.set_device(0)
        _comms[ranks] = ([ep.Comm(ranks, r) for r in range(ranks)], [torch.cuda.Stream() for _ in range(ranks)])
    return _comms[ranks]


_layers = {}


def _outputs(case, rows, local_experts, counts, dev=DEV):
    """What a dispatch writes.  Zero-filled: rows that no route is placed in stay as they are."""
    h, payload = case["hidden"], case["payload"]
    o = dict(rows=torch.zeros((rows, h), dtype=TORCH_TYPE[case["dtype"]] if payload == "none" else torch.uint8, device=dev),
             assist=torch.zeros((rows, 4), dtype=torch.int32, device=dev),
             token_nums=torch.zeros((local_experts,), dtype=torch.int64, device=dev),
             counts=torch.zeros((counts,), dtype=torch.int32, device=dev), scales=None)
    if payload != "none":
        shape, dtype = _scale_shape(payload, rows, h)
        o["scales"] = torch.zeros(shape, dtype=dtype, device=dev)
    return o


def _generator(seed, dev=DEV):
    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    return g


def prepare(case, seed):
    torch.cuda.set_device(0)
    gen = _generator(seed)
    s = dict(case=case)
    if case["kind"] == "plan":
        return _prepare_plan(case, seed, s)
    bs, h, k, e, ranks = case["tokens"], case["hidden"], case["top_k"], case["experts"], case["ranks"]
    tdt = TORCH_TYPE[case["dtype"]]
    if case["kind"] == "graph":
        return _prepare_graph(case, gen, s)
    if case["kind"] == "layer":
        key = (e, k, h)
        if key not in _layers:
            _layers[key] = layer.MoeEpLayer(e, k, h)
        s["layer"] = _layers[key]
        s["x"] = _rows(case, bs, gen)
        s["ids"], s["weights"] = _routing(case, bs, DEV, gen)
        return s
    s["comms"], s["streams"] = _handles(ranks)
    s["ranks"] = []
    for _ in range(ranks):
        r = dict(x=_rows(case, bs, gen), y=torch.zeros((bs, h), dtype=tdt, device=DEV))
        r["ids"], r["weights"] = _routing(case, bs, DEV, gen)
        local = e // ranks
        r.update(_outputs(case, ranks * bs * k, local, 1 if case["kind"] == "mvp" else local * ranks))
        if case["masked"]:
            r["mask"] = (torch.arange(bs, device=DEV) < _active(case)).to(torch.uint8)
        if case["shared"]:
            r["shared"] = _rows(case, bs, gen)
        if case["kind"] in ("ref", "mvp") and case["payload"] != "none":
            # these combines take rows of the output type, not the payload: what an expert stage computed from it
            r["expert_out"] = torch.randn(bs * k, h, device=DEV, generator=gen).to(tdt)
        if case["kind"] == "ex":
            r["row_map"] = torch.zeros((bs, k), dtype=torch.int32, device=DEV)
            if case["flags"]:
                r["tile_flags"] = torch.zeros(((bs * k + 63) // 64,), dtype=torch.int64, device=DEV)
                r["status"] = torch.zeros((1,), dtype=torch.int32, device=DEV)
        s["ranks"].append(r)
    return s


class _Graph:
    """Layers captured on a communicator and a stream of their own."""

    def __init__(self):
        self.comm, self.stream, self.graph = ep.Comm(1, 0), torch.cuda.Stream(), torch.cuda.CUDAGraph()

    def __del__(self):
        try:
            torch.cuda.synchronize()
            self.comm.destroy()
        except Exception:
            pass


def _prepare_graph(case, gen, s):
    bs, h, k, e = case["tokens"], case["hidden"], case["top_k"], case["experts"]
    g = _Graph()
    s["x"] = _rows(case, bs, gen)
    s["layers"] = []
    for _ in range(GRAPH_LAYERS):
        r = _outputs(case, bs * k, e, e)
        r["ids"], r["weights"] = _routing(case, bs, DEV, gen)
        r["row_map"] = torch.zeros((bs, k), dtype=torch.int32, device=DEV)
        r["y"] = torch.zeros((bs, h), dtype=TORCH_TYPE[case["dtype"]], device=DEV)
        if s["layers"]:
            r["rows"] = s["layers"][0]["rows"]       # one receive buffer for every layer
        s["layers"].append(r)

    def layers():
        x = s["x"]
        for r in s["layers"]:
            _run_ex(case, dict(r, x=x), g.comm, g.stream)
            x = r["y"]

    torch.cuda.synchronize()
    layers()
    torch.cuda.synchronize()
    with torch.cuda.graph(g.graph, stream=g.stream):
        layers()
    torch.cuda.synchronize()
    s["graph"] = g
    return s


def _plan_ids(case, seed):
    gen = _generator(seed, "cpu")
    ranks, s, e, k = case["ranks"], case["tokens"], case["experts"], case["top_k"]
    return torch.topk(torch.rand(ranks, s, e, generator=gen), k, dim=2).indices.to(torch.int32)


def _prepare_plan(case, seed, s):
    ranks, tokens, k, h, e = case["ranks"], case["tokens"], case["top_k"], case["hidden"], case["experts"]
    gen = _generator(seed)
    plan = workloads.moonep_home_plan(_plan_ids(case, seed), e)
    nvs = plan["nvs"]
    local = workloads.moonep_dst_local(plan["dst"], nvs)
    s["comms"], s["streams"] = _handles(ranks)
    s["ranks"] = []
    for r in range(ranks):
        t = dict(dst=plan["dst"][r].to(DEV), dst_local=local[r].to(DEV),
                 groups=torch.zeros((nvs, 3), dtype=torch.int32, device=DEV),
                 loffs=torch.zeros((nvs,), dtype=torch.int32, device=DEV),
                 counts=torch.zeros((2,), dtype=torch.int32, device=DEV),
                 status=torch.zeros((8,), dtype=torch.int32, device=DEV),
                 x=_rows(case, tokens, gen), weights=torch.rand(tokens, k, device=DEV, generator=gen),
                 rows=torch.zeros((nvs, h), dtype=torch.bfloat16, device=DEV),
                 row_weights=torch.zeros((nvs,), dtype=torch.float32, device=DEV),
                 y=torch.zeros((tokens, h), dtype=torch.bfloat16, device=DEV),
                 y_weights=torch.zeros((tokens, k), dtype=torch.float32, device=DEV))
        t["plan"] = mp.plan(tokens * k, ranks, e, 1, nvs, k, t["dst"], t["groups"], t["loffs"], t["counts"], t["status"])
        if case["backward"]:
            t["grad_y"] = _rows(case, tokens, gen)
            t["grad_rows"] = torch.zeros_like(t["rows"])
            t["grad_x"] = torch.zeros_like(t["x"])

        def desc(name, dtype, shape, t=t):
            return mp.tensor(t[name], dtype, shape)

        t["fwd"] = ((desc("x", mp.DT_BF16, (tokens, h)), desc("rows", mp.DT_BF16, (nvs, h)), desc("y", mp.DT_BF16, (tokens, h))),
                    (desc("weights", mp.DT_FP32, (tokens, k)), desc("row_weights", mp.DT_FP32, (nvs,)),
                     desc("y_weights", mp.DT_FP32, (tokens, k))))
        if case["backward"]:
            t["bwd"] = (desc("grad_y", mp.DT_BF16, (tokens, h)), desc("grad_rows", mp.DT_BF16, (nvs, h)),
                        desc("grad_x", mp.DT_BF16, (tokens, h)))
        s["ranks"].append(t)
    return s


# ---- one pass ------------------------------------------------------------------------------------------------------
def _run_ex(case, r, comm, stream):
    bs, h, k, e = case["tokens"], case["hidden"], case["top_k"], case["experts"]
    dt, q = EP_TYPE[case["dtype"]], QUANT[case["payload"]]
    flags = r.get("tile_flags")
    tile_rows = 64 if flags is not None else 0
    st, epoch = ep.dispatch_memory_ex(r["x"], r["ids"], comm, bs, h, k, e, r["rows"], r["assist"], r["token_nums"],
                                      r["counts"], dt, stream, quant_mode=q, expert_capacity=_capacity(case),
                                      dynamic_scales=r["scales"], row_index_map=r["row_map"], tile_flags=flags,
                                      tile_rows=tile_rows)
    ep.check(st, "dispatch")
    ep.check(ep.combine_memory_ex(r["rows"], r["assist"], r["counts"], comm, bs, h, k, e, r["y"], dt, stream,
                                  expert_out_quant_mode=q, expert_out_scales=r["scales"], expert_scales=r["weights"],
                                  row_index_map=r["row_map"], tile_flags=flags, tile_rows=tile_rows,
                                  flag_epoch=epoch if flags is not None else 0, device_status=r.get("status")), "combine")


def _run_ref(case, s):
    bs, h, k, e = case["tokens"], case["hidden"], case["top_k"], case["experts"]
    dt, q = EP_TYPE[case["dtype"]], QUANT[case["payload"]]
    mask_type = ep.MASK_TOKEN if case["masked"] else ep.MASK_NONE
    for r, comm, stream in zip(s["ranks"], s["comms"], s["streams"]):
        ep.check(ep.dispatch_memory_v2(r["x"], r["ids"], comm, bs, h, k, e, r["rows"], r["assist"], r["token_nums"],
                                       r["counts"], dt, stream, active_mask=r.get("mask"), active_mask_type=mask_type,
                                       quant_mode=q, dynamic_scales=r["scales"],
                                       expand_x_dtype=ep.DT_FP8E4M3 if q else ep.DT_RESERVED), "dispatch")
    for r, comm, stream in zip(s["ranks"], s["comms"], s["streams"]):
        ep.check(ep.combine_memory_v2(r.get("expert_out", r["rows"]), r["assist"], r["counts"], comm, bs, h, k, e, r["y"], dt,
                                      stream, expert_scales=r["weights"], active_mask=r.get("mask"),
                                      active_mask_type=mask_type, shared_expert_x=r.get("shared"), quant_mode=q), "combine")


def _run_mvp(case, s):
    bs, h, k, e = case["tokens"], case["hidden"], case["top_k"], case["experts"]
    dt, q = EP_TYPE[case["dtype"]], QUANT[case["payload"]]
    r, comm, stream = s["ranks"][0], s["comms"][0], s["streams"][0]
    ep.check(ep.dispatch_v2(r["x"], r["ids"], comm, bs, h, k, e, r["rows"], r["assist"], r["token_nums"], r["counts"],
                            ep.DT_INT8 if q else dt, stream, quant_mode=q, dynamic_scales=r["scales"]), "dispatch")
    ep.check(ep.combine_v2(r.get("expert_out", r["rows"]), r["assist"], r["counts"], comm, bs, h, k, e, r["y"], dt, stream),
             "combine")


def _run_plan(case, s):
    calls = list(zip(s["ranks"], s["comms"], s["streams"]))
    for t, comm, stream in calls:
        (x, rows, _), (w, rw, _) = t["fwd"]
        ep.check(mp.dispatch_v1(comm, t["plan"], x, rows, stream, weights_sk=w, weights_nvs=rw, flags=mp.FLAG_BUILD_DEDUP),
                 "dispatch")
    for t, comm, stream in calls:
        (_, rows, y), (_, rw, yw) = t["fwd"]
        ep.check(mp.combine_v1(comm, t["plan"], t["dst_local"], rows, y, stream, weights_nvs=rw, weights_sk=yw), "combine")
    if case["backward"]:
        for t, comm, stream in calls:
            ep.check(mp.dispatch_v1(comm, t["plan"], t["bwd"][0], t["bwd"][1], stream), "dispatch of gradients")
        for t, comm, stream in calls:
            ep.check(mp.combine_v1(comm, t["plan"], t["dst_local"], t["bwd"][1], t["bwd"][2], stream), "combine of gradients")


def _written(r):
    return [r["rows"], r["scales"], r["assist"], r["token_nums"], r["counts"], r["y"]]


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "layer":
        quant = {"none": None, "int8": "int8", "fp8": "fp8_block128"}[case["payload"]]
        moe = state["layer"]
        d = moe.dispatch(state["x"], state["ids"], quant=quant)
        y = moe.combine(d.expand_x, d, state["weights"], dtype=TORCH_TYPE[case["dtype"]], expert_out_scales=d.scales,
                        expert_out_quant=quant)
        return [d.expand_x, d.scales, d.assist, d.send_counts, d.token_nums, d.row_map, y]
    if kind == "graph":
        state["graph"].graph.replay()
        per_layer = [[r["assist"], r["token_nums"], r["counts"], r["row_map"], r["y"]] for r in state["layers"]]
        return [state["layers"][0]["rows"], per_layer]
    if kind == "plan":
        _run_plan(case, state)
        names = ["rows", "row_weights", "y", "y_weights", "groups", "loffs", "counts", "status"]
        if case["backward"]:
            names += ["grad_rows", "grad_x"]
        return [[t[n] for n in names] for t in state["ranks"]]
    if kind == "ex":
        _run_ex(case, state["ranks"][0], state["comms"][0], state["streams"][0])
        return [_written(r) + [r["row_map"], r.get("status")] for r in state["ranks"]]
    (_run_mvp if kind == "mvp" else _run_ref)(case, state)
    return [_written(r) for r in state["ranks"]]


# ---- what a pass cannot do without ---------------------------------------------------------------------------------
def _kept_rows(case):
    """Rows that find a place.  Under a capacity limit that follows from the experts' popularity, sampled here."""
    n = _active(case) * case["top_k"]
    cap = _capacity(case)
    if cap == 0:
        return n
    sample = 4096
    ids, _ = _routing(case, sample, "cpu", _generator(1, "cpu"))
    load = torch.bincount(ids.reshape(-1).long(), minlength=case["experts"]).float() * (case["tokens"] / sample)
    return int(load.clamp(max=cap).sum())


def work(case):
    bs, h, k, e, ranks = case["tokens"], case["hidden"], case["top_k"], case["experts"], case["ranks"]
    if case["kind"] == "plan":
        d, c = workloads.moonep_algorithmic_bytes(bs, k, h)
        d2, c2 = workloads.moonep_algorithmic_bytes(bs, k, h, with_weights=False)
        return {"bytes": ranks * (d + c + (d2 + c2 if case["backward"] else 0)), "flops": ranks * bs * k * h * (2 if case["backward"] else 1)}
    rows, active = _kept_rows(case), _active(case)
    wide = rows * h * 2
    payload = wide
    if case["payload"] != "none":
        shape, dtype = _scale_shape(case["payload"], rows, h)
        payload = rows * h + shape[0] * shape[1] * dtype.itemsize
    combine_rows = payload if case["kind"] in ("ex", "layer") else wide
    dispatch = active * h * 2 + bs * k * 4 + payload + rows * 16 + e * 12
    combine = combine_rows + rows * (4 if case["kind"] in ("ex", "layer", "graph") else 16) + bs * h * 2
    combine += 0 if case["kind"] == "mvp" else bs * k * 4
    combine += active * h * 2 if case["shared"] else 0
    times = GRAPH_LAYERS if case["kind"] == "graph" else ranks
    return {"bytes": times * (dispatch + combine), "flops": times * rows * h * 2}


def tolerance(case):
    """Every output is defined bit for bit: positions and counts are whole numbers, payloads and scales have one rounding
    rule, and sums are taken in slot order in fp32 with one rounding at the end."""
    return "exact"
