"""Dispatch + combine captured in a HIP graph (torch.cuda.graph on the session's stream) and replayed.

Steady-state calls allocate nothing and record no memset, so they can be captured once scratch has been sized by an
eager call.  Every replay runs on fresh inputs, with eager calls and synchronisations in between, and is compared
bit for bit with the eager result on the same inputs.  Readiness flags are left out on purpose: their epoch is a
kernel argument fixed at capture time, so a replay would find the previous replay's words already "ready".
"""
import numpy as np
import pytest
import torch

from gpu_harness import DEV, Session
from tilexr_amd import ep, moonep as mp, workloads

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name,bs,quant", [("C2", 128, "none"), ("C3", 700, "none"), ("C4", 600, "int8"),
                                           ("C5", 900, "fp8_block128")])
def test_graph_replays_match_eager(name, bs, quant):
    w = workloads.scaled(workloads.CONFIGS[name], bs)
    h, K, E = w.h, w.top_k, w.experts
    q = {"none": ep.Q_NONE, "int8": ep.Q_TOKEN_INT8, "fp8_block128": ep.Q_FP8_BLOCK128}[quant]
    n = bs * K
    with Session() as s:
        d_x = torch.empty((bs, h), dtype=torch.bfloat16, device=DEV)
        d_ids = torch.empty((bs, K), dtype=torch.int32, device=DEV)
        d_w = torch.empty((bs, K), dtype=torch.float32, device=DEV)
        expand_x = torch.empty((n, h * 2 if q == ep.Q_NONE else h), dtype=torch.uint8, device=DEV)
        assist = torch.empty((n, 4), dtype=torch.int32, device=DEV)
        tn = torch.empty((E,), dtype=torch.int64, device=DEV)
        sc = torch.empty((E,), dtype=torch.int32, device=DEV)
        rm = torch.empty((bs, K), dtype=torch.int32, device=DEV)
        y = torch.empty((bs, h), dtype=torch.bfloat16, device=DEV)
        scales = None
        if q == ep.Q_TOKEN_INT8:
            scales = torch.empty((n, 1), dtype=torch.float32, device=DEV)
        elif q == ep.Q_FP8_BLOCK128:
            scales = torch.empty((n, (h + 127) // 128), dtype=torch.float32, device=DEV)

        def load(seed):
            ws = workloads.Workload(w.name, 1, bs, h, K, E, x_dist=w.x_dist, routing=w.routing, zipf_s=w.zipf_s, seed=seed)
            ids, wt = workloads.make_routing(ws)
            d_x.copy_(workloads.make_x(ws).to(DEV))
            d_ids.copy_(ids.to(DEV))
            d_w.copy_(wt.to(DEV))

        def step():
            st, _ = ep.dispatch_memory_ex(d_x, d_ids, s.comm, bs, h, K, E, expand_x, assist, tn, sc, ep.DT_BF16, s.stream,
                                          quant_mode=q, expert_capacity=w.capacity, dynamic_scales=scales,
                                          row_index_map=rm)
            assert st == 0
            assert ep.combine_memory_ex(expand_x, assist, sc, s.comm, bs, h, K, E, y, ep.DT_BF16, s.stream,
                                        expert_out_quant_mode=q, expert_out_scales=scales, expert_scales=d_w,
                                        row_index_map=rm) == 0

        load(1)
        step()                      # sizes the scratch: nothing is allocated from here on
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=s.stream):
            step()
        torch.cuda.synchronize()
        for seed in (11, 12, 13, 14):
            load(seed)
            for t in (expand_x, assist, rm, y):
                t.fill_(0x5a if t.dtype == torch.uint8 else 7)
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            got = [t.clone() for t in (expand_x, assist, tn, sc, rm, y)]
            rows = int(sc[-1].item())
            for t in (expand_x, assist, rm, y):
                t.fill_(0x33 if t.dtype == torch.uint8 else 9)
            torch.cuda.synchronize()
            step()                  # eager work between the replays, on the same communicator
            torch.cuda.synchronize()
            want = (expand_x, assist, tn, sc, rm, y)
            assert int(sc[-1].item()) == rows
            for g, e, part in zip(got, want, ("rows", "assist", "token_nums", "send_counts", "row_map", "y")):
                if part in ("rows", "assist"):
                    g, e = g[:rows], e[:rows]
                assert torch.equal(g.view(torch.uint8), e.view(torch.uint8)), f"seed {seed}: {part}"


@pytest.mark.parametrize("memory", [True, False])
def test_replays_without_a_row_map_forget_the_rows_of_the_replay_before(memory):
    """More than 2048 routes and no row map: combine inverts the assist table.  Every replay leaves other routes without a
    row (ids that name no expert); two layers of the graph share the table."""
    bs, h, K, E = 700, 64, 4, 16
    dtype, tdt = (ep.DT_BF16, torch.bfloat16) if memory else (ep.DT_FP16, torch.float16)
    gen = torch.Generator(device=DEV).manual_seed(3)
    x = torch.empty((bs, h), dtype=tdt, device=DEV)
    layers = [dict(ids=torch.empty((bs, K), dtype=torch.int32, device=DEV), rows=torch.empty((bs * K, h), dtype=tdt, device=DEV),
                   assist=torch.empty((bs * K, 4), dtype=torch.int32, device=DEV),
                   nums=torch.empty((E,), dtype=torch.int64, device=DEV), counts=torch.empty((E,), dtype=torch.int32, device=DEV),
                   y=torch.empty((bs, h), dtype=tdt, device=DEV)) for _ in range(2)]

    def load():
        x.copy_(torch.randn(bs, h, device=DEV, generator=gen))
        for t in layers:
            ids = torch.randint(0, E, (bs, K), device=DEV, generator=gen, dtype=torch.int32)
            t["ids"].copy_(torch.where(torch.rand(bs, K, device=DEV, generator=gen) < 0.4, -1, ids))
            t["y"].fill_(7)
        torch.cuda.synchronize()

    # the eager calls have a communicator of their own: on the graph's they would write the table's words anew
    with Session() as s, Session() as eager:
        def step(on):
            for t in layers:
                call = ep.dispatch_memory if memory else ep.dispatch
                assert call(x, t["ids"], on.comm, bs, h, K, E, t["rows"], t["nums"], t["counts"], t["assist"], dtype, on.stream) == 0
                call = ep.combine_memory if memory else ep.combine
                assert call(t["rows"], t["assist"], t["counts"], on.comm, bs, h, K, E, t["y"], dtype, on.stream) == 0

        load()
        step(s)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=s.stream):
            step(s)
        torch.cuda.synchronize()
        for _ in range(4):
            load()
            graph.replay()
            torch.cuda.synchronize()
            got = [t["y"].clone() for t in layers]
            for t in layers:
                t["y"].fill_(9)
            torch.cuda.synchronize()
            step(eager)
            torch.cuda.synchronize()
            for g, t in zip(got, layers):
                assert torch.equal(g, t["y"])


def test_replays_of_a_logical_world_forget_the_rows_of_the_replay_before():
    """Two ranks on one captured stream (their eager calls are made on another one)."""
    R, bs, h, K, E = 2, 60, 64, 2, 8
    gen = torch.Generator(device=DEV).manual_seed(4)
    new = lambda *shape, dtype=torch.int32: torch.empty(shape, dtype=dtype, device=DEV)
    ranks = [dict(x=new(bs, h, dtype=torch.bfloat16), ids=new(bs, K), rows=new(R * bs * K, h, dtype=torch.bfloat16),
                  assist=new(R * bs * K, 4), nums=new(E // R, dtype=torch.int64), counts=new(E), y=new(bs, h, dtype=torch.bfloat16))
             for _ in range(R)]

    def load():
        for t in ranks:
            t["x"].copy_(torch.randn(bs, h, device=DEV, generator=gen))
            ids = torch.randint(0, E, (bs, K), device=DEV, generator=gen, dtype=torch.int32)
            t["ids"].copy_(torch.where(torch.rand(bs, K, device=DEV, generator=gen) < 0.5, -1, ids))
            t["y"].fill_(7)
        torch.cuda.synchronize()

    def step(comms, stream):
        for c, t in zip(comms, ranks):
            assert ep.dispatch_memory(t["x"], t["ids"], c, bs, h, K, E, t["rows"], t["nums"], t["counts"], t["assist"], ep.DT_BF16,
                                      stream) == 0
        for c, t in zip(comms, ranks):
            assert ep.combine_memory(t["rows"], t["assist"], t["counts"], c, bs, h, K, E, t["y"], ep.DT_BF16, stream) == 0

    torch.cuda.set_device(0)
    captured, eager = [ep.Comm(R, r) for r in range(R)], [ep.Comm(R, r) for r in range(R)]
    first, stream = torch.cuda.Stream(), torch.cuda.Stream()
    load()
    step(captured, first)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        step(captured, stream)
    for _ in range(4):
        load()
        graph.replay()
        torch.cuda.synchronize()
        got = [t["y"].clone() for t in ranks]
        step(eager, first)
        torch.cuda.synchronize()
        for g, t in zip(got, ranks):
            assert torch.equal(g, t["y"])
    for c in captured + eager:
        c.destroy()


def test_replays_of_plan_driven_stages_follow_the_plan_as_it_stands():
    """One rank; the plan's words are rewritten between the replays, so that other rows are named, and rows that no route
    names any more come out as zeros.  The expected outputs are torch's."""
    S, K, H, NVS = 64, 4, 64, 400
    gen = torch.Generator().manual_seed(5)
    comm = ep.Comm(1, 0)
    first, stream = torch.cuda.Stream(), torch.cuda.Stream()
    dst, dst_local = torch.zeros(S * K, dtype=torch.int32, device=DEV), torch.zeros(NVS, dtype=torch.int32, device=DEV)
    groups, loffs = torch.zeros((NVS, 3), dtype=torch.int32, device=DEV), torch.zeros(NVS, dtype=torch.int32, device=DEV)
    counts, status = torch.zeros(2, dtype=torch.int32, device=DEV), torch.zeros(4, dtype=torch.int32, device=DEV)
    x, rows = torch.zeros((S, H), dtype=torch.bfloat16, device=DEV), torch.zeros((NVS, H), dtype=torch.bfloat16, device=DEV)
    y = torch.zeros((S, H), dtype=torch.bfloat16, device=DEV)
    plan = mp.plan(S * K, 1, K, 1, NVS, K, dst, groups, loffs, counts, status)

    def load():
        at = torch.randperm(NVS, generator=gen)[:S * K].to(torch.int32)
        words = at.clone().view(S, K)
        words[:, 1:] = -words[:, 1:] - 1            # the later routes of a token are duplicates
        dst.copy_(words.flatten().to(DEV))
        back = torch.full((NVS,), -1, dtype=torch.int32)
        back[at.long()] = torch.arange(S * K, dtype=torch.int32)
        dst_local.copy_(back.to(DEV))
        x.copy_(torch.randn(S, H, generator=gen).to(DEV))
        for t in (rows, y):
            t.fill_(7)
        torch.cuda.synchronize()
        return at.long().to(DEV)

    def step(on):
        tensors = [mp.tensor(t, mp.DT_BF16, tuple(t.shape)) for t in (x, rows, y)]
        assert mp.dispatch_v1(comm, plan, tensors[0], tensors[1], on, flags=mp.FLAG_BUILD_DEDUP) == 0
        assert mp.combine_v1(comm, plan, dst_local, tensors[1], tensors[2], on) == 0

    load()
    step(first)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        step(stream)
    for _ in range(4):
        at = load()
        graph.replay()
        torch.cuda.synchronize()
        want = torch.zeros_like(rows)
        want[at] = x.repeat_interleave(K, dim=0)
        assert torch.equal(rows, want)
        assert torch.equal(y, (K * x.float()).to(torch.bfloat16))      # K equal rows: a power of two times the row
    comm.destroy()
