"""One layer called on one stream after another, torch's default stream, streams of torch's own, a wrapped one and a
capturing one among them: every call sees the inputs its stream has written and the scratch of no other call."""
import ctypes

import pytest
import torch

from test_gpu_layer import torch_combine_k_ordered, torch_dispatch
from tilexr_amd import ep, layer

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
BS, H, K, E = 700, 512, 8, 32


def inputs(seed):
    g = torch.Generator().manual_seed(seed)
    ids = torch.stack([torch.randperm(E, generator=g)[:K] for _ in range(BS)]).to(torch.int32)
    return (torch.randn(BS, H, generator=g).to(torch.bfloat16).to(DEV), ids.to(DEV), torch.rand(BS, K, generator=g).to(DEV))


def check(x, ids, weights, d, y):
    rows, assist, counts, row_map = torch_dispatch(x, ids, E)
    assert torch.equal(d.expand_x.view(torch.int16), rows.view(torch.int16))
    assert torch.equal(d.assist, assist) and torch.equal(d.token_nums, counts) and torch.equal(d.row_map, row_map)
    ref = torch_combine_k_ordered(rows, row_map, weights).to(torch.bfloat16)
    assert torch.equal(y.view(torch.int16), ref.view(torch.int16))


def test_calls_on_changing_streams():
    wrapped = torch.cuda.Stream()
    schedule = [torch.cuda.default_stream(), torch.cuda.Stream(), torch.cuda.ExternalStream(wrapped.cuda_stream),
                torch.cuda.default_stream(), torch.cuda.ExternalStream(wrapped.cuda_stream), torch.cuda.Stream()]
    given = [inputs(i) for i in range(len(schedule))]
    torch.cuda.synchronize()
    done = []
    with layer.MoeEpLayer(E, K, H) as moe:
        for stream, (x, ids, weights) in zip(schedule, given):
            with torch.cuda.stream(stream):
                late = torch.zeros_like(x)
                late.copy_(x, non_blocking=True)        # written on this stream just ahead of the call
                d = moe.dispatch(late, ids)
                y = moe.combine(d.expand_x, d, weights)
            del late
            done.append((d, y))
        # dispatch on one stream, combine on another
        with torch.cuda.stream(schedule[1]):
            d = moe.dispatch(given[0][0], given[0][1])
        with torch.cuda.stream(schedule[5]):
            y = moe.combine(d.expand_x, d, given[0][2])
        torch.cuda.synchronize()
        for (x, ids, weights), (got, out) in zip(given + given[:1], done + [(d, y)]):
            check(x, ids, weights, got, out)


def test_eager_calls_on_two_streams_run_one_after_the_other():
    x, ids, weights = inputs(9)
    other = inputs(10)
    first, second = torch.cuda.Stream(), torch.cuda.Stream()
    with layer.MoeEpLayer(E, K, H) as moe:
        moe.dispatch(x, ids, capacity=8)            # scratch of this size
        torch.cuda.synchronize()
        reached = torch.cuda.Event()
        with torch.cuda.stream(first):
            torch.cuda._sleep(50_000_000)
            a = moe.dispatch(x, ids, capacity=8)
            reached.record()
        with torch.cuda.stream(second):
            b = moe.dispatch(*other[:2], capacity=8)
        second.synchronize()
        assert reached.query()                      # the first call, behind some 20 ms of sleep, has run
        for d, given in ((a, ids), (b, other[1])):
            want = torch.bincount(given.flatten().long(), minlength=E).clamp(max=8)
            assert torch.equal(d.token_nums, want)


def test_captured_call_replays():
    x, ids, weights = inputs(11)
    other = inputs(12)
    with layer.MoeEpLayer(E, K, H) as moe:
        moe.combine(moe.dispatch(x, ids).expand_x, moe.dispatch(x, ids), weights)       # scratch of this size
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            d = moe.dispatch(x, ids)
            y = moe.combine(d.expand_x, d, weights)
        for replay in range(3):
            x.copy_(inputs(20 + replay)[0])
            eager = moe.dispatch(other[0], other[1])
            out = moe.combine(eager.expand_x, eager, other[2])
            graph.replay()
            torch.cuda.synchronize()
            check(x, ids, weights, d, y)
            check(*other, eager, out)


def test_two_branches_of_one_capture():
    """Two micro-batches on forked streams of one capture.  With a capacity limit a dispatch of this size takes the count
    launch, which hands histograms and its ticket from workgroup to workgroup through the layer's scratch."""
    batches = [inputs(31), inputs(32)]
    capacity = BS * K // E
    side = torch.cuda.Stream()

    def step(moe, x, ids, weights):
        d = moe.dispatch(x, ids, capacity=capacity)
        return d, moe.combine(d.expand_x, d, weights)

    def results(d, y):
        rows = d.rows()
        return [d.expand_x[:rows].clone(), d.assist[:rows].clone(), d.send_counts.clone(), d.token_nums.clone(), d.row_map.clone(),
                y.clone()]

    with layer.MoeEpLayer(E, K, H) as moe:
        step(moe, *batches[0])                      # scratch of this size
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            main = torch.cuda.current_stream()
            side.wait_stream(main)
            first = step(moe, *batches[0])
            with torch.cuda.stream(side):
                second = step(moe, *batches[1])
            main.wait_stream(side)
        for replay in range(3):
            for (x, _, _), seed in zip(batches, (40 + replay, 50 + replay)):
                x.copy_(inputs(seed)[0])
            eager = [results(*step(moe, *b)) for b in batches]
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            for (d, y), want in zip((first, second), eager):
                for got, expected in zip(results(d, y), want):
                    assert torch.equal(got, expected)


def test_calls_of_one_capture_are_one_chain():
    """Whether the two micro-batches of a capture are ordered, from the captured graph itself: it begins with one kernel,
    where two unordered branches begin with two."""
    hip = ctypes.CDLL("libamdhip64.so")
    batches = [inputs(33), inputs(34)]
    side = torch.cuda.Stream()
    with layer.MoeEpLayer(E, K, H) as moe:
        moe.dispatch(*batches[0][:2], capacity=8)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph(keep_graph=True)
        with torch.cuda.graph(graph):
            main = torch.cuda.current_stream()
            side.wait_stream(main)
            kept = [moe.dispatch(*batches[0][:2], capacity=8)]
            with torch.cuda.stream(side):
                kept.append(moe.dispatch(*batches[1][:2], capacity=8))
            main.wait_stream(side)
        roots = ctypes.c_size_t(0)
        assert hip.hipGraphGetRootNodes(ctypes.c_void_p(graph.raw_cuda_graph()), None, ctypes.byref(roots)) == 0
        assert roots.value == 1


def test_default_stream_handle_is_taken_and_null_is_not():
    x, ids, _ = inputs(3)
    n = BS * K
    rows = torch.empty((n, H), dtype=torch.bfloat16, device=DEV)
    assist, counts = torch.empty((n, 4), dtype=torch.int32, device=DEV), torch.empty(E, dtype=torch.int32, device=DEV)
    nums = torch.empty(E, dtype=torch.int64, device=DEV)
    comm = ep.Comm(1, 0)
    args = (x, ids, comm, BS, H, K, E, rows, nums, counts, assist, ep.DT_BF16)
    assert ep.dispatch_memory(*args, None) == ep.ERR_PARA_CHECK_FAIL
    assert ep.dispatch_memory(*args, ep.STREAM_LEGACY) == ep.SUCCESS
    want = torch_dispatch(x, ids, E)
    assert torch.equal(rows.view(torch.int16), want[0].view(torch.int16)) and torch.equal(assist, want[1])
    torch.cuda.synchronize()
    comm.destroy()
