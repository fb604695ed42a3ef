"""Logical worlds at the edges of their launches: more segments than a copying workgroup adds up itself, more ranks than
one launch takes, rows on both sides of 4 KiB (a wave or a workgroup per row), sends of one launch and of two, every row
on one rank (its workgroups go round again), and all ranks on one stream (no events between them)."""
import numpy as np
import pytest
import torch

import test_gpu_multi_rank as multi
from oracle import ep as O
from tilexr_amd import ep

pytestmark = pytest.mark.gpu

SHAPES = [
    (2, 40, 64, 4, 256),         # 256 segments per rank: the most a copying workgroup adds up
    (2, 40, 64, 4, 258),         # 258: a plan launch ahead
    (17, 9, 64, 2, 34),          # one rank more than a launch takes
    (2, 260, 2048, 8, 32),       # 2080 routes: send in two launches; rows of exactly 4 KiB
    (3, 20, 2056, 2, 9),         # rows just wider
]


@pytest.mark.parametrize("shape", SHAPES)
def test_memory_route_world(shape):
    multi.test_memory_dispatch_and_combine_across_ranks(shape, ep.DT_BF16)


@pytest.mark.parametrize("dtype", [ep.DT_BF16, ep.DT_FP16])
@pytest.mark.parametrize("shape", [(3, 20, 1032, 4, 9), (2, 320, 2048, 2, 8), (2, 321, 1536, 2, 8), (2, 512, 1040, 3, 8),
                                   (2, 513, 1040, 3, 8)])
def test_rows_in_one_slice_and_in_two(shape, dtype):
    """Combines of rows of 129 to 256 vectors on both sides of the numbers of tokens up to which they are cut."""
    multi.test_memory_dispatch_and_combine_across_ranks(shape, dtype)


@pytest.mark.parametrize("shape", [(2, 20, 64, 2, 514), (17, 9, 64, 2, 34), (3, 20, 2056, 2, 9)])
def test_mvp_route_world(shape):
    multi.test_mvp_dispatch_and_combine_across_ranks(shape)


@pytest.mark.parametrize("one_stream", [False, True])
def test_every_row_on_one_rank(one_stream):
    R, bs, h, K, E = 4, 60, 136, 4, 32
    rng = np.random.default_rng(5)
    ids = np.stack([np.stack([rng.permutation(8)[:K] for _ in range(bs)]) for _ in range(R)]).astype(np.int32) + 8
    xt, xb = multi.rand_x(rng, R, bs, h, ep.DT_BF16)
    with multi.World(R) as w:
        if one_stream:
            w.streams = [w.streams[0]] * R
        for _ in range(2):                       # the second exchange reuses the first one's staging
            outs = multi.run_dispatch(w, True, xt, ids, bs, h, K, E, ep.DT_BF16)
            case = O.Case(R, bs, h, K, E, token_nums_type=1)
            for r in range(R):
                multi.check_rank(outs[r], O.mem_dispatch(case, r, xb, ids), "send_counts")
            ys = [torch.full((bs, h), 7.0, dtype=torch.bfloat16, device=multi.DEV) for _ in range(R)]
            torch.cuda.synchronize()
            for r in range(R):
                assert ep.combine_memory_v2(outs[r]["expand_x"], outs[r]["assist"], outs[r]["counts"], w.comms[r], bs, h, K, E,
                                            ys[r], ep.DT_BF16, w.streams[r]) == 0
            w.sync()
            eo = np.stack([o["expand_x"].cpu().numpy().view(np.uint16) for o in outs])
            assist = np.stack([o["assist"].cpu().numpy() for o in outs])
            counts = np.stack([o["counts"].cpu().numpy() for o in outs])
            for r in range(R):
                assert np.array_equal(multi.bits16(ys[r]), O.mem_combine(case, r, eo, assist, counts)), f"rank {r}"


@pytest.mark.parametrize("memory", [True, False])
def test_sizes_in_turn_leave_no_rows_behind(memory):
    """A large, a small and the large size again, the last with a rank whose routes name no expert: its outputs are zero,
    whatever the small exchange, whose slots lie elsewhere in the same tables, has written there."""
    R, h, K, E = 8, 64, 2, 16
    rng = np.random.default_rng(12)
    dtype, tdt = (ep.DT_BF16, torch.bfloat16) if memory else (ep.DT_FP16, torch.float16)
    with multi.World(R) as w:
        for round_ in range(3):
            for bs in (64, 9, 64, 17, 64):
                ids = multi.rand_ids(rng, R, bs, K, E)
                ids[0] = -1
                xt, _ = multi.rand_x(rng, R, bs, h, dtype)
                outs = multi.run_dispatch(w, memory, xt, ids, bs, h, K, E, dtype)
                ys = [torch.full((bs, h), 7.0, dtype=tdt, device=multi.DEV) for _ in range(R)]
                torch.cuda.synchronize()
                for r in range(R):
                    call = ep.combine_memory_v2 if memory else ep.combine_v2
                    assert call(outs[r]["expand_x"].view(tdt), outs[r]["assist"], outs[r]["counts"], w.comms[r], bs, h, K, E, ys[r],
                                dtype, w.streams[r]) == 0
                w.sync()
                assert not ys[0].any()
                assert ys[1].any()


def test_work_between_a_ranks_call_and_the_last_ones_runs_ahead_of_the_outputs():
    """Rank 0 fills its outputs, and writes the combine weights, on its own stream after its call: the second half, which
    the last caller's stream runs, comes behind that."""
    R, bs, h, K, E = 2, 50, 256, 4, 8
    rng = np.random.default_rng(8)
    ids = multi.rand_ids(rng, R, bs, K, E)
    xt, xb = multi.rand_x(rng, R, bs, h, ep.DT_BF16)
    weights = rng.random((R, bs, K)).astype(np.float32)
    case = O.Case(R, bs, h, K, E, token_nums_type=1)
    wants = [O.mem_dispatch(case, r, xb, ids) for r in range(R)]
    with multi.World(R) as w:
        outs = multi.run_dispatch(w, True, xt, ids, bs, h, K, E, ep.DT_BF16)        # scratch of this size
        dev_ids = [multi.to_dev(ids[r]) for r in range(R)]
        dev_w = [torch.zeros((bs, K), device=multi.DEV) for _ in range(R)]
        given = [multi.to_dev(weights[r]) for r in range(R)]
        ys = [torch.full((bs, h), 7.0, dtype=torch.bfloat16, device=multi.DEV) for _ in range(R)]
        torch.cuda.synchronize()
        for r in range(R):
            o = outs[r]
            assert ep.dispatch_memory_v2(xt[r], dev_ids[r], w.comms[r], bs, h, K, E, o["expand_x"], o["assist"], o["token_nums"],
                                         o["counts"], ep.DT_BF16, w.streams[r]) == 0
            if r == 0:
                with torch.cuda.stream(w.streams[0]):
                    torch.cuda._sleep(2_000_000)
                    for name in ("expand_x", "assist", "counts"):
                        o[name].fill_(-77)
        w.sync()
        for r in range(R):
            multi.check_rank(outs[r], wants[r], "send_counts")
        for r in range(R):
            assert ep.combine_memory_v2(outs[r]["expand_x"], outs[r]["assist"], outs[r]["counts"], w.comms[r], bs, h, K, E, ys[r],
                                        ep.DT_BF16, w.streams[r], expert_scales=dev_w[r]) == 0
            with torch.cuda.stream(w.streams[r]):
                if r == 0:
                    torch.cuda._sleep(2_000_000)
                    dev_w[0].copy_(given[0])
        w.sync()
        eo = np.stack([o["expand_x"].cpu().numpy().view(np.uint16) for o in outs])
        assist = np.stack([o["assist"].cpu().numpy() for o in outs])
        counts = np.stack([o["counts"].cpu().numpy() for o in outs])
        assert np.array_equal(multi.bits16(ys[0]), O.mem_combine(case, 0, eo, assist, counts, expert_scales=weights[0]))
