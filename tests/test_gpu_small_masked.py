"""Masked dispatch in one launch, at the sizes where it can go wrong: one token, a mask of all or none, tokens on both
sides of a workgroup's 256 mask bytes and of the four batches a lane has in flight, the largest table, routes that do not
cover the experts' count outputs, a capacity limit, readiness flags."""
import numpy as np
import pytest
import torch

from gpu_harness import DEV, Session, alloc_dispatch_outputs, fetch, to_dev
from oracle import ep as O
from tilexr_amd import ep
from test_gpu_parity import check_dispatch, ids_for, x_for

pytestmark = pytest.mark.gpu

CASES = [
    # bs, h, K, E, share of the mask that is set, capacity, flags
    (1, 7168, 8, 256, 1.0, 0, False),
    (3, 64, 4, 16, 0.0, 0, False),
    (200, 1024, 8, 256, 0.8, 0, True),
    (257, 64, 7, 32, 0.5, 0, False),
    (256, 4096, 8, 64, 0.99, 0, False),          # 2048 routes: the most one launch takes
    (1025, 16, 1, 8, 0.7, 0, False),
    (2048, 8, 1, 5, 0.3, 0, True),
    (100, 8192, 6, 64, 0.6, 3, False),           # capacity: a workgroup per token
    (9, 40, 3, 100, 0.7, 0, True),               # fewer routes than experts
]


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("mask_type", [ep.MASK_TOKEN, ep.MASK_EXPERT])
def test_masked_small_dispatch_matches_oracle(case, mask_type):
    bs, h, K, E, share, capacity, flags = case
    rng = np.random.default_rng(bs + h + mask_type)
    ids = ids_for(rng, bs, K, E, invalid=0.1)
    mask = (rng.random((bs, K) if mask_type == ep.MASK_EXPERT else bs) < share).astype(np.uint8)
    xt, xb = x_for(rng, bs, h, ep.DT_BF16)
    with Session() as s:
        out = alloc_dispatch_outputs(bs, h, K, E)
        counts = torch.full((E,), -1, dtype=torch.int32, device=DEV)
        words = torch.zeros(((bs * K + 15) // 16,), dtype=torch.int64, device=DEV) if flags else None
        st, epoch = ep.dispatch_memory_ex(xt, to_dev(ids), s.comm, bs, h, K, E, out["expand_x"], out["assist"],
                                          out["token_nums"], counts, ep.DT_BF16, s.stream, expert_capacity=capacity,
                                          active_mask=to_dev(mask), active_mask_type=mask_type,
                                          row_index_map=out["row_map"], tile_flags=words, tile_rows=16 if flags else 0)
        assert st == 0
        s.sync()
        assert ep.last_kernel_name(s.comm, ep.K_SCATTER).startswith("ep_dispatch_small")
        got = fetch(out, "send_counts", counts)
        want = O.mem_dispatch(O.Case(1, bs, h, K, E, mask_type=mask_type, token_nums_type=1, capacity=capacity), 0, xb[None],
                              ids[None], mask[None])
        check_dispatch(got, want)
        n = want["rows"]
        assert np.array_equal(got["send_counts"], want["send_counts"])
        rows = np.full((bs, K), -1, np.int32)
        rows[want["assist"][:n, 1], want["assist"][:n, 2]] = np.arange(n)
        assert np.array_equal(got["row_map"], rows)
        if flags:
            tiles = [min(16, n - t) for t in range(0, n, 16)]
            assert words.cpu().numpy()[:len(tiles)].tolist() == [(epoch << 32) | t for t in tiles]
