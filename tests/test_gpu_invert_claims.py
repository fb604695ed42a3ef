"""Combine without a row map on tables in which many rows claim the same slot (only a corrupted table does): the highest
row has to win whatever order the threads run in, for tables that a launch of their own inverts (more than 2048 tuples)."""
import numpy as np
import pytest
import torch

from gpu_harness import DEV, Session, bits16, to_dev
from oracle import ep as O
from tilexr_amd import ep
from test_gpu_parity import x_for

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("slots", [1, 7, 300])
def test_the_highest_of_many_claims_wins(slots):
    bs, h, K, E = 600, 64, 8, 16
    n = bs * K
    rng = np.random.default_rng(slots)
    claimed = rng.choice(n, slots, replace=False)[rng.integers(0, slots, n)]
    assist = np.zeros((n, 4), np.int32)
    assist[:, 1], assist[:, 2] = claimed // K, claimed % K
    assist[rng.random(n) < 0.05, 0] = 1                     # of another rank: not looked at
    counts = np.full(E, n, np.int32)
    xt, xb = x_for(rng, n, h, ep.DT_BF16)
    w = (0.25 + rng.random((bs, K))).astype(np.float32)
    case = O.Case(1, bs, h, K, E, dtype=ep.DT_BF16)
    want = O.mem_combine(case, 0, xb[None], assist[None], counts[None], expert_scales=w)
    with Session() as s:
        for _ in range(3):                                  # a later call's epoch replaces an earlier one's claims
            y = torch.full((bs, h), 9.0, dtype=torch.bfloat16, device=DEV)
            torch.cuda.synchronize()
            st = ep.combine_memory_v2(xt, to_dev(assist), to_dev(counts), s.comm, bs, h, K, E, y, ep.DT_BF16, s.stream,
                                      expert_scales=to_dev(w))
            assert st == 0
            s.sync()
            assert np.array_equal(bits16(y), want)
