"""One-launch routing of the MVP route, at the sizes where it can go wrong: one route, both sides of a workgroup's 1024
routes and of the 4096 ids it takes with one load per lane, experts 0 only, no valid id at all, more experts than routes,
tables that are not aligned for the vector loads (the count launch takes those ids) or the tuple stores."""
import numpy as np
import pytest
import torch

from gpu_harness import DEV, Session, alloc_dispatch_outputs, fetch, to_dev
from oracle import ep as O
from tilexr_amd import ep
from test_gpu_parity import check_dispatch, ids_for, x_for

pytestmark = pytest.mark.gpu

CASES = [
    # bs, h, K, E, share of invalid ids
    (1, 64, 1, 1, 0.0),
    (3, 72, 5, 2000, 0.3),
    (128, 64, 8, 16, 0.1),         # 1024 routes: exactly one workgroup's
    (205, 16, 5, 7, 0.1),          # 1025
    (1365, 8, 3, 64, 0.0),         # 4095
    (512, 32, 8, 64, 0.5),         # 4096
    (241, 16, 17, 33, 0.2),        # 4097
    (1100, 1000, 6, 64, 1.0),      # nothing to place
    (1501, 4096, 6, 1, 0.4),       # one expert, token rows read ahead
    (4099, 16, 8, 256, 0.05),      # a second batch of loads (32 792 routes)
]


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("nums_type", [0, 1])
def test_one_launch_mvp_routing_matches_oracle(case, nums_type):
    bs, h, K, E, invalid = case
    rng = np.random.default_rng(bs + h + K + nums_type)
    ids = ids_for(rng, bs, K, E, invalid=invalid)
    if invalid == 1.0:
        ids[:] = rng.choice([-1, E, np.iinfo(np.int32).min, np.iinfo(np.int32).max], (bs, K))
    xt, xb = x_for(rng, bs, h, ep.DT_FP16)
    want = O.mvp_dispatch(O.Case(1, bs, h, K, E, dtype=O.DT_FP16, token_nums_type=nums_type), 0, xb[None], ids[None])
    with Session(legacy_routing=False) as s:
        for shift_ids, shift_assist in ((0, 0), (0, 1), (1, 0)):
            out = alloc_dispatch_outputs(bs, h, K, E)
            counts = torch.full((1,), -1, dtype=torch.int32, device=DEV)
            table = torch.zeros(bs * K + 4, dtype=torch.int32, device=DEV)
            table[shift_ids:shift_ids + bs * K] = to_dev(ids).reshape(-1)
            assist = torch.full((bs * K * 4 + 4,), -77, dtype=torch.int32, device=DEV)
            torch.cuda.synchronize()
            st = ep.dispatch_v2(xt, table[shift_ids:], s.comm, bs, h, K, E, out["expand_x"], assist[shift_assist:],
                                out["token_nums"], counts, ep.DT_FP16, s.stream, token_nums_type=nums_type)
            assert st == 0
            s.sync()
            assert ep.last_kernel_name(s.comm, ep.K_COUNT) == ("ep_route_count_kernel" if shift_ids else "ep_route_compact_kernel")
            n = want["rows"]
            got = assist.cpu().numpy()[shift_assist:shift_assist + bs * K * 4].reshape(-1, 4)
            assert np.array_equal(got[:n], want["assist"][:n])
            assert np.all(got[n:] == -77)
            out["assist"] = assist[shift_assist:shift_assist + bs * K * 4].reshape(-1, 4)
            got = fetch(out, "recv_counts", counts)
            check_dispatch(got, want)
            assert np.array_equal(got["recv_counts"], want["recv_counts"])


@pytest.mark.parametrize("bs,K,E,kernel", [(2, 4, 1024, "ep_route_compact_kernel"), (2, 4, 1025, "ep_route_count_kernel"),
                                           (2047, 1, 2048, "ep_route_count_kernel"), (256, 8, 2048, "ep_route_compact_kernel")])
def test_many_experts_and_few_routes_keep_the_count_launch(bs, K, E, kernel):
    rng = np.random.default_rng(bs + E)
    ids = ids_for(rng, bs, K, E, invalid=0.1)
    xt, xb = x_for(rng, bs, 64, ep.DT_FP16)
    want = O.mvp_dispatch(O.Case(1, bs, 64, K, E, dtype=O.DT_FP16, token_nums_type=1), 0, xb[None], ids[None])
    with Session() as s:
        out = alloc_dispatch_outputs(bs, 64, K, E)
        counts = torch.full((1,), -1, dtype=torch.int32, device=DEV)
        ids_dev = to_dev(ids)
        torch.cuda.synchronize()
        assert ep.dispatch_v2(xt, ids_dev, s.comm, bs, 64, K, E, out["expand_x"], out["assist"], out["token_nums"], counts,
                              ep.DT_FP16, s.stream, token_nums_type=1) == 0
        s.sync()
        assert ep.last_kernel_name(s.comm, ep.K_COUNT) == kernel
        check_dispatch(fetch(out, "recv_counts", counts), want)
