"""Decode-sized calls of the MVP route in one launch: both sides of the largest table and number of experts, one route, more
experts than routes, nothing to place, rows on both sides of what a lane holds, int8 rows.  Against the oracle."""
import numpy as np
import pytest
import torch

from gpu_harness import DEV, Session, alloc_dispatch_outputs, fetch, to_dev
from oracle import ep as O
from test_gpu_parity import check_dispatch, ids_for, x_for
from tilexr_amd import ep

pytestmark = pytest.mark.gpu

SMALL, VEC = "ep_dispatch_small_route_kernel", "ep_scatter_vec_kernel"


@pytest.mark.parametrize("bs,h,k,e,invalid,plain,int8", [
    (1, 8, 1, 1, 0.0, SMALL, SMALL), (3, 72, 5, 512, 0.3, SMALL, SMALL), (3, 72, 5, 513, 0.3, VEC, VEC),
    (256, 64, 8, 16, 0.1, SMALL, SMALL), (257, 64, 8, 16, 0.1, VEC, VEC), (100, 1000, 6, 64, 1.0, SMALL, SMALL),
    (19, 4104, 6, 64, 0.05, SMALL, SMALL), (256, 2048, 8, 64, 0.0, SMALL, VEC), (5, 8200, 2, 7, 0.2, SMALL, VEC), (30, 2048, 12, 33, 0.1, SMALL, SMALL)])
@pytest.mark.parametrize("nums_type", [0, 1])
def test_dispatch(bs, h, k, e, invalid, plain, int8, nums_type):
    rng = np.random.default_rng(bs + h + k + nums_type)
    ids = ids_for(rng, bs, k, e, invalid=invalid)
    xt, xb = x_for(rng, bs, h, ep.DT_FP16, scale=3.0)
    with Session() as s:
        for quant, kernel in ((ep.Q_NONE, plain), (ep.Q_TOKEN_INT8, int8)):
            out = alloc_dispatch_outputs(bs, h, k, e, quant=quant)
            counts = torch.full((1,), -1, dtype=torch.int32, device=DEV)
            assert ep.dispatch_v2(xt, to_dev(ids), s.comm, bs, h, k, e, out["expand_x"], out["assist"], out["token_nums"],
                                  counts, ep.DT_FP16 if quant == ep.Q_NONE else ep.DT_INT8, s.stream, quant_mode=quant,
                                  token_nums_type=nums_type, dynamic_scales=out["scales"]) == 0
            s.sync()
            assert ep.last_kernel_name(s.comm, ep.K_SCATTER) == kernel
            got = fetch(out, "recv_counts", counts)
            want = O.mvp_dispatch(O.Case(1, bs, h, k, e, dtype=O.DT_FP16, quant_mode=quant, token_nums_type=nums_type), 0,
                                  xb[None], ids[None])
            check_dispatch(got, want)
            assert np.array_equal(got["recv_counts"], want["recv_counts"])
            if quant != ep.Q_NONE:
                assert np.array_equal(got["scales"][:want["rows"], 0], want["dyn_scales"][:want["rows"]])


@pytest.mark.parametrize("bs,h,k", [(384, 16384, 2), (383, 16384, 2), (1537, 8192, 1), (1540, 8184, 1)])
def test_rows_on_both_sides_of_those_that_are_kept(bs, h, k):
    """24 MiB of rows of whole lines and more are written through and kept, others stream."""
    e = 16
    rng = np.random.default_rng(bs + h)
    ids = ids_for(rng, bs, k, e, invalid=0.02)
    xt, xb = x_for(rng, bs, h, ep.DT_FP16)
    with Session() as s:
        out = alloc_dispatch_outputs(bs, h, k, e)
        counts = torch.full((1,), -1, dtype=torch.int32, device=DEV)
        for _ in range(2):
            assert ep.dispatch_v2(xt, to_dev(ids), s.comm, bs, h, k, e, out["expand_x"], out["assist"], out["token_nums"],
                                  counts, ep.DT_FP16, s.stream) == 0
        s.sync()
        assert ep.last_kernel_name(s.comm, ep.K_SCATTER) == SMALL
        got = fetch(out, "recv_counts", counts)
    want = O.mvp_dispatch(O.Case(1, bs, h, k, e, dtype=O.DT_FP16), 0, xb[None], ids[None])
    check_dispatch(got, want)
    assert np.array_equal(got["recv_counts"], want["recv_counts"])
