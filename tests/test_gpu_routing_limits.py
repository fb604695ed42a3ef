"""The one-launch routing under a capacity limit and under a token-prefix mask, at the edges of its tables: parts and slots
that are nearly empty, experts that nobody names, that overflow and that take everything, limits of one and beyond
the count, masks that are empty, whole, or end within a load.  Against the oracle and the count + place routing."""
import numpy as np
import pytest
import torch

from gpu_harness import DEV, Session, alloc_dispatch_outputs, fetch, to_dev
from oracle import ep as O
from test_gpu_parity import check_dispatch, x_for
from tilexr_amd import ep

pytestmark = pytest.mark.gpu


def _run(legacy, xt, xb, ids, e, nums_type, capacity=0, mask=None, quant=ep.Q_NONE):
    bs, k = ids.shape
    h = xb.shape[1]
    with Session(legacy_routing=legacy) as s:
        out = alloc_dispatch_outputs(bs, h, k, e, quant=quant)
        counts = torch.full((e,), -1, dtype=torch.int32, device=DEV)
        st, _ = ep.dispatch_memory_ex(
            xt, to_dev(ids), s.comm, bs, h, k, e, out["expand_x"], out["assist"], out["token_nums"], counts, ep.DT_BF16, s.stream,
            token_nums_type=nums_type, expert_capacity=capacity, row_index_map=out["row_map"], quant_mode=quant,
            dynamic_scales=out["scales"], active_mask=to_dev(mask),
            active_mask_type=ep.MASK_NONE if mask is None else ep.MASK_TOKEN)
        assert st == 0
        s.sync()
        assert ep.last_kernel_name(s.comm, ep.K_COUNT) == ("ep_route_count_kernel" if legacy else "ep_route_rows_kernel")
        got = fetch(out, "send_counts", counts)
    case = O.Case(1, bs, h, k, e, quant_mode=quant, token_nums_type=nums_type, capacity=capacity,
                  mask_type=ep.MASK_NONE if mask is None else ep.MASK_TOKEN)
    want = O.mem_dispatch(case, 0, xb[None], ids[None], None if mask is None else mask[None])
    check_dispatch(got, want)
    n = want["rows"]
    assert np.array_equal(got["send_counts"], want["send_counts"])
    rows = np.full((bs, k), -1, np.int32)
    rows[want["assist"][:n, 1], want["assist"][:n, 2]] = np.arange(n)
    assert np.array_equal(got["row_map"], rows)


SHAPES = [(2049, 1, 1, 0.0), (700, 3, 5, 0.1), (513, 4, 300, 0.02), (1025, 8, 64, 0.0), (4097, 2, 16, 1.0), (6000, 5, 9, 0.05),
          (4096, 8, 512, 0.01), (2048, 16, 2048, 0.01)]


@pytest.mark.parametrize("bs,k,e,invalid", SHAPES)
@pytest.mark.parametrize("limit", ["one", "mean", "most"])
@pytest.mark.parametrize("legacy", [False, True])
def test_capacity(bs, k, e, invalid, limit, legacy):
    rng = np.random.default_rng(bs + k + e)
    ids = rng.integers(0, max(e - 1, 1), (bs, k)).astype(np.int32)       # nobody names the last expert, many the second
    ids[rng.random((bs, k)) < 0.3] = min(1, e - 1)
    bad = rng.random(ids.shape) < invalid
    ids[bad] = rng.choice([-1, e, 2 ** 31 - 1, -2 ** 31], size=int(bad.sum()))
    capacity = {"one": 1, "mean": max(1, bs * k // e), "most": bs * k + 5}[limit]
    xt, xb = x_for(rng, bs, 16, ep.DT_BF16)
    for nums_type in (0, 1):
        _run(legacy, xt, xb, ids, e, nums_type, capacity=capacity)
    if limit == "mean":
        _run(legacy, xt, xb, ids, e, 1, capacity=capacity, quant=ep.Q_TOKEN_INT8)


@pytest.mark.parametrize("bs,k,e", [(16384, 1, 64), (2048, 8, 64), (2100, 5, 7), (2500, 1, 1024), (2500, 1, 1025), (1024, 16, 2048)])
@pytest.mark.parametrize("first", ["low", "high"])
def test_capacity_when_every_token_goes_the_same_way(bs, k, e, first):
    """All lanes count the same expert at once; both layouts of the counters, up to their last key."""
    rng = np.random.default_rng(bs + k + e)
    start = 0 if first == "low" else e - k - 1 if e > k else 0
    ids = np.tile(np.arange(start, start + k, dtype=np.int32), (bs, 1))
    ids[rng.integers(0, bs, 20), rng.integers(0, k, 20)] = e - 1
    xt, xb = x_for(rng, bs, 16, ep.DT_BF16)
    for capacity in (1, bs // 3, bs * k):
        _run(False, xt, xb, ids, e, 1, capacity=capacity)


@pytest.mark.parametrize("bs,k,e,invalid", SHAPES)
@pytest.mark.parametrize("active", ["none", "one", "some", "all"])
@pytest.mark.parametrize("legacy", [False, True])
def test_prefix_mask(bs, k, e, invalid, active, legacy):
    rng = np.random.default_rng(bs + k + e)
    ids = rng.integers(0, e, (bs, k)).astype(np.int32)
    bad = rng.random(ids.shape) < invalid
    ids[bad] = rng.choice([-1, e, 2 ** 31 - 1, -2 ** 31], size=int(bad.sum()))
    some = bs * 3 // 5 + 1
    mask = (np.arange(bs) < {"none": 0, "one": 1, "some": some, "all": bs}[active]).astype(np.uint8)
    if active == "some":
        mask = rng.permutation(mask) * rng.integers(1, 256, bs).astype(np.uint8)       # the sum counts, not the places
    xt, xb = x_for(rng, bs, 16, ep.DT_BF16)
    for nums_type in (0, 1):
        _run(legacy, xt, xb, ids, e, nums_type, mask=mask)
