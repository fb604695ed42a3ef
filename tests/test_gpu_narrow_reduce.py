"""Combine of few tokens with rows of 129 to 256 vectors, which are cut in two slices: the narrowest and widest such rows,
a second slice of one vector, one token, and the numbers of tokens on both sides of where slicing ends."""
import pytest
import torch

from gpu_harness import DEV, Session
from tilexr_amd import ep

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,torch_dtype", [(ep.DT_BF16, torch.bfloat16), (ep.DT_FP16, torch.float16)])
@pytest.mark.parametrize("bs,h,K,E", [(1, 2048, 8, 16), (3, 1032, 8, 16), (7, 2040, 1, 8), (130, 1536, 9, 32), (1024, 2048, 2, 16),
                                      (1025, 2048, 2, 16), (640, 1032, 2, 16), (641, 2048, 1, 16), (1024, 1032, 3, 16),
                                      (1025, 2048, 3, 16)])
def test_matches_sums_in_slot_order(bs, h, K, E, dtype, torch_dtype):
    gen = torch.Generator(device=DEV).manual_seed(bs + h)
    x = torch.randn(bs, h, device=DEV, generator=gen).to(torch_dtype)
    ids = torch.randint(-1, E, (bs, K), device=DEV, generator=gen, dtype=torch.int32)       # -1: no expert, no row
    w = torch.rand(bs, K, device=DEV, generator=gen)
    rows = torch.zeros(bs * K, h, dtype=torch_dtype, device=DEV)
    assist = torch.zeros(bs * K, 4, dtype=torch.int32, device=DEV)
    nums = torch.zeros(E, dtype=torch.int64, device=DEV)
    counts = torch.zeros(E, dtype=torch.int32, device=DEV)
    row_map = torch.zeros(bs, K, dtype=torch.int32, device=DEV)
    y = torch.full((bs, h), 7.0, dtype=torch_dtype, device=DEV)
    torch.cuda.synchronize()
    with Session() as s:
        st, _ = ep.dispatch_memory_ex(x, ids, s.comm, bs, h, K, E, rows, assist, nums, counts, dtype, s.stream, row_index_map=row_map)
        assert st == 0
        assert ep.combine_memory_ex(rows, assist, counts, s.comm, bs, h, K, E, y, dtype, s.stream, expert_scales=w,
                                    row_index_map=row_map) == 0
        s.sync()
    want = torch.zeros(bs, h, device=DEV)
    for k in range(K):      # products and sums rounded apart, in slot order, as the combine defines them: equal bit for bit
        term = w[:, k:k + 1] * x.float()
        want = torch.where(ids[:, k:k + 1] >= 0, want + term, want)
    assert torch.equal(y, want.to(torch_dtype))
