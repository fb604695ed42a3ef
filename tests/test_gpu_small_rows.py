"""Single-launch dispatch on both sides of the size up to which its rows are left to the L2, with and without a mask, in both
counts of ids per lane: rows, row map and the combine that follows on the same stream, eagerly and replayed from a graph with the
inputs changed in between."""
import pytest
import torch

from gpu_harness import DEV, Session
from tilexr_amd import ep

pytestmark = pytest.mark.gpu

CASES = [
    # tokens, columns, top_k: 2.5 MiB of token rows and rows are 1 310 720 elements
    (1, 8, 1), (3, 1024, 8), (142, 1024, 8), (160, 1024, 8), (146, 1024, 8), (20, 7168, 8), (21, 7168, 8), (9, 16384, 8),
    (79, 8192, 1), (80, 8192, 1), (81, 8192, 1), (250, 1024, 8), (7, 1000, 5),
]


@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("case", CASES)
def test_rows_and_sums_of_small_calls(case, masked):
    bs, h, k = case
    experts = 64
    gen = torch.Generator(device=DEV)
    gen.manual_seed(bs * 7 + h + k)
    with Session() as s:
        x = torch.empty(bs, h, dtype=torch.bfloat16, device=DEV)
        ids = torch.empty(bs, k, dtype=torch.int32, device=DEV)
        w = torch.empty(bs, k, dtype=torch.float32, device=DEV)
        mask = (torch.arange(bs, device=DEV) < max(1, bs * 3 // 4)).to(torch.uint8) if masked else None
        rows = torch.zeros(bs * k, h, dtype=torch.bfloat16, device=DEV)
        assist = torch.zeros(bs * k, 4, dtype=torch.int32, device=DEV)
        nums = torch.zeros(experts, dtype=torch.int64, device=DEV)
        counts = torch.zeros(experts, dtype=torch.int32, device=DEV)
        row_map = torch.zeros(bs, k, dtype=torch.int32, device=DEV)
        y = torch.zeros(bs, h, dtype=torch.bfloat16, device=DEV)

        def fill():
            x.copy_(torch.randn(bs, h, device=DEV, generator=gen))
            ids.copy_(torch.topk(torch.rand(bs, experts, device=DEV, generator=gen), k, dim=1).indices)
            w.copy_(torch.rand(bs, k, device=DEV, generator=gen))
            torch.cuda.synchronize()

        def call():
            st, _ = ep.dispatch_memory_ex(x, ids, s.comm, bs, h, k, experts, rows, assist, nums, counts, ep.DT_BF16, s.stream,
                                          row_index_map=row_map, active_mask=mask,
                                          active_mask_type=ep.MASK_TOKEN if masked else ep.MASK_NONE)
            assert st == 0
            assert ep.combine_memory_ex(rows, assist, counts, s.comm, bs, h, k, experts, y, ep.DT_BF16, s.stream,
                                        expert_scales=w, row_index_map=row_map) == 0

        def check():
            live = torch.ones(bs, dtype=torch.bool, device=DEV) if mask is None else mask.bool()
            flat = torch.where(live[:, None], ids, experts).reshape(-1).long()
            order = torch.sort(flat, stable=True).indices
            want_map = torch.empty_like(order)
            want_map[order] = torch.arange(order.numel(), device=DEV)
            want_map = torch.where(flat < experts, want_map, -1).reshape(bs, k)
            assert torch.equal(row_map.long(), want_map)
            total = torch.zeros(bs, h, dtype=torch.float32, device=DEV)
            for slot in range(k):
                at = row_map[:, slot].long()
                assert torch.equal(rows[at[live]], x[live])
                total = torch.where(live[:, None], total + x.float() * w[:, slot:slot + 1], total)
            assert torch.equal(y, total.to(torch.bfloat16))

        fill()
        call()
        s.sync()
        assert ep.last_kernel_name(s.comm, ep.K_SCATTER) == "ep_dispatch_small_route_kernel"
        check()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=s.stream):
            call()
        for _ in range(3):
            fill()
            graph.replay()
            torch.cuda.synchronize()
            check()
