"""Which kernel copies the rows and how they are stored goes by sizes: plain rows on both sides of what the memory-side cache
takes, rows that end within a 128-byte line on both sides of what is worth keeping, block fp8 rows on both sides of twice
that cache, with and without readiness flags.  Rows are compared bit for bit with the token rows (plain), or with the rows of
a call that places every token once (quantised), at the places a stable sort of the ids gives."""
import pytest
import torch

from gpu_harness import DEV, Session
from tilexr_amd import ep

pytestmark = pytest.mark.gpu

CASES = [
    # tokens, columns, top_k, experts, payload, kernel
    (1029, 4104, 39, 64, "none", "ep_scatter_vec_kernel"),          # 314 MiB
    (1029, 4104, 40, 64, "none", "ep_scatter_route_kernel"),        # 322 MiB
    (1023, 4104, 41, 64, "none", "ep_scatter_vec_kernel"),          # 328 MiB of fewer than 1024 tokens
    (2097, 1000, 8, 16, "none", "ep_scatter_vec_kernel"),           # 32 MiB less 2432 bytes: streams
    (2098, 1000, 8, 16, "none", "ep_scatter_vec_kernel"),
    (687, 2560, 3, 16, "none", "ep_scatter_vec_kernel"),            # 320 vectors: the narrowest rows with a cap
    (411, 4104, 5, 16, "none", "ep_scatter_vec_kernel"),            # 513 vectors
    (1000, 16384, 3, 8, "none", "ep_scatter_vec_kernel"),           # the widest rows
    (1400, 16384, 8, 64, "none", "ep_scatter_route_kernel"),        # ... published in two parts
    (2600, 8200, 8, 64, "none", "ep_scatter_route_kernel"),         # a second part of one vector
    (1100, 8200, 8, 64, "none", "ep_scatter_vec_kernel"),           # published whole
    (1000, 1048, 5, 16, "int8", "ep_scatter_vec_kernel"),
    (4100, 1040, 8, 16, "int8", "ep_scatter_vec_kernel"),           # ends within a line, 32 MiB and more: ordinary stores
    (1200, 7176, 4, 16, "none", "ep_scatter_vec_kernel"),
    (16384, 4096, 8, 64, "fp8", "ep_scatter_vec_kernel"),           # exactly 512 MiB
    (16385, 4096, 8, 64, "fp8", "ep_scatter_vec_kernel"),
    # rows that the scatter resolves itself (too many routes x experts for the one-launch routing), on both sides of the vectors
    # stored from which a cap of four and of two workgroups per compute unit pays
    (2100, 3576, 8, 600, "none", "ep_scatter_vec_kernel"),
    (2100, 3584, 8, 600, "none", "ep_scatter_vec_kernel"),
    (2100, 4600, 8, 600, "none", "ep_scatter_vec_kernel"),
    (2100, 4608, 8, 600, "none", "ep_scatter_vec_kernel"),
]
QUANT = {"none": ep.Q_NONE, "int8": ep.Q_TOKEN_INT8, "fp8": ep.Q_FP8_BLOCK128}


def _dispatch(s, x, ids, experts, payload, flags):
    bs, h = x.shape
    k = ids.shape[1]
    n = bs * k
    o = dict(rows=torch.full((n, h), 7, dtype=torch.bfloat16 if payload == "none" else torch.uint8, device=DEV),
             scales=None, row_map=torch.full((bs, k), -1, dtype=torch.int32, device=DEV))
    if payload != "none":
        o["scales"] = torch.zeros((n, 1 if payload == "int8" else (h + 127) // 128), dtype=torch.float32, device=DEV)
    assist = torch.zeros((n, 4), dtype=torch.int32, device=DEV)
    nums = torch.zeros((experts,), dtype=torch.int64, device=DEV)
    counts = torch.zeros((experts,), dtype=torch.int32, device=DEV)
    words = torch.zeros(((n + 63) // 64,), dtype=torch.int64, device=DEV) if flags else None
    torch.cuda.synchronize()
    st, epoch = ep.dispatch_memory_ex(x, ids, s.comm, bs, h, k, experts, o["rows"], assist, nums, counts, ep.DT_BF16, s.stream,
                                      quant_mode=QUANT[payload], dynamic_scales=o["scales"], row_index_map=o["row_map"],
                                      tile_flags=words, tile_rows=64 if flags else 0)
    assert st == 0
    s.sync()
    if flags:
        tiles = torch.arange(words.numel(), device=DEV)
        assert torch.equal(words, (epoch << 32) | torch.clamp(n - tiles * 64, max=64))
    return o


@pytest.mark.parametrize("flags", [False, True])
@pytest.mark.parametrize("case", CASES)
def test_rows_are_whole_whatever_stores_them(case, flags):
    bs, h, k, experts, payload, kernel = case
    gen = torch.Generator(device=DEV)
    gen.manual_seed(bs + h + k)
    x = torch.randn(bs, h, device=DEV, generator=gen).to(torch.bfloat16)
    ids = torch.topk(torch.rand(bs, experts, device=DEV, generator=gen), k, dim=1).indices.to(torch.int32).contiguous()
    with Session() as s:
        got = _dispatch(s, x, ids, experts, payload, flags)
        assert ep.last_kernel_name(s.comm, ep.K_SCATTER) == kernel
        order = torch.sort(ids.reshape(-1).long(), stable=True).indices        # route of every row
        rows_of = torch.empty_like(order)
        rows_of[order] = torch.arange(order.numel(), device=DEV)
        assert torch.equal(got["row_map"].reshape(-1).long(), rows_of)
        want, scales = x, None
        if payload != "none":
            once = _dispatch(s, x, torch.zeros((bs, 1), dtype=torch.int32, device=DEV), 1, payload, False)
            want, scales = once["rows"], once["scales"]
        for slot in range(k):
            at = got["row_map"][:, slot].long()
            assert torch.equal(got["rows"][at], want), slot
            assert scales is None or torch.equal(got["scales"][at], scales), slot
