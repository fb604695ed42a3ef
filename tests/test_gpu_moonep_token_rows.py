"""Per-token scatter of the plan-driven Dispatch: row widths on both sides of every geometry (lanes per token, vectors per lane,
slices of a row), tokens that do not fill the last group of eight workgroups, several ranks, plans that are built, also where
another launch leaves the chunk totals, and saved ones.  Compared with the oracle bit for bit."""
import numpy as np
import pytest

from oracle import moonep as M
from tilexr_amd import ep
from tilexr_amd import moonep as mp
import moonep_cases as MC
from test_gpu_moonep import World, check_dispatch, random_rows

pytestmark = pytest.mark.gpu

CASES = [
    # world, s, k, h, slack rows
    (1, 1, 1, 8, 0),
    (1, 33, 3, 1024, 5),        # 128 vectors: two per lane of a wave
    (2, 31, 5, 1032, 2),        # 129
    (1, 65, 2, 2048, 0),        # 256: four per lane of a wave
    (3, 7, 4, 2056, 9),         # 257: the workgroup, two per lane
    (2, 17, 2, 4096, 1),        # 512
    (1, 9, 8, 4104, 3),         # 513
    (2, 8, 3, 8192, 0),         # 1024: one slice
    (1, 11, 2, 8200, 4),        # 1025: two, the second of one vector
    (1, 5, 32, 16384, 7),
    (2, 1100, 8, 64, 9000),     # more chunks than a plan workgroup adds up itself
    (1, 17, 4, 4096, 1),        # 512 vectors held by a workgroup: four workgroups to a compute unit
    (1, 17, 4, 4104, 1),        # 513: two
    (2, 40, 4, 1024, 0),        # 512, of four tokens
    (2, 40, 4, 1032, 0),        # 516
    (2, 40, 3, 1032, 0),        # 516 stored three times
    (1, 50, 4, 1000, 3),        # rows that end within a 128-byte line, four and more to a token: ordinary stores
    (2, 33, 3, 520, 1),         # ... fewer: streaming ones
    (1, 21, 3, 4104, 2),
    (1, 21, 1, 2008, 0),
]


@pytest.mark.parametrize("world,s,k,h,slack", CASES)
def test_token_rows_match_oracle(world, s, k, h, slack):
    rng = np.random.default_rng(world + 10 * s + k + h)
    sh = M.Shape(world, s, k, h, s * k + slack)
    dst = MC.random_dst(sh, rng, duplicates=True)
    hidden = random_rows(rng, (world, s, h))
    weights = rng.standard_normal((world, s * k)).astype(np.float32)
    want = M.dispatch_world(sh, dst, hidden, weights, flags=M.FLAG_BUILD_DEDUP)
    with World(world) as w:
        plans = w.plan_tensors(sh, dst)
        for flags in (mp.FLAG_BUILD_DEDUP, 0, mp.FLAG_BUILD_DEDUP):
            if flags:
                for p in plans:
                    for name in ("groups", "loffs", "counts"):
                        p[name].fill_(-7)
            res = w.dispatch(sh, plans, hidden, weights, flags=flags)
            w.sync()
            assert ep.last_kernel_name(w.comms[0], ep.K_SCATTER) == "moon_scatter_token_kernel"
            check_dispatch(sh, res, plans, want, fresh=flags != 0)


@pytest.mark.parametrize("s,k,kernel", [
    (3291, 8, "moon_scatter_token_kernel"),     # 360 MiB of rows less 48 KiB: kept for Combine
    (3292, 8, "moon_scatter_kernel"),           # more: token rows read ahead, a workgroup per route
    (7606, 4, "moon_scatter_kernel"),           # 104 MiB of token rows less 12 KiB
    (7607, 4, "moon_scatter_token_kernel"),     # more: not read ahead
])
def test_sizes_pick_the_scatter(s, k, kernel):
    """The library's own choice, at the knob's default, on both sides of both of its lines; built and saved plans."""
    rng = np.random.default_rng(s)
    sh = M.Shape(1, s, k, 7168, s * k)
    dst = MC.random_dst(sh, rng, duplicates=True)
    hidden = random_rows(rng, (1, s, 7168))
    weights = rng.standard_normal((1, s * k)).astype(np.float32)
    want = M.dispatch_world(sh, dst, hidden, weights, flags=M.FLAG_BUILD_DEDUP)
    with World(1) as w:
        plans = w.plan_tensors(sh, dst)
        for flags in (mp.FLAG_BUILD_DEDUP, 0):
            res = w.dispatch(sh, plans, hidden, weights, flags=flags)
            w.sync()
            assert ep.last_kernel_name(w.comms[0], ep.K_SCATTER) == kernel
            check_dispatch(sh, res, plans, want, fresh=flags != 0)
