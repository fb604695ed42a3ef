"""Dispatches whose scatter launch builds the plan, fills the rows nobody copies to and writes the status: sizes at the edges
of a plan workgroup's 256 rows and of the totals it looks at, more routes per token than it reads at once, several ranks, and
saved plans whose copies the launch makes from the primaries' token rows.  Compared with the oracle bit for bit."""
import numpy as np
import pytest

import moonep_cases as MC
from oracle import moonep as M
from tilexr_amd import moonep as mp
from test_gpu_moonep import World, check_dispatch, random_rows, row_cache  # noqa: F401  (row_cache: both scatter kernels)

pytestmark = pytest.mark.gpu

CASES = [
    # world, s, k, h, rows beyond the routes
    (1, 32, 8, 64, 0),          # 256 rows: one workgroup, all its threads
    (1, 32, 8, 64, 1),          # 257: the second has one row, which no route names
    (1, 51, 5, 64, 0),          # 255
    (2, 64, 8, 1032, 1),        # 513, two ranks: the last plan to be built writes both statuses
    (3, 40, 9, 64, 600),        # nine routes per token, read eight at a time; most rows unnamed
    (4, 30, 32, 64, 3),
    (1, 100, 3, 520, 1748),     # 2048 rows, runs of 16 of them to a wave; most unnamed, in pieces of one pass and more
    (2, 100, 3, 520, 1749),     # 2049
    (1, 8192, 8, 8, 7),         # 257 workgroups: a thread looks at two totals
    (1, 65536, 8, 8, 0),        # 2048 workgroups
    (1, 65536, 8, 8, 1),        # 2049
    (1, 131072, 8, 8, 0),       # 4096: the most of rows this narrow
    (1, 131072, 8, 8, 1),       # one more: launches behind the copies
]


@pytest.mark.parametrize("world,s,k,h,slack", CASES)
def test_built_and_saved_plans(world, s, k, h, slack, row_cache):  # noqa: F811
    rng = np.random.default_rng(world + s + k)
    sh = M.Shape(world, s, k, h, s * k + slack)
    dst = MC.random_dst(sh, rng, duplicates=True)
    hidden = random_rows(rng, (world, s, h))
    weights = rng.standard_normal((world, s * k)).astype(np.float32)
    want = M.dispatch_world(sh, dst, hidden, weights, flags=M.FLAG_BUILD_DEDUP)
    with World(world) as w:
        plans = w.plan_tensors(sh, dst)
        for flags in (mp.FLAG_BUILD_DEDUP, mp.FLAG_BUILD_DEDUP, 0):
            if flags:
                for p in plans:
                    for name in ("groups", "loffs", "counts"):
                        p[name].fill_(-7)
            res = w.dispatch(sh, plans, hidden, weights, flags=flags)
            w.sync()
            check_dispatch(sh, res, plans, want, fresh=flags != 0)


@pytest.mark.parametrize("world,s,k,slack", [(1, 51, 5, 0), (2, 64, 8, 1), (3, 100, 9, 600), (1, 8192, 8, 7)])
def test_a_chunk_whose_totals_do_not_come(world, s, k, slack, row_cache, monkeypatch):  # noqa: F811
    """No look at another workgroup's word: every thread adds up the chunks before its own from their rows' records, as it would
    after so many looks."""
    monkeypatch.setenv("TILEXR_MOONEP_PLAN_POLLS", "0")
    rng = np.random.default_rng(world + s + k)
    sh = M.Shape(world, s, k, 64, s * k + slack)
    dst = MC.random_dst(sh, rng, duplicates=True)
    hidden = random_rows(rng, (world, s, sh.h))
    want = M.dispatch_world(sh, dst, hidden, flags=M.FLAG_BUILD_DEDUP)
    with World(world) as w:
        plans = w.plan_tensors(sh, dst)
        res = w.dispatch(sh, plans, hidden, flags=mp.FLAG_BUILD_DEDUP)
        w.sync()
        check_dispatch(sh, res, plans, want, fresh=True)


@pytest.mark.parametrize("world,s,k,h", [(1, 40, 4, 64), (2, 33, 3, 4104)])
def test_saved_plans_that_disagree_with_the_routes(world, s, k, h, row_cache):  # noqa: F811
    """A plan is data: it may list a row that a route of its own names, an unnamed row, or another token's row as the primary.
    Whatever a route writes there, the row comes out as its primary's; a primary no route writes is zeros."""
    rng = np.random.default_rng(s)
    sh = M.Shape(world, s, k, h, s * k + 4)
    dst = MC.random_dst(sh, rng, duplicates=False)
    hidden = random_rows(rng, (world, s, h))
    dup = M.DupPlan.empty(sh)
    for q in range(world):
        named = np.unique(dst[(dst >= q * sh.nvs) & (dst < (q + 1) * sh.nvs)] - q * sh.nvs)
        unnamed = np.setdiff1d(np.arange(sh.nvs), named)
        assert len(named) > 6 and len(unnamed) > 2
        # two rows of routes and an unnamed one follow a named primary; a row of a route follows an unnamed primary
        dup.groups[q, :2] = [[named[0], 0, 3], [unnamed[1], 3, 1]]
        dup.loffs[q, :4] = [named[3], unnamed[0], named[5], named[6]]
        dup.counts[q] = [2, 4]
    want = M.dispatch_world(sh, dst, hidden, flags=0, dup=dup)
    assert all((want[0][q][dup.loffs[q, 3]] == 0).all() for q in range(world))
    with World(world) as w:
        plans = w.plan_tensors(sh, dst, dup=dup)
        res = w.dispatch(sh, plans, hidden, flags=0)
        w.sync()
        check_dispatch(sh, res, plans, want, fresh=False)


def test_largest_plan_of_wide_rows():
    """8192 workgroups: a thread looks at 32 totals.  The plan does not depend on the rows' width, nor do the rows matter here."""
    s, k, h = 262144, 8, 512
    dst = MC.random_dst(M.Shape(1, s, k, 8, s * k), np.random.default_rng(s), duplicates=True)
    want = M.dispatch_world(M.Shape(1, s, k, 8, s * k), dst, np.zeros((1, s, 8), np.uint16), flags=M.FLAG_BUILD_DEDUP)[3]
    sh = M.Shape(1, s, k, h, s * k)
    with World(1) as w:
        plans = w.plan_tensors(sh, dst)
        w.dispatch(sh, plans, np.zeros((1, s, h), np.uint16), flags=mp.FLAG_BUILD_DEDUP)
        w.sync()
        groups, places = (int(c) for c in plans[0]["counts"].cpu())
        assert [groups, places] == want.counts[0].tolist() and int(plans[0]["status"][0]) == 2000
        np.testing.assert_array_equal(plans[0]["groups"].cpu().numpy()[:groups], want.groups[0, :groups])
        np.testing.assert_array_equal(plans[0]["loffs"].cpu().numpy()[:places], want.loffs[0, :places])
