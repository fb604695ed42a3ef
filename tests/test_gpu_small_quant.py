"""Decode-sized calls of quantised rows, a dispatch and a combine of one launch each: both sides of the largest table and
width they take, rows narrower than a workgroup, more experts than routes, masks, readiness flags of every payload, MXFP8
exchange with and without infinities.  Bit for bit against the oracle."""
import numpy as np
import pytest
import torch

from gpu_harness import DEV, Session, alloc_dispatch_outputs, bits16, fetch, to_dev
from oracle import ep as O
from test_gpu_mx_blocks import as_tensor, edge_rows, mx_round_trip, rows_with_infinities, values
from test_gpu_parity import check_dispatch, ids_for, x_for
from tilexr_amd import ep

pytestmark = pytest.mark.gpu

SMALL, GENERAL = "ep_dispatch_small_route_kernel", "ep_scatter_vec_kernel"
MODES = [(ep.Q_TOKEN_INT8, None), (ep.Q_MXFP8, ep.DT_FP8E4M3), (ep.Q_MXFP8, ep.DT_FP8E5M2), (ep.Q_FP8_BLOCK128, None)]


@pytest.mark.parametrize("bs,h,k,e,kernel", [
    (1, 8, 1, 3, SMALL), (3, 136, 2, 1500, SMALL), (9, 4096, 6, 64, SMALL), (7, 4104, 5, 16, SMALL), (33, 8192, 8, 64, SMALL),
    (11, 8200, 2, 8, GENERAL), (256, 64, 8, 32, SMALL), (257, 64, 8, 32, GENERAL)])
@pytest.mark.parametrize("dtype", [ep.DT_BF16, ep.DT_FP16])
@pytest.mark.parametrize("quant,fp8", MODES)
@pytest.mark.parametrize("mask_type", [ep.MASK_NONE, ep.MASK_TOKEN, ep.MASK_EXPERT])
def test_dispatch(bs, h, k, e, kernel, dtype, quant, fp8, mask_type):
    rng = np.random.default_rng(bs + h + quant + mask_type)
    ids = ids_for(rng, bs, k, e, invalid=0.05)
    xt, xb = x_for(rng, bs, h, dtype, scale=2.0)
    mask = None
    if mask_type != ep.MASK_NONE:
        mask = (rng.random((bs,) if mask_type == ep.MASK_TOKEN else (bs, k)) < 0.7).astype(np.uint8)
    case = O.Case(1, bs, h, k, e, dtype=dtype, quant_mode=quant, out_dtype=fp8 or O.DT_FP8E4M3, mask_type=mask_type)
    with Session() as s:
        out = alloc_dispatch_outputs(bs, h, k, e, quant=quant)
        counts = torch.zeros((e,), dtype=torch.int32, device=DEV)
        flags = torch.zeros(((bs * k + 63) // 64,), dtype=torch.int64, device=DEV)
        st, epoch = ep.dispatch_memory_ex(
            xt, to_dev(ids), s.comm, bs, h, k, e, out["expand_x"], out["assist"], out["token_nums"], counts, dtype, s.stream,
            quant_mode=quant, dynamic_scales=out["scales"], expand_x_dtype=fp8, row_index_map=out["row_map"],
            active_mask=to_dev(mask), active_mask_type=mask_type, tile_flags=flags, tile_rows=64)
        assert st == 0
        s.sync()
        assert ep.last_kernel_name(s.comm, ep.K_SCATTER) == kernel
        got = fetch(out, "send_counts", counts)
        want = O.mem_dispatch(case, 0, xb[None], ids[None], None if mask is None else mask[None])
        check_dispatch(got, want)
        n = want["rows"]
        assert np.array_equal(got["send_counts"], want["send_counts"])
        assert np.array_equal(got["scales"][:n], want["dyn_scales"][:n])
        tiles = [min(64, n - t) for t in range(0, n, 64)]
        assert flags.cpu().tolist() == [(epoch << 32) | t for t in tiles] + [0] * (len(flags) - len(tiles))
        if quant != ep.Q_MXFP8 and h % 16 == 0:
            # every row reported landed: the combine on the same stream finds all words and reads what is there
            w = (0.5 + rng.random((bs, k))).astype(np.float32)
            y = torch.full((bs, h), 7.0, dtype=xt.dtype, device=DEV)
            status = torch.zeros((1,), dtype=torch.int32, device=DEV)
            assert ep.combine_memory_ex(
                out["expand_x"], out["assist"], counts, s.comm, bs, h, k, e, y, dtype, s.stream, expert_out_quant_mode=quant,
                expert_out_scales=out["scales"], expert_scales=to_dev(w), row_index_map=out["row_map"], tile_flags=flags,
                tile_rows=64, flag_epoch=epoch, device_status=status) == 0
            s.sync()
            wy = O.mem_combine(O.Case(1, bs, h, k, e, dtype=dtype), 0, want["expand_x"][None], want["assist"][None],
                               want["send_counts"][None], expert_scales=w, in_quant=quant, in_scales=want["dyn_scales"])
            assert int(status) == 0 and np.array_equal(bits16(y), wy)


@pytest.mark.parametrize("bs,h,k,kernel", [
    (1, 32, 1, "ep_reduce_small_kernel"), (37, 1024, 3, "ep_reduce_small_kernel"), (16, 16384, 9, "ep_reduce_small_kernel"),
    (256, 96, 8, "ep_reduce_small_kernel"), (257, 96, 8, "ep_reduce_vec_kernel")])
@pytest.mark.parametrize("dtype", [ep.DT_BF16, ep.DT_FP16])
@pytest.mark.parametrize("comm", [ep.Q_MXFP8, ep.Q_COMM_E5M2])
@pytest.mark.parametrize("infinite", [False, True])
def test_mx_exchange(bs, h, k, kernel, dtype, comm, infinite):
    e = 32
    rng = np.random.default_rng(bs + h + comm)
    ids = ids_for(rng, bs, k, e)
    _, xb = x_for(rng, bs, h, dtype)
    d = O.mem_dispatch(O.Case(1, bs, h, k, e, dtype=dtype), 0, xb[None], ids[None])
    eo = (rows_with_infinities if infinite else edge_rows)(rng, bs * k, h, dtype)
    mask = (np.arange(bs) < max(1, bs - 3)).astype(np.uint8)
    _, shared = x_for(rng, bs, h, dtype)
    w = rng.standard_normal((bs, k)).astype(np.float32)
    with Session() as s:
        d_eo, d_shared = as_tensor(eo, dtype), as_tensor(shared, dtype)
        y = torch.full((bs, h), 7.0, dtype=d_eo.dtype, device=DEV)
        assert ep.combine_memory_v2(d_eo, to_dev(d["assist"]), to_dev(d["send_counts"]), s.comm, bs, h, k, e, y, dtype, s.stream,
                                    expert_scales=to_dev(w), active_mask=to_dev(mask), active_mask_type=ep.MASK_TOKEN,
                                    shared_expert_x=d_shared, quant_mode=comm) == 0
        s.sync()
        assert ep.last_kernel_name(s.comm, ep.K_REDUCE) == kernel
        if infinite:
            # (the oracle's codec takes finite values)
            fp8 = ep.DT_FP8E4M3 if comm == ep.Q_MXFP8 else ep.DT_FP8E5M2
            back = mx_round_trip(eo, dtype, fp8)[2]
            row = np.empty((bs, k), np.int64)
            row[d["assist"][:, 1], d["assist"][:, 2]] = np.arange(bs * k)
            acc = np.zeros((bs, h), np.float32)
            with np.errstate(invalid="ignore", over="ignore"):
                for slot in range(k):
                    acc = acc + back[row[:, slot]] * w[:, slot:slot + 1]
                acc = acc + d_shared.float().cpu().numpy()
            if dtype == ep.DT_FP16:
                acc = np.clip(acc, -65504.0, 65504.0)
            want = bits16(torch.from_numpy(np.where(mask[:, None] != 0, acc, np.float32(0))).to(y.dtype))
        else:
            want = O.mem_combine(O.Case(1, bs, h, k, e, dtype=dtype, mask_type=ep.MASK_TOKEN), 0, eo[None], d["assist"][None],
                                 d["send_counts"][None], expert_scales=w, token_mask=mask, shared_expert_x=shared, comm_quant=comm)
        assert np.array_equal(values(bits16(y), dtype), values(want, dtype))


@pytest.mark.parametrize("bs,kernel", [(40, SMALL), (1100, GENERAL)])
@pytest.mark.parametrize("dtype", [ep.DT_BF16, ep.DT_FP16])
def test_int8_of_numbers_that_are_not_finite(bs, kernel, dtype):
    """A NaN does not take part in its row's maximum and becomes -128; in a row with an infinity, whose scale is infinite, so does
    the infinity, and what is finite becomes 0.  (The oracle takes finite rows.)"""
    h, k, e = 136, 2, 8
    rng = np.random.default_rng(bs)
    ids = ids_for(rng, bs, k, e)
    xt, _ = x_for(rng, bs, h, dtype, scale=2.0)
    plain = xt.clone()
    xt[::3, 5], xt[::3, h - 1] = float("nan"), -float("nan")
    xt[1::3, 7] = float("inf")
    plain[::3, 5] = plain[::3, h - 1] = 0.0
    with Session() as s:
        got = []
        for x in (xt, plain):
            out = alloc_dispatch_outputs(bs, h, k, e, quant=ep.Q_TOKEN_INT8)
            counts = torch.zeros((e,), dtype=torch.int32, device=DEV)
            assert ep.dispatch_memory_ex(x, to_dev(ids), s.comm, bs, h, k, e, out["expand_x"], out["assist"], out["token_nums"],
                                         counts, dtype, s.stream, quant_mode=ep.Q_TOKEN_INT8, dynamic_scales=out["scales"],
                                         row_index_map=out["row_map"])[0] == 0
            s.sync()
            assert ep.last_kernel_name(s.comm, ep.K_SCATTER) == kernel
            got.append(fetch(out, "send_counts", counts))
    token = got[0]["assist"][:, 1]
    want, scales = got[1]["expand_x"].view(np.int8).copy(), got[1]["scales"].copy()
    nan, inf = token % 3 == 0, token % 3 == 1
    want[nan, 5] = want[nan, h - 1] = -128
    want[inf] = 0
    want[inf, 7] = -128
    scales[inf] = np.inf
    assert np.array_equal(got[0]["expand_x"].view(np.int8), want)
    assert np.array_equal(got[0]["scales"], scales)
