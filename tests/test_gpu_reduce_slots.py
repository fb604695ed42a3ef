"""Slots of a token that the lanes of a wave look up, and put in order, for themselves: counts of slots on both sides of what
is read at once, up to one per lane; rows that are missing; rows whose order is not the slots'; one, two and four waves to a
token; several tokens to a workgroup, the last one not full.  Bit for bit against the oracle."""
import numpy as np
import pytest
import torch

from gpu_harness import DEV, Session, bits16, to_dev
from oracle import ep as O
from tilexr_amd import ep
from test_gpu_parity import ids_for, x_for

pytestmark = pytest.mark.gpu


def _lose(rng, d, bs, k):
    keep = rng.random((bs, k)) < rng.random((bs, 1))
    keep[0], keep[1], keep[2, :k - 1], keep[2, k - 1] = True, False, False, True
    assist = d["assist"].copy()
    assist[~keep[assist[:, 1], assist[:, 2]], 1] = -1
    return assist


@pytest.mark.parametrize("k", [1, 4, 5, 6, 7, 32])
@pytest.mark.parametrize("h", [64, 1040, 2064, 4096, 4112])
@pytest.mark.parametrize("quant", [ep.Q_TOKEN_INT8, ep.Q_FP8_BLOCK128])
@pytest.mark.parametrize("dtype", [ep.DT_BF16, ep.DT_FP16])
def test_quantised_rows_by_slots(k, h, quant, dtype):
    bs, experts = 67, 40
    rng = np.random.default_rng(k * 10000 + h + quant)
    ids = ids_for(rng, bs, k, experts)
    _, xb = x_for(rng, bs, h, dtype, scale=2.0)
    d = O.mem_dispatch(O.Case(1, bs, h, k, experts, dtype=dtype, quant_mode=quant), 0, xb[None], ids[None])
    assist = _lose(rng, d, bs, k)
    w = (0.5 + rng.random((bs, k))).astype(np.float32)
    tdt = torch.bfloat16 if dtype == ep.DT_BF16 else torch.float16
    with Session() as s:
        y = torch.full((bs, h), 7.0, dtype=tdt, device=DEV)
        args = [to_dev(v) for v in (d["expand_x"], assist, d["send_counts"], d["dyn_scales"], w)]
        torch.cuda.synchronize()
        assert ep.combine_memory_ex(args[0], args[1], args[2], s.comm, bs, h, k, experts, y, dtype, s.stream,
                                    expert_out_quant_mode=quant, expert_out_scales=args[3], expert_scales=args[4]) == 0
        s.sync()
        assert ep.last_kernel_name(s.comm, ep.K_REDUCE) == "ep_reduce_quant_kernel"
        want = O.mem_combine(O.Case(1, bs, h, k, experts, dtype=dtype), 0, d["expand_x"][None], assist[None],
                             d["send_counts"][None], expert_scales=w, in_quant=quant, in_scales=d["dyn_scales"])
        assert np.array_equal(bits16(y), want)


@pytest.mark.parametrize("h", [64, 2048, 4112, 16384])
@pytest.mark.parametrize("k", [2, 6])
@pytest.mark.parametrize("quant,edge", [(ep.Q_TOKEN_INT8, 511.875), (ep.Q_FP8_BLOCK128, 146.25)])
def test_fp16_rows_that_saturate(h, k, quant, edge):
    """A row's largest magnitude (128 or 448 times its scale) on both sides of the 65520 from which rounding to fp16 has to
    saturate, beside rows that stay far below; infinite and NaN scales; zero and negative ones."""
    bs, experts = 48, 8
    rng = np.random.default_rng(h + k + quant)
    ids = ids_for(rng, bs, k, experts)
    _, xb = x_for(rng, bs, h, ep.DT_FP16, scale=2.0)
    d = O.mem_dispatch(O.Case(1, bs, h, k, experts, dtype=ep.DT_FP16, quant_mode=quant), 0, xb[None], ids[None])
    payload = d["expand_x"].view(np.uint8).copy()
    payload[:, ::5] = 0x80 if quant == ep.Q_TOKEN_INT8 else 0x7e        # -128, 448
    payload[:, 1::5] = 0x7f if quant == ep.Q_TOKEN_INT8 else 0xfe       # 127, -448
    edge = np.float32(edge)
    some = np.array([1.0, 0.0, np.nextafter(edge, np.float32(0)), edge, np.nextafter(edge, np.float32(1e9)), -edge, 3e4, 1e-6,
                     np.inf, -np.inf, np.nan], np.float32)
    scales = np.ones_like(d["dyn_scales"])
    odd = rng.random(scales.shape) < 0.3
    scales[odd] = rng.choice(some, int(odd.sum()))
    w = (0.5 + rng.random((bs, k))).astype(np.float32)
    with Session() as s:
        y = torch.full((bs, h), 7.0, dtype=torch.float16, device=DEV)
        args = [to_dev(v) for v in (payload, d["assist"], d["send_counts"], scales, w)]
        torch.cuda.synchronize()
        assert ep.combine_memory_ex(args[0], args[1], args[2], s.comm, bs, h, k, experts, y, ep.DT_FP16, s.stream,
                                    expert_out_quant_mode=quant, expert_out_scales=args[3], expert_scales=args[4]) == 0
        s.sync()
        want = O.mem_combine(O.Case(1, bs, h, k, experts, dtype=ep.DT_FP16), 0, payload[None], d["assist"][None],
                             d["send_counts"][None], expert_scales=w, in_quant=quant, in_scales=scales)
        got, want = bits16(y), want.view(np.uint16).reshape(bs, h)
        nan = (want & 0x7fff) > 0x7c00
        assert nan.any() and not nan.all() and ((want & 0x7fff) == 0x7bff).any()
        assert np.array_equal((got & 0x7fff) > 0x7c00, nan)             # (a NaN's sign is the adder's choice of operand)
        assert np.array_equal(got[~nan], want[~nan])


@pytest.mark.parametrize("bs,h,k", [(5, 64, 8), (700, 64, 5), (41, 1024, 64), (300, 1032, 8), (65, 4104, 33), (3, 16384, 2)])
def test_sums_in_the_order_of_the_rows(bs, h, k):
    """The MVP route adds rows in ascending row order; here the rows of a token stand in any order of its slots."""
    experts = 64
    rng = np.random.default_rng(bs + h + k)
    ids = ids_for(rng, bs, k, experts)
    _, xb = x_for(rng, bs, h, ep.DT_FP16, scale=2.0)
    case = O.Case(1, bs, h, k, experts, dtype=O.DT_FP16)
    d = O.mvp_dispatch(case, 0, xb[None], ids[None])
    assist = _lose(rng, d, bs, k)[rng.permutation(bs * k)]
    rows = xb[rng.integers(0, bs, bs * k)]
    counts = np.array([bs * k], np.int32)
    with Session() as s:
        y = torch.full((bs, h), 7.0, dtype=torch.float16, device=DEV)
        args = [to_dev(v) for v in (rows, assist, counts)]
        torch.cuda.synchronize()
        assert ep.combine_v2(args[0], args[1], args[2], s.comm, bs, h, k, experts, y, ep.DT_FP16, s.stream) == 0
        s.sync()
        assert np.array_equal(bits16(y), O.mvp_combine(case, 0, rows[None], assist[None], counts[None]))


@pytest.mark.parametrize("bs,h,k", [(2950, 8016, 1), (12007, 2064, 2), (23611, 1008, 1), (5801, 4096, 2)])
@pytest.mark.parametrize("quant", [ep.Q_TOKEN_INT8, ep.Q_FP8_BLOCK128])
@pytest.mark.parametrize("dtype", [ep.DT_BF16, ep.DT_FP16])
def test_several_tokens_to_a_wave(bs, h, k, quant, dtype):
    """One or two slots and outputs of 47 MB and more: slices that end within a row, tokens that do not fill the last wave,
    lost rows, masked tokens, a shared expert; in places scales whose rows saturate in fp16, and NaN codes."""
    _reduce_few(bs, h, k, quant, dtype, "ep_reduce_quant_few_kernel")


@pytest.mark.parametrize("bs,h,k,kernel", [
    (3301, 7168, 1, "few_"), (3301, 7184, 1, ""), (3005, 7920, 2, ""), (3005, 7936, 2, "few_"), (1777, 13312, 2, "few_"),
    (1777, 13328, 2, ""), (1777, 13440, 1, "few_")])
def test_rows_that_end_within_a_line(bs, h, k, kernel):
    """Both sides of the widths at which such rows take one token to a wave."""
    _reduce_few(bs, h, k, ep.Q_TOKEN_INT8, ep.DT_BF16, f"ep_reduce_quant_{kernel}kernel")


def _reduce_few(bs, h, k, quant, dtype, kernel):
    experts = 16
    rng = np.random.default_rng(bs + h + quant)
    ids = ids_for(rng, bs, k, experts)
    d = O.mem_dispatch(O.Case(1, bs, 16, k, experts), 0, np.zeros((1, bs, 16), np.uint16), ids[None])
    assist = _lose(rng, d, bs, k)
    n = bs * k
    payload = rng.integers(0, 256, (n, h), dtype=np.uint8)
    if quant == ep.Q_FP8_BLOCK128:
        payload[(payload & 0x7f) == 0x7f] = 0x30
        payload[rng.integers(0, n, 50), rng.integers(0, h, 50)] = rng.choice([0x7f, 0xff], 50)
    scales = rng.random((n, 1 if quant == ep.Q_TOKEN_INT8 else (h + 127) // 128)).astype(np.float32)
    scales[rng.integers(0, n, 60), rng.integers(0, scales.shape[1], 60)] = rng.choice(np.array([140, 147, 500, 512, 1e5], np.float32), 60)
    w = (0.5 + rng.random((bs, k))).astype(np.float32)
    mask = (rng.random(bs) < 0.9).astype(np.uint8)
    _, shared = x_for(rng, bs, h, dtype)
    with Session() as s:
        y = torch.full((bs, h), 7.0, dtype=torch.bfloat16 if dtype == ep.DT_BF16 else torch.float16, device=DEV)
        args = [to_dev(v) for v in (payload, assist, d["send_counts"], scales, w, mask, shared.view(np.int16))]
        torch.cuda.synchronize()
        assert ep.combine_memory_ex(args[0], args[1], args[2], s.comm, bs, h, k, experts, y, dtype, s.stream,
                                    expert_out_quant_mode=quant, expert_out_scales=args[3], expert_scales=args[4],
                                    active_mask=args[5], active_mask_type=ep.MASK_TOKEN, shared_expert_x=args[6]) == 0
        s.sync()
        assert ep.last_kernel_name(s.comm, ep.K_REDUCE) == kernel
        got = bits16(y)
    want = O.mem_combine(O.Case(1, bs, h, k, experts, dtype=dtype, mask_type=ep.MASK_TOKEN), 0, payload[None], assist[None],
                         d["send_counts"][None], expert_scales=w, token_mask=mask, shared_expert_x=shared, in_quant=quant,
                         in_scales=scales).view(np.uint16).reshape(bs, h)
    infinity = 0x7f80 if dtype == ep.DT_BF16 else 0x7c00
    nan = (want & 0x7fff) > infinity
    assert nan.any() == (quant == ep.Q_FP8_BLOCK128)
    assert np.array_equal((got & 0x7fff) > infinity, nan)       # (a NaN's sign is the adder's choice of operand)
    assert np.array_equal(got[~nan], want[~nan])
