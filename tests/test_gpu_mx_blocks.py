"""MXFP8 blocks at the edges of the codec, dispatch output and combine exchange, against the oracle bit for bit: blocks of
subnormals, blocks whose largest elements saturate, a clamped shared exponent, NaNs (blocks that are not finite take
another path in the kernels), blocks of zeros, and a last block of fewer than 32 columns.  Infinities are left out: the
kernels derive a block's exponent from their exponent field, the oracle gives such a block the largest exponent.
"""
import numpy as np
import pytest
import torch

from gpu_harness import DEV, Session, alloc_dispatch_outputs, bits16, fetch, to_dev
from oracle import ep as O
from tilexr_amd import ep

pytestmark = pytest.mark.gpu


def edge_rows(rng, rows, h, dtype):
    """16-bit patterns, block by block of one of the kinds above."""
    mant = 7 if dtype == ep.DT_BF16 else 10
    top = (1 << (15 - mant)) - 1                                  # exponent field of infinities and NaNs
    out = np.zeros((rows, h), np.uint16)
    for r in range(rows):
        for b in range(0, h, 32):
            n = min(32, h - b)
            kind = rng.integers(0, 8)
            sign = rng.integers(0, 2, n).astype(np.uint16) << 15
            m = rng.integers(0, 1 << mant, n)
            if kind == 0:
                e = np.zeros(n, np.int64)                         # subnormals
            elif kind == 1:
                e = np.full(n, rng.integers(1, top))              # one binade: the upper eighth of it saturates
                m |= 7 << (mant - 3)
            elif kind == 2:
                e = rng.integers(0, 18, n)                        # shared exponent at or near its lower clamp (bf16)
            elif kind == 3:
                e = np.full(n, top)                               # NaNs among finite elements
                e[n // 2:] = rng.integers(0, top, n - n // 2)
                m |= 1
            elif kind == 4:
                continue                                          # zeros
            else:
                hi = rng.integers(1, top)
                e = np.clip(hi - rng.integers(0, 14, n), 0, top - 1)
            out[r, b:b + n] = sign | (e.astype(np.uint16) << mant) | m.astype(np.uint16)
    return out


def as_tensor(bits, dtype):
    return torch.from_numpy(bits.view(np.int16)).view(torch.bfloat16 if dtype == ep.DT_BF16 else torch.float16).to(DEV)


def values(bits, dtype):
    """Finite and infinite patterns as they are, every NaN as one value (its payload is the adder's choice)."""
    nan = (bits & 0x7fff) > (0x7f80 if dtype == ep.DT_BF16 else 0x7c00)
    return np.where(nan, np.uint16(0xffff), bits)


@pytest.mark.parametrize("dtype", [ep.DT_BF16, ep.DT_FP16])
@pytest.mark.parametrize("fp8,comm", [(ep.DT_FP8E4M3, ep.Q_MXFP8), (ep.DT_FP8E5M2, ep.Q_COMM_E5M2)])
@pytest.mark.parametrize("h", [32, 1000, 1024, 2016, 7168])
def test_mx_blocks_at_the_edges(dtype, fp8, comm, h):
    bs, K, E = 37, 3, 8
    rng = np.random.default_rng(h + dtype + 7 * comm)
    ids = np.stack([rng.permutation(E)[:K] for _ in range(bs)]).astype(np.int32)
    xb = edge_rows(rng, bs, h, dtype)
    x = as_tensor(xb, dtype)
    with Session() as s:
        out = alloc_dispatch_outputs(bs, h, K, E, quant=ep.Q_MXFP8)
        counts = torch.zeros((E,), dtype=torch.int32, device=DEV)
        assert ep.dispatch_memory_v2(x, to_dev(ids), s.comm, bs, h, K, E, out["expand_x"], out["assist"], out["token_nums"],
                                     counts, dtype, s.stream, quant_mode=ep.Q_MXFP8, dynamic_scales=out["scales"],
                                     expand_x_dtype=fp8) == 0
        s.sync()
        got = fetch(out, "send_counts", counts)
        want = O.mem_dispatch(O.Case(1, bs, h, K, E, dtype=dtype, quant_mode=O.Q_MXFP8, out_dtype=fp8), 0, xb[None], ids[None])
        assert np.array_equal(got["assist"], want["assist"])
        assert np.array_equal(got["expand_x"], want["expand_x"])
        assert np.array_equal(got["scales"], want["dyn_scales"])
        if h % 32 != 0:
            return                                                # the exchange takes whole blocks only
        eo = edge_rows(rng, bs * K, h, dtype)
        w = rng.standard_normal((bs, K)).astype(np.float32)
        y = torch.full((bs, h), 7.0, dtype=x.dtype, device=DEV)
        d_eo = as_tensor(eo, dtype)
        assert ep.combine_memory_v2(d_eo, out["assist"], counts, s.comm, bs, h, K, E, y, dtype, s.stream,
                                    expert_scales=to_dev(w), quant_mode=comm) == 0
        s.sync()
        wy = O.mem_combine(O.Case(1, bs, h, K, E, dtype=dtype), 0, eo[None], want["assist"][None], want["send_counts"][None],
                           expert_scales=w, comm_quant=comm)
        assert np.array_equal(values(bits16(y), dtype), values(wy, dtype))
