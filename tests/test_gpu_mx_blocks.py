"""MXFP8 blocks at the edges of the codec, dispatch output and combine exchange, against the oracle bit for bit: blocks of
subnormals, blocks whose largest elements saturate, a clamped shared exponent, NaNs (blocks that are not finite take
another path in the kernels), blocks of zeros, and a last block of fewer than 32 columns.

Blocks with infinities are compared with the software codec's rule, written out here (mx_round_trip): the kernels derive a
block's exponent from the exponent field of its largest element, an infinity's too, where the oracle gives such a block
the largest exponent.  tests/cxx/mx_convert_check.hip compares the scaled converts, which take every other block, with the
software codec for every block maximum and every element under it.
"""
import os
import subprocess

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


def mx_round_trip(bits, dtype, fp8):
    """The software codec on 16-bit patterns [rows, h], h a multiple of 32: codes, scale bytes and the fp32 values that
    come back.  A block's exponent is its largest number's (NaNs do not take part) less that of the largest code; what
    then passes the largest code, infinities among it, gets that code."""
    emax, largest, out = (8, 448.0, torch.float8_e4m3fn) if fp8 == ep.DT_FP8E4M3 else (15, 57344.0, torch.float8_e5m2)
    x = torch.from_numpy(bits.view(np.int16)).view(torch.bfloat16 if dtype == ep.DT_BF16 else torch.float16).to(torch.float32).numpy()
    x = x.reshape(x.shape[0], -1, 32)
    top = np.fmax.reduce(np.abs(x), axis=2, initial=0.0).view(np.uint32)
    se = np.where(top == 0, -127, np.clip((top >> 23).astype(np.int64) - 127 - emax, -127, 127))
    with np.errstate(invalid="ignore"):
        scaled = np.clip(np.ldexp(x, -se[:, :, None].astype(np.int32)), -largest, largest)
    codes = torch.from_numpy(scaled.astype(np.float32)).to(out)
    raw = codes.view(torch.uint8).numpy()
    raw = np.where(np.isnan(x), (x.view(np.uint32) >> 24).astype(np.uint8) & np.uint8(0x80) | np.uint8(0x7f), raw)
    back = torch.from_numpy(np.ascontiguousarray(raw)).view(out).to(torch.float32).numpy()
    with np.errstate(over="ignore"):
        back = back * np.exp2(se.astype(np.float64)).astype(np.float32)[:, :, None]
    return raw.reshape(bits.shape), (se + 127).astype(np.uint8), back.reshape(bits.shape)


def rows_with_infinities(rng, rows, h, dtype):
    """Per block one of: finite, a single infinity, both infinities, nothing else, beside a NaN, beside zeros, and the
    largest finite pattern, which is one below the infinity's."""
    inf = 0x7f80 if dtype == ep.DT_BF16 else 0x7c00
    out = rng.integers(0, inf, (rows, h)).astype(np.uint16) | (rng.integers(0, 2, (rows, h)).astype(np.uint16) << 15)
    for r in range(rows):
        for b in range(0, h, 32):
            block = out[r, b:b + 32]
            kind = rng.integers(0, 8)
            at = rng.permutation(32)
            if kind in (1, 2, 5):
                block[at[0]] = inf | (rng.integers(0, 2) << 15)
            if kind == 2:
                block[at[1]] = inf | (~block[at[0]] & 0x8000)
            elif kind == 3:
                block[:] = inf | (block & 0x8000)
            elif kind == 4:
                block[at[0]], block[at[1]] = inf, 0xffff
            elif kind == 5:
                block[at[1:]] &= 0x8000
            elif kind == 6:
                block[at[0]] = (inf - 1) | (block[at[0]] & 0x8000)
    return out


@pytest.mark.parametrize("dtype", [ep.DT_BF16, ep.DT_FP16])
@pytest.mark.parametrize("fp8,comm", [(ep.DT_FP8E4M3, ep.Q_MXFP8), (ep.DT_FP8E5M2, ep.Q_COMM_E5M2)])
@pytest.mark.parametrize("h", [32, 1024, 2016, 7168])
def test_mx_blocks_with_infinities(dtype, fp8, comm, h):
    bs, K, E = 29, 3, 8
    rng = np.random.default_rng(h + dtype + 7 * comm)
    ids = np.stack([rng.permutation(E)[:K] for _ in range(bs)]).astype(np.int32)
    xb, eo = rows_with_infinities(rng, bs, h, dtype), rows_with_infinities(rng, bs * K, h, dtype)
    w = rng.standard_normal((bs, K)).astype(np.float32)
    x, d_eo = as_tensor(xb, dtype), as_tensor(eo, dtype)
    with Session() as s:
        out = alloc_dispatch_outputs(bs, h, K, E, quant=ep.Q_MXFP8)
        counts = torch.zeros((E,), dtype=torch.int32, device=DEV)
        assert ep.dispatch_memory_v2(x, to_dev(ids), s.comm, bs, h, K, E, out["expand_x"], out["assist"], out["token_nums"],
                                     counts, dtype, s.stream, quant_mode=ep.Q_MXFP8, dynamic_scales=out["scales"],
                                     expand_x_dtype=fp8) == 0
        y = torch.full((bs, h), 7.0, dtype=x.dtype, device=DEV)
        assert ep.combine_memory_v2(d_eo, out["assist"], counts, s.comm, bs, h, K, E, y, dtype, s.stream,
                                    expert_scales=to_dev(w), quant_mode=comm) == 0
        s.sync()
        got = fetch(out, "send_counts", counts)
        token = got["assist"][:, 1]
        codes, scales, _ = mx_round_trip(xb, dtype, fp8)
        assert np.array_equal(got["expand_x"], codes[token])
        assert np.array_equal(got["scales"][:, :h // 32], scales[token])
        back = mx_round_trip(eo, dtype, fp8)[2]
        acc = np.zeros((bs, h), np.float32)
        row = np.empty((bs, K), np.int64)
        row[token, got["assist"][:, 2]] = np.arange(bs * K)
        with np.errstate(invalid="ignore", over="ignore"):
            for k in range(K):
                acc = acc + back[row[:, k]] * w[:, k:k + 1]
        if dtype == ep.DT_FP16:
            acc = np.clip(acc, -65504.0, 65504.0)                 # the output saturates
        want = torch.from_numpy(acc).to(x.dtype)
        assert np.array_equal(values(bits16(y), dtype), values(bits16(want), dtype))


ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.parametrize("element", ["bf16", "fp16"])
@pytest.mark.parametrize("code", ["e4m3", "e5m2"])
def test_scaled_converts_are_the_software_codec(element, code):
    check = os.path.join(ROOT, "tests", "cxx", "bin", "mx_convert_check")
    if not os.path.exists(check):
        pytest.fail(f"{check} is missing: build it with `make -C tilexr_amd/csrc` (or __graft_entry__.build())")
    print(f"mx convert check {element} {code}", flush=True)
    run = subprocess.run([check, element, code], capture_output=True, text=True, timeout=100)
    last = run.stdout.strip().splitlines()[-1] if run.stdout.strip() else ""
    assert run.returncode == 0, run.stdout[-2000:] + run.stderr[-2000:]
    assert last.startswith(f"OK {element} {code}:"), last
