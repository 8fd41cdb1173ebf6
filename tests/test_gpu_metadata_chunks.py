"""The page-a-wavefront metadata build (16-row pages of 128 16-bit channels)
against the oracle, bit for bit: sizes around a page and a window, values that
stress the ordering (zeros of both signs, infinities, NaNs of both signs) and
the INT4 quotient (rows on a code grid, denormal and huge ranges, constant
rows), and operands the launch hands to the row routine (odd alignment)."""

from __future__ import annotations

import numpy as np
import pytest
import torch
from helpers import TORCH_DT, from_bits, same_bits, to_bits

import oracle

pytestmark = pytest.mark.gpu

D, BS = 128, 16


def _keys(T: int, dtype: str, seed: int) -> torch.Tensor:
    g = torch.Generator().manual_seed(seed)
    k = torch.randn((T, D), generator=g)
    grid = torch.randint(0, 31, (T, D), generator=g).float()
    for t in range(T):
        kind = t % 16
        if kind == 1:    # every value a multiple of half a code: quotients on and beside the ties
            k[t] = grid[t] * 0.5 * 2.0 ** int(torch.randint(-8, 8, (1,), generator=g))
        elif kind == 3:  # tiny ranges: denormal scales, or below the clamp
            k[t] *= 2.0 ** int(torch.randint(-24 if dtype == "f16" else -120, -10, (1,), generator=g))
        elif kind == 5:
            k[t] *= 1e4 if dtype == "f16" else 1e30
        elif kind == 7:
            k[t] = 0.5
    k = k.to(TORCH_DT[dtype])
    bits = k.view(torch.int16)
    inf = 0x7C00 if dtype == "f16" else 0x7F80
    for t, d, v in ((9, 1, inf + 1), (10, 2, inf - 0x8000 + 1), (11, 5, inf), (12, 7, inf - 0x8000), (13, 0, inf)):
        for base in range(0, T, 64):
            if base + t < T:
                bits[base + t, d] = v if v < 0x8000 else v - 0x10000
    for base in range(0, T, 48):
        k[base] = -0.0
        k[base, 3] = 0.0
    return k


def _check(keys: torch.Tensor, dtype: str, sink: int, pages: bool, quant: bool, entry_pad: int = 0, offset: int = 0):
    from headinfer import kernels

    dev = torch.device("cuda", 0)
    E, T, _ = keys.shape
    P = (T - sink) // BS if T > sink else 0
    flat = torch.zeros(E * (T * D + entry_pad) + offset, dtype=keys.dtype, device=dev)
    kd = flat[offset:].as_strided((E, T, D), (T * D + entry_pad, D, 1))
    kd.copy_(keys)
    pmin = torch.full((E, P + 1, D), 7.0, dtype=keys.dtype, device=dev)
    pmax = torch.full_like(pmin, 7.0)
    packed = torch.full((E, T + 3, D // 2), 0xAB, dtype=torch.uint8, device=dev)
    scale = torch.full((E, T + 3), 7.0, dtype=keys.dtype, device=dev)
    minimum = torch.full_like(scale, 7.0)
    kernels.build_page_metadata(kd, sink=sink, block_size=BS, page_min=pmin if pages else None,
                                page_max=pmax if pages else None, packed=packed if quant else None,
                                scale=scale if quant else None, minimum=minimum if quant else None)
    torch.cuda.synchronize()
    for e in range(E):
        omin, omax, opk, osc, omn = oracle.build_page_metadata(to_bits(keys[e]), dtype, sink, BS)
        if pages and P:
            assert same_bits(pmin[e, :P], from_bits(omin, dtype)) and same_bits(pmax[e, :P], from_bits(omax, dtype))
        assert bool((pmin[e, P if pages else 0:] == 7.0).all())
        if quant:
            assert np.array_equal(packed[e, :T].cpu().numpy(), opk)
            assert same_bits(scale[e, :T], from_bits(osc, dtype)) and same_bits(minimum[e, :T], from_bits(omn, dtype))
            assert bool((packed[e, T:] == 0xAB).all()) and bool((scale[e, T:] == 7.0).all())


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("T,sink", [(1, 64), (15, 0), (16, 0), (17, 0), (63, 64), (64, 64), (65, 64), (79, 64),
                                    (80, 64), (81, 64), (130, 17), (1000, 64), (1031, 33)])
def test_metadata_chunks(T, sink, dtype):
    keys = torch.stack([_keys(T, dtype, seed=T + e) for e in range(2)])
    for pages, quant in ((True, True), (True, False), (False, True)):
        _check(keys, dtype, sink, pages, quant)


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_metadata_chunks_alignment(dtype):
    """Entry strides and bases that are and are not whole 16-byte units."""
    keys = torch.stack([_keys(200, dtype, seed=e) for e in range(3)])
    for pad, offset in ((8, 0), (0, 8), (2, 0), (0, 2), (4, 4)):
        _check(keys, dtype, 64, True, True, entry_pad=pad, offset=offset)


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_metadata_chunks_every_scale(dtype):
    """Rows whose scale takes every mantissa of the type, each row holding 126 values between its ends: the quotient's
    rounding is the division's."""
    g = torch.Generator().manual_seed(5)
    mant = 1024 if dtype == "f16" else 128
    top = 15.0 * (1.0 + torch.arange(mant) / mant) * 2.0 ** torch.randint(-6, 6, (mant,), generator=g)
    keys = torch.rand((mant, D), generator=g) * top[:, None]
    keys[:, 0], keys[:, 1] = 0.0, top
    _check(keys.to(TORCH_DT[dtype])[None], dtype, 64, True, True)
