"""The prompt attention at the ends of its operands' range, both kernels and
both types: rows whose first keys weigh nothing, scores of any finite size,
scales down to the smallest float, values up to the largest bfloat16, long rows
and row strides past the wide kernel's offsets.

Limit: a row is a convex combination of V rows and its weights and output are
each rounded once to the 16-bit type, whose unit roundoff is u = 2^-8 (bf16) or
2^-11 (fp16): |error| <= 2 u max |v|, and 2^-12 max |v| for the fp32 terms and
fp16's weights below 2^-14 (at most 2^-25 each, 600 rows)."""

from __future__ import annotations

import math

import pytest
import torch

pytestmark = pytest.mark.gpu

U = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}
# one head: blocks of 128 rows; 512 heads of one: 512 and more blocks of 256 rows, the wide kernel
KERNELS = pytest.mark.parametrize("heads", [1, 512], ids=["narrow", "wide"])
DTYPES = pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
SCALE = 128 ** -0.5


def _randn(shape, dtype, seed):
    return torch.randn(shape, generator=torch.Generator(device="cuda").manual_seed(seed), device="cuda").to(dtype)


def _reference(q, k, v, scale):
    """Float64, q/k/v [S, 128] of one head."""
    S = q.shape[0]
    s = (q.double() @ k.double().T) * scale
    future = torch.ones((S, S), dtype=torch.bool, device=q.device).triu(1)
    return torch.softmax(s.masked_fill(future, -math.inf), dim=-1) @ v.double()


def _attention(q, k, v, scale, heads):
    """[S, 128] of one head, computed `heads` times over one KV head: every copy gives the same bits."""
    from headinfer import kernels

    S = q.shape[0]
    out = kernels.prefill_attention(q[None, None].expand(1, heads, -1, -1), k[None, None], v[None, None], scale)
    out = out.view(S, heads, 128)
    assert torch.equal(out.view(torch.int16), out[:, :1].expand_as(out).contiguous().view(torch.int16))
    return out[:, 0]


def _close(out, ref, v, dtype):
    assert torch.equal(out.isnan(), ref.isnan())
    limit = (2 * U[dtype] + 2.0 ** -12) * float(v.double().abs().max())
    assert float((out.double() - ref).nan_to_num().abs().max()) <= limit


@KERNELS
@DTYPES
@pytest.mark.parametrize("S,n", [(200, 63), (200, 64), (300, 128), (300, 130), (450, 257)])
def test_leading_keys_of_minus_infinity(S, n, dtype, heads):
    """The first n keys score -inf in every row: rows that see another key are finite, the others 0 / 0."""
    q, k, v = (_randn((S, 128), dtype, seed=i) for i in range(3))
    q[:, 0] = 1.0
    k[:n, 0] = -math.inf
    ref = _reference(q, k, v, SCALE)
    assert bool(ref[:n].isnan().all()) and bool(ref[n:].isfinite().all())
    _close(_attention(q, k, v, SCALE, heads), ref, v, dtype)


@KERNELS
def test_leading_keys_past_the_float_range(heads):
    """bfloat16 products below -3.4e38 in every second row, finite scores in the others of the wavefront."""
    S, n = 300, 130
    q, k, v = (_randn((S, 128), torch.bfloat16, seed=i) for i in range(3))
    q[:, 0] = 0.0
    q[::2, 0] = 3e38
    k[:, 0] = 0.0
    k[:n, 0] = -3e38
    out, ref = _attention(q, k, v, SCALE, heads), _reference(q, k, v, SCALE)
    keep = torch.arange(S, device="cuda") % 2 == 1
    keep[n:] = True
    _close(out[keep], ref[keep], v, torch.bfloat16)


@KERNELS
@DTYPES
@pytest.mark.parametrize("size", [1.0, 100.0, 1000.0, 6000.0, 20000.0, 60000.0])
@pytest.mark.parametrize("sign", [1.0, -1.0])
def test_large_scores(size, sign, dtype, heads):
    """Equal scores of up to 5e10 average their rows; scores that differ by more than the range of the exponential
    pick one row, wherever in the prompt it is."""
    S = 300
    v = _randn((S, 128), dtype, seed=1)
    q = torch.full((S, 128), size, device="cuda").to(dtype)
    k = sign * q
    _close(_attention(q, k, v, SCALE, heads), _reference(q, k, v, SCALE), v, dtype)
    if size < 1000.0:
        return
    # eight key sizes a factor 2^-1 .. 2^-8 apart, in no order
    k = k * torch.exp2(-1.0 - torch.randint(0, 8, (S, 1), generator=torch.Generator(device="cuda").manual_seed(2),
                                            device="cuda")).to(dtype)
    _close(_attention(q, k, v, SCALE, heads), _reference(q, k, v, SCALE), v, dtype)


@KERNELS
@DTYPES
@pytest.mark.parametrize("scale", [1e-20, 2.4e-38, 1e-39, 2.0 ** -149])
def test_tiny_scales(scale, dtype, heads):
    """Down to the smallest positive float a row is the plain average of what it sees."""
    q, k, v = (_randn((300, 128), dtype, seed=i) for i in range(3))
    _close(_attention(q, k, v, scale, heads), _reference(q, k, v, scale), v, dtype)


@pytest.mark.parametrize("scale", [2.0 ** -150, 1e-50, 3e38, 1e39])
def test_scales_outside_the_float_range(scale):
    """A scale that is not a float, or whose product with log2 e is not, goes to the torch path as a type that the
    kernels do not take does."""
    from headinfer import kernels, mp

    q, k, v = (_randn((1, 1, 80, 128), torch.bfloat16, seed=i) for i in range(3))
    assert not kernels.prefill_attention_fits(q, k, v, scale)
    out = mp._prefill_attention(q * 1e-15, k * 1e-15, v, scale)
    odd = torch.zeros((1, 1, 80, 129), dtype=torch.bfloat16, device="cuda")[..., :128].copy_(k * 1e-15)
    want = mp._prefill_attention(q * 1e-15, odd, v, scale)
    assert torch.equal(out.isnan(), want.isnan()) and torch.equal(out.nan_to_num(), want.nan_to_num())


@KERNELS
@pytest.mark.parametrize("size", [1e30, 1e36, 1e38])
@pytest.mark.parametrize("spread", [0.0, 1.0, 8.0])
def test_large_values(size, spread, heads):
    """V near the top of bfloat16's range: the weights' sum before the division may exceed 1 by the prompt's length."""
    S = 600
    q, k, v = (_randn((S, 128), torch.bfloat16, seed=i) for i in range(3))
    v = (v.float().clamp(-3, 3) * size).to(torch.bfloat16)
    out, ref = _attention(q * spread, k, v, SCALE, heads), _reference(q * spread, k, v, SCALE)
    _close(out, ref, v, torch.bfloat16)


@KERNELS
def test_large_values_beside_ordinary_ones(heads):
    """A row that sees no large value keeps its precision beside rows that do; infinities and NaN stay where they are."""
    S = 400
    q, k, v = (_randn((S, 128), torch.bfloat16, seed=i) for i in range(3))
    small = _reference(q, k, v, SCALE)
    v[200:300] = 3e38
    ref = _reference(q, k, v, SCALE)
    top = v.clone()
    v[300, 5] = math.inf
    v[301, 6] = math.nan
    out = _attention(q, k, v, SCALE, heads)
    # (rows 256 .. 300 share a tile of keys with the infinity: 0 times it is a NaN, as in torch's products)
    _close(out[:192], small[:192], v[:200], torch.bfloat16)
    _close(out[192:256], ref[192:256], top, torch.bfloat16)
    assert bool(out[301:, 5].isinf().all()) and bool(out[301:, 6].isnan().all())
    _close(out[301:, 7:], ref[301:, 7:], top, torch.bfloat16)


@KERNELS
@DTYPES
def test_row_strides_on_both_sides_of_the_wide_offsets(dtype, heads):
    """K/V rows up to 2^24 elements apart go to the wide kernel, rows further apart to the other: the same row by row."""
    from headinfer import kernels

    S, far = 20, 1 << 24
    q, k, v = (_randn((S, 128), dtype, seed=i) for i in range(3))
    ref = _reference(q, k, v, SCALE)
    flat = torch.empty((S - 1) * (far + 8) + 256, dtype=dtype, device="cuda")
    for stride in (far, far + 8):
        both = flat.as_strided((2, S, 128), (128, stride, 1))
        both[0], both[1] = k, v
        for kk, vv in ((both[0], v), (k, both[1]), (both[0], both[1])):
            assert kernels.prefill_attention_fits(q[None, None], kk[None, None], vv[None, None], SCALE)
            _close(_attention(q, kk, vv, SCALE, heads), ref, v, dtype)


@DTYPES
@pytest.mark.parametrize("heads", [1, 8], ids=["narrow", "wide"])  # 157 blocks of 128 rows, 632 of 256
@pytest.mark.parametrize("spread", [0.1, 3.0])
def test_long_rows(spread, dtype, heads):
    """20000 rows: the sums are chains of at most S / 2 fp32 additions, 2^-24 each, 2^-10 max |v| in all; fp16 weights
    below 2^-14 add S 2^-25."""
    S = 20000
    q, k, v = (_randn((S, 128), dtype, seed=i) for i in range(3))
    q, v = q * spread, v + 1.0
    out = _attention(q, k, v, SCALE, heads)
    rows = torch.cat([torch.arange(0, S, 997, device="cuda"), torch.arange(S - 40, S, device="cuda")])
    s = (q[rows].double() @ k.double().T) * SCALE
    s.masked_fill_(torch.arange(S, device="cuda")[None] > rows[:, None], -math.inf)
    ref = torch.softmax(s, dim=-1) @ v.double()
    limit = (2 * U[dtype] + 2.0 ** -10 + (S * 2.0 ** -25 if dtype == torch.float16 else 0.0)) * float(v.abs().max())
    assert float((out[rows].double() - ref).abs().max()) <= limit
    # 2-norm: two independent roundings, each uniform within +- u / m of the value for a mantissa m in [1, 2), an rms
    # of u / sqrt(6)
    assert float((out[rows].double() - ref).norm() / ref.norm()) <= 0.6 * U[dtype]
