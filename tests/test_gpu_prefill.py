"""The prompt attention kernel against float64, and its dispatch against the
general torch path.

Tolerance: the weights and the output are each rounded once to the 16-bit type
(unit roundoff 2 U: 2^-8 for bf16, 2^-11 for fp16, whose weights below 2^-14 round
by up to 2^-25 instead); a row's output is a convex combination of V rows, so
|error| <= (4 U + fp32 terms + 2^-25 S in fp16) max |v|.  The 3 U max |v| asserted
here is tighter than that bound: the weights' roundings differ in sign, and these
inputs keep to it."""

from __future__ import annotations

import math

import pytest
import torch

pytestmark = pytest.mark.gpu

U = {torch.bfloat16: 2.0 ** -9, torch.float16: 2.0 ** -12}  # half the unit roundoff


def _inputs(S, G, R, dtype, seed, scale=1.0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    # laid out as the projections give them: rows of all heads, viewed per head
    x = [torch.randn((1, S, h, 128), generator=g, device="cuda").to(dtype).transpose(1, 2) for h in (G * R, G, G)]
    return x[0] * scale, x[1], x[2]


def _reference(q, k, v, scale):
    _, Hq, S, D = q.shape
    R = Hq // k.shape[1]
    future = torch.ones((S, S), dtype=torch.bool, device=q.device).triu(1)
    out = torch.empty((S, Hq, D), dtype=torch.float64, device=q.device)
    for h in range(Hq):
        s = (q[0, h].double() @ k[0, h // R].double().T) * scale
        out[:, h] = torch.softmax(s.masked_fill(future, -math.inf), dim=-1) @ v[0, h // R].double()
    return out.view(1, S, Hq * D)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("S,G,R", [(1, 1, 1), (2, 8, 4), (31, 2, 3), (32, 1, 2), (33, 2, 2), (63, 1, 1), (64, 2, 2),
                                   (65, 1, 8), (127, 4, 7), (128, 1, 1), (129, 2, 2), (255, 1, 2), (513, 2, 4),
                                   (1500, 1, 2),
                                   # the wide kernel, from 512 blocks of 256 rows on: one key tile to several, every
                                   # parity of the last one, wavefronts that end before others
                                   (1, 128, 16), (256, 256, 8), (257, 128, 8), (31, 64, 8), (64, 128, 4), (65, 64, 8),
                                   (127, 64, 8), (129, 128, 4), (193, 64, 8), (320, 64, 8), (449, 64, 8), (577, 32, 8)])
def test_prefill_attention(S, G, R, dtype):
    from headinfer import kernels

    q, k, v = _inputs(S, G, R, dtype, seed=S, scale=3.0)  # peaked rows: the running maximum moves
    out = kernels.prefill_attention(q, k, v, 128 ** -0.5)
    ref = _reference(q, k, v, 128 ** -0.5)
    assert out.shape == (1, S, G * R * 128) and out.dtype == dtype
    assert float((out.double() - ref).abs().max()) <= 3 * U[dtype] * float(v.double().abs().max())


def test_prefill_attention_rising_scores_and_infinities():
    """Scores that grow with the key position move the maximum on every tile; an infinite key row takes the rows that
    see it to what torch's softmax gives."""
    from headinfer import kernels

    S = 400
    q, k, v = _inputs(S, 1, 1, torch.bfloat16, seed=1)
    ramp = torch.linspace(0.0, 4.0, S, device="cuda").to(torch.bfloat16)
    k = k + q[:, :, -1:] * ramp[None, None, :, None]
    q = q * 0 + q[:, :, -1:]
    out, ref = kernels.prefill_attention(q, k, v, 128 ** -0.5), _reference(q, k, v, 128 ** -0.5)
    assert float((out.double() - ref).abs().max()) <= 3 * U[torch.bfloat16] * float(v.double().abs().max())
    k = k.clone()
    k[:, :, 250] = math.inf
    out, ref = kernels.prefill_attention(q, k, v, 128 ** -0.5), _reference(q, k, v, 128 ** -0.5)
    assert torch.equal(out.isnan().any(dim=-1), ref.isnan().any(dim=-1))
    fine = ~ref.isnan()
    assert float((out.double() - ref)[fine].abs().max()) <= 3 * U[torch.bfloat16] * float(v.double().abs().max())


def test_wide_kernel_rising_scores_and_infinities():
    """The same of the wide kernel: the maximum moves on every tile, and an infinite key row among later finite ones."""
    from headinfer import kernels

    S, G, R = 600, 64, 4  # 768 blocks of 256 rows
    q, k, v = _inputs(S, 1, 1, torch.bfloat16, seed=6)
    ramp = torch.linspace(0.0, 4.0, S, device="cuda").to(torch.bfloat16)
    k = k + q[:, :, -1:] * ramp[None, None, :, None]
    q = q * 0 + q[:, :, -1:]
    for inf in (False, True):
        if inf:
            k[:, :, 250] = math.inf
        ref = _reference(q, k, v, 128 ** -0.5)
        out = kernels.prefill_attention(*(t.expand(-1, h, -1, -1).contiguous() for t, h in ((q, G * R), (k, G), (v, G))),
                                        128 ** -0.5).view(1, S, G * R, 128)
        assert torch.equal(out, out[:, :, :1].expand_as(out)) or inf
        out = out[:, :, 0]
        assert torch.equal(out.isnan().any(dim=-1), ref.isnan().any(dim=-1))
        fine = ~ref.isnan()
        assert float((out.double() - ref)[fine].abs().max()) <= 3 * U[torch.bfloat16] * float(v.double().abs().max())


def test_prefill_dispatch_matches_the_general_path():
    """Every operand form the dispatch accepts gives the general path's result; forms it does not take go there."""
    from headinfer import kernels, mp

    S, G, R, sc = 300, 2, 4, 128 ** -0.5
    q, k, v = _inputs(S, G, R, torch.bfloat16, seed=3)
    general = mp._prefill_attention(q.float(), k.float(), v.float(), sc)
    tol = 6 * U[torch.bfloat16] * float(v.float().abs().max())
    wide = torch.zeros((1, S, G * R + 2 * G, 136), dtype=torch.bfloat16, device="cuda")
    forms = [(q, k, v), tuple(t.contiguous() for t in (q, k, v))]
    parts, h = [], 0
    for t in (q, k, v):  # one fused projection output with padded heads
        n = t.shape[1]
        wide[0, :, h:h + n, :128] = t[0].transpose(0, 1)
        parts.append(wide[:, :, h:h + n, :128].transpose(1, 2))
        h += n
    forms.append(tuple(parts))
    for f in forms:
        assert kernels.prefill_attention_fits(*f, sc)
        assert float((mp._prefill_attention(*f, sc).float() - general).abs().max()) <= tol
    odd = torch.zeros((1, G, S, 129), dtype=torch.bfloat16, device="cuda")[..., :128]
    odd.copy_(k)
    for f in ((q, odd, v), (q.float(), k.float(), v.float()), (q, k.flip(3).flip(3)[..., ::1].half(), v)):
        assert not kernels.prefill_attention_fits(*f, sc)
    assert not kernels.prefill_attention_fits(q, k, v, 0.0)
    assert float((mp._prefill_attention(q, odd, v, sc).float() - general).abs().max()) <= tol


def test_prefill_attention_keeps_derivatives():
    """Backward and forward derivatives still go through the torch path."""
    from torch.autograd import forward_ad

    from headinfer import mp

    q, k, v = (t.contiguous() for t in _inputs(40, 1, 2, torch.bfloat16, seed=4))
    q.requires_grad_(True)
    mp._prefill_attention(q, k, v, 128 ** -0.5).float().sum().backward()
    assert q.grad is not None and bool(q.grad.isfinite().all())
    with torch.no_grad(), forward_ad.dual_level():
        dual = forward_ad.make_dual(v, torch.ones_like(v))
        assert forward_ad.unpack_dual(mp._prefill_attention(q.detach(), k, dual, 128 ** -0.5)).tangent is not None
