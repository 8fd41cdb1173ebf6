"""The prompt's cache write in one launch (K rotation, K/V rows, page min/max,
INT4 keys) and the attention that rotates q itself, against the general path:
the eager rotation, a copy and the metadata build.  Every value is a copy or a
16-bit rounding of the same expression, so the results are the same bits."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

D = 128


def _rotate(x, cos, sin):
    half = torch.cat((-x[..., D // 2:], x[..., :D // 2]), dim=-1)
    return x * cos[:, None] + half * sin[:, None]


def _tables(S, dtype, device, seed=9):
    g = torch.Generator(device=device).manual_seed(seed)
    # all four halves differ: nothing relies on cos[d] == cos[d + 64]
    return [torch.randn((1, S, D), generator=g, device=device).to(dtype) for _ in range(2)]


def _kv(G, S, dtype, device, layout, scale, seed=3):
    g = torch.Generator(device=device).manual_seed(seed + S)
    out = []
    for _ in range(2):
        x = torch.randn((1, S, G, D), generator=g, device=device) * scale
        x = x.to(dtype).transpose(1, 2)
        if layout == "heads":
            x = x.contiguous()
        elif layout == "padded":
            wide = torch.zeros((1, S, G + 1, D + 8), dtype=dtype, device=device)[:, :, 1:, :D].transpose(1, 2)
            x = wide.copy_(x)
        out.append(x)
    return out


def _bits(t):
    return t.contiguous().view(torch.int16 if t.element_size() == 2 else torch.uint8)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("T,sink,G,layout,scale", [
    (1, 64, 1, "rows", 1.0), (2, 0, 3, "heads", 1.0), (15, 0, 2, "rows", 1.0), (16, 0, 2, "padded", 1.0),
    (17, 0, 1, "rows", 1.0), (63, 64, 2, "heads", 1.0), (64, 64, 2, "rows", 1.0), (65, 64, 2, "rows", 1.0),
    (79, 64, 8, "padded", 1.0), (80, 64, 8, "rows", 1.0), (81, 70, 4, "heads", 1.0), (1000, 64, 8, "rows", 1.0),
    (777, 5, 3, "rows", 1e-6), (333, 64, 2, "rows", 3e4)])
def test_prompt_kv_is_the_general_path(dev, dtype, T, sink, G, layout, scale):
    from headinfer import kernels

    if dtype == torch.bfloat16:  # subnormal products, and sums past the range
        scale = {1e-6: 1e-39, 3e4: 2e38}.get(scale, scale)
    k, v = _kv(G, T, dtype, dev, layout, scale)
    cos, sin = _tables(T, dtype, dev)
    P = (T - sink) // 16 if T > sink else 0
    rows = T + 7

    def buffers():
        return dict(k=torch.zeros((G, rows, D), dtype=dtype, device=dev), v=torch.zeros((G, rows, D), dtype=dtype, device=dev),
                    page_min=torch.zeros((G, P + 1, D), dtype=dtype, device=dev),
                    page_max=torch.zeros((G, P + 1, D), dtype=dtype, device=dev),
                    packed=torch.zeros((G, rows, D // 2), dtype=torch.uint8, device=dev),
                    scale=torch.zeros((G, rows), dtype=dtype, device=dev),
                    minimum=torch.zeros((G, rows), dtype=dtype, device=dev))

    for int4 in (True, False):
        names = ("page_min", "page_max") + (("packed", "scale", "minimum") if int4 else ())
        want, got = buffers(), buffers()
        want["k"][:, :T], want["v"][:, :T] = _rotate(k, cos, sin)[0], v[0]
        if P or int4:
            kernels.build_page_metadata(want["k"][:, :T], sink=sink, block_size=16, **{n: want[n] for n in names})
        kernels.prompt_kv(k, v, cos, sin, got["k"], got["v"], sink=sink, block_size=16, **{n: got[n] for n in names})
        nan = want["k"].isnan()
        assert torch.equal(nan, got["k"].isnan())
        for n in want:
            a, b = want[n], got[n]
            if n == "k":
                a, b = a.masked_fill(nan, 0), b.masked_fill(nan, 0)
            assert torch.equal(_bits(a), _bits(b)), (n, int4)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("S,G,R", [(1, 1, 1), (33, 2, 3), (130, 1, 8), (700, 2, 4), (257, 128, 8)])
def test_attention_rotates_q(dev, dtype, S, G, R):
    from headinfer import kernels

    g = torch.Generator(device=dev).manual_seed(S)
    q, k, v = (torch.randn((1, S, h, D), generator=g, device=dev).to(dtype).transpose(1, 2) for h in (G * R, G, G))
    cos, sin = _tables(S, dtype, dev)
    want = kernels.prefill_attention(_rotate(q, cos, sin), k, v, D ** -0.5)
    got = kernels.prefill_attention(q, k, v, D ** -0.5, rope=(cos, sin))
    assert torch.equal(_bits(want), _bits(got))


class _Cfg:
    num_key_value_heads, num_attention_heads, hidden_size = 2, 6, 768


def _layer(dtype, dev, seed=5):
    from headinfer.mp import mp_headinfer

    class LlamaOneLayer(torch.nn.Module):
        def __init__(self):
            super().__init__()
            self.config = _Cfg()
            self.model = torch.nn.Module()
            attn = torch.nn.Module()
            attn.config, attn.head_dim, attn.scaling = self.config, D, D ** -0.5
            for name, n in (("q_proj", 768), ("k_proj", 256), ("v_proj", 256), ("o_proj", 768)):
                setattr(attn, name, torch.nn.Linear(768, n, bias=False, device=dev, dtype=dtype))
            layer = torch.nn.Module()
            layer.self_attn = attn
            self.model.layers = torch.nn.ModuleList([layer])

    torch.manual_seed(seed)
    return mp_headinfer(LlamaOneLayer().eval()).model.layers[0].self_attn


def _cache(kind, residency, dtype, dev, S, own=True, **more):
    from headinfer.quest_offload_cache import QuestTopKOffloadedCache
    from headinfer.twilight_offload_cache import TwilightMatchedBudgetOffloadedCache

    base = QuestTopKOffloadedCache if kind == "quest" else TwilightMatchedBudgetOffloadedCache
    calls = []

    class Traced(base):  # a subclass of a program's own: its per-entry update is the one that runs
        def update(self, key_states, value_states, layer_idx, cache_kwargs=None):
            calls.append(layer_idx)
            return super().update(key_states, value_states, layer_idx, cache_kwargs)

    twilight = dict(candidate_token_budget=256, budget_mode="dynamic") if kind == "twilight" else {}
    cache = (base if own else Traced)(num_cache_entries=2, max_cache_len=S + 40, head_dim=D, num_query_heads_per_kv=3,
                                      dtype=dtype, device=dev, kv_residency=residency, **twilight, **more)
    return cache, calls


@pytest.mark.parametrize("kind", ["quest", "twilight"])
@pytest.mark.parametrize("residency", ["hbm", "host"])
@pytest.mark.parametrize("S,more", [(2, {}), (50, {}), (451, {}), (600, dict(update_metadata_on_decode=True)),
                                    (600, dict(block_size=32))])
def test_prompt_layer_is_the_per_entry_path(dev, kind, residency, S, more):
    if kind == "twilight" and more.get("block_size", 16) != 16:
        more = {}
    dtype = torch.bfloat16
    attn = _layer(dtype, dev)
    g = torch.Generator(device=dev).manual_seed(S)
    hidden = torch.randn((1, S, 768), generator=g, device=dev).to(dtype)
    cos, sin = _tables(S, dtype, dev)
    got, want = _cache(kind, residency, dtype, dev, S, **more), _cache(kind, residency, dtype, dev, S, own=False, **more)
    with torch.no_grad():
        outs = [attn(hidden, position_embeddings=(cos, sin), past_key_values=c[0])[0] for c in (got, want)]
        assert want[1] == [0, 1]
        torch.cuda.synchronize()
        assert torch.equal(_bits(outs[0]), _bits(outs[1]))
        a, b = got[0], want[0]
        assert torch.equal(_bits(a._key_cache[:, :S]), _bits(b._key_cache[:, :S]))
        assert torch.equal(_bits(a._value_cache[:, :S]), _bits(b._value_cache[:, :S]))
        P = max(0, (S - 64) // more.get("block_size", 16))
        for n in ("_page_min", "_page_max"):
            assert getattr(a, n).shape == getattr(b, n).shape
            assert torch.equal(_bits(getattr(a, n)[:, :P]), _bits(getattr(b, n)[:, :P]))
        if kind == "twilight":
            for n in ("_packed", "_qscale", "_qmin"):
                assert torch.equal(_bits(getattr(a, n)[:, :S]), _bits(getattr(b, n)[:, :S]))
        assert a._logical_lengths == b._logical_lengths and a.get_seq_length() == b.get_seq_length() == S
        # a second prompt and a prompt past the capacity are refused as before
        for c in (a, b):
            with pytest.raises(ValueError, match="chunked"):
                attn(hidden[:, :30], position_embeddings=(cos[:, :30], sin[:, :30]), past_key_values=c)
        for own in (True, False):
            c, _ = _cache(kind, residency, dtype, dev, S - 41 if S > 41 else 1, own=own)
            if S > 41:
                with pytest.raises(RuntimeError, match="capacity"):
                    attn(hidden, position_embeddings=(cos, sin), past_key_values=c)


def test_prompt_forms_that_take_the_general_path(dev):
    """A wanted derivative, and tables off the 16-byte grid."""
    from headinfer import mp

    S, dtype = 100, torch.bfloat16
    attn = _layer(dtype, dev)
    hidden = torch.randn((1, S, 768), device=dev).to(dtype)
    cos, sin = _tables(S, dtype, dev)
    cache, _ = _cache("quest", "hbm", dtype, dev, S)
    q, k, v = (torch.randn((1, h, S, D), device=dev).to(dtype) for h in (6, 2, 2))
    assert mp._fused_prompt(cache, q, k, v, cos, sin, D ** -0.5)
    odd = torch.zeros((1, S, D + 4), dtype=dtype, device=dev)[..., 4:].copy_(cos)
    assert not mp._fused_prompt(cache, q, k, v, odd, sin, D ** -0.5)
    assert not mp._fused_prompt(cache, q, k, v, cos.float(), sin.float(), D ** -0.5)
    assert not mp._fused_prompt(cache, q.requires_grad_(True), k, v, cos, sin, D ** -0.5)
    cache.update = type(cache).update.__get__(cache)  # an instance's own update
    assert not mp._fused_prompt(cache, q.detach(), k, v, cos, sin, D ** -0.5)
    fresh, _ = _cache("quest", "hbm", dtype, dev, S)
    fused, _ = _cache("quest", "hbm", dtype, dev, S)
    with torch.no_grad():
        a = attn(hidden, position_embeddings=(odd, sin), past_key_values=fresh)[0]
        b = attn(hidden, position_embeddings=(cos, sin), past_key_values=fused)[0]
    assert torch.equal(_bits(a), _bits(b))
