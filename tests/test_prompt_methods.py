"""The one-launch prompt write stands in for three per-entry methods: wherever a
program replaces one of them, its own runs."""

from __future__ import annotations

import pytest
import torch


def _classes():
    from headinfer.quest_offload_cache import QuestTopKOffloadedCache
    from headinfer.twilight_offload_cache import TwilightMatchedBudgetOffloadedCache

    return QuestTopKOffloadedCache, TwilightMatchedBudgetOffloadedCache


def test_replaced_prompt_methods_are_seen(monkeypatch):
    from headinfer.quest_offload_cache import _prompt_methods_replaced

    def replaced(cls, **own):
        cache = object.__new__(cls)
        vars(cache).update(own)
        return _prompt_methods_replaced(cache)

    quest, twilight = _classes()
    assert not replaced(quest) and not replaced(twilight)
    for base in (quest, twilight):
        assert not replaced(type("Plain", (base,), {"extra": 1}))
        assert not replaced(type("Mixed", (base, type("After", (), {"update": None})), {}))
        for name in ("update", "_build_metadata", "_write_prompt"):
            original = getattr(base, name)

            def own(self, *args, original=original):
                return original(self, *args)

            assert replaced(base, **{name: own})
            assert replaced(type("Own", (base,), {name: own}))
            assert replaced(type("Own", (type("Before", (), {name: own}), base), {}))
            with monkeypatch.context() as m:
                m.setattr(base, name, own)
                assert replaced(base) and replaced(twilight) and replaced(type("Sub", (base,), {}))
            assert not replaced(base) and not replaced(twilight)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", [0, 1])
@pytest.mark.parametrize("where", ["class", "base", "plain subclass"])
def test_prompt_through_replaced_methods(dev, monkeypatch, kind, where):
    from headinfer import mp

    base, S, G = _classes()[kind], 100, 2
    calls, fused = [], []
    target = _classes()[0] if where == "base" else base
    original = target.update

    def traced(self, key_states, value_states, layer_idx, cache_kwargs=None):
        calls.append(layer_idx)
        return original(self, key_states, value_states, layer_idx, cache_kwargs)

    if where == "plain subclass":
        base = type("Plain", (base,), {})
    else:
        monkeypatch.setattr(target, "update", traced)
    run = base.update_prompt_layer
    monkeypatch.setattr(base, "update_prompt_layer", lambda self, *args: fused.append(1) or run(self, *args))
    cache = base(num_cache_entries=G, max_cache_len=S, head_dim=128, num_query_heads_per_kv=2, dtype=torch.bfloat16,
                 device=dev, kv_residency="hbm")
    attn = torch.nn.Module()
    attn.head_dim, attn.scaling, attn._headinfer_entry0 = 128, 128 ** -0.5, 0
    for name, n in (("q_proj", 512), ("k_proj", 256), ("v_proj", 256), ("o_proj", 512)):
        setattr(attn, name, torch.nn.Linear(512, n, bias=False, device=dev, dtype=torch.bfloat16))
    cos, sin = (torch.randn((1, S, 128), device=dev).to(torch.bfloat16) for _ in range(2))
    hidden = torch.randn((1, S, 512), device=dev).to(torch.bfloat16)
    with torch.no_grad():
        mp._fast_forward(attn, hidden, position_embeddings=(cos, sin), past_key_values=cache)
    assert (calls, fused) == (([], [1]) if where == "plain subclass" else ([0, 1], []))
    assert cache.get_seq_length() == S
