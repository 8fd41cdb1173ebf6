"""update_prompt_layer refuses what the per-entry update refuses before it
touches the cache: lengths, order, metadata and slab stay as they were, and the
prompt can still be given afterwards."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

D, S, G = 128, 100, 2


def _cache(kind, residency, dev, **more):
    from headinfer.quest_offload_cache import QuestTopKOffloadedCache
    from headinfer.twilight_offload_cache import TwilightMatchedBudgetOffloadedCache

    cls = QuestTopKOffloadedCache if kind == "quest" else TwilightMatchedBudgetOffloadedCache
    kw = dict(num_cache_entries=2 * G, max_cache_len=S + 20, head_dim=D, num_query_heads_per_kv=2,
              dtype=torch.bfloat16, device=dev, kv_residency=residency)
    return cls(**{**kw, **more})


def _operands(dev, S=S, G=G, dtype=torch.bfloat16, D=D):
    k, v = (torch.randn((1, G, S, D), device=dev).to(dtype) for _ in range(2))
    cos, sin = (torch.randn((1, S, D), device=dev).to(dtype) for _ in range(2))
    return [k, v, cos, sin]


def _state(cache):
    return (list(cache._logical_lengths), cache._bookkeeping.expected_next_entry, cache._bookkeeping.write_position,
            cache._seen_tokens, cache._prompt_length, list(cache._initialized), cache.get_seq_length(),
            cache._page_min is None)


@pytest.mark.parametrize("kind", ["quest", "twilight"])
@pytest.mark.parametrize("residency", ["hbm", "host"])
def test_refused_prompt_leaves_the_cache_as_it_was(dev, kind, residency):
    cache = _cache(kind, residency, dev)
    fine = _operands(dev)
    fresh = _state(cache)
    k, v, cos, sin = fine
    off = torch.zeros((1, S, D + 4), dtype=k.dtype, device=dev)[..., 4:]
    for operands in (_operands(dev, dtype=torch.float16), _operands(dev, D=64), [k, v[:, :, :-1], cos, sin],
                     [k, v, cos[:, :-1], sin], [k, v, cos, sin.float()], [k, v, off, sin], [k, v.cpu(), cos, sin],
                     [k[0], v[0], cos, sin]):
        with pytest.raises(ValueError):
            cache.update_prompt_layer(0, *operands)
        assert _state(cache) == fresh
    with pytest.raises(ValueError, match="strict"):
        cache.update_prompt_layer(1, *fine)
    with pytest.raises(ValueError, match="strict"):  # the last head past the cache's entries
        cache.update_prompt_layer(0, *_operands(dev, G=2 * G + 1))
    with pytest.raises(RuntimeError, match="capacity"):
        cache.update_prompt_layer(0, *_operands(dev, S=S + 21))
    assert _state(cache) == fresh
    cache.update_prompt_layer(0, *fine)
    one = _state(cache)
    with pytest.raises(RuntimeError, match="unequal"):
        cache.update_prompt_layer(G, *_operands(dev, S=S - 1))
    assert _state(cache) == one
    cache.update_prompt_layer(G, *fine)
    both = _state(cache)
    assert both[0] == [S] * (2 * G) and both[1] == 0 and both[3] == both[4] == S
    with pytest.raises(ValueError, match="chunked"):
        cache.update_prompt_layer(0, *_operands(dev, S=10))
    assert _state(cache) == both
    torch.cuda.synchronize()
    assert torch.equal(cache._value_cache[:G, :S].cpu(), v[0].cpu())
    assert torch.equal(cache._key_cache[:G, :S], cache._key_cache[G:, :S])


@pytest.mark.parametrize("residency", ["hbm", "host"])
def test_refused_page_size(dev, residency):
    cache = _cache("quest", residency, dev, block_size=32)
    fresh = _state(cache)
    with pytest.raises(ValueError):
        cache.update_prompt_layer(0, *_operands(dev))
    assert _state(cache) == fresh
