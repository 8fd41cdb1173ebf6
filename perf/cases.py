"""What the framework's speed is measured on: the sparse-decode KV path and the prompt path that feeds it.

Every case is one pass of work that a serving program does through the public entry points:

* ``quest``     one decode step of a few layers: Quest page selection, sparse GQA attention over the selected pages with
                the decode token appended (KV in HBM, or in pinned host memory read over the host link);
* ``ragged``    the same step for several requests of different lengths at once, with the page metadata kept current;
* ``twilight``  one decode step of a few layers: Quest B0, INT4 QK, top-p (dynamic or matched budgets), union attention;
* ``gqa_rows``  one layer through the row-list form of Twilight (selection, K/V gather, varlen attention), called eagerly
                with the union's lengths read back, as the GQA-group branch of the model patch does;
* ``metadata``  the page min/max and INT4 keys of a prompt, every KV head of a layer at once;
* ``prefill``   one patched attention layer over a whole prompt: projections, RoPE, cache fill, causal attention;
* ``token``     one decode token through whole decoder layers and the LM head (the fused decode-step projections).

Decode steps are captured once and replayed, as a serving loop keeps them.  Sizes are those of the benchmark's workloads
(Llama-3-8B-shaped: 8 KV heads of 4 query heads; Qwen2.5-7B-like: 4 KV heads of 7; head_dim 128, 16-row pages, sink 64,
recent 256).  All values are synthetic and made from the seed.
"""

from __future__ import annotations

import math
import sys
from pathlib import Path

import torch

ROOT = Path(__file__).resolve().parent.parent
for _p in (str(ROOT), str(ROOT / "twilight-cpu-gpu-offloading_amd")):
    if _p not in sys.path:
        sys.path.insert(0, _p)

D, SINK, RECENT, BS = 128, 64, 256, 16
DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16}


# ------------------------------------------------------------------ the cases
def listed() -> list[dict]:
    return [
        # a short chat context: every launch is latency
        dict(name="quest-4k", kind="quest", context=4096, layers=8, kv_heads=8, q_per_kv=4, pages=16, dtype="f16",
             residency="hbm"),
        # the benchmark's headline layer
        dict(name="quest-32k", kind="quest", context=32768, layers=8, kv_heads=8, q_per_kv=4, pages=128, dtype="f16",
             residency="hbm"),
        # the offloaded cache: K/V in pinned host memory, selected pages read over the host link
        dict(name="quest-64k-host", kind="quest", context=65536, layers=2, kv_heads=8, q_per_kv=4, pages=128,
             dtype="f16", residency="host"),
        # eight requests of 16K to 128K decoded in the same launches
        dict(name="ragged-8-requests", kind="ragged", requests=8, shortest=16384, longest=131072, layers=2, kv_heads=4,
             q_per_kv=7, pages=128, dtype="bf16"),
        # the Twilight layer with the reference's two budget modes
        dict(name="twilight-32k-dynamic", kind="twilight", context=32768, layers=8, kv_heads=8, q_per_kv=4,
             candidates=4096, top_p=0.95, mode="dynamic", dtype="bf16"),
        dict(name="twilight-32k-matched", kind="twilight", context=32768, layers=8, kv_heads=8, q_per_kv=4,
             candidates=4096, top_p=0.95, mode="matched", dtype="bf16"),
        # the GQA-group branch of the patched model, eager, one layer
        dict(name="gqa-rows-32k", kind="gqa_rows", context=32768, kv_heads=8, q_per_kv=4, candidates=4096, top_p=0.95,
             dtype="bf16"),
        # the end of a prompt: page min/max and INT4 keys of one layer
        dict(name="metadata-32k", kind="metadata", tokens=32768, kv_heads=8, int4=True, dtype="bf16"),
        # a prompt through one attention layer: a short question, and a long document
        dict(name="prefill-2k", kind="prefill", tokens=2048, kv_heads=8, q_per_kv=4, cache="quest", dtype="bf16"),
        dict(name="prefill-32k", kind="prefill", tokens=32768, kv_heads=8, q_per_kv=4, cache="twilight",
             dtype="bf16"),
        # one generated token through whole layers and the LM head
        dict(name="token-32k", kind="token", context=32768, layers=2, kv_heads=8, q_per_kv=4, hidden=4096,
             intermediate=14336, vocab=128256, pages=128, bias=False, dtype="bf16"),
    ]


def _log(rng, lo: int, hi: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng) -> dict:
    kind = rng.choice(["quest", "quest", "ragged", "twilight", "twilight", "gqa_rows", "metadata", "prefill",
                       "prefill", "token"])
    kv_heads, q_per_kv = rng.choice([(8, 4), (8, 4), (4, 7), (8, 8), (2, 6)])
    dtype = rng.choice(["f16", "bf16"])
    if kind == "quest":
        residency = rng.choice(["hbm", "hbm", "hbm", "host"])
        context = _log(rng, 2048, 65536 if residency == "host" else 131072)
        return dict(kind=kind, context=context, layers=2 if residency == "host" or context > 65536 else 8,
                    kv_heads=kv_heads, q_per_kv=q_per_kv, pages=min(_log(rng, 16, 256), (context - 320) // BS // 2),
                    dtype=dtype, residency=residency)
    if kind == "ragged":
        shortest = _log(rng, 2048, 32768)
        return dict(kind=kind, requests=rng.randint(2, 8), shortest=shortest, longest=_log(rng, shortest, 131072),
                    layers=2, kv_heads=4, q_per_kv=rng.choice([4, 7]), pages=_log(rng, 32, 128), dtype=dtype)
    if kind == "twilight":
        context = _log(rng, 4096, 131072)
        return dict(kind=kind, context=context, layers=2 if context > 65536 else 8, kv_heads=kv_heads,
                    q_per_kv=q_per_kv, candidates=min(rng.choice([2048, 4096, 8192]), (context - 320) // 32 * BS),
                    top_p=round(rng.uniform(0.85, 0.98), 3), mode=rng.choice(["dynamic", "matched"]), dtype=dtype)
    if kind == "gqa_rows":
        context = _log(rng, 4096, 65536)
        return dict(kind=kind, context=context, kv_heads=kv_heads, q_per_kv=q_per_kv,
                    candidates=min(rng.choice([2048, 4096]), (context - 320) // 32 * BS),
                    top_p=round(rng.uniform(0.85, 0.98), 3), dtype=dtype)
    if kind == "metadata":
        return dict(kind=kind, tokens=_log(rng, 512, 131072), kv_heads=kv_heads, int4=rng.random() < 0.7, dtype=dtype)
    if kind == "prefill":
        return dict(kind=kind, tokens=_log(rng, 256, 24576), kv_heads=kv_heads,
                    q_per_kv=q_per_kv if kv_heads * q_per_kv <= 32 else 4, cache=rng.choice(["quest", "twilight"]),
                    dtype=dtype)
    wide = rng.random() < 0.5
    return dict(kind="token", context=_log(rng, 4096, 65536), layers=2, kv_heads=8 if wide else 4,
                q_per_kv=4 if wide else 7, hidden=4096 if wide else 3584, intermediate=14336 if wide else 18944,
                vocab=128256 if wide else 152064, pages=_log(rng, 32, 128), bias=not wide, dtype=dtype)


# ------------------------------------------------------------------ geometry
def _window(length: int) -> tuple[int, int]:
    sink_end = min(SINK, length)
    return sink_end, max(sink_end, length - (RECENT - 1))


def _pages(length: int) -> tuple[int, int]:
    """(scored pages, complete pages) of a history of `length` tokens."""
    sink_end, recent_start = _window(length)
    complete = max(0, length - SINK) // BS
    return min((recent_start - sink_end) // BS, complete), complete


def _request_lengths(case: dict) -> list[int]:
    n = case["requests"]
    ratio = case["longest"] / case["shortest"]
    return [int(case["shortest"] * ratio ** (i / max(1, n - 1))) for i in range(n)]


def _matched_pages(length: int) -> int:
    """The default matched budget: 5% of the eligible pages, per query head."""
    sink_end, recent_start = _window(length)
    return min((recent_start - sink_end) // BS, max(1, math.ceil(0.05 * (recent_start - sink_end) / BS)))


# ------------------------------------------------------------------ inputs (torch only)
def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device="cuda").manual_seed(seed)


def _randn(gen, *shape, dtype=torch.float32):
    return torch.randn(shape, generator=gen, device="cuda", dtype=dtype)


def _keys(gen, q: torch.Tensor, rows: int, pages: int, relevance: str, dtype) -> torch.Tensor:
    """Keys [G, rows, D] with the structure real heads show: a few pages that answer the query (planted), or a Zipf
    relevance over all pages; the planted form also has a few outlier channels."""
    G = q.shape[0]
    k = _randn(gen, G, rows, D)
    u = q.float().mean(dim=1)
    u = u / u.norm(dim=-1, keepdim=True)
    if relevance == "planted":
        n = min(16, pages)
        at = torch.rand((G, pages), generator=gen, device="cuda").argsort(dim=1)[:, :n]
        idx = (SINK + at[:, :, None] * BS + torch.arange(BS, device="cuda")).reshape(G, -1)
        noise = 0.1 * _randn(gen, G, idx.shape[1], D)
        k.scatter_(1, idx[:, :, None].expand(-1, -1, D), 3.0 * u[:, None] + noise)
        k[:, :, torch.randperm(D, generator=gen, device="cuda")[:4]] *= 8.0
    else:
        rank = torch.rand((G, pages), generator=gen, device="cuda").argsort(dim=1).float() + 1.0
        w = (4.0 * rank ** -1.1).repeat_interleave(BS, dim=1)
        k[:, SINK:SINK + pages * BS] += w[:, :, None] * u[:, None]
    return k.to(dtype)


def _decode_inputs(case: dict, seed: int, lengths: list[int], relevance: str) -> dict:
    """q [layers, G, R, D], K/V [layers, G, Lmax, D] and the decode tokens [layers, G, D]; group g has lengths[g]
    tokens of history, and one spare row."""
    gen, dt = _gen(seed), DTYPES[case["dtype"]]
    G, R, n = len(lengths), case["q_per_kv"], case.get("layers", 1)
    Lmax = max(lengths) + 1
    q = _randn(gen, n, G, R, D).to(dt)
    k = torch.empty((n, G, Lmax, D), dtype=dt, device="cuda")
    v = torch.empty_like(k)
    for i in range(n):
        if len(set(lengths)) == 1:
            k[i] = _keys(gen, q[i], Lmax, _pages(lengths[0])[0], relevance, dt)
        else:
            for g, L in enumerate(lengths):
                k[i, g, :L + 1] = _keys(gen, q[i, g:g + 1], L + 1, _pages(L)[0], relevance, dt)[0]
                k[i, g, L + 1:] = 0
        v[i] = _randn(gen, G, Lmax, D, dtype=dt)
    return dict(q=q, k=k, v=v, cur_k=_randn(gen, n, G, D).to(dt), cur_v=_randn(gen, n, G, D).to(dt))


def _weights(case: dict, gen, dt) -> dict:
    H, I, G, R = case["hidden"], case["intermediate"], case["kv_heads"], case["q_per_kv"]
    nq = (G * R + 2 * G) * D
    layers = []
    for _ in range(case["layers"]):
        layers.append(dict(
            norm1=(1.0 + 0.1 * _randn(gen, H)).to(dt), norm2=(1.0 + 0.1 * _randn(gen, H)).to(dt),
            qkv=_randn(gen, nq, H, dtype=dt).mul_(H ** -0.5), o=_randn(gen, H, G * R * D, dtype=dt).mul_(H ** -0.5),
            gate_up=_randn(gen, 2 * I, H, dtype=dt).mul_(H ** -0.5),
            down=_randn(gen, H, I, dtype=dt).mul_(I ** -0.5),
            bias=0.1 * _randn(gen, nq, dtype=dt) if case["bias"] else None))
    return dict(layers=layers, norm=(1.0 + 0.1 * _randn(gen, H)).to(dt),
                head=_randn(gen, case["vocab"], H, dtype=dt).mul_(H ** -0.5))


def _rope_tables(positions: int, dt) -> tuple[torch.Tensor, torch.Tensor]:
    inv = 500000.0 ** (-torch.arange(0, D, 2, device="cuda", dtype=torch.float64) / D)
    ang = torch.arange(positions, device="cuda", dtype=torch.float64)[:, None] * inv
    ang = torch.cat([ang, ang], dim=1)
    return ang.cos().to(dt), ang.sin().to(dt)


def _token_inputs(case: dict, seed: int) -> dict:
    dt, L = DTYPES[case["dtype"]], case["context"]
    s = _decode_inputs(case, seed, [L] * case["kv_heads"], "planted")
    gen = _gen(seed + 7919)
    s.update(_weights(case, gen, dt))
    s["h"] = _randn(gen, 1, case["hidden"]).to(dt)
    s["cos"], s["sin"] = _rope_tables(L + 1, dt)
    return s


class _Projections(torch.nn.Module):
    """The projections of one attention layer of the decoder model that the patch serves."""

    def __init__(self, config, dt, gen, bias: bool):
        super().__init__()
        self.config, self.head_dim, self.scaling = config, D, D ** -0.5
        H, nq, nk = config.hidden_size, config.num_attention_heads * D, config.num_key_value_heads * D
        for name, n_out, n_in in (("q_proj", nq, H), ("k_proj", nk, H), ("v_proj", nk, H), ("o_proj", H, nq)):
            lin = torch.nn.Linear(n_in, n_out, bias=bias and name != "o_proj", device="cuda", dtype=dt)
            with torch.no_grad():
                lin.weight.copy_(_randn(gen, n_out, n_in, dtype=dt).mul_(n_in ** -0.5))
                if lin.bias is not None:
                    lin.bias.copy_(0.1 * _randn(gen, n_out, dtype=dt))
            setattr(self, name, lin)


class _Config:
    pass


class LlamaPromptLayer(torch.nn.Module):
    """A decoder-only model reduced to its attention layers, as ``mp_headinfer`` patches them."""

    def __init__(self, config, dt, gen):
        super().__init__()
        self.config = config
        self.model = torch.nn.Module()
        layer = torch.nn.Module()
        layer.self_attn = _Projections(config, dt, gen, bias=False)
        self.model.layers = torch.nn.ModuleList([layer])


def _prefill_inputs(case: dict, seed: int) -> dict:
    gen, dt, S = _gen(seed), DTYPES[case["dtype"]], case["tokens"]
    cfg = _Config()
    cfg.num_key_value_heads, cfg.num_attention_heads = case["kv_heads"], case["kv_heads"] * case["q_per_kv"]
    cfg.hidden_size = cfg.num_attention_heads * D
    model = LlamaPromptLayer(cfg, dt, gen).eval()
    hidden = _randn(gen, 1, S, cfg.hidden_size, dtype=dt)
    cos, sin = _rope_tables(S, dt)
    return dict(model=model, hidden=hidden, cos=cos[None], sin=sin[None])


# ------------------------------------------------------------------ prepare
def _capture(s: dict, step) -> None:
    """The step as a replayable graph (warmed up eagerly first, so workspaces exist).  The graph holds addresses, so the
    state keeps the step too, with every tensor that it names."""
    with torch.no_grad():
        step()
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            step()
    torch.cuda.synchronize()
    s.update(graph=graph, step=step)


def _metadata(case: dict, s: dict, lengths: list[int], int4: bool) -> None:
    from headinfer import kernels

    n, G = s["k"].shape[:2]
    P = max(_pages(L)[1] for L in lengths)
    s["pmin"] = torch.zeros((n, G, P, D), dtype=s["k"].dtype, device="cuda")
    s["pmax"] = torch.zeros_like(s["pmin"])
    if int4:
        rows = s["k"].shape[2]
        s["packed"] = torch.zeros((n, G, rows, D // 2), dtype=torch.uint8, device="cuda")
        s["scale"] = torch.zeros((n, G, rows), dtype=s["k"].dtype, device="cuda")
        s["minimum"] = torch.zeros_like(s["scale"])
    for i in range(n):
        quant = dict(packed=s["packed"][i], scale=s["scale"][i], minimum=s["minimum"][i]) if int4 else {}
        if len(set(lengths)) == 1:
            kernels.build_page_metadata(s["k"][i, :, :lengths[0]], sink=SINK, block_size=BS, page_min=s["pmin"][i],
                                        page_max=s["pmax"][i], **quant)
            continue
        for g, L in enumerate(lengths):
            kernels.build_page_metadata(s["k"][i, g, :L], sink=SINK, block_size=BS, page_min=s["pmin"][i, g],
                                        page_max=s["pmax"][i, g])


def _pinned(t: torch.Tensor) -> torch.Tensor:
    h = torch.empty(t.shape, dtype=t.dtype, pin_memory=True)
    h.copy_(t)
    return h


def _prepare_quest(case: dict, seed: int) -> dict:
    from headinfer import kernels

    L, G, R = case["context"], case["kv_heads"], case["q_per_kv"]
    s = _decode_inputs(case, seed, [L] * G, "planted")
    _metadata(case, s, [L] * G, int4=False)
    P = _pages(L)[0]
    k = min(case["pages"], P)
    if case["residency"] == "host":
        s["k"], s["v"] = _pinned(s["k"]), _pinned(s["v"])
    qf = s["q"].float()
    s["bits"] = torch.zeros((case["layers"], G, R, kernels.sel_bits_words(P)), dtype=torch.int32, device="cuda")
    s["out"] = torch.empty_like(s["q"])

    def step():
        for i in range(case["layers"]):
            kernels.quest_select_bits(qf[i], s["pmin"][i, :, :P], s["pmax"][i, :, :P], k, s["bits"][i])
            kernels.decode_attention_pages_bits(s["q"][i], s["k"][i], s["v"][i], s["bits"][i], P,
                                                max_pages=min(P, R * k), sink=SINK, recent=RECENT, block_size=BS,
                                                length=L, append=True, cur_k=s["cur_k"][i], cur_v=s["cur_v"][i],
                                                out=s["out"][i])

    _capture(s, step)
    s["outputs"] = dict(out=s["out"], selected=s["bits"], k_row=s["k"][:, :, L], v_row=s["v"][:, :, L])
    return s


def _prepare_ragged(case: dict, seed: int) -> dict:
    from headinfer import kernels

    H, R = case["kv_heads"], case["q_per_kv"]
    lens = [L for L in _request_lengths(case) for _ in range(H)]
    s = _decode_inputs(case, seed, lens, "planted")
    _metadata(case, s, lens, int4=False)
    G, n = len(lens), case["layers"]
    P = s["pmin"].shape[2]
    k = min(case["pages"], P)
    W = min(P, R * k)
    at = torch.tensor(lens, dtype=torch.int32, device="cuda")
    qf = s["q"].float()
    s["out"] = torch.empty_like(s["q"])
    s["plan"] = torch.zeros((n, G, W), dtype=torch.int32, device="cuda")
    s["masks"] = torch.zeros((n, G, W), dtype=torch.uint8, device="cuda")
    s["counts"] = torch.zeros((n, G), dtype=torch.int32, device="cuda")

    def step():
        for i in range(n):
            kernels.quest_select_ragged(qf[i], s["pmin"][i], s["pmax"][i], at, k, sink=SINK, recent=RECENT,
                                        block_size=BS, plan_pages=s["plan"][i], plan_masks=s["masks"][i],
                                        plan_counts=s["counts"][i])
            kernels.decode_attention_pages_ragged(s["q"][i], s["k"][i], s["v"][i], s["plan"][i], s["counts"][i], at,
                                                  plan_masks=s["masks"][i], max_pages=W, sink=SINK, recent=RECENT,
                                                  block_size=BS, append=True, cur_k=s["cur_k"][i],
                                                  cur_v=s["cur_v"][i], out=s["out"][i])
            kernels.update_page_metadata_ragged(s["k"][i], at, first_entry=0, sink=SINK, block_size=BS,
                                                page_min=s["pmin"][i], page_max=s["pmax"][i])

    _capture(s, step)
    rows = [s[t][:, g, lens[g]] for t in ("k", "v") for g in range(0, G, H)]
    s["outputs"] = dict(out=s["out"], counts=s["counts"], page_min=s["pmin"], page_max=s["pmax"],
                        appended=rows)
    return s


def _prepare_twilight(case: dict, seed: int) -> dict:
    from headinfer import kernels

    L, G, R, n = case["context"], case["kv_heads"], case["q_per_kv"], case["layers"]
    s = _decode_inputs(case, seed, [L] * G, "zipf")
    _metadata(case, s, [L] * G, int4=True)
    P = _pages(L)[0]
    b0 = min(P, case["candidates"] // BS)
    matched = case["mode"] == "matched"
    target = min(_matched_pages(L), b0) * BS * R if matched else 0
    qf = s["q"].float()
    words = (kernels.union_record_words(P) + 3) & ~3
    s["rec"] = torch.zeros((n, G, words), dtype=torch.int32, device="cuda")
    s["desired"] = torch.zeros((n, G, R), dtype=torch.int32, device="cuda")
    s["out"] = torch.empty_like(s["q"])

    def step():
        for i in range(n):
            kernels.twilight_select_fused(qf[i], s["pmin"][i, :, :P], s["pmax"][i, :, :P], s["packed"][i],
                                          s["scale"][i], s["minimum"][i], b0, s["rec"][i], top_p=case["top_p"],
                                          sink=SINK, recent=RECENT, block_size=BS, length=L, desired=s["desired"][i],
                                          budget_mode=case["mode"], target_total=target)
            kernels.decode_attention_union(s["q"][i], s["k"][i], s["v"][i], s["rec"][i], P, max_pages=min(P, R * b0),
                                           sink=SINK, recent=RECENT, block_size=BS, length=L, append=True,
                                           cur_k=s["cur_k"][i], cur_v=s["cur_v"][i], out=s["out"][i])

    _capture(s, step)
    s["outputs"] = dict(out=s["out"], desired=s["desired"], record=s["rec"][:, :, :kernels.union_record_words(P)],
                        k_row=s["k"][:, :, L], v_row=s["v"][:, :, L])
    return s


def _prepare_gqa_rows(case: dict, seed: int) -> dict:
    L, G, R = case["context"], case["kv_heads"], case["q_per_kv"]
    s = _decode_inputs(case, seed, [L] * G, "zipf")
    _metadata(case, s, [L] * G, int4=True)
    P = _pages(L)[0]
    b0 = min(P, case["candidates"] // BS)
    W = min(P, R * b0)
    dt, i32 = s["q"].dtype, torch.int32
    s.update(P=P, b0=b0, qf=s["q"][0].float(), cu_q=torch.arange(G + 1, dtype=i32, device="cuda"),
             sel=torch.empty((G, R, b0), dtype=i32, device="cuda"),
             plan=torch.empty((G, W), dtype=i32, device="cuda"),
             masks=torch.empty((G, W), dtype=torch.uint8, device="cuda"),
             plan_counts=torch.empty((G,), dtype=i32, device="cuda"),
             rows=torch.empty((G, L + 1), dtype=i32, device="cuda"),
             counts=torch.empty((G,), dtype=i32, device="cuda"),
             flat_k=torch.zeros((G * (L + 1), D), dtype=dt, device="cuda"),
             flat_v=torch.zeros((G * (L + 1), D), dtype=dt, device="cuda"),
             cu=torch.empty((G + 1,), dtype=i32, device="cuda"))
    return s


def _prepare_metadata(case: dict, seed: int) -> dict:
    gen, dt, T, G = _gen(seed), DTYPES[case["dtype"]], case["tokens"], case["kv_heads"]
    keys = _keys(gen, _randn(gen, G, 4, D).to(dt), T, _pages(T)[0], "planted", dt)
    P = _pages(T)[1]
    s = dict(keys=keys, pmin=torch.empty((G, P, D), dtype=dt, device="cuda"))
    s["pmax"] = torch.empty_like(s["pmin"])
    if case["int4"]:
        s.update(packed=torch.empty((G, T, D // 2), dtype=torch.uint8, device="cuda"),
                 scale=torch.empty((G, T), dtype=dt, device="cuda"),
                 minimum=torch.empty((G, T), dtype=dt, device="cuda"))
    return s


def _prepare_prefill(case: dict, seed: int) -> dict:
    from headinfer.mp import mp_headinfer

    s = _prefill_inputs(case, seed)
    mp_headinfer(s["model"])
    s["attn"] = s["model"].model.layers[0].self_attn
    return s


def _prepare_token(case: dict, seed: int) -> dict:
    from headinfer import kernels

    s = _token_inputs(case, seed)
    L, G, R, H, n = case["context"], case["kv_heads"], case["q_per_kv"], case["hidden"], case["layers"]
    _metadata(case, s, [L] * G, int4=False)
    P, dt, Hq = _pages(L)[0], s["h"].dtype, G * R
    k = min(case["pages"], P)

    def empty(*shape, dtype=dt):
        return torch.empty(shape, dtype=dtype, device="cuda")

    position = torch.full((1,), L, dtype=torch.long, device="cuda")
    qkv = [empty(1, (Hq + 2 * G) * D) for _ in range(n)]
    q32, m, o, down = empty(Hq, D, dtype=torch.float32), empty(1, case["intermediate"]), empty(1, H), empty(1, H)
    res = [empty(1, H) for _ in range(2 * n + 1)]
    attn = [empty(G, R, D) for _ in range(n)]
    bits = torch.zeros((G, R, kernels.sel_bits_words(P)), dtype=torch.int32, device="cuda")
    logits = empty(1, case["vocab"])

    def step():
        h, delta = s["h"], None
        for i, w in enumerate(s["layers"]):
            h_out = res[2 * i] if delta is not None else None
            kernels.rms_norm_gemv(h, delta, w["norm1"], 1e-5, h_out, w["qkv"], w["bias"], qkv[i], epilogue="rope",
                                  rope=(Hq, G, s["cos"], s["sin"], position), q32=q32)
            h = h if h_out is None else h_out
            x = qkv[i][0]
            kernels.quest_select_bits(q32.view(G, R, D), s["pmin"][i, :, :P], s["pmax"][i, :, :P], k, bits)
            kernels.decode_attention_pages_bits(x[:Hq * D].view(G, R, D), s["k"][i], s["v"][i], bits, P,
                                                max_pages=min(P, R * k), sink=SINK, recent=RECENT, block_size=BS,
                                                length=L, append=True, cur_k=x[Hq * D:(Hq + G) * D].view(G, D),
                                                cur_v=x[(Hq + G) * D:].view(G, D), out=attn[i])
            kernels.gemv(attn[i].view(1, Hq * D), w["o"], None, o)
            kernels.rms_norm_gemv(h, o, w["norm2"], 1e-5, res[2 * i + 1], w["gate_up"], None, m, epilogue="silu")
            h = res[2 * i + 1]
            kernels.gemv(m, w["down"], None, down)
            delta = down
        kernels.rms_norm_gemv(h, delta, s["norm"], 1e-5, res[2 * n], s["head"], None, logits)

    _capture(s, step)
    # the first layer's attention: a later layer's selection may turn on the rounding of the layers before it
    s["outputs"] = dict(logits=logits, hidden=res[2 * n], attention=attn[0])
    return s


def prepare(case: dict, seed: int) -> dict:
    state = {"quest": _prepare_quest, "ragged": _prepare_ragged, "twilight": _prepare_twilight,
             "gqa_rows": _prepare_gqa_rows, "metadata": _prepare_metadata, "prefill": _prepare_prefill,
             "token": _prepare_token}[case["kind"]](case, seed)
    state["case"] = case
    return state


# ------------------------------------------------------------------ run
def _run_gqa_rows(s: dict) -> dict:
    from headinfer import kernels, mp

    case, L = s["case"], s["case"]["context"]
    G = case["kv_heads"]
    kernels.quest_select(s["qf"], s["pmin"][0, :, :s["P"]], s["pmax"][0, :, :s["P"]], s["b0"], sel_pages=s["sel"],
                         plan_pages=s["plan"], plan_masks=s["masks"], plan_counts=s["plan_counts"])
    logits = kernels.twilight_qk(s["qf"], s["packed"][0], s["scale"][0], s["minimum"][0], s["plan"], s["masks"],
                                 s["plan_counts"], s["b0"], sink=SINK, block_size=BS)
    kernels.twilight_select(logits, s["sel"], top_p=case["top_p"], budget_mode="dynamic", rows=s["rows"],
                            row_counts=s["counts"], sink=SINK, recent=RECENT, block_size=BS, length=L)
    k, v = s["k"][0], s["v"][0]
    kernels.gather_union(k.view(-1, D), v.view(-1, D), s["rows"], s["counts"], s["cur_k"][0], s["cur_v"][0],
                         s["flat_k"], s["flat_v"], s["cu"], entry_row0=0, entry_row_step=L + 1, max_count=L)
    kernels.append_kv(s["cur_k"][0], s["cur_v"][0], k, v, first_entry=0, position=L)
    cu = s["cu"].tolist()  # the branch returns the union's lengths as Python ints
    lengths = [b - a for a, b in zip(cu, cu[1:])]
    out = mp._flash_attention_varlen_forward(s["q"][0], s["flat_k"][:cu[-1]].unsqueeze(1),
                                             s["flat_v"][:cu[-1]].unsqueeze(1), s["cu_q"], s["cu"], 1, max(lengths),
                                             dropout=0.0, is_causal=True)
    return dict(out=out, cu=s["cu"], packed_k=s["flat_k"], packed_v=s["flat_v"])


def _run_prefill(s: dict) -> dict:
    from headinfer.quest_offload_cache import QuestTopKOffloadedCache
    from headinfer.twilight_offload_cache import TwilightMatchedBudgetOffloadedCache

    case, S = s["case"], s["case"]["tokens"]
    kind = QuestTopKOffloadedCache if case["cache"] == "quest" else TwilightMatchedBudgetOffloadedCache
    # a prompt is prefilled into a cache of its own
    cache = kind(num_cache_entries=case["kv_heads"], max_cache_len=S + 64, head_dim=D,
                 num_query_heads_per_kv=case["q_per_kv"], dtype=s["hidden"].dtype, device=s["hidden"].device,
                 sink_tokens=SINK, recent_tokens=RECENT, block_size=BS, kv_residency="hbm",
                 **({} if case["cache"] == "quest" else dict(candidate_token_budget=4096, budget_mode="dynamic")))
    with torch.no_grad():
        out, _ = s["attn"](s["hidden"], position_embeddings=(s["cos"], s["sin"]), past_key_values=cache)
    got = dict(out=out, k=cache._key_cache[:, :S], v=cache._value_cache[:, :S], page_min=cache._page_min,
               page_max=cache._page_max)
    if case["cache"] == "twilight":
        got.update(packed=cache._packed, scale=cache._qscale, minimum=cache._qmin)
    return got


def run(state: dict):
    kind = state["case"]["kind"]
    if kind == "gqa_rows":
        return _run_gqa_rows(state)
    if kind == "prefill":
        return _run_prefill(state)
    if kind == "metadata":
        from headinfer import kernels

        quant = {n: state[n] for n in ("packed", "scale", "minimum") if n in state}
        kernels.build_page_metadata(state["keys"], sink=SINK, block_size=BS, page_min=state["pmin"],
                                    page_max=state["pmax"], **quant)
        return dict(page_min=state["pmin"], page_max=state["pmax"], **quant)
    state["graph"].replay()
    return state["outputs"]


# ------------------------------------------------------------------ work
def _union_pages(P: int, k: int, heads: int) -> float:
    """Pages that `heads` heads of a group choose between them when each takes k of P: the expectation for independent
    choices, less the share that heads of one group have in common (measured 0.73 to 0.8 of it)."""
    return 0.78 * P * (1.0 - (1.0 - min(k, P) / P) ** heads)


def _attention_work(rows: float, groups: int, heads: int) -> tuple[float, float]:
    return rows * 2 * D * 2 + 2 * groups * heads * D * 2 + 8 * groups * D, rows * heads * 4 * D


def work(case: dict) -> dict:
    kind, G, R, e = case["kind"], case["kv_heads"], case.get("q_per_kv", 1), 2
    fixed = SINK + RECENT
    if kind in ("quest", "token"):
        P = _pages(case["context"])[0]
        rows = G * (_union_pages(P, case["pages"], R) * BS + fixed)
        b, f = _attention_work(rows, G, R)
        b, f = b + 2 * P * D * e * G + 4 * G * R * D, f + 4 * P * D * G * R
        if kind == "token":
            H, I = case["hidden"], case["intermediate"]
            params = (G * R + 2 * G) * D * H + H * G * R * D + 3 * H * I
            b, f = b + params * e, f + 2 * params
            head = case["vocab"] * H
            return {"bytes": case["layers"] * b + head * e, "flops": case["layers"] * f + 2 * head}
        return {"bytes": case["layers"] * b, "flops": case["layers"] * f}
    if kind == "ragged":
        b = f = 0.0
        for L in _request_lengths(case):
            P = _pages(L)[0]
            rows = G * (_union_pages(P, case["pages"], R) * BS + fixed)
            x, y = _attention_work(rows, G, R)
            b, f = b + x + 2 * P * D * e * G, f + y + 4 * P * D * G * R
        return {"bytes": case["layers"] * b, "flops": case["layers"] * f}
    if kind in ("twilight", "gqa_rows"):
        P = _pages(case["context"])[0]
        b0 = min(P, case["candidates"] // BS)
        cand = _union_pages(P, b0, R) * BS
        # dynamic budgets at top-p 0.95 keep about 0.8 of the candidates; matched ones 5% of the history a head
        kept = 0.8 * cand if case.get("mode", "dynamic") == "dynamic" else \
            min(cand, 0.78 * R * _matched_pages(case["context"]) * BS)
        b, f = _attention_work(G * (kept + fixed), G, R)
        b += 2 * P * D * e * G + G * cand * (D // 2 + 2 * e)
        f += 4 * P * D * G * R + 2 * cand * D * G * R
        if kind == "gqa_rows":
            b += 2 * G * (kept + fixed) * 2 * D * e  # the packed K/V, written and read
        n = case.get("layers", 1)
        return {"bytes": n * b, "flops": n * f}
    if kind == "metadata":
        T = case["tokens"]
        b = G * (T * D * e + 2 * _pages(T)[1] * D * e + (T * (D // 2 + 2 * e) if case["int4"] else 0))
        return {"bytes": b, "flops": 0.0}
    S, Hq = case["tokens"], G * R
    H = Hq * D
    proj = (Hq + 2 * G) * D * H + H * H
    b = 2 * S * H * e + proj * e + 2 * S * G * D * e + G * 2 * _pages(S)[1] * D * e
    b += S * G * (D // 2 + 2 * e) if case["cache"] == "twilight" else 0
    return {"bytes": b, "flops": 2 * S * proj + 4 * D * Hq * S * (S + 1) / 2}


# ------------------------------------------------------------------ tolerance and the 64-bit reference
def tolerance(case: dict):
    """Selections, counts, copied rows and metadata are whole values or copies: the same.  Attention accumulates in 32
    bits and rounds its probabilities and results to the K/V type; the prompt layer's projections do too."""
    kind = case["kind"]
    if kind == "metadata":
        return "exact"
    half = case["dtype"] == "f16"
    if kind == "prefill":  # 6.4e-4 and 5.4e-3 from 64 bits
        return {"rel": 2.5e-3 if half else 2e-2, "differ": 0.0}
    if kind == "token":    # 1.2e-2 from 64 bits in bf16
        return {"rel": 8e-3 if half else 3e-2, "differ": 0.0}
    return {"rel": 1e-3 if half else 8e-3, "differ": 0.0}  # 2.1e-4 and 2.0e-3 from 64 bits


def _minmax64(keys: torch.Tensor, T: int):
    """Page min and max of the complete pages of keys [G, >= T, D]."""
    P = _pages(T)[1]
    p = keys[:, SINK:SINK + P * BS].reshape(keys.shape[0], P, BS, D)
    return p.amin(dim=2), p.amax(dim=2)


def _score64(q, pmin, pmax):
    q = q.double()
    return q.clamp(min=0) @ pmax.double().transpose(-1, -2) + q.clamp(max=0) @ pmin.double().transpose(-1, -2)


def _page_rows(pages: torch.Tensor) -> torch.Tensor:
    return (SINK + pages[:, None] * BS + torch.arange(BS, device=pages.device)).reshape(-1)


def _attend64(q, k, v, rows, visible=None):
    """softmax(q k^T / sqrt(D)) v of one group over `rows`, q [R, D], visible [R, rows] or None."""
    s = q.double() @ k[rows].double().T / math.sqrt(D)
    if visible is not None:
        s = s.masked_fill(~visible, float("-inf"))
    return torch.softmax(s, dim=-1) @ v[rows].double()


def _with_token(k, v, cur_k, cur_v, L):
    k, v = k.clone(), v.clone()
    k[L], v[L] = cur_k, cur_v
    return k, v


def _quest_group64(q, k, v, pmin, pmax, L, budget):
    """One group's Quest attention: every head its own top pages, the windows and the decode token (row L of k/v)."""
    dev, R = q.device, q.shape[0]
    P = min(_pages(L)[0], pmin.shape[0])
    sink_end, recent_start = _window(L)
    top = _score64(q, pmin[:P], pmax[:P]).topk(min(budget, P), dim=-1).indices
    member = torch.zeros((R, P), dtype=torch.bool, device=dev).scatter_(1, top, True)
    pages = member.any(dim=0).nonzero()[:, 0]
    head, tail = torch.arange(sink_end, device=dev), torch.arange(recent_start, L + 1, device=dev)
    rows = torch.cat([head, _page_rows(pages), tail])
    ones = torch.ones((R, 1), dtype=torch.bool, device=dev)
    visible = torch.cat([ones.expand(-1, len(head)), member[:, pages].repeat_interleave(BS, dim=1),
                         ones.expand(-1, len(tail))], dim=1)
    return _attend64(q, k, v, rows, visible)


def _int4_64(keys: torch.Tensor) -> torch.Tensor:
    """Keys [T, D] after per-token affine INT4 (range rounded to the key type), dequantised."""
    dt = keys.dtype
    lo, hi = keys.amin(dim=-1, keepdim=True), keys.amax(dim=-1, keepdim=True)
    scale = ((hi - lo).float().clamp_min(1e-9) / 15.0).to(dt).float()
    code = torch.round((keys.float() - lo.float()) / scale).clamp(0, 15)
    return code.double() * scale.double() + lo.double()


def _matched64(desired: list[int], target: int, capacity: int) -> list[int]:
    """`target` rows split over the heads in proportion to their top-p counts (largest remainder, at least one each)."""
    n, total = len(desired), float(sum(desired))
    raw = [(target - n) * d / total for d in desired]
    got = [1 + min(capacity - 1, math.floor(r)) for r in raw]
    while sum(got) < target:
        i = min((i for i in range(n) if got[i] < capacity), key=lambda i: (-(raw[i] - math.floor(raw[i])), -desired[i], i))
        got[i], raw[i] = got[i] + 1, float(math.floor(raw[i]))
    return got


def _twilight_rows64(q, k, pmin, pmax, L, candidates, top_p, matched):
    """The union of one group's kept rows with the windows, ascending (without the decode token)."""
    dev, R = q.device, q.shape[0]
    P = _pages(L)[0]
    sink_end, recent_start = _window(L)
    b0 = min(P, candidates // BS)
    pages = _score64(q, pmin[:P], pmax[:P]).topk(b0, dim=-1).indices.sort(dim=-1).values
    est = q.double() @ _int4_64(k[:L]).T / math.sqrt(D)
    keep = torch.zeros(L, dtype=torch.bool, device=dev)
    keep[:sink_end] = True
    keep[recent_start:] = True
    order, desired = [], []
    for r in range(R):
        rows = _page_rows(pages[r])
        logit, at = est[r, rows].sort(descending=True, stable=True)
        cum = torch.softmax(logit, dim=0).cumsum(dim=0)
        desired.append(min(len(rows), int((cum < top_p).sum()) + 1))
        order.append(rows[at])
    counts = desired
    if matched:
        counts = _matched64(desired, min(_matched_pages(L), b0) * BS * R, b0 * BS)
    for rows, c in zip(order, counts):
        keep[rows[:c]] = True
    return keep.nonzero()[:, 0]


def _exact_quest(case, seed):
    L, G = case["context"], case["kv_heads"]
    s = _decode_inputs(case, seed, [L] * G, "planted")
    out = torch.empty(s["q"].shape, dtype=torch.float64, device="cuda")
    for i in range(case["layers"]):
        pmin, pmax = _minmax64(s["k"][i], L)
        for g in range(G):
            k, v = _with_token(s["k"][i, g], s["v"][i, g], s["cur_k"][i, g], s["cur_v"][i, g], L)
            out[i, g] = _quest_group64(s["q"][i, g], k, v, pmin[g], pmax[g], L, case["pages"])
    return dict(out=out, selected=None, k_row=s["cur_k"].double(), v_row=s["cur_v"].double())


def _exact_ragged(case, seed):
    H = case["kv_heads"]
    lens = [L for L in _request_lengths(case) for _ in range(H)]
    s = _decode_inputs(case, seed, lens, "planted")
    out = torch.empty(s["q"].shape, dtype=torch.float64, device="cuda")
    P = max(_pages(L)[1] for L in lens)
    budget = min(case["pages"], P)
    page_min = torch.zeros((case["layers"], len(lens), P, D), dtype=torch.float64, device="cuda")
    page_max = torch.zeros_like(page_min)
    for i in range(case["layers"]):
        for g, L in enumerate(lens):
            k, v = _with_token(s["k"][i, g], s["v"][i, g], s["cur_k"][i, g], s["cur_v"][i, g], L)
            pmin, pmax = _minmax64(k[None], L)
            out[i, g] = _quest_group64(s["q"][i, g], k, v, pmin[0], pmax[0], L, budget)
            lo, hi = _minmax64(k[None], L + 1)  # the decode token may complete a page
            n = min(P, lo.shape[1])
            page_min[i, g, :n], page_max[i, g, :n] = lo[0, :n].double(), hi[0, :n].double()
    rows = [s[t][:, g].double() for t in ("cur_k", "cur_v") for g in range(0, len(lens), H)]
    return dict(out=out, counts=None, page_min=page_min, page_max=page_max, appended=rows)


def _exact_twilight(case, seed):
    L, G, n = case["context"], case["kv_heads"], case.get("layers", 1)
    s = _decode_inputs(case, seed, [L] * G, "zipf")
    out = torch.empty(s["q"].shape, dtype=torch.float64, device="cuda")
    for i in range(n):
        pmin, pmax = _minmax64(s["k"][i], L)
        for g in range(G):
            rows = _twilight_rows64(s["q"][i, g], s["k"][i, g], pmin[g], pmax[g], L, case["candidates"],
                                    case["top_p"], case.get("mode") == "matched")
            rows = torch.cat([rows, torch.tensor([L], device=rows.device)])
            k, v = _with_token(s["k"][i, g], s["v"][i, g], s["cur_k"][i, g], s["cur_v"][i, g], L)
            out[i, g] = _attend64(s["q"][i, g], k, v, rows)
    if case["kind"] == "gqa_rows":
        return dict(out=out[0], cu=None, packed_k=None, packed_v=None)
    return dict(out=out, desired=None, record=None, k_row=s["cur_k"].double(), v_row=s["cur_v"].double())


def _exact_metadata(case, seed):
    s = _prepare_metadata(case, seed)
    lo, hi = _minmax64(s["keys"], case["tokens"])
    got = dict(page_min=lo.double(), page_max=hi.double())
    if case["int4"]:
        k = s["keys"]
        mn, mx = k.amin(dim=-1), k.amax(dim=-1)
        scale = (mx.double() - mn.double()).clamp_min(1e-9) / 15.0
        got.update(packed=None, scale=scale, minimum=mn.double())
    return got


def _rope64(x, cos, sin):
    half = D // 2
    return x * cos + torch.cat([-x[..., half:], x[..., :half]], dim=-1) * sin


def _exact_prefill(case, seed):
    s = _prefill_inputs(case, seed)
    S, G, R = case["tokens"], case["kv_heads"], case["q_per_kv"]
    attn = s["model"].model.layers[0].self_attn
    x = s["hidden"][0].double()

    def proj(lin, heads):
        return (x @ lin.weight.double().T).view(S, heads, D).transpose(0, 1)

    cos, sin = s["cos"][0].double(), s["sin"][0].double()
    q = _rope64(proj(attn.q_proj, G * R), cos, sin).view(G, R, S, D)
    k = _rope64(proj(attn.k_proj, G), cos, sin)
    v = proj(attn.v_proj, G)
    out = torch.empty((S, G * R * D), dtype=torch.float64, device="cuda")
    col = torch.arange(S, device="cuda")
    for g in range(G):
        for r in range(R):
            for a in range(0, S, 8192):
                b = min(S, a + 8192)
                sc = (q[g, r, a:b] @ k[g, :b].T) / math.sqrt(D)
                sc.masked_fill_(col[None, :b] > col[a:b, None], float("-inf"))
                at = (g * R + r) * D
                out[a:b, at:at + D] = torch.softmax(sc, dim=-1) @ v[g, :b]
    out = out @ attn.o_proj.weight.double().T
    lo, hi = _minmax64(k, S)
    got = dict(out=out[None], k=k, v=v, page_min=lo, page_max=hi)
    if case["cache"] == "twilight":
        mn, mx = k.amin(dim=-1), k.amax(dim=-1)
        got.update(packed=None, scale=(mx - mn).clamp_min(1e-9) / 15.0, minimum=mn)
    return got


def _exact_token(case, seed):
    s = _token_inputs(case, seed)
    L, G, R = case["context"], case["kv_heads"], case["q_per_kv"]
    Hq = G * R

    def norm(x, w):
        return x * torch.rsqrt(x.square().mean(dim=-1, keepdim=True) + 1e-5) * w.double()

    h, attention = s["h"].double(), None
    cos, sin = s["cos"][L].double(), s["sin"][L].double()
    for i, w in enumerate(s["layers"]):
        qkv = (norm(h, w["norm1"]) @ w["qkv"].double().T)[0]
        if w["bias"] is not None:
            qkv = qkv + w["bias"].double()
        qkv = qkv.view(Hq + 2 * G, D)
        q = _rope64(qkv[:Hq], cos, sin).view(G, R, D)
        kn, vn = _rope64(qkv[Hq:Hq + G], cos, sin), qkv[Hq + G:]
        pmin, pmax = _minmax64(s["k"][i], L)
        got = torch.empty((G, R, D), dtype=torch.float64, device="cuda")
        for g in range(G):
            k, v = _with_token(s["k"][i, g].double(), s["v"][i, g].double(), kn[g], vn[g], L)
            got[g] = _quest_group64(q[g], k, v, pmin[g], pmax[g], L, case["pages"])
        attention = got if attention is None else attention
        h = h + got.view(1, Hq * D) @ w["o"].double().T
        gu = norm(h, w["norm2"]) @ w["gate_up"].double().T
        I = case["intermediate"]
        h = h + (torch.nn.functional.silu(gu[:, :I]) * gu[:, I:]) @ w["down"].double().T
    return dict(logits=norm(h, s["norm"]) @ s["head"].double().T, attention=attention, hidden=h)


def exact(case: dict, seed: int):
    """What run() returns, in 64 bits, by plain torch."""
    with torch.no_grad():
        return {"quest": _exact_quest, "ragged": _exact_ragged, "twilight": _exact_twilight,
                "gqa_rows": _exact_twilight, "metadata": _exact_metadata, "prefill": _exact_prefill,
                "token": _exact_token}[case["kind"]](case, seed)
