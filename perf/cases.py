"""Timing cases of the attention and KV-cache paths, as an agent's inference loop calls them.

A case is a dict of plain values. ``listed()`` gives the fixed ones, ``draw(rng)`` one more of the same
ranges, ``prepare(case, seed)`` what a program holds before the call, ``run(state)`` one pass through the
package's public entry points, ``work(case)`` the bytes and operations that a pass cannot do without,
``tolerance(case)`` how far another correct implementation's outputs may lie, and ``exact(case, seed)``
the outputs in float64 by plain torch.

Kinds:
- ``decode``: one decode call of the registered attention on a cache (one layer of a token).
- ``decode_graph``: the decode attention of every layer of a token, prepared once and captured.
- ``decode_ragged``: a batch of sequences of different lengths, one decode call.
- ``append``: a token's cache append and attention in every layer (the eager decode loop).
- ``paged_step``: the same over a paged cache of several sequences.
- ``prefill``: the prefill attention of one forward pass, layer after layer: a whole prompt (``causal``), a
  chunk on top of a cache (``chunk``) or a left-padded batch of prompts (``padded``).
- ``splice``: a span of the cached context is dropped and as many new tokens are appended.
- ``paged_turn``: the same on a paged cache, with the new tokens' attention.
"""
import math

import torch

from threadcut_amd import attention, flash_decode, kv, paged, workloads
from threadcut_amd.match import Split

D = 128
SCALE = D ** -0.5
DEV = "cuda"
DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}


def listed():
    return [
        # The smallest call: one layer of one token, 1536 tokens cached (32 query heads over 8 KV heads).
        dict(name="decode_1536", kind="decode", batch=1, q_heads=32, kv_heads=8, tokens=1536, dtype="fp16"),
        # A token's 36 layers at 10240 cached tokens, prepared once and replayed.
        dict(name="decode_graph_10240", kind="decode_graph", layers=36, batch=1, q_heads=32, kv_heads=8,
             tokens=10240, dtype="fp16"),
        # Serving 16 conversations of 1k to 32k tokens at once.
        dict(name="decode_ragged_16", kind="decode_ragged", batch=16, q_heads=32, kv_heads=8, tokens=32768,
             shortest=1024, dtype="bf16"),
        # The eager decode loop of a batch: each layer's row is written while it is attended (16 query heads over
        # 8 KV heads, an odd length).
        dict(name="append_8x4001", kind="append", layers=8, batch=8, q_heads=16, kv_heads=8, tokens=4001,
             dtype="bf16"),
        # The decode loop over a paged cache of four sequences.
        dict(name="paged_step_4x5000", kind="paged_step", layers=8, batch=4, q_heads=32, kv_heads=8, tokens=5000,
             page_tokens=64, dtype="fp16"),
        # The engine's chunk of 2048 tokens on the 7716 tokens that a prune kept.
        dict(name="prefill_chunk_2048", kind="prefill", layers=4, batch=1, q_heads=32, kv_heads=8, queries=2048,
             past=7716, mask="chunk", dtype="fp16"),
        # A short prompt on an empty cache.
        dict(name="prefill_prompt_1100", kind="prefill", layers=4, batch=1, q_heads=32, kv_heads=8, queries=1100,
             past=0, mask="causal", dtype="fp16"),
        # A short tool result on a long conversation.
        dict(name="prefill_turn_93", kind="prefill", layers=4, batch=1, q_heads=32, kv_heads=8, queries=93,
             past=9000, mask="chunk", dtype="fp16"),
        # A left-padded batch of prompts (16 query heads over 8 KV heads).
        dict(name="prefill_padded_4", kind="prefill", layers=4, batch=4, q_heads=16, kv_heads=8, queries=1500,
             past=0, mask="padded", dtype="bf16"),
        # A long tool result is dropped from a 14336-token conversation: the suffix moves further than its length.
        dict(name="splice_far", kind="splice", layers=36, kv_heads=8, tokens=14336, a=2048, gap=6620, dtype="fp16"),
        # A short one: the suffix overlaps its old place.
        dict(name="splice_near", kind="splice", layers=28, kv_heads=8, tokens=9000, a=700, gap=333, dtype="bf16"),
        # The same turn on a paged cache, with the new tokens' attention.
        dict(name="paged_turn_600", kind="paged_turn", layers=12, q_heads=32, kv_heads=8, tokens=8200, a=1500,
             gap=600, page_tokens=64, dtype="fp16"),
    ]


def _span(rng, lo, hi):
    """A whole number of [lo, hi], even over the logarithm."""
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(["decode", "decode_graph", "decode_ragged", "append", "paged_step", "prefill", "prefill",
                       "prefill", "splice", "paged_turn"])
    q_heads, kv_heads = rng.choice([(32, 8), (32, 8), (16, 8), (8, 8), (64, 8), (8, 2), (16, 4)])
    c = dict(kind=kind, q_heads=q_heads, kv_heads=kv_heads, dtype=rng.choice(["fp16", "fp16", "bf16"]))
    if kind == "decode":
        c.update(batch=rng.choice([1, 1, 1, 2, 5, 12, 32]), tokens=_span(rng, 40, 16000))
    elif kind == "decode_graph":
        c.update(layers=rng.choice([8, 28, 36]), batch=rng.choice([1, 1, 3]), tokens=_span(rng, 200, 16000))
    elif kind == "decode_ragged":
        top = _span(rng, 2000, 32768)
        c.update(batch=rng.randint(2, 16), tokens=top, shortest=_span(rng, 16, top // 2))
    elif kind == "append":
        c.update(layers=rng.randint(2, 8), batch=_span(rng, 1, 16), tokens=_span(rng, 60, 8000))
    elif kind == "paged_step":
        c.update(layers=rng.randint(2, 8), batch=_span(rng, 1, 8), tokens=_span(rng, 100, 8000),
                 page_tokens=rng.choice([16, 32, 64, 64, 128]))
    elif kind == "prefill":
        mask = rng.choice(["causal", "chunk", "chunk", "padded"])
        if mask == "chunk":
            c.update(queries=_span(rng, 2, 2048), past=_span(rng, 100, 9000), batch=1)
        else:
            c.update(queries=_span(rng, 20, 2048), past=0, batch=rng.randint(2, 4) if mask == "padded" else 1)
        c.update(layers=rng.randint(1, 4), mask=mask)
        if c["q_heads"] > 32:
            c["layers"] = 1
    elif kind == "splice":
        n = _span(rng, 400, 14336)
        a = rng.randint(0, n // 3)
        c.update(layers=rng.choice([8, 28, 36]), tokens=n, a=a, gap=_span(rng, 8, n - a - 40))
        del c["q_heads"]
    else:
        n = _span(rng, 600, 9000)
        a = rng.randint(0, n // 3)
        c.update(layers=rng.randint(2, 12), tokens=n, a=a, gap=_span(rng, 8, min(2048, n - a - 40)),
                 page_tokens=rng.choice([16, 32, 64, 64, 128]))
    return c


class _Config:
    """What a cache asks of a model's configuration."""

    def __init__(self, layers):
        self.num_hidden_layers = layers

    def get_text_config(self, decoder=True):
        return self


def _randn(gen, shape, case):
    return torch.randn(shape, generator=gen, device=DEV, dtype=torch.float32).to(DTYPES[case["dtype"]])


def _rows(gen, case, batch, heads, n):
    """Projections of n new tokens as a model hands them over: [b, heads, n, d], a transposed view."""
    return _randn(gen, (batch, n, heads, D), case).transpose(1, 2)


def _inputs(case, seed):
    """Every random tensor of a case, from the seed alone."""
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    kind, hkv, n = case["kind"], case["kv_heads"], case.get("tokens", 0)
    hq, layers, b = case.get("q_heads", 0), case.get("layers", 1), case.get("batch", 1)
    x = {}
    if kind == "prefill":
        n = case["past"] + case["queries"]
    if kind == "decode_ragged":
        x["lens"] = torch.randint(case["shortest"], n + 1, (b,), generator=g, device=DEV).to(torch.int32)
        x["lens"][0] = n
    if kind == "paged_step":  # between half and all of `tokens`
        x["lens"] = torch.randint(n - n // 2, n + 1, (b,), generator=g, device=DEV).tolist()
    if kind == "prefill" and case["mask"] == "padded":
        x["pads"] = torch.randint(0, case["queries"] // 2 + 1, (b,), generator=g, device=DEV)
        x["pads"][0] = 0
    x["k"] = [_randn(g, (b, hkv, n, D), case) for _ in range(layers)]
    x["v"] = [_randn(g, (b, hkv, n, D), case) for _ in range(layers)]
    new = {"append": 1, "paged_step": 1, "splice": case.get("gap"), "paged_turn": case.get("gap")}.get(kind)
    if new:
        x["kn"] = [_rows(g, case, b, hkv, new) for _ in range(layers)]
        x["vn"] = [_rows(g, case, b, hkv, new) for _ in range(layers)]
    if kind != "splice":
        queries = case["queries"] if kind == "prefill" else case["gap"] if kind == "paged_turn" else 1
        x["q"] = [_rows(g, case, b, hq, queries) for _ in range(layers)]
    return x


def _mask(case, x):
    """Boolean [b|1, 1, q, n] as transformers builds it, or None."""
    if case["kind"] == "paged_turn":
        return workloads.causal_mask(case["gap"], case["tokens"], device=DEV).contiguous()
    if case["mask"] == "causal":
        return None
    n = case["past"] + case["queries"]
    m = workloads.causal_mask(case["queries"], n, device=DEV)
    if case["mask"] == "padded":
        m = m & (torch.arange(n, device=DEV)[None, :] >= x["pads"][:, None])[:, None, None, :]
    return m.contiguous()


def _split(case):
    return Split(case["a"], case["a"] + case["gap"], case["tokens"] - case["a"] - case["gap"])


def prepare(case, seed):
    x = _inputs(case, seed)
    kind, layers = case["kind"], case.get("layers", 1)
    st = {"case": case, "kind": kind, "q": x.get("q"), "kn": x.get("kn"), "vn": x.get("vn")}
    if kind in ("decode", "prefill"):
        caches = [kv.GrowingLayer() for _ in range(layers)]
        for c, k, v in zip(caches, x["k"], x["v"]):  # two updates: the buffers then hold more than the cached tokens
            c.update(k[:, :, :-1], v[:, :, :-1])
            c.update(k[:, :, -1:], v[:, :, -1:])
        st["caches"] = caches
        if kind == "prefill":
            st["mask"] = _mask(case, x)
    elif kind == "decode_ragged":
        b, hkv = case["batch"], case["kv_heads"]
        st.update(k=x["k"][0], v=x["v"][0], lens=x["lens"], q=x["q"][0].reshape(b, hkv, -1, D))
    elif kind == "decode_graph":
        b, hkv = case["batch"], case["kv_heads"]
        qs = [q.reshape(b, hkv, -1, D) for q in x["q"]]
        outs = [torch.empty_like(q) for q in qs]
        plans, space = [], None
        for q, k, v, o in zip(qs, x["k"], x["v"], outs):
            plans.append(flash_decode.DecodePlan(q, k, v, SCALE, o, workspace=space))
            space = plans[0].workspace
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            for p in plans:
                p.run()
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            for p in plans:
                p.run()
        st.update(plans=plans, graph=graph, outs=outs)
    elif kind == "append":
        cache = kv.new_cache(_Config(layers), fused_append=True)
        for i in range(layers):
            cache.update(x["k"][i], x["v"][i], i)
        st["cache"] = cache
        run(st)  # the buffers have grown past the first step
    elif kind == "paged_step":
        b, P = case["batch"], case["page_tokens"]
        pages = b * (-(-case["tokens"] // P) + 2)
        c = paged.PagedKV(layers, case["kv_heads"], pages, P, batch=b, dtype=DTYPES[case["dtype"]], device=DEV)
        for at in range(0, case["tokens"], 512):  # the sequences arrive in turns, so their pages mix
            for i, n in enumerate(x["lens"]):
                if at < n:
                    c.append(i, [k[i, :, at:min(n, at + 512)] for k in x["k"]],
                             [v[i, :, at:min(n, at + 512)] for v in x["v"]])
        st.update(cache=c, inv_freq=workloads.inv_freq().to(DEV))
    elif kind == "splice":
        cache = kv.new_cache(_Config(layers), slab=True)
        for i in range(layers):
            cache.update(x["k"][i], x["v"][i], i)
        st.update(cache=cache, split=_split(case), inv_freq=workloads.inv_freq().to(DEV))
    else:
        P = case["page_tokens"]
        cache = paged.new_paged_cache(_Config(layers), -(-case["tokens"] // P) + -(-case["gap"] // P) + 4, P)
        for i in range(layers):
            cache.update(x["k"][i], x["v"][i], i)
        st.update(cache=cache, split=_split(case), inv_freq=workloads.inv_freq().to(DEV), mask=_mask(case, x))
    return st


def run(st):
    kind = st["kind"]
    if kind == "decode":
        c = st["caches"][0]
        return attention.attention(None, st["q"][0], c.keys, c.values, None)[0]
    if kind == "prefill":
        return [attention.attention(None, q, c.keys, c.values, st["mask"])[0] for q, c in zip(st["q"], st["caches"])]
    if kind == "decode_ragged":
        return flash_decode.decode_attention_batched(st["q"], st["k"], st["v"], SCALE, lens=st["lens"])
    if kind == "decode_graph":
        st["graph"].replay()
        return st["outs"]
    cache = st["cache"]
    if kind == "append":
        outs, n = [], cache.get_seq_length()
        for i, q in enumerate(st["q"]):
            k, v = cache.update(st["kn"][i], st["vn"][i], i)
            outs.append(attention.attention(None, q, k, v, None)[0])
            outs += [k, v]
        cache.crop(n)  # the token is taken back (a rejected draft)
        return outs
    if kind == "paged_step":
        b, hkv = st["case"]["batch"], st["case"]["kv_heads"]
        cache.reserve_step()
        outs = [cache.decode_append(i, q.reshape(b, hkv, -1, D), st["kn"][i], st["vn"][i], SCALE)
                for i, q in enumerate(st["q"])]
        for i in range(b):  # the token is taken back
            n = cache.length(i)
            cache.prune(i, Split(n - 1, n, 0), st["inv_freq"])
        return {"out": outs, "k": cache.k_pools, "v": cache.v_pools}
    kv.splice(cache, st["split"], st["inv_freq"])
    if kind == "splice":
        for i in range(st["case"]["layers"]):
            cache.update(st["kn"][i], st["vn"][i], i)
        layer = cache.layers[0]
        return layer.slab.tensor[..., :layer.n, :]
    outs = []
    for i, q in enumerate(st["q"]):
        k, v = cache.update(st["kn"][i], st["vn"][i], i)
        outs.append(attention.attention(None, q, k, v, st["mask"])[0])
    return {"out": outs, "k": list(paged.state_of(cache).kv.k_pools), "v": list(paged.state_of(cache).kv.v_pools)}


def _visible(q, n):
    """(query, key) pairs that q causal queries at the end of n keys see."""
    return q * n - q * (q - 1) // 2


def work(case):
    kind, hkv, layers, b = case["kind"], case["kv_heads"], case.get("layers", 1), case.get("batch", 1)
    hq, n = case.get("q_heads", 0), case.get("tokens", 0)
    row = 2 * D  # bytes of one head's row
    if kind in ("decode", "decode_graph", "append"):
        keys, q = b * n, b
    elif kind == "decode_ragged":
        keys, q = n + (b - 1) * (n + case["shortest"]) // 2, b
    elif kind == "paged_step":
        keys, q = b * (n - n // 4), b
    elif kind == "prefill":
        q = b * case["queries"]
        n = case["past"] + case["queries"]
        keys = b * n
        pairs = b * _visible(case["queries"], n)
        if case["mask"] == "padded":  # pads average a quarter of the prompt
            pairs = _visible(n, n) + (b - 1) * _visible(3 * n // 4, 3 * n // 4)
        masked = 0 if case["mask"] == "causal" else (b if case["mask"] == "padded" else 1) * case["queries"] * n
        return {"bytes": layers * (2 * hkv * keys + 2 * hq * q) * row + masked, "flops": layers * 4 * D * hq * pairs}
    elif kind == "splice":
        c = case["tokens"] - case["a"] - case["gap"]
        return {"bytes": layers * 2 * 2 * hkv * row * (c + case["gap"]), "flops": layers * 3 * D * hkv * c}
    else:
        c, q = n - case["a"] - case["gap"], case["gap"]
        moved = 2 * hkv * c + 4 * hkv * q
        return {"bytes": layers * (moved + 2 * hkv * n + 2 * hq * q) * row + q * n,
                "flops": layers * 4 * D * hq * _visible(q, n)}
    new = 4 * hkv * b if kind in ("append", "paged_step") else 0
    return {"bytes": layers * (2 * hkv * keys + 2 * hq * q + new) * row, "flops": layers * 4 * D * hq * keys}


def tolerance(case):
    if case["kind"] == "splice":
        return "exact"  # rows are moved, and rotated in fp32 by one fixed order of operations
    # Outputs rounded to the storage type, the weights too in prefill: measured against float64 at up to 3.5e-4
    # (fp16) and 2e-3 (bf16).
    return {"rel": 1.4e-3} if case["dtype"] == "fp16" else {"rel": 8e-3}


def _attend(q, k, v, vis):
    """float64 [b, q, hq, d] of q [b, hq, q, d] over k/v [b, hkv, n, d]; vis bool [b|1, q, n] or None."""
    b, hq, ql, _ = q.shape
    g = hq // k.shape[1]
    out = torch.zeros((b, ql, hq, D), dtype=torch.float64, device=q.device)
    for i in range(b):
        ok = None if vis is None else vis[i if vis.shape[0] > 1 else 0]
        for h in range(hq):
            s = q[i, h].double() @ k[i, h // g].double().t() * SCALE
            if ok is not None:
                s = s.masked_fill(~ok, float("-inf"))
            out[i, :, h] = torch.softmax(s, -1).nan_to_num() @ v[i, h // g].double()
    return out


def _rotated(k, delta):
    """Keys moved by `delta` positions, in float64."""
    angle = (delta * workloads.inv_freq()).double().to(k.device)
    cos, sin = angle.cos(), angle.sin()
    lo, hi = k[..., :D // 2].double(), k[..., D // 2:].double()
    return torch.cat((lo * cos - hi * sin, hi * cos + lo * sin), -1)


def exact(case, seed):
    x = _inputs(case, seed)
    kind = case["kind"]
    if kind == "decode":
        return _attend(x["q"][0], x["k"][0], x["v"][0], None)
    if kind == "decode_graph":
        b, hkv = case["batch"], case["kv_heads"]
        return [_attend(q, k, v, None).reshape(b, hkv, -1, D) for q, k, v in zip(x["q"], x["k"], x["v"])]
    if kind == "decode_ragged":
        b, hkv = case["batch"], case["kv_heads"]
        out = [_attend(x["q"][0][i:i + 1], x["k"][0][i:i + 1, :, :n], x["v"][0][i:i + 1, :, :n], None)
               for i, n in enumerate(x["lens"].tolist())]
        return torch.cat(out).reshape(b, hkv, -1, D)
    if kind == "append":
        outs = []
        for q, k, v, kn, vn in zip(x["q"], x["k"], x["v"], x["kn"], x["vn"]):
            k, v = torch.cat((k, kn), 2), torch.cat((v, vn), 2)
            outs += [_attend(q, k, v, None), k.double(), v.double()]
        return outs
    if kind == "paged_step":  # the pools' rows are copies, whose places the page table gives
        b, hkv = case["batch"], case["kv_heads"]
        outs = []
        for q, k, v, kn, vn in zip(x["q"], x["k"], x["v"], x["kn"], x["vn"]):
            one = [_attend(q[i:i + 1], torch.cat((k[i:i + 1, :, :n], kn[i:i + 1]), 2),
                           torch.cat((v[i:i + 1, :, :n], vn[i:i + 1]), 2), None) for i, n in enumerate(x["lens"])]
            outs.append(torch.cat(one).reshape(b, hkv, -1, D))
        return {"out": outs, "k": None, "v": None}
    if kind == "prefill":
        m = _mask(case, x)
        if m is None:
            m = workloads.causal_mask(case["queries"], case["queries"], device=DEV)
        return [_attend(q, k, v, m[:, 0]) for q, k, v in zip(x["q"], x["k"], x["v"])]
    s = _split(case)
    spliced = []
    for k, v, kn, vn in zip(x["k"], x["v"], x["kn"], x["vn"]):
        spliced.append((torch.cat((k[:, :, :s.a].double(), _rotated(k[:, :, s.c0:], -s.gap), kn.double()), 2),
                        torch.cat((v[:, :, :s.a].double(), v[:, :, s.c0:].double(), vn.double()), 2)))
    if kind == "splice":
        return torch.stack([torch.stack(kv_) for kv_ in spliced])
    m = _mask(case, x)[:, 0]
    return {"out": [_attend(q, k, v, m) for q, (k, v) in zip(x["q"], spliced)], "k": None, "v": None}
