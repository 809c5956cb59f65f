"""The calls this framework is timed on: what a serving program has it do, through the same objects
such a program holds (``AttnBackend`` over an ``MHAKVCache``, ``GDNBackend`` over a ``MambaStatePool``).

Kinds of case, each one pass of

* ``step``    a whole decode step of a small model: metadata from the slot table, then for every layer
              q/k norm + rotary embedding + KV-store + decode attention;
* ``decode``  one layer of a decode step: KV-store of one new token per request, then attention;
* ``extend``  one layer of a prefill, chunked prefill or speculative-verify step: KV-store of the new
              tokens, then attention under one of the four masks;
* ``gdn``     one linear-attention layer: the gated delta rule over the new tokens (``single``: one
              token per request) with the recurrent state of every request updated in place.

Request lengths are uniform between the case's ``*_lo`` and ``*_hi``, drawn from its ``lens`` number, so
that a case is one set of shapes; the seed of ``prepare`` decides values, slots and page order.
"""
import math
import os
import random
import sys
from types import SimpleNamespace

import torch

# the package folder lies under the root this file is used from
sys.path.insert(1, os.path.abspath("mini-sglang-mlx_amd"))

from mini_sglang_amd import roofline  # noqa: E402
from mini_sglang_amd.attention import AttnBackend, GDNBackend  # noqa: E402
from mini_sglang_amd.kvcache import MambaStateConfig, MambaStatePool, MHAKVCache  # noqa: E402

PAGE = 16
GDN_DIM = 128
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16}


def _attn(name, kind, batch, heads, kv, ext=(1, 1), d=128, dtype="bf16", layers=1, window=0, cross=False, lens=1):
    """``kv``: tokens in the cache before this step (shortest, longest request); ``ext``: new ones."""
    case = {"kind": kind, "batch": batch, "n_q": heads[0], "n_kv": heads[1], "d": d, "dtype": dtype,
            "layers": layers, "kv_lo": kv[0], "kv_hi": kv[1], "ext_lo": ext[0], "ext_hi": ext[1],
            "window": window, "cross": cross, "lens": lens}
    return dict(case, name=name) if name else case


def _gdn(name, batch, ext, single, hk=16, hv=32, lens=1):
    case = {"kind": "gdn", "batch": batch, "hk": hk, "hv": hv, "ext_lo": ext[0], "ext_hi": ext[1],
            "single": single, "lens": lens}
    return dict(case, name=name) if name else case


def listed():
    return [
        # interactive use of a small model: four chats, every layer of one decode step
        _attn("step_small", "step", 4, (16, 8), (36, 1022), layers=28),
        # a loaded server in steady state: 64 requests of ordinary length
        _attn("decode_batch", "decode", 64, (32, 8), (1023, 8191)),
        # long documents: 16 requests of 32 K to 128 K tokens, 64 query heads
        _attn("decode_long", "decode", 16, (64, 8), (32767, 131071)),
        # the full-attention layer of a hybrid model: head_dim 256, few kv heads, half precision, short ragged chats
        _attn("decode_d256_half", "decode", 24, (16, 2), (127, 4095), d=256, dtype="f16"),
        # chunked prefill: 512 new tokens each on cached prefixes of very different length
        _attn("extend_chunks", "extend", 8, (32, 8), (0, 16384), ext=(512, 512)),
        # fresh prompts of odd lengths, nothing cached
        _attn("prompts_ragged", "extend", 6, (32, 8), (0, 0), ext=(237, 3333), lens=3),
        # one long conversation goes on: the launch is small for the chip
        _attn("extend_one_long", "extend", 1, (32, 8), (32768, 32768), ext=(509, 509)),
        # prefill of the head_dim 256 layer
        _attn("extend_d256", "extend", 4, (24, 4), (0, 8192), ext=(237, 2048), d=256),
        # speculative verify: eight draft tokens per request
        _attn("verify", "extend", 32, (32, 8), (2048, 8192), ext=(8, 8)),
        # the same on a sliding-window layer
        _attn("verify_window", "extend", 32, (32, 8), (2048, 8192), ext=(8, 8), window=1024),
        # linear-attention layer of a hybrid model, prefill of a few prompts
        _gdn("gdn_prefill", 4, (64, 4096), False, lens=8),
        # and its decode step
        _gdn("gdn_decode", 64, (1, 1), True),
    ]


def _log(rng, lo, hi):
    """An integer in [lo, hi], its logarithm uniform."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _cost(case):
    w = work(case)
    return w["bytes"] / 6e12 + w["flops"] / 1e15


def draw(rng):
    most = {}  # by family of kinds: the recurrence is a long chain for few bytes and operations
    for c in listed():
        most[c["kind"] == "gdn"] = max(_cost(c), most.get(c["kind"] == "gdn", 0.0))
    while True:
        kind, lens = rng.choice(("step", "decode", "decode", "extend", "extend", "verify", "gdn", "gdn")), rng.randrange(1 << 16)
        d = rng.choice((128, 128, 128, 256))
        heads = rng.choice(((16, 8), (32, 8), (64, 8)) if d == 128 else ((16, 2), (16, 4), (24, 4), (32, 2)))
        if kind == "step":
            top = _log(rng, 16, 2047)
            case = _attn("", "step", _log(rng, 1, 16), (16, 8), (_log(rng, 1, top), top), layers=28, lens=lens)
        elif kind == "decode":
            top = _log(rng, 64, 131071)
            case = _attn("", "decode", _log(rng, 1, 256), heads, (_log(rng, max(1, top // 16), top), top), d=d,
                         dtype=rng.choice(("bf16", "bf16", "f16")), lens=lens)
        elif kind == "extend":
            new, cached = _log(rng, 16, 4096), rng.choice((0, _log(rng, 64, 131072)))
            # most layers are causal; some models have sliding windows, drafts see both sides
            window, cross = rng.choice(((0, False),) * 5 + ((1024, False), (0, True), (1024, True)))
            case = _attn("", "extend", _log(rng, 1, 32), heads, (rng.randint(0, cached), cached), (_log(rng, 9, new) if new > 9 else new, new),
                         d=d, window=window, cross=cross, lens=lens)
        elif kind == "verify":
            n, top = rng.randint(2, 16), _log(rng, 256, 16384)
            case = _attn("", "extend", _log(rng, 1, 64), heads, (_log(rng, max(1, top // 16), top), top), (n, n), d=d,
                         window=rng.choice((0, 0, 1024)), lens=lens)
        elif rng.random() < 0.5:
            case = _gdn("", _log(rng, 1, 256), (1, 1), True, lens=lens)
        else:
            top = _log(rng, 8, 4000)
            case = _gdn("", _log(rng, 1, 16), (_log(rng, max(1, top // 64), top), top), False, lens=lens)
        if _cost(case) <= most[case["kind"] == "gdn"]:
            return case


def _lengths(case):
    r = random.Random(case["lens"])
    ext = [r.randint(case["ext_lo"], case["ext_hi"]) for _ in range(case["batch"])]
    kv = [r.randint(case["kv_lo"], case["kv_hi"]) for _ in range(case["batch"])] if "kv_lo" in case else []
    return ext, kv


def _attention_state(case, g, dev):
    ext, cached = _lengths(case)
    total = [c + e for c, e in zip(cached, ext)]
    n_q, n_kv, d, layers, dtype = case["n_q"], case["n_kv"], case["d"], case["layers"], DTYPES[case["dtype"]]

    # slots: pages in random order, half as many again as the requests fill
    pages = [-(-t // PAGE) for t in total]
    order = torch.randperm(int(1.5 * sum(pages)) + 1, generator=g, device=dev).to(torch.int32)
    table = torch.zeros((case["batch"] + 1, max(pages) * PAGE), dtype=torch.int32, device=dev)
    within, at = torch.arange(PAGE, dtype=torch.int32, device=dev), 0
    for b, n in enumerate(pages):
        table[b, :n * PAGE] = (order[at:at + n, None] * PAGE + within).view(-1)
        at += n
    cache = MHAKVCache(n_kv, layers, d, order.numel() * PAGE, dtype, device=dev)
    for layer in range(layers):
        cache.k_cache(layer).normal_(generator=g)
        cache.v_cache(layer).normal_(generator=g)
    reqs = [SimpleNamespace(table_idx=b, cached_len=c, device_len=t, extend_len=e) for b, (c, t, e) in enumerate(zip(cached, total, ext))]
    batch = SimpleNamespace(reqs=reqs, padded_reqs=reqs, is_prefill=case["kind"] == "extend", attn_metadata=None,
                            out_loc=torch.cat([table[b, c:t] for b, (c, t) in enumerate(zip(cached, total))]).contiguous())
    backend = AttnBackend(SimpleNamespace(head_dim=d), cache, table)
    if case["kind"] != "step":  # elsewhere the step's metadata is there when its layers run
        backend.prepare_metadata(batch)
    # every layer's projections: heads of q, k and v side by side, as one matrix product leaves them
    qkv = torch.empty((layers, sum(ext), n_q + 2 * n_kv, d), dtype=dtype, device=dev).normal_(generator=g)
    parts = [(x[:, :n_q], x[:, n_q:n_q + n_kv], x[:, n_q + n_kv:]) for x in qkv]
    if case["kind"] != "step":  # norm and rotary embedding have left q contiguous
        parts = [(q.contiguous(), k.contiguous(), v) for q, k, v in parts]
    norms = (1 + 0.1 * torch.randn((2, layers, d), generator=g, device=dev)).to(dtype)
    return SimpleNamespace(case=case, backend=backend, cache=cache, batch=batch, parts=parts, norms=norms)


def _gdn_state(case, g, dev):
    ext, _ = _lengths(case)
    n, hk, hv, d = sum(ext), case["hk"], case["hv"], GDN_DIM
    pool = MambaStatePool(MambaStateConfig(num_slots=case["batch"], num_layers=1, conv_shapes=[[(3, (2 * hk + hv) * d)]],
                                           temporal_shapes=[(hv, d, d)]), device=dev)
    pool.temporal_state(0).normal_(std=0.1, generator=g)
    unit = lambda t: t / t.norm(dim=-1, keepdim=True)  # noqa: E731
    rand = lambda *s: torch.randn(s, generator=g, device=dev)  # noqa: E731
    q, k = (unit(rand(n, hk, d)) * d ** -0.5).bfloat16(), unit(rand(n, hk, d)).bfloat16()
    # heads forget at very different rates: from thousands of tokens to less than one
    rate = torch.exp(torch.rand(hv, generator=g, device=dev) * math.log(400.0) + math.log(0.01))
    decay = torch.exp(-rate * torch.nn.functional.softplus(rand(n, hv))).bfloat16()
    slots = (torch.randperm(case["batch"], generator=g, device=dev) + 1).tolist()
    batch = SimpleNamespace(reqs=[SimpleNamespace(mamba_slot=s, extend_len=e) for s, e in zip(slots, ext)],
                            is_decode=case["single"], mamba_slot_ids=None, mamba_prefill_indptr=None)
    backend = GDNBackend(pool)
    backend.prepare_batch(batch)
    return SimpleNamespace(case=case, backend=backend, pool=pool, batch=batch,
                           inputs=(q, k, rand(n, hv, d).bfloat16(), decay, torch.sigmoid(rand(n, hv)).bfloat16()))


def prepare(case, seed):
    dev = torch.device("cuda", torch.cuda.current_device())
    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    return (_gdn_state if case["kind"] == "gdn" else _attention_state)(case, g, dev)


def run(state):
    case, backend, batch = state.case, state.backend, state.batch
    if case["kind"] == "gdn":
        return backend.forward(*state.inputs, 0, batch), state.pool.temporal_state(0)
    if case["kind"] == "step":
        backend.prepare_metadata(batch)
        out = [backend.forward_fused_norm_rope(q, k, v, state.norms[0, layer], state.norms[1, layer], layer, batch,
                                               rms_norm_eps=1e-6, rope_base=1e6)
               for layer, (q, k, v) in enumerate(state.parts)]
    else:
        q, k, v = state.parts[0]
        out = [backend.forward(q, k, v, 0, batch, is_cross_attention=case["cross"], sliding_window_size=case["window"])]
    return out + [state.cache.k_cache(layer) for layer in (0, case["layers"] - 1)] + [state.cache.v_cache(layer) for layer in (0, case["layers"] - 1)]


def work(case):
    ext, cached = _lengths(case)
    n = sum(ext)
    if case["kind"] == "gdn":
        hk, hv, d = case["hk"], case["hv"], GDN_DIM
        state = 2 * case["batch"] * hv * d * d * 4
        # per token and value head: decay, state times key, rank-one update, state times query
        return {"bytes": state + n * (2 * hk * d * 2 + 2 * hv * d * 2 + 2 * hv * 2), "flops": n * hv * 7 * d * d}
    total = [c + e for c, e in zip(cached, ext)]
    args = (cached, ext, total, case["n_q"])
    mask = (case["cross"], case["window"])
    one = roofline.attention_bytes(*args, case["n_kv"], case["d"], *mask)
    new = roofline.store_bytes(n, case["n_kv"], case["d"])
    layers = case["layers"]
    meta = 8 * sum(total) if case["kind"] == "step" else 0
    return {"bytes": layers * (one + new) + meta, "flops": layers * _flops(cached, ext, case)}


def _flops(cached, ext, case):
    """4 d per visible (query, key) pair and query head, in closed form for every query of a request."""
    pairs, w = 0, case["window"]
    for c, e in zip(cached, ext):
        if case["cross"]:
            seen = e * (c + e)
        else:
            seen = e * c + e * (e + 1) // 2
        if w:  # less what lies before the window: key j of query i where j <= c + i - w
            first = max(0, w - c)  # the first query with such keys
            m = max(0, e - first)
            seen -= m * (c + first - w) + m * (m + 1) // 2
        pairs += seen
    return 4 * case["d"] * case["n_q"] * pairs


def tolerance(case):
    """bf16 results with fp32 sums: a bf16 step is 2^-8 of the value, softmax weights are bf16 too.
    The recurrence is fp32 throughout, only its result is rounded."""
    if case["kind"] == "gdn":
        return {"rel": 3e-3, "max": 2e-2}
    return {"rel": 1e-2, "max": 0.1}
