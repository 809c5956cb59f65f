"""Requests that list the slots of other requests' new tokens, or one of their own twice: without ``own_slots`` every row is
in the pool before the attention starts, so a step is exactly the store and the attention called one after the other."""
from types import SimpleNamespace

import pytest
import torch

from mini_sglang_amd.attention import AttnBackend
from mini_sglang_amd.kvcache import MHAKVCache
from mini_sglang_amd_kernel import extend_step, paged_decode_attention, paged_prefill_attention, qk_norm_rope_store, store_kv_cache

pytestmark = pytest.mark.gpu

N_Q, N_KV = 16, 8


def _step(gpu, d, cached, ext):
    """Requests whose rows of the slot table share what they have in common: request b > 0 has the new slots of request 0
    among its cached ones, and the last request lists its own new slot in front as well."""
    total = [c + e for c, e in zip(cached, ext)]
    table = (torch.randperm(len(total) * 1200, generator=torch.Generator().manual_seed(sum(total)))[:len(total) * 1100]
             .reshape(len(total), 1100).to(torch.int32))
    for b in range(1, len(total)):
        n = min(ext[0], cached[b])
        table[b, cached[b] - n:cached[b]] = table[0, cached[0]:cached[0] + n]
    table[-1, 0] = table[-1, total[-1] - 1]
    table = table.to(gpu)
    cache = MHAKVCache(N_KV, 1, d, len(total) * 1200, torch.bfloat16, device=gpu)
    g = torch.Generator(device=gpu)
    g.manual_seed(d)
    out_loc = torch.cat([table[b, c:t] for b, (c, t) in enumerate(zip(cached, total))]).contiguous()
    for pool in (cache.k_cache(0), cache.v_cache(0)):
        pool.normal_(generator=g)
        pool[out_loc.long()] = float("nan")  # what a row read too early would show
    reqs = [SimpleNamespace(table_idx=b, cached_len=c, device_len=t, extend_len=e) for b, (c, t, e) in enumerate(zip(cached, total, ext))]
    batch = SimpleNamespace(padded_reqs=reqs, attn_metadata=None, out_loc=out_loc, own_slots=False)
    q, k, v = (torch.randn((sum(ext), n, d), generator=g, device=gpu).bfloat16() for n in (N_Q, N_KV, N_KV))
    weights = [(1 + 0.1 * torch.randn(d, generator=g, device=gpu)).bfloat16() for _ in range(2)]
    return AttnBackend(SimpleNamespace(head_dim=d), cache, table), cache, batch, (q, k, v), weights


def _same(a, b):
    assert torch.equal(a.view(torch.int16), b.view(torch.int16))


@pytest.mark.parametrize("d", [128, 256])
@pytest.mark.parametrize("cached", [[4, 40, 700, 33], [0, 1, 64, 1000], [1000] * 12])
@pytest.mark.parametrize("norm", [False, True])
def test_decode(gpu, d, cached, norm):
    backend, cache, batch, (q, k, v), (qw, kw) = _step(gpu, d, cached, [1] * len(cached))
    batch.is_prefill = False
    backend.prepare_metadata(batch)
    m = batch.attn_metadata
    kc, vc = cache.k_cache(0).clone(), cache.v_cache(0).clone()
    print(f"decode with shared slots d{d} {cached[:4]} norm={norm}", flush=True)
    if norm:
        got = backend.forward_fused_norm_rope(q, k, v, qw, kw, 0, batch, rms_norm_eps=1e-6, rope_base=1e6)
        q = qk_norm_rope_store(q, k, v, qw, kw, m.positions, batch.out_loc, kc, vc, eps=1e-6, rope_base=1e6)
    else:
        got = backend.forward(q, k, v, 0, batch)
        store_kv_cache(kc, vc, batch.out_loc, k, v)
    want = paged_decode_attention(q, kc, vc, m.kv_indptr, m.kv_indices, m.num_kv_splits, backend.sm_scale, m.max_kv_splits)
    assert bool(torch.isfinite(got).all())
    _same(got, want)
    _same(cache.k_cache(0), kc)
    _same(cache.v_cache(0), vc)


@pytest.mark.parametrize("d", [128, 256])
@pytest.mark.parametrize("cached,ext", [([30, 200, 8, 64], [8] * 4), ([0, 90, 700], [40, 60, 9]), ([0, 64, 600], [300, 200, 77])])
@pytest.mark.parametrize("window", [0, 50])
def test_extend(gpu, d, cached, ext, window):
    backend, cache, batch, (q, k, v), _ = _step(gpu, d, cached, ext)
    batch.is_prefill = True
    backend.prepare_metadata(batch)
    m = batch.attn_metadata
    pools = [(cache.k_cache(0).clone(), cache.v_cache(0).clone()) for _ in range(2)]
    print(f"extend with shared slots d{d} {cached} + {ext} window={window}", flush=True)
    got = backend.forward(q, k, v, 0, batch, sliding_window_size=window)
    by_hand = extend_step(q, k, v, batch.out_loc, *pools[0], m.qo_indptr, m.kv_indptr, m.kv_indices, m.prefix_lens,
                          sm_scale=backend.sm_scale, max_len_extend=m.max_len_extend, sliding_window_size=window, own_slots=False)
    store_kv_cache(*pools[1], batch.out_loc, k, v)
    want = paged_prefill_attention(q, *pools[1], m.qo_indptr, m.kv_indptr, m.kv_indices, m.prefix_lens, backend.sm_scale,
                                   m.max_len_extend, sliding_window_size=window)
    assert bool(torch.isfinite(got).all())
    _same(got, want)
    _same(by_hand, want)
    for pool, ours in ((pools[1][0], cache.k_cache(0)), (pools[1][1], cache.v_cache(0))):
        _same(ours, pool)
