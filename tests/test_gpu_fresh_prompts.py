"""Prompts with nothing cached whose rows the attention launch stores itself: output and pool are, bit for bit, those of the store and
the attention called one after the other.  Groups whose blocks' own tokens are a tile, part of one, or several; last blocks that are
not full; windows and cross attention; rows that belong to no request; rows whose slots are not the ones listed; requests that see no key."""
import numpy as np
import pytest
import torch

from mini_sglang_amd_kernel import _lib, extend_step, paged_prefill_attention, store_kv_cache

pytestmark = pytest.mark.gpu

D = 128


def _one_launch(ext, n_q, n_kv, cross, window):
    """Whether the call goes in one launch at all (some workspace is wanted then)."""
    return _lib.load().msgl_extend_step_workspace_bytes(len(ext), sum(ext), sum(ext), n_q, n_kv, D, max(ext), int(cross), window) > 0


def _check(gpu, ext, heads, window=0, cross=False, change=None, front=0, strided=False, pad=0, hidden=(), keyless=False):
    n_q, n_kv = heads
    g = torch.Generator(device=gpu)
    g.manual_seed(sum(ext) + n_q)
    total = sum(ext)
    slots = 2 * total + 5
    ids = torch.randperm(slots, generator=g, device=gpu)[:total].to(torch.int32)
    out_loc = ids.clone()
    rand = lambda *s: torch.randn(s, generator=g, device=gpu).bfloat16()  # noqa: E731
    q = rand(total, n_q, D)
    kv = rand(total, 2 * n_kv, D) if strided else None
    k, v = (kv[:, :n_kv], kv[:, n_kv:]) if strided else (rand(total, n_kv, D), rand(total, n_kv, D))
    # (`pad`: heads between a slot's rows and the next slot's; with enough of them offsets have 64 bits)
    pools = [torch.empty((slots, n_kv + pad, D), dtype=torch.bfloat16, device=gpu)[:, :n_kv].copy_(rand(slots, n_kv, D)) for _ in range(2)]
    starts = np.cumsum([front] + list(ext[:-1]) + [ext[-1] - front])  # with rows in front of the first request, its last one is shorter
    ip = torch.tensor(starts, dtype=torch.int32, device=gpu)
    prefix = torch.zeros(len(ext), dtype=torch.int32, device=gpu)
    kv_ip = ip
    for b in hidden:  # the window lies behind all of the request's keys
        prefix[b] = 5000
    if keyless:  # the first request lists no keys, the second as many more, which are in the pool
        kv_ip = ip.clone()
        kv_ip[1] = 0
        prefix[1] = ext[0]
        ids[:ext[0]] = torch.arange(slots, device=gpu, dtype=torch.int32)[~torch.isin(torch.arange(slots, device=gpu), out_loc.long())][:ext[0]]
    if change == "slot":  # a key of a request is a row of the pool that no row goes to
        ids[total // 2] = next(s for s in range(slots) if not bool((out_loc == s).any()))
    elif change == "outside":  # a row that goes nowhere
        out_loc[total // 3] = -1
    assert _one_launch(ext, n_q, n_kv, cross, window)
    print(f"fresh {ext[:6]} heads {heads} window {window} cross {cross} {change} front {front} hidden {hidden} {keyless}", flush=True)
    want_pools = [p.clone() for p in pools]
    store_kv_cache(*want_pools, out_loc, k, v)
    want = paged_prefill_attention(q, *want_pools, ip, kv_ip, ids, prefix, sm_scale=D ** -0.5, max_len_extend=max(ext),
                                   is_cross_attention=cross, sliding_window_size=window)
    got = extend_step(q, k, v, out_loc, *pools, ip, kv_ip, ids, prefix, sm_scale=D ** -0.5, max_len_extend=max(ext),
                      is_cross_attention=cross, sliding_window_size=window)
    torch.cuda.synchronize()
    for a, b in zip(pools, want_pools):
        assert torch.equal(a.view(torch.int16), b.view(torch.int16))
    lo, hi = int(starts[0]), int(starts[-1])
    assert torch.equal(got[lo:hi].view(torch.int16), want[lo:hi].view(torch.int16))


@pytest.mark.parametrize("heads", [(8, 8), (16, 8), (24, 8), (32, 8), (64, 8), (32, 4), (16, 2), (8, 1)])
@pytest.mark.parametrize("ext", [[1500, 1, 1399, 63, 1300, 64, 65, 700, 3301], [2100] * 4])
def test_as_store_and_attention(gpu, heads, ext):
    _check(gpu, ext, heads)


@pytest.mark.parametrize("window,cross", [(1, False), (70, False), (1024, False), (0, True), (300, True)])
@pytest.mark.parametrize("heads", [(16, 8), (32, 8)])
def test_masks(gpu, heads, window, cross):
    _check(gpu, [1700, 129, 1999, 901], heads, window, cross)


@pytest.mark.parametrize("change", [None, "slot", "outside"])
@pytest.mark.parametrize("front", [0, 7])
def test_rows_that_are_not_the_keys(gpu, change, front):
    _check(gpu, [1300, 900, 64, 1100], (32, 8), change=change, front=front, strided=change is None)


@pytest.mark.parametrize("heads", [(32, 8), (16, 2)])
@pytest.mark.parametrize("hidden", [(0,), (1, 3), (0, 1, 2, 3)])
def test_requests_whose_keys_the_window_hides(gpu, hidden, heads):
    _check(gpu, [1300] * 4, heads, window=1024, hidden=hidden)
    _check(gpu, [1700, 64, 1999, 901], heads, window=300, hidden=hidden)


@pytest.mark.parametrize("heads", [(32, 8), (16, 2)])
def test_request_without_keys(gpu, heads):
    _check(gpu, [700, 1300, 900, 1500], heads, keyless=True)


def test_wide_pool(gpu):
    _check(gpu, [1300, 900, 64, 1100], (32, 8), pad=2500)
    _check(gpu, [1300, 900, 64, 1100], (32, 8), pad=2500, change="slot")


@pytest.mark.parametrize("batch,length,heads", [(4, 1030, (32, 8)), (3, 2049, (16, 8)), (1, 4100, (32, 4))])
def test_prompts_of_one_length(gpu, batch, length, heads):
    """Their blocks go in order of length as those of others do; against attention in fp32."""
    n_q, n_kv = heads
    g = torch.Generator(device=gpu)
    g.manual_seed(length)
    rand = lambda *s: torch.randn(s, generator=g, device=gpu).bfloat16()  # noqa: E731
    total = batch * length
    q, k, v = rand(total, n_q, D), rand(total, n_kv, D), rand(total, n_kv, D)
    ids = torch.randperm(total + 3, generator=g, device=gpu)[:total].to(torch.int32)
    pools = [torch.zeros((total + 3, n_kv, D), dtype=torch.bfloat16, device=gpu) for _ in range(2)]
    for pool, rows in zip(pools, (k, v)):
        pool[ids.long()] = rows
    ip = torch.arange(0, total + 1, length, dtype=torch.int32, device=gpu)
    print(f"prompts of one length {batch} x {length} {heads}", flush=True)
    got = paged_prefill_attention(q, *pools, ip, ip, ids, torch.zeros(batch, dtype=torch.int32, device=gpu), sm_scale=D ** -0.5, max_len_extend=length)
    mask = torch.full((length, length), float("-inf"), device=gpu).triu(1)
    for b in range(batch):
        rows = slice(b * length, (b + 1) * length)
        for h in range(n_q):
            at = h // (n_q // n_kv)
            p = torch.softmax(q[rows, h].float() @ k[rows, at].float().t() * D ** -0.5 + mask, dim=-1)
            want = p @ v[rows, at].float()
            # weights and results are bf16: 2^-8 of a value below 5, twice
            assert (got[rows, h].float() - want).abs().max() <= 2e-2
