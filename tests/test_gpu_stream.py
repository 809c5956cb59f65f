"""Decode and verify with keys and values read past the caches: the same bits as read the plain way, at lengths around the
pieces that the lanes exchange (8 and 16 rows, tiles of 32 and 64 keys), in segments and in shares, with the new tokens' rows
stored inside and masks.  The plain way is checked against the CPU oracle elsewhere; here one launch beyond the line is too."""
import pytest
import torch

import oracle
from mini_sglang_amd.workloads import build_workload
from mini_sglang_amd_kernel import _lib, decode_step, paged_decode_attention, paged_prefill_attention

pytestmark = pytest.mark.gpu


def _both(tuning, launch):
    out = []
    for kib in (-1, 1):
        tuning(_lib.TUNE_STREAM, kib)
        out.append(launch())
    torch.cuda.synchronize()
    return out


def _same(a, b):
    return torch.equal(a.view(torch.int16), b.view(torch.int16))


LENS = [[1], [7, 8, 9, 15, 16, 17, 0, 23, 24, 25, 31, 32, 33], [63, 64, 65, 71, 72, 73, 95, 96, 97, 127, 128, 129], [1500, 2, 700]]


@pytest.mark.parametrize("lens", LENS)
@pytest.mark.parametrize("n_q,n_kv,d", [(16, 8, 128), (8, 1, 128), (32, 2, 256), (24, 4, 256)])
@pytest.mark.parametrize("shares", [-1, 64 | 1 << 20])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_decode(gpu, tuning, lens, n_q, n_kv, d, shares, dtype):
    g = build_workload("stream", "decode", seed=len(lens) + d, n_q=n_q, n_kv=n_kv, head_dim=d, kv_lens=lens).to(gpu)
    q, kc, vc = (t.to(dtype) for t in (g.q, g.k_cache, g.v_cache))
    tuning(_lib.TUNE_SHARES, shares)
    print(f"stream decode {lens[:4]} {n_q}/{n_kv} d{d} {dtype} shares {shares}", flush=True)
    plain, stream = _both(tuning, lambda: paged_decode_attention(q, kc, vc, g.kv_indptr, g.kv_indices, g.num_kv_splits, g.sm_scale, 32))
    assert bool(plain.isfinite().all()) and _same(plain, stream)


@pytest.mark.parametrize("q_len,n_q,n_kv,d", [(4, 32, 8, 128), (8, 32, 8, 128), (12, 32, 8, 128), (5, 64, 8, 128), (4, 16, 4, 256), (2, 24, 4, 256),
                                                (16, 32, 8, 128), (6, 24, 4, 256)])
@pytest.mark.parametrize("shares", [-1, 128 | 1 << 20])
@pytest.mark.parametrize("cross,window", [(False, 0), (True, 0), (False, 100), (True, 100)])
def test_verify(gpu, tuning, q_len, n_q, n_kv, d, shares, cross, window):
    lens = [q_len, q_len + 7, 16 + q_len, 65, 300, 1030]
    g = build_workload("stream", "prefill", seed=q_len, n_q=n_q, n_kv=n_kv, head_dim=d, kv_lens=lens,
                       extend_lens=[q_len, 1, q_len, q_len - 1, q_len, q_len], is_cross_attention=cross, sliding_window_size=window).to(gpu)
    tuning(_lib.TUNE_SHARES, shares)
    print(f"stream verify q{q_len} d{d} cross {cross} window {window} shares {shares}", flush=True)
    plain, stream = _both(tuning, lambda: paged_prefill_attention(
        g.q, g.k_cache, g.v_cache, g.qo_indptr, g.kv_indptr, g.kv_indices, g.prefix_lens, g.sm_scale, q_len,
        is_cross_attention=cross, sliding_window_size=window))
    assert bool(plain.isfinite().all()) and _same(plain, stream)


@pytest.mark.parametrize("d", [128, 256])
@pytest.mark.parametrize("shares", [-1, 64 | 1 << 20])
@pytest.mark.parametrize("norm", [False, True])
def test_decode_step(gpu, tuning, d, shares, norm):
    if norm and shares < 0:
        pytest.skip("norm weights: shares only")
    lens = [1, 8, 9, 16, 17, 33, 64, 65, 200, 1100]
    g = build_workload("stream", "decode", seed=d, n_q=16, n_kv=4, head_dim=d, kv_lens=lens).to(gpu)
    r = torch.Generator(device=gpu)
    r.manual_seed(d)
    k, v = (torch.randn((len(lens), 4, d), generator=r, device=gpu).bfloat16() for _ in range(2))
    loc = g.kv_indices[g.kv_indptr[1:].long() - 1].contiguous()
    w = (1 + 0.2 * torch.randn((2, d), generator=r, device=gpu)).bfloat16()
    more = dict(q_weight=w[0], k_weight=w[1], positions=(g.kv_indptr[1:] - g.kv_indptr[:-1] - 1).int(), eps=1e-6, rope_base=1e6) if norm else {}
    tuning(_lib.TUNE_SHARES, shares)
    if shares < 0:
        tuning(_lib.TUNE_SEGMENTS, 5)
        tuning(_lib.TUNE_MIN_SEGMENT, 64)

    def step():
        kc, vc = g.k_cache.clone(), g.v_cache.clone()
        out = decode_step(g.q, k, v, loc, kc, vc, g.kv_indptr, g.kv_indices, g.num_kv_splits, sm_scale=g.sm_scale, **more)
        assert out is not None
        return out, kc, vc

    print(f"stream decode step d{d} shares {shares} norm {norm}", flush=True)
    plain, stream = _both(tuning, step)
    assert all(_same(a, b) for a, b in zip(plain, stream))


@pytest.mark.parametrize("d", [128, 256])
def test_beyond_the_line(gpu, d):
    """From 80 MiB of keys and values on by itself: 90 MiB against the oracle."""
    n_kv = 8 * 128 // d
    lens = [22000, 513, 527]
    wl = build_workload("stream", "decode", seed=d, n_q=2 * n_kv, n_kv=n_kv, head_dim=d, kv_lens=lens, pool_factor=1.0)
    want = oracle.paged_decode_attention(wl.q, wl.k_cache, wl.v_cache, wl.kv_indptr, wl.kv_indices, wl.num_kv_splits, wl.sm_scale,
                                         wl.max_kv_splits, return_f32=True)[1]
    g = wl.to(gpu)
    print(f"stream beyond the line d{d}", flush=True)
    diff = (paged_decode_attention(g.q, g.k_cache, g.v_cache, g.kv_indptr, g.kv_indices, g.num_kv_splits, g.sm_scale, 32).float().cpu() - want).abs()
    assert float(diff.max()) <= 2e-2 and float(diff.mean()) <= 2e-3  # as for the plain way


def _common_prefix(gpu, batch, common, own, heads, d, ext, dtype=torch.bfloat16):
    """Requests whose first `common` keys are in the same slots, and the rest in slots of their own."""
    n_q, n_kv = heads
    g = torch.Generator(device=gpu)
    g.manual_seed(batch + common)
    slots = torch.randperm(common + own * batch, generator=g, device=gpu).int()
    idx = torch.cat([torch.cat([slots[:common], slots[common + b * own:common + (b + 1) * own]]) for b in range(batch)])
    rand = lambda *s: torch.randn(s, generator=g, device=gpu).to(dtype)  # noqa: E731
    kc, vc, q = rand(slots.numel(), n_kv, d), rand(slots.numel(), n_kv, d), rand(batch * ext, n_q, d)
    indptr = torch.arange(batch + 1, dtype=torch.int32, device=gpu) * (common + own)
    if ext == 1:
        splits = torch.ones(batch, dtype=torch.int32, device=gpu)
        return lambda: paged_decode_attention(q, kc, vc, indptr, idx, splits, d ** -0.5, 32)
    qo = torch.arange(batch + 1, dtype=torch.int32, device=gpu) * ext
    prefix = torch.full((batch,), common + own - ext, dtype=torch.int32, device=gpu)
    return lambda: paged_prefill_attention(q, kc, vc, qo, indptr, idx, prefix, d ** -0.5, ext)


# no keys of a request's own before the first tile, in the middle of one, and none but its own behind the first; more requests than lanes
@pytest.mark.parametrize("batch,common,own", [(1, 100, 30), (2, 64, 40), (5, 1000, 33), (3, 1, 700), (70, 90, 17), (130, 40, 9)])
@pytest.mark.parametrize("heads,d,ext", [((16, 8), 128, 1), ((32, 8), 128, 8), ((8, 1), 256, 1), ((16, 4), 256, 6)])
@pytest.mark.parametrize("shares", [-1, 64 | 1 << 20])
def test_common_prefixes(gpu, tuning, batch, common, own, heads, d, ext, shares):
    tuning(_lib.TUNE_SHARES, shares)
    if d == 256 and ext > 1 and shares < 0:
        tuning(_lib.TUNE_SMALLQ_MAXCOLS, 64)
    print(f"common prefix {batch} x {common} + {own} {heads} d{d} x {ext} shares {shares}", flush=True)
    plain, stream = _both(tuning, _common_prefix(gpu, batch, common, own, heads, d, ext))
    assert bool(plain.isfinite().all()) and _same(plain, stream)


def test_common_prefixes_come_from_the_caches(gpu, tuning):
    """What one request has read, the others find: 80 MiB in all, of which 64 requests read 1088.  (Past the caches 1.3-1.4 times the time.)"""
    launch = _common_prefix(gpu, 64, 4096, 256, (32, 8), 128, 1)

    def us():
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        for _ in range(20):
            launch()
        b.record()
        b.synchronize()
        return a.elapsed_time(b) * 50

    times = {-1: [], 0: []}
    for _ in range(5):
        for kib in times:
            tuning(_lib.TUNE_STREAM, kib)
            launch()
            times[kib].append(us())
    assert min(times[0]) <= 1.15 * min(times[-1]), times
