"""Shares: the arithmetic on the way to a workgroup's share, where its terms are no powers of two (head groups, groups of q
heads, share lengths) and where a request ends beside a share's end, against the CPU oracle."""
import pytest
import torch

import oracle
from mini_sglang_amd.workloads import build_workload
from mini_sglang_amd_kernel import _lib, paged_decode_attention, paged_prefill_attention

pytestmark = pytest.mark.gpu


def _close(got, want):  # bf16 results of N(0, 1) inputs: half a bf16 step of values up to 4, and the weights' rounding
    diff = (got.float().cpu() - want).abs()
    assert float(diff.max()) <= 2e-2 and float(diff.mean()) <= 2e-3, (float(diff.max()), float(diff.mean()))


@pytest.mark.parametrize("n_q,n_kv,d", [(15, 3, 128), (42, 6, 128), (12, 12, 128), (22, 2, 128), (15, 5, 256), (39, 3, 256)])
@pytest.mark.parametrize("share,heads", [(0, 0), (33, 1), (100, 1), (341, 2), (96, 4)])
def test_decode(gpu, tuning, n_q, n_kv, d, share, heads):
    lens = [1, 32, 33, 34, 99, 100, 101, 340, 341, 342, 700, 0, 1023]
    wl = build_workload("cuts", "decode", seed=n_q + share, n_q=n_q, n_kv=n_kv, head_dim=d, kv_lens=lens)
    want = oracle.paged_decode_attention(wl.q, wl.k_cache, wl.v_cache, wl.kv_indptr, wl.kv_indices, wl.num_kv_splits,
                                         wl.sm_scale, wl.max_kv_splits, return_f32=True)[1]
    g = wl.to(gpu)
    tuning(_lib.TUNE_SHARES, share | heads << 20)
    print(f"share cuts decode {n_q}/{n_kv} d{d} cut {share} x {heads}", flush=True)
    _close(paged_decode_attention(g.q, g.k_cache, g.v_cache, g.kv_indptr, g.kv_indices, g.num_kv_splits, g.sm_scale, 32), want)


@pytest.mark.parametrize("n_q,n_kv,q_len", [(15, 3, 3), (42, 6, 6), (18, 2, 5), (7, 1, 2)])
@pytest.mark.parametrize("share", [0, 100, 341])
@pytest.mark.parametrize("cross,window", [(False, 0), (True, 0), (False, 90)])
def test_short_query_blocks(gpu, tuning, n_q, n_kv, q_len, share, cross, window):
    kv = [q_len, 100, 101, 341, 342, 1030]
    wl = build_workload("cuts", "prefill", seed=n_q + q_len, n_q=n_q, n_kv=n_kv, kv_lens=kv, extend_lens=[q_len, 1, q_len, q_len - 1, q_len, q_len],
                        is_cross_attention=cross, sliding_window_size=window)
    args = lambda w: (w.q, w.k_cache, w.v_cache, w.qo_indptr, w.kv_indptr, w.kv_indices, w.prefix_lens, w.sm_scale, q_len)
    mask = dict(is_cross_attention=cross, sliding_window_size=window)
    want = oracle.paged_prefill_attention(*args(wl), **mask, return_f32=True)[1]
    g = wl.to(gpu)
    tuning(_lib.TUNE_SHARES, share | 1 << 20 if share else 0)
    print(f"share cuts verify {n_q}/{n_kv} q{q_len} {mask} cut {share}", flush=True)
    _close(paged_prefill_attention(*args(g), **mask), want)


@pytest.mark.parametrize("lens,n_q,n_kv", [([20001], 16, 2), ([1907, 812], 24, 4), ([129], 32, 2), ([7000, 1, 255, 4100], 16, 2), ([5200], 16, 4)])
def test_few_wide_heads(gpu, lens, n_q, n_kv):
    """As many shares to a request as fit the chip: up to 53 here, put together 16 at a time."""
    wl = build_workload("wide heads", "decode", seed=len(lens), n_q=n_q, n_kv=n_kv, head_dim=256, kv_lens=lens)
    want = oracle.paged_decode_attention(wl.q, wl.k_cache, wl.v_cache, wl.kv_indptr, wl.kv_indices, wl.num_kv_splits,
                                         wl.sm_scale, wl.max_kv_splits, return_f32=True)[1]
    g = wl.to(gpu)
    print(f"wide heads {lens} {n_q}/{n_kv}", flush=True)
    for _ in range(2):
        _close(paged_decode_attention(g.q, g.k_cache, g.v_cache, g.kv_indptr, g.kv_indices, g.num_kv_splits, g.sm_scale, 32), want)


def test_a_window_of_very_many_requests(gpu):
    """17000 requests, 8 queries each: partials of more than 2 GiB in all, one share to a request."""
    few, times, q_len, window = 34, 500, 8, 200
    kv = [240 + 3 * i for i in range(few)]
    wl = build_workload("many windows", "prefill", seed=34, n_q=32, n_kv=8, kv_lens=kv, extend_lens=[q_len] * few, sliding_window_size=window)
    want = oracle.paged_prefill_attention(wl.q, wl.k_cache, wl.v_cache, wl.qo_indptr, wl.kv_indptr, wl.kv_indices, wl.prefix_lens, wl.sm_scale,
                                          q_len, sliding_window_size=window, return_f32=True)[1]
    g = wl.to(gpu)
    indptr = lambda n: torch.cat([torch.zeros(1, dtype=torch.int64), torch.tensor(n * times).cumsum(0)]).int().to(gpu)  # noqa: E731
    print("share cuts: 17000 windows", flush=True)
    got = paged_prefill_attention(g.q.repeat(times, 1, 1), g.k_cache, g.v_cache, indptr([q_len] * few), indptr(kv), g.kv_indices.repeat(times),
                                  g.prefix_lens.repeat(times), g.sm_scale, q_len, sliding_window_size=window).view(times, *want.shape)
    _close(got[0], want)
    _close(got[-1], want)
    assert bool((got == got[0]).all())  # every request its own bits, wherever it stands
