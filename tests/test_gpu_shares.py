"""Decode and short query blocks as shares of each request's keys, one launch: against the CPU oracle
at the sizes where the cut can go wrong (one share, two, more shares than are loaded together, requests
without keys, more than one wave of requests, every number of kv heads per workgroup), for default
and forced cuts, and replayed from a graph."""
import pytest
import torch

import oracle
from mini_sglang_amd.workloads import build_workload
from mini_sglang_amd_kernel import _lib, paged_decode_attention, paged_prefill_attention

pytestmark = pytest.mark.gpu


def _close(got, want, what):
    diff = (got.float().cpu() - want).abs()
    assert float(diff.max()) <= 2e-2 and float(diff.mean()) <= 2e-3, (what, float(diff.max()), float(diff.mean()))


def _decode(g):
    return paged_decode_attention(g.q, g.k_cache, g.v_cache, g.kv_indptr, g.kv_indices, g.num_kv_splits, g.sm_scale, 32)


DECODE = [  # kv lengths, q heads, kv heads, head_dim, share_len, kv heads per workgroup (0: the default cut)
    ([1], 16, 8, 128, 0, 0),
    ([37, 128, 500, 1023], 16, 8, 128, 0, 0),
    ([31, 32, 33, 127, 128, 129, 0, 257], 32, 8, 128, 128, 1),
    ([2100, 5], 64, 4, 128, 128, 1),     # 17 shares, 16 columns
    ([2100, 5, 64], 32, 8, 128, 64, 8),  # a wave per share and head
    ([700] * 3, 8, 2, 128, 256, 2),
    ([1 + i % 90 for i in range(150)], 16, 8, 128, 0, 0),
    ([600, 0, 1, 255, 256, 257], 16, 2, 256, 0, 0),
    ([1500, 40], 24, 4, 256, 64, 4),
]


@pytest.mark.parametrize("lens,n_q,n_kv,d,share,heads", DECODE)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_decode(gpu, tuning, lens, n_q, n_kv, d, share, heads, dtype):
    wl = build_workload("shares", "decode", seed=len(lens) + d, n_q=n_q, n_kv=n_kv, head_dim=d, kv_lens=lens)
    for name in ("q", "k_cache", "v_cache"):
        setattr(wl, name, getattr(wl, name).to(dtype))
    want = oracle.paged_decode_attention(wl.q.bfloat16() if dtype == torch.bfloat16 else wl.q.float().bfloat16(),
                                         wl.k_cache.bfloat16(), wl.v_cache.bfloat16(), wl.kv_indptr, wl.kv_indices,
                                         wl.num_kv_splits, wl.sm_scale, wl.max_kv_splits, return_f32=True)[1]
    g = wl.to(gpu)
    tuning(_lib.TUNE_SHARES, share | heads << 20)
    print(f"shares decode {lens[:4]} {n_q}/{n_kv} d{d} {dtype} cut {share} x {heads}", flush=True)
    first = _decode(g)
    _close(first, want, "decode")
    for _ in range(3):  # the count words are as good as new after every launch
        assert torch.equal(_decode(g), first)


@pytest.mark.parametrize("q_len,n_q,n_kv,d,share", [(2, 16, 8, 128, 128), (8, 32, 8, 128, 256), (11, 32, 8, 128, 512),
                                                    (3, 16, 4, 256, 128)])
@pytest.mark.parametrize("cross,window", [(False, 0), (True, 0), (False, 200), (True, 200)])
def test_short_query_blocks(gpu, tuning, q_len, n_q, n_kv, d, share, cross, window):
    kv = [q_len, q_len + 1, 300, 1030, 31 + q_len]
    wl = build_workload("shares", "prefill", seed=q_len, n_q=n_q, n_kv=n_kv, head_dim=d, kv_lens=kv,
                        extend_lens=[q_len, 1, q_len, q_len, q_len - 1], is_cross_attention=cross, sliding_window_size=window)
    args = lambda w: (w.q, w.k_cache, w.v_cache, w.qo_indptr, w.kv_indptr, w.kv_indices, w.prefix_lens, w.sm_scale, q_len)
    mask = dict(is_cross_attention=cross, sliding_window_size=window)
    want = oracle.paged_prefill_attention(*args(wl), **mask, return_f32=True)[1]
    g = wl.to(gpu)
    for cut in (0, share | 1 << 20, share | 2 << 20):
        tuning(_lib.TUNE_SHARES, cut)
        print(f"shares verify q{q_len} d{d} {mask} cut {cut:#x}", flush=True)
        _close(paged_prefill_attention(*args(g), **mask), want, f"cut {cut:#x}")


def test_replayed_from_a_graph(gpu, tuning):
    wl = build_workload("shares", "decode", seed=3, n_q=32, n_kv=8, kv_lens=[37, 900, 2000])
    g = wl.to(gpu)
    tuning(_lib.TUNE_SHARES, 128 | 1 << 20)
    want = _decode(g)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        _decode(g)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = _decode(g)
    for _ in range(5):
        out.zero_()
        graph.replay()
        assert torch.equal(_decode(g), want)  # eager work between the replays
        torch.cuda.synchronize()
        assert torch.equal(out, want)
