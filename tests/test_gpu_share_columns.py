"""Short query blocks whose columns go to several workgroups of a share: both ends of every number of them, blocks shorter than the longest (some
workgroups have no column then), one share to a request and several, windows, masks off, requests without keys or rows, against the CPU
oracle; and the store of the launch's own rows, which one of those workgroups does."""
import pytest

import oracle
from _util import assert_close_bf16
from mini_sglang_amd.workloads import build_workload
from mini_sglang_amd_kernel import _lib, paged_prefill_attention
from test_gpu_decode_step import test_extend_one_launch_is_two as _one_launch_is_two

pytestmark = pytest.mark.gpu

CASES = [  # n_q, n_kv, head_dim, kv lengths, query tokens, window
    (49, 1, 128, [700, 1900], [1, 1], 0), (32, 4, 128, [3000, 260, 900], [8, 3, 1], 0), (32, 8, 128, [1500, 800, 2200, 400], [16, 5, 13, 4], 1024),
    (64, 8, 128, [500, 700], [8, 7], 0), (64, 8, 128, [500, 1700], [9, 12], 0), (48, 6, 128, [2600, 130, 900], [16, 2, 9], 513),
    (32, 8, 128, [2000, 700, 90], [8, 5, 2], 0), (64, 8, 128, [900, 400, 250], [5, 6, 1], 300), (34, 2, 128, [1500], [1], 0),
    (48, 6, 128, [2600], [7], 513), (24, 3, 128, [900, 0, 7], [7, 0, 7], 0),
    (17, 1, 256, [600], [1], 0), (8, 1, 256, [3000, 130, 700], [4, 3, 2], 0), (24, 4, 256, [420, 900], [6, 1], 129), (16, 4, 256, [4100, 300], [9, 12], 0),
    (32, 2, 256, [700, 640, 5], [10, 7, 5], 0), (16, 2, 256, [1000] * 6 + [9], [16] * 6 + [3], 200), (40, 2, 256, [2000, 300], [8, 2], 0),
]


@pytest.mark.parametrize("n_q,n_kv,d,kv,ext,window", CASES)
@pytest.mark.parametrize("cross", [False, True])
@pytest.mark.parametrize("share", [0, 64, 100000])  # share lengths: chosen, short, one share to a request
def test_against_the_oracle(gpu, tuning, n_q, n_kv, d, kv, ext, window, cross, share):
    tuning(_lib.TUNE_SHARES, share)
    wl = build_workload("columns", "prefill", seed=sum(kv), n_q=n_q, n_kv=n_kv, head_dim=d, kv_lens=kv, extend_lens=ext)
    args = lambda w: (w.q, w.k_cache, w.v_cache, w.qo_indptr, w.kv_indptr, w.kv_indices, w.prefix_lens, w.sm_scale, max(ext))  # noqa: E731
    masks = dict(is_cross_attention=cross, sliding_window_size=window)
    want = oracle.paged_prefill_attention(*args(wl), **masks, return_f32=True)[1]
    print(f"share columns {n_q}/{n_kv} d{d} {kv[:3]} x {ext[:3]} window {window} {cross} share {share}", flush=True)
    g = wl.to(gpu)
    for _ in range(2):
        assert_close_bf16(paged_prefill_attention(*args(g), **masks).cpu(), want, "columns in several workgroups")


STORES = [  # cached, new tokens, n_q, n_kv, head_dim
    ([700, 300, 900], [8, 3, 8], 32, 4, 128), ([400, 700], [16, 1], 32, 8, 128), ([900, 200, 0], [8, 7, 5], 64, 8, 128), ([900, 300, 250], [16, 3, 10], 64, 8, 128),
    ([700, 300, 900], [8, 3, 5], 32, 8, 128), ([1900, 300], [5, 1], 64, 8, 128),
    ([600], [2], 24, 2, 256), ([900, 140], [5, 12], 16, 4, 256), ([800, 300, 700], [10, 0, 4], 32, 2, 256), ([500, 600], [33, 9], 8, 2, 256),
]


@pytest.mark.parametrize("cached,ext,n_q,n_kv,d", STORES)
# share 0: the plan that such a call has, a workgroup to each tile of columns; else two tiles to one at head_dim 128
@pytest.mark.parametrize("share,cross,window", [(0, False, 0), (0, True, 0), (0, False, 600)] +
                         [(s, *m) for s in (64, 96) for m in ((False, 0), (True, 0), (False, 100))])
@pytest.mark.parametrize("places", ["last", "mixed"])
def test_one_launch_is_two(gpu, tuning, cached, ext, n_q, n_kv, d, share, cross, window, places):
    batch, keys, tiles = len(ext), sum(ext) + sum(cached), -(-max(ext) * n_q // n_kv // 16)
    if share == 0:
        if window:
            keys = min(keys, batch * (window + max(ext) + 15))
        assert keys > 192 * batch and keys * n_kv * tiles <= (400 if d == 256 else 512) * 256 and 4 * batch * n_kv <= 3 * (256 // (8 * tiles) * 8)
        assert _lib.load().msgl_extend_step_workspace_bytes(batch, sum(ext), sum(ext) + sum(cached), n_q, n_kv, d, max(ext), int(cross), window) > 0
    shares_only = lambda knob, value: tuning(knob, value) if share and knob == _lib.TUNE_SHARES else None  # noqa: E731
    _one_launch_is_two(gpu, shares_only, cached, ext, n_q, n_kv, d, share, 0, cross, window, places)


# around the lines up to which launches go this way: workgroups, keys in all, keys of a request, columns
@pytest.mark.parametrize("d,batch,keys,n_q,n_kv,q_len", [
    (256, 64, 200, 8, 2, 6), (256, 65, 200, 8, 2, 6), (256, 32, 150, 8, 1, 14), (256, 33, 150, 8, 1, 14), (256, 1, 25600, 16, 2, 4), (256, 1, 25664, 16, 2, 4),
    (256, 2, 128, 16, 2, 4), (256, 2, 129, 16, 2, 4), (256, 2, 600, 32, 2, 10), (256, 2, 600, 32, 2, 11), (128, 12, 193, 32, 8, 16), (128, 13, 193, 32, 8, 16),
    (128, 1, 8192, 32, 8, 16), (128, 1, 8193, 32, 8, 16), (128, 2, 192, 64, 8, 7), (128, 2, 193, 64, 8, 7), (128, 2, 500, 64, 8, 8), (128, 2, 500, 64, 8, 9),
    (128, 1, 4096, 64, 8, 16), (128, 1, 4097, 64, 8, 16), (128, 6, 500, 64, 8, 16), (128, 7, 500, 64, 8, 16), (128, 1, 500, 64, 8, 17),
    (128, 12, 300, 32, 8, 8), (128, 13, 300, 32, 8, 8), (128, 1, 8192, 32, 8, 8), (128, 1, 8193, 32, 8, 8), (128, 7, 300, 64, 8, 6), (128, 8, 300, 64, 8, 6), (128, 9, 300, 64, 8, 6)])
def test_the_lines(gpu, d, batch, keys, n_q, n_kv, q_len):
    wl = build_workload("lines", "prefill", seed=keys, n_q=n_q, n_kv=n_kv, head_dim=d, kv_lens=[keys] * batch, extend_lens=[q_len] * batch)
    args = lambda w: (w.q, w.k_cache, w.v_cache, w.qo_indptr, w.kv_indptr, w.kv_indices, w.prefix_lens, w.sm_scale, q_len)  # noqa: E731
    print(f"lines d{d} {batch} x {keys} {n_q}/{n_kv} x {q_len}", flush=True)
    got = paged_prefill_attention(*args(wl.to(gpu))).cpu()
    assert_close_bf16(got, oracle.paged_prefill_attention(*args(wl), return_f32=True)[1], "lines")
