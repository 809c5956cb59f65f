"""Decode and verify at head_dim 128 whose shares have the length that costs least: one and few requests in more than 16 shares, one to three
tiles of columns, lengths around whole shares, a long request among short ones, against the CPU oracle; and that such decode steps take
one launch."""
import pytest

import oracle
from _util import assert_close_bf16
from mini_sglang_amd.workloads import build_workload
from mini_sglang_amd_kernel import _lib, paged_decode_attention, paged_prefill_attention

pytestmark = pytest.mark.gpu

CASES = [  # kv lengths, q heads, kv heads, query tokens
    ([12000], 16, 2, 1), ([6143], 8, 1, 1), ([6144, 6145, 1], 32, 4, 1), ([9000, 5], 16, 1, 1), ([300] * 9 + [11000], 16, 8, 1),
    ([7000, 7001], 8, 1, 6), ([5000, 40], 16, 2, 4), ([9000, 120, 2500], 32, 4, 5), ([4100, 4000, 17], 32, 8, 9), ([2000 + 37 * i for i in range(12)], 8, 8, 1)]


@pytest.mark.parametrize("lens,n_q,n_kv,q_len", CASES)
def test_against_the_oracle(gpu, lens, n_q, n_kv, q_len):
    print(f"share lengths {lens[:3]} {n_q}/{n_kv} x {q_len}", flush=True)
    if q_len == 1:
        wl = build_workload("lengths", "decode", seed=len(lens), n_q=n_q, n_kv=n_kv, kv_lens=lens)
        args = lambda w: (w.q, w.k_cache, w.v_cache, w.kv_indptr, w.kv_indices, w.num_kv_splits, w.sm_scale, 32)  # noqa: E731
        want, op = oracle.paged_decode_attention(*args(wl), return_f32=True)[1], paged_decode_attention
        assert _lib.load().msgl_decode_step_workspace_bytes(len(lens), sum(lens), n_q, n_kv, 128, 1) > 0
    else:
        wl = build_workload("lengths", "prefill", seed=len(lens), n_q=n_q, n_kv=n_kv, kv_lens=lens, extend_lens=[min(q_len, n) for n in lens])
        args = lambda w: (w.q, w.k_cache, w.v_cache, w.qo_indptr, w.kv_indptr, w.kv_indices, w.prefix_lens, w.sm_scale, q_len)  # noqa: E731
        want, op = oracle.paged_prefill_attention(*args(wl), return_f32=True)[1], paged_prefill_attention
    g = wl.to(gpu)
    for _ in range(3):
        assert_close_bf16(op(*args(g)).cpu(), want, "share lengths")
