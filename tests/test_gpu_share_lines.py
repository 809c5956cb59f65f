"""Decode launches on both sides of the sizes from which the keys go in segments instead of shares, against the CPU oracle."""
import math

import pytest
import torch

import oracle
from mini_sglang_amd.workloads import build_workload
from mini_sglang_amd_kernel import paged_decode_attention

pytestmark = pytest.mark.gpu

LINES = [  # kv lengths, q heads, kv heads, head_dim
    ([513 + 3 * (i % 9) for i in range(101)], 16, 8, 128),  # 205 MiB, heads four by four
    ([513 + 3 * (i % 9) for i in range(104)], 16, 8, 128),  # 211
    ([2048] * 26, 32, 8, 128), ([2048] * 26 + [33], 32, 8, 128),  # 208 and a little more
    ([12288], 64, 8, 128), ([12289], 64, 8, 128),
    ([4000, 9000, 1], 16, 4, 128),  # 12 units
    ([20001, 17], 16, 4, 128),      # 8 of them, of some length
    ([9000, 300, 7000], 16, 4, 256), ([9000, 300], 24, 4, 256),
    ([32768, 40000, 17, 5000, 30000, 23200], 16, 4, 256), ([32768, 40000, 17, 5000, 30000, 23400], 16, 4, 256),  # 255 and 256
    ([9000] * 6, 16, 4, 256), ([9000] * 5 + [4000], 16, 4, 256)
]


@pytest.mark.parametrize("lens,n_q,n_kv,d", LINES)
def test_decode(gpu, lens, n_q, n_kv, d):
    wl = build_workload("share lines", "decode", seed=len(lens), n_q=n_q, n_kv=n_kv, head_dim=d, kv_lens=lens)
    want = oracle.paged_decode_attention(wl.q, wl.k_cache, wl.v_cache, wl.kv_indptr, wl.kv_indices, wl.num_kv_splits, wl.sm_scale,
                                         wl.max_kv_splits, return_f32=True)[1]
    g = wl.to(gpu)
    print(f"share lines {len(lens)} requests of {lens[0]} {n_q}/{n_kv} d{d}", flush=True)
    for _ in range(2):
        got = paged_decode_attention(g.q, g.k_cache, g.v_cache, g.kv_indptr, g.kv_indices, g.num_kv_splits, g.sm_scale, 32)
        diff = (got.float().cpu() - want).abs()
        for i, n in enumerate(lens):
            # the result rounded once, and each weight once: their errors, at most 2^-9 of terms that are about n^-0.5 of
            # a value together, are independent, so that 8 of them side by side is beyond what can occur
            assert (diff[i] <= 2.0 ** -8 * want[i].abs() + 2.0 ** -6 / math.sqrt(n)).all(), (i, float(diff[i].max()))
