"""Short query blocks under a sliding window that most requests exceed, as shares of the window: one share per
request and several, one to three column tiles, several kv heads to a workgroup, requests shorter than the window,
windows that start inside a block of 16 keys; against the oracle."""
import pytest

import oracle
from _util import assert_close_bf16
from mini_sglang_amd.workloads import build_workload

pytestmark = pytest.mark.gpu

# (n_q, n_kv, head_dim, query tokens, kv lengths, window)
CASES = [
    (32, 8, 128, 8, [3000, 1100, 1031, 9, 2048] + [2500] * 27, 1024),  # one share per request
    (32, 8, 128, 4, [5000, 1700, 300], 1024),                           # several shares
    (16, 8, 128, 2, [900 + 37 * i for i in range(70)], 200),            # several kv heads to a workgroup
    (32, 8, 128, 12, [2600] * 5 + [12, 13, 700], 513),                  # three column tiles
    (16, 4, 256, 3, [700, 900, 1500, 3, 65], 129),
    (64, 8, 128, 5, [1300, 2200], 100),                                 # three column tiles, few requests
    (32, 8, 128, 8, [450 + 7 * (i % 50) for i in range(200)], 200),     # more requests than the chip has room for
    (64, 8, 128, 2, [9 + 5 * (i % 90) for i in range(400)], 128),       # as many, some shorter than the window
    (16, 2, 256, 2, [420 + i for i in range(430)], 100),
]


@pytest.mark.parametrize("n_q,n_kv,d,q_len,kv,window", CASES)
def test_against_the_oracle(gpu, n_q, n_kv, d, q_len, kv, window):
    from mini_sglang_amd_kernel import paged_prefill_attention

    wl = build_workload("ws", "prefill", seed=len(kv) + q_len, n_q=n_q, n_kv=n_kv, head_dim=d, kv_lens=kv,
                        extend_lens=[q_len - (i % 3 == 2) for i in range(len(kv))], sliding_window_size=window)
    args = lambda w: (w.q, w.k_cache, w.v_cache, w.qo_indptr, w.kv_indptr, w.kv_indices, w.prefix_lens, w.sm_scale, q_len)
    want = oracle.paged_prefill_attention(*args(wl), sliding_window_size=window, return_f32=True)[1]
    print(f"{n_q}/{n_kv} d{d} batch {len(kv)} x {q_len} window {window}", flush=True)
    got = paged_prefill_attention(*args(wl.to(gpu)), sliding_window_size=window)
    assert_close_bf16(got.cpu(), want, "shares of a window")
