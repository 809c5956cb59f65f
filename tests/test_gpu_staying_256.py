"""Workgroups of the head_dim 256 extend kernel that stay for several blocks, against the CPU oracle: blocks of one step and of
many, with few rows and without keys, groups that fill a block with whole queries or not, windows, both sides visible, rows
whose offsets have 64 bits; and on both sides of the number of rounds from which they stay."""
import pytest
import torch

from _gpu_util import run_gpu, run_oracle
from _util import assert_close_bf16
from mini_sglang_amd.workloads import build_workload
from mini_sglang_amd_kernel import paged_prefill_attention

pytestmark = pytest.mark.gpu


def _mixed(n, longest):
    return [1 + (i * 97) % longest for i in range(n - 2)] + [longest, 0]


CASES = [  # q heads, kv heads, extends, cached, window, cross, every third request's keys hidden by the window
    (8, 8, _mixed(64, 300), [0] * 64, 0, False, False),
    (24, 4, _mixed(64, 300), [(i * 131) % 700 for i in range(64)], 0, False, False),
    (16, 2, _mixed(64, 500), [(i * 131) % 300 for i in range(64)], 100, False, False),
    (16, 2, _mixed(64, 500), [(i * 131) % 300 for i in range(64)], 100, False, True),
    (16, 4, _mixed(50, 300), [(i * 61) % 200 for i in range(50)], 0, True, False),
    (32, 2, _mixed(30, 320), [(i * 61) % 200 for i in range(30)], 64, True, True),
    (16, 1, _mixed(32, 300), [(i * 17) % 90 for i in range(32)], 0, False, False),
    (10, 2, _mixed(64, 300), [(i * 17) % 90 for i in range(64)], 0, False, False),
    # 1.4 and 1.6 rounds, and one long extend beside short ones
    (16, 4, [190] * 14 + [150], [(i * 61) % 500 for i in range(15)], 0, False, False),
    (16, 4, [220] * 14 + [150], [(i * 61) % 500 for i in range(15)], 0, False, False),
    (32, 8, [1300] + [16] * 14 + [0], [(i * 61) % 500 for i in range(16)], 0, False, False),
    # prefixes: under a window that most requests exceed, and beside blocks that fill their XCDs
    (24, 4, _mixed(64, 300), [(i * 131) % 700 for i in range(64)], 200, False, False),
    (16, 1, _mixed(32, 300), [0] * 32, 0, False, False),
    (10, 2, _mixed(64, 300), [64 + (i * 17) % 90 for i in range(64)], 64, False, False),
    (32, 8, [1024, 1100], [300, 40], 0, False, False),
    (16, 4, [200, 333, 128, 1] * 6, [0] * 24, 400, True, False),  # all keys seen
]


def _workload(n_q, n_kv, extends, prefixes, window, is_cross):
    return build_workload("s", "prefill", seed=len(extends) + n_kv, n_q=n_q, n_kv=n_kv, head_dim=256,
                          kv_lens=[p + e for p, e in zip(prefixes, extends)], extend_lens=extends,
                          pool_factor=1.1, store_new=True, sliding_window_size=window, is_cross_attention=is_cross)


@pytest.mark.parametrize("n_q,n_kv,extends,prefixes,window,is_cross,hidden", CASES)
def test_against_the_oracle(gpu, n_q, n_kv, extends, prefixes, window, is_cross, hidden):
    wl = _workload(n_q, n_kv, extends, prefixes, window, is_cross)
    if hidden:
        wl.prefix_lens[::3] += 5000
    print(f"{n_q}/{n_kv} batch={len(extends)} window={window} cross={is_cross} hidden={hidden}", flush=True)
    got, _ = run_gpu(wl, gpu)
    want, _ = run_oracle(wl)
    assert torch.isfinite(got.float()).all()
    assert_close_bf16(got, want, "blocks of workgroups that stay vs oracle")
    for _ in range(5):  # a stage refilled under a reader would show as unequal bits
        assert torch.equal(run_gpu(wl, gpu)[0], got)


def test_wide_rows_and_values_that_are_not_finite(gpu):
    g = _workload(24, 4, _mixed(64, 300), [(i * 131) % 700 for i in range(64)], 0, False).to(gpu)
    run = lambda q, k, v: paged_prefill_attention(q, k, v, g.qo_indptr, g.kv_indptr, g.kv_indices, g.prefix_lens, g.sm_scale,  # noqa: E731
                                                  g.max_len_extend)
    want = run(g.q, g.k_cache, g.v_cache)
    slots = g.k_cache.shape[0]
    heads = (1 << 32) // (slots * 512) + 8  # between two slots' rows: offsets past 4 GiB
    wide = [torch.empty((slots, heads, 256), dtype=torch.bfloat16, device=gpu)[:, :4].copy_(c) for c in (g.k_cache, g.v_cache)]
    assert torch.equal(run(g.q, *wide), want)
    # one query of every request: nobody else's row sees it, whichever block comes next
    q, at = g.q.clone(), g.qo_indptr[:-2].long()
    q[at] = float("nan")
    got, others = run(q, g.k_cache, g.v_cache), torch.ones(q.shape[0], dtype=torch.bool, device=gpu)
    others[at] = False
    assert torch.equal(got[others], want[others]) and torch.isnan(got[at].float()).all()
