"""Query blocks of an extend in order of length: every block of every request has to come up exactly once,
whatever the kv heads (1, 2, 4 or a multiple of 8 of them: the XCDs share a head, or have several), with
empty and one-token requests, requests of one length, and as many requests as the order holds (64) or more."""
import pytest
import torch

from _gpu_util import run_gpu, run_oracle
from _util import assert_close_bf16
from mini_sglang_amd.workloads import build_workload

pytestmark = pytest.mark.gpu

# (n_q, n_kv, head_dim, extends, prefixes, window, cross): all of them more blocks than compute units
CASES = [
    (16, 1, 128, [700, 1, 513, 900, 300, 64, 33, 255] + [512] * 4, [100, 0, 3000, 0, 10, 65, 0, 640] + [0] * 4, 0, False),
    (32, 2, 256, [700, 16, 0, 1, 513], [300, 1000, 50, 0, 64], 0, False),
    (16, 4, 256, [900, 3, 260, 64, 513, 700], [0, 2000, 64, 63, 700, 130], 256, False),
    (32, 8, 128, [640, 65, 1, 257, 500, 384], [0, 800, 31, 64, 1000, 0], 0, False),
    (32, 8, 128, [640, 65, 1, 257, 500, 384], [0, 800, 31, 64, 1000, 0], 0, True),
    (16, 16, 128, [300, 0, 256, 257, 900, 515], [0, 70, 0, 128, 300, 5], 128, False),
    (8, 8, 128, [300] * 63 + [1], [i * 3 for i in range(64)], 0, False),
    (8, 8, 128, [300] * 64 + [2], [i % 7 for i in range(65)], 0, False),
    (32, 8, 128, [300] * 4, [0] * 4, 0, False),
]


@pytest.mark.parametrize("n_q,n_kv,d,extends,prefixes,window,is_cross", CASES)
def test_every_block_once(gpu, n_q, n_kv, d, extends, prefixes, window, is_cross):
    wl = build_workload("l", "prefill", seed=len(extends) + n_kv, n_q=n_q, n_kv=n_kv, head_dim=d,
                        kv_lens=[p + e for p, e in zip(prefixes, extends)], extend_lens=extends,
                        pool_factor=1.1, store_new=True, sliding_window_size=window, is_cross_attention=is_cross)
    print(f"{n_q}/{n_kv} d={d} batch={len(extends)} window={window} cross={is_cross}", flush=True)
    got, _ = run_gpu(wl, gpu)
    want, _ = run_oracle(wl)
    assert torch.isfinite(got.float()).all()
    assert_close_bf16(got, want, "blocks in order of length vs oracle")


# Enough blocks for workgroups that stay and take one in each of several rounds: blocks of one tile and of many, so
# that the moves that start a stream run over several blocks, partly filled ones, and ones without keys
def _mixed(n, longest):
    return [1 + (i * 97) % longest for i in range(n - 2)] + [longest, 0]


STAY = [  # the last column: every third request's queries sit so far behind its keys that the window hides all of them
    (8, 8, _mixed(64, 300), [0] * 64, 0, False, False),
    (8, 8, _mixed(64, 300), [(i * 131) % 700 for i in range(64)], 0, False, False),
    (8, 8, _mixed(64, 600), [(i * 131) % 300 for i in range(64)], 100, False, False),
    (8, 8, _mixed(64, 600), [(i * 131) % 300 for i in range(64)], 100, False, True),
    (8, 8, _mixed(64, 300), [(i * 61) % 200 for i in range(64)], 0, True, False),
    (24, 8, _mixed(30, 520), [(i * 61) % 200 for i in range(30)], 64, True, False),
    (24, 8, _mixed(30, 520), [(i * 61) % 200 for i in range(30)], 64, True, True),
    (6, 2, _mixed(64, 400), [(i * 17) % 90 for i in range(64)], 0, False, False),
    (16, 1, _mixed(32, 500), [(i * 17) % 90 for i in range(32)], 0, False, False),
    # about two rounds of blocks: of even extends, and of one long one beside short ones, whose grid has many more
    (6, 2, _mixed(64, 700), [(i * 17) % 90 for i in range(64)], 0, False, False),
    (16, 1, _mixed(32, 600), [(i * 17) % 90 for i in range(32)], 0, False, False),
    (16, 4, [380] * 30, [(i * 61) % 500 for i in range(30)], 0, False, False),
    (64, 8, [1700] + [16] * 14 + [0], [(i * 61) % 500 for i in range(16)], 0, False, False),
]


@pytest.mark.parametrize("n_q,n_kv,extends,prefixes,window,is_cross,hidden", STAY)
def test_workgroups_that_stay(gpu, n_q, n_kv, extends, prefixes, window, is_cross, hidden):
    wl = build_workload("s", "prefill", seed=len(extends) + n_kv, n_q=n_q, n_kv=n_kv, head_dim=128,
                        kv_lens=[p + e for p, e in zip(prefixes, extends)], extend_lens=extends,
                        pool_factor=1.1, store_new=True, sliding_window_size=window, is_cross_attention=is_cross)
    if hidden:
        wl.prefix_lens[::3] += 5000
    print(f"{n_q}/{n_kv} batch={len(extends)} window={window} cross={is_cross} hidden={hidden}", flush=True)
    got, _ = run_gpu(wl, gpu)
    want, _ = run_oracle(wl)
    assert torch.isfinite(got.float()).all()
    assert_close_bf16(got, want, "blocks of workgroups that stay vs oracle")
    for _ in range(5):  # a tile refilled under a reader would show as unequal bits
        assert torch.equal(run_gpu(wl, gpu)[0], got)
