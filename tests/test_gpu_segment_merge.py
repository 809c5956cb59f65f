"""The merge of segments' partials that takes many rows to a workgroup: heads that do not fill its lanes, up to four, up to
eight and more items of a request, requests without keys, capped rows, both head sizes and partial types."""
import pytest
import torch

from _gpu_util import run_gpu, run_oracle
from _util import assert_close_bf16
from mini_sglang_amd.workloads import build_workload
from test_gpu_decode import _as_half

pytestmark = pytest.mark.gpu

# kind, n_q, n_kv, head_dim, kv lens, extends, segments
SHAPES = [
    ("decode", 24, 4, 128, [900, 1, 300, 0, 700], None, 16),
    ("decode", 10, 2, 128, [1500, 70], None, 9),
    ("decode", 6, 1, 256, [600, 0, 129], None, 8),
    ("decode", 32, 8, 128, [400 + 13 * i for i in range(40)], None, 208),
    ("decode", 24, 4, 256, [200] * 50, None, 208),
    ("prefill", 32, 8, 128, [500, 64, 3000, 130], [3, 1, 8, 4], 16),
    ("prefill", 12, 4, 128, [2100, 40], [5, 2], 16),
    ("prefill", 64, 8, 128, [700] * 9, [2] * 9, 64),
]


@pytest.mark.parametrize("kind,n_q,n_kv,d,kv,ext,segments", SHAPES)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_against_the_oracle(gpu, tuning, kind, n_q, n_kv, d, kv, ext, segments, dtype):
    from mini_sglang_amd_kernel import _lib

    if dtype == torch.float16 and kind == "prefill":
        pytest.skip("prefill is bf16")
    wl = build_workload("t", kind, seed=sum(kv) + n_q, n_q=n_q, n_kv=n_kv, head_dim=d, kv_lens=kv, pool_factor=1.2,
                        **({"extend_lens": ext, "store_new": True} if ext else {}))
    like = wl
    if dtype == torch.float16:
        like, wl = _as_half(wl)
    tuning(_lib.TUNE_SHARES, -1)
    tuning(_lib.TUNE_SEGMENTS, segments)
    tuning(_lib.TUNE_MIN_SEGMENT, 64)
    print(f"segment merge {kind} {n_q}/{n_kv} d{d} {kv[:4]} {dtype}", flush=True)
    got, _ = run_gpu(wl, gpu)
    want, _ = run_oracle(like)
    assert_close_bf16(got, want, "segments merged")
