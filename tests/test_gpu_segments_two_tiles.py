"""Segments at head_dim 256 with 17 to 32 columns in one wave, whose Q is in LDS, with up to 64 in two, and one tile a wave on little work:
lengths around a tile of 32 keys,
requests without keys or rows, windows, no mask, rows by whole lines and as operands, against the CPU oracle; the launches that go this way for
their size, against plain float64 products, and the same without a workspace."""
import pytest
import torch

import oracle
from _util import assert_close_bf16
from mini_sglang_amd.workloads import build_workload
from mini_sglang_amd_kernel import _lib, paged_prefill_attention

pytestmark = pytest.mark.gpu

# n_q, n_kv, kv lengths, query tokens, window, segments; from 64 MiB of keys and values on (65536 of one kv head) two tiles share a wave
CASES = [
    (17, 1, [31, 32, 33, 65440], [1, 1, 1, 1], 0, 40), (8, 1, [700, 64, 65, 3, 65000], [4, 3, 2, 3, 4], 0, 64), (32, 8, [300, 0, 1000, 7000], [8, 0, 5, 8], 100, 7),
    (16, 4, [16000] + [45] * 9, [5] + [7] * 9, 0, 60), (24, 4, [129, 96, 16200], [5, 1, 4], 129, 5), (32, 2, [6560] * 5, [2] * 5, 0, 208),
    (33, 1, [536, 65000], [1, 1], 0, 32), (16, 2, [800, 300, 31, 31700], [8, 5, 3, 7], 0, 90), (24, 4, [400, 16100], [10, 9], 200, 6),
    (32, 8, [64, 128, 8100], [12, 9, 16], 0, 4), (8, 2, [700, 64, 65, 3], [8, 3, 2, 3], 0, 3), (16, 2, [800, 300], [8, 5], 0, 9),
]


@pytest.mark.parametrize("n_q,n_kv,kv,ext,window,segments", CASES)
@pytest.mark.parametrize("cross", [False, True])
@pytest.mark.parametrize("stream", [-1, 1])
def test_against_the_oracle(gpu, tuning, n_q, n_kv, kv, ext, window, segments, cross, stream):
    for knob, value in ((_lib.TUNE_SMALLQ_MAXCOLS, 64), (_lib.TUNE_SEGMENTS, segments), (_lib.TUNE_MIN_SEGMENT, 64), (_lib.TUNE_STREAM, stream)):
        tuning(knob, value)
    wl = build_workload("tiles", "prefill", seed=sum(kv), n_q=n_q, n_kv=n_kv, head_dim=256, kv_lens=kv, extend_lens=ext)
    args = lambda w: (w.q, w.k_cache, w.v_cache, w.qo_indptr, w.kv_indptr, w.kv_indices, w.prefix_lens, w.sm_scale, max(ext))  # noqa: E731
    masks = dict(is_cross_attention=cross, sliding_window_size=window)
    want = oracle.paged_prefill_attention(*args(wl), **masks, return_f32=True)[1]
    print(f"two tiles {n_q}/{n_kv} {kv[:3]} x {ext[:3]} window {window} {cross} segments {segments} stream {stream}", flush=True)
    g = wl.to(gpu)
    for _ in range(2):
        assert_close_bf16(paged_prefill_attention(*args(g), **masks).cpu(), want, "two tiles a wave")


@pytest.mark.parametrize("n_q,n_kv,kv,q_len,window", [(32, 8, [19000, 13800], 8, 0), (16, 4, [40000, 25600, 9], 6, 0), (16, 2, [140000], 3, 0),
                                                      (32, 8, [17000, 17000], 5, 16000), (32, 8, [17000, 17000], 5, 16400)])
@pytest.mark.parametrize("room", [True, False])
def test_large_launches(gpu, n_q, n_kv, kv, q_len, window, room):
    print(f"large {n_q}/{n_kv} {kv} x {q_len} window {window} {room}", flush=True)
    wl = build_workload("large", "prefill", seed=len(kv), n_q=n_q, n_kv=n_kv, head_dim=256, kv_lens=kv, extend_lens=[q_len] * len(kv)).to(gpu)
    assert sum(kv) * n_kv * 1024 >= 256 << 20
    if room:
        got = paged_prefill_attention(wl.q, wl.k_cache, wl.v_cache, wl.qo_indptr, wl.kv_indptr, wl.kv_indices, wl.prefix_lens, wl.sm_scale, q_len,
                                      sliding_window_size=window)
    else:  # what needs no workspace elsewhere needs none here
        got = torch.empty_like(wl.q)
        ptr = lambda t: t.data_ptr()  # noqa: E731
        rc = _lib.load().msgl_paged_prefill_attention(
            ptr(wl.q), ptr(wl.k_cache), ptr(wl.v_cache), ptr(wl.qo_indptr), ptr(wl.kv_indptr), ptr(wl.kv_indices), ptr(wl.prefix_lens), ptr(got), None, 0,
            len(kv), q_len * len(kv), sum(kv), n_q, n_kv, 256, wl.k_cache.shape[0], wl.k_cache.stride(0), wl.v_cache.stride(0), wl.sm_scale, q_len, 0,
            window, _lib.MSGL_DTYPE_BF16, torch.cuda.current_stream().cuda_stream)
        assert rc == 0
    torch.cuda.synchronize()
    group, want = n_q // n_kv, torch.empty(wl.q.shape, dtype=torch.float64)
    for b, n in enumerate(kv):
        rows = wl.kv_indices[int(wl.kv_indptr[b]):int(wl.kv_indptr[b]) + n].long()
        at, pos = torch.arange(n, device=gpu), torch.arange(n - q_len, n, device=gpu)
        seen = (at[None] <= pos[:, None]) & ((at[None] > pos[:, None] - window) if window else True)
        for h in range(n_kv):
            k, v = (c[rows, h].double() for c in (wl.k_cache, wl.v_cache))
            for e in range(group):
                q = wl.q[b * q_len:(b + 1) * q_len, h * group + e].double()
                weight = torch.softmax((q @ k.t().contiguous() * wl.sm_scale).masked_fill(~seen, float("-inf")), -1)
                want[b * q_len:(b + 1) * q_len, h * group + e] = (weight @ v).cpu()
    assert_close_bf16(got.cpu(), want.float(), "large launches")


# A call gives the same for values of V that IEEE half does not hold whatever its size: below the line the tile kernel takes it, above it segments do
@pytest.mark.parametrize("kv", [[40000, 25000, 90], [40000, 26000, 90]])
@pytest.mark.parametrize("scale", [1e5, 1e-6])
def test_values_beyond_half(gpu, kv, scale):
    n_q, n_kv, q_len = 16, 4, 6
    wl = build_workload("range", "prefill", seed=len(kv), n_q=n_q, n_kv=n_kv, head_dim=256, kv_lens=kv, extend_lens=[q_len] * len(kv)).to(gpu)
    assert (sum(kv) * n_kv * 1024 >= 256 << 20) == (kv[1] == 26000)
    v = ((1 + 0.1 * wl.v_cache.float()) * scale).bfloat16()
    not_finite = [(0, 1000, 1, 5, float("inf")), (1, 20000, 2, 250, float("-inf")), (1, 300, 0, 77, float("nan")), (0, 39000, 3, 128, float("nan"))]
    for b, at, h, dim, value in not_finite:
        v[int(wl.kv_indices[int(wl.kv_indptr[b]) + at]), h, dim] = value
    got = paged_prefill_attention(wl.q, wl.k_cache, v, wl.qo_indptr, wl.kv_indptr, wl.kv_indices, wl.prefix_lens, wl.sm_scale, q_len).double().cpu()
    group, want = n_q // n_kv, torch.empty(wl.q.shape, dtype=torch.float64)
    for b, n in enumerate(kv):
        rows = wl.kv_indices[int(wl.kv_indptr[b]):int(wl.kv_indptr[b]) + n].long()
        seen = torch.arange(n, device=gpu)[None] <= torch.arange(n - q_len, n, device=gpu)[:, None]
        for h in range(n_kv):
            k, vals = wl.k_cache[rows, h].double(), v[rows, h].double()
            for e in range(group):
                q = wl.q[b * q_len:(b + 1) * q_len, h * group + e].double()
                weight = torch.softmax((q @ k.t().contiguous() * wl.sm_scale).masked_fill(~seen, float("-inf")), -1)
                want[b * q_len:(b + 1) * q_len, h * group + e] = (weight @ vals.nan_to_num(0, 0, 0)).cpu()
        for _, at, h, dim, value in (x for x in not_finite if x[0] == b):
            want[b * q_len:(b + 1) * q_len, h * group:(h + 1) * group, dim] = value
    finite = want.isfinite()
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got[want.isinf()], want[want.isinf()])
    # values of one sign: weights rounded to bf16 and the result, 2^-9 each, and as much again for the exponentials
    assert ((got - want).abs()[finite] <= 2.0 ** -7 * want.abs()[finite]).all()
