"""What ``msgl_decode_step`` and ``msgl_extend_step`` refuse, and with which code.  Host code only: the pointers are made up,
so this runs where no GPU is visible, and a call that passes every check ends with MSGL_ERR_LAUNCH for want of a device."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.skipif(torch.cuda.device_count() > 0, reason="made-up pointers: only where nothing can be launched")

OK, NULL, HEAD_DIM, HEAD_RATIO, GROUP, DTYPE, WORKSPACE, SHAPE, ALIGNMENT, LAUNCH = 0, -1, -2, -3, -4, -5, -8, -9, -10, -11
WINDOW = -7
FAKE, ODD = 0x1000, 0x1008  # 16-byte aligned and not


def _decode(**change):
    a = dict(q=FAKE, k=FAKE, v=FAKE, q_stride0=2048, k_stride0=1024, v_stride0=1024, q_weight=None, k_weight=None, positions=None,
             out_loc=FAKE, k_cache=FAKE, v_cache=FAKE, kv_indptr=FAKE, kv_indices=FAKE, out=FAKE, workspace=FAKE, workspace_bytes=1 << 30,
             batch=4, total_kv=2000, n_q=16, n_kv=8, head_dim=128, num_slots=1 << 16, kc_stride0=1024, vc_stride0=1024, sm_scale=0.1,
             eps=1e-6, rope_base=1e6, dtype=0, stream=None)
    from mini_sglang_amd_kernel import _lib

    assert set(change) <= set(a)
    return _lib.load().msgl_decode_step(*(a | change).values())


def _extend(**change):
    a = dict(q=FAKE, k=FAKE, v=FAKE, k_stride0=1024, v_stride0=1024, out_loc=FAKE, k_cache=FAKE, v_cache=FAKE, qo_indptr=FAKE, kv_indptr=FAKE,
             kv_indices=FAKE, prefix_lens=FAKE, out=FAKE, workspace=FAKE, workspace_bytes=1 << 30, batch=4, total_q=20, total_kv=2000, n_q=16,
             n_kv=8, head_dim=128, num_slots=1 << 16, kc_stride0=1024, vc_stride0=1024, sm_scale=0.1, max_len_extend=5, cross=0, window=0,
             dtype=0, stream=None)
    from mini_sglang_amd_kernel import _lib

    assert set(change) <= set(a)
    return _lib.load().msgl_extend_step(*(a | change).values())


NORM = dict(q_weight=FAKE, k_weight=FAKE, positions=FAKE)
COMMON = [
    (dict(), LAUNCH), (dict(head_dim=64), HEAD_DIM), (dict(n_q=0), SHAPE), (dict(n_kv=0), SHAPE), (dict(n_q=12), HEAD_RATIO), (dict(dtype=7), DTYPE),
    (dict(kc_stride0=1000), SHAPE), (dict(vc_stride0=1016), SHAPE), (dict(kc_stride0=1028), ALIGNMENT), (dict(k_stride0=1016), SHAPE),
    (dict(v_stride0=0), SHAPE), (dict(k_stride0=1028), ALIGNMENT), (dict(v_stride0=1025), ALIGNMENT), (dict(num_slots=0), SHAPE),
    (dict(q=ODD), ALIGNMENT), (dict(k=ODD), ALIGNMENT), (dict(v=ODD), ALIGNMENT), (dict(out=ODD), ALIGNMENT), (dict(k_cache=ODD), ALIGNMENT),
    (dict(workspace=None), WORKSPACE), (dict(workspace=ODD), WORKSPACE), (dict(workspace_bytes=0), WORKSPACE),
    *((dict([(name, None)]), NULL) for name in ("q", "k", "v", "out", "out_loc", "k_cache", "v_cache", "kv_indptr", "kv_indices")),
]
DECODE = COMMON + [
    (dict(batch=0), OK), (dict(batch=-1), SHAPE), (dict(total_kv=-1), SHAPE), (dict(q_stride0=2040), SHAPE), (dict(q_stride0=2052), ALIGNMENT),
    (dict(n_q=136, q_stride0=1 << 15), GROUP), (dict(dtype=1), LAUNCH), (NORM, LAUNCH), (NORM | dict(dtype=1), DTYPE), (NORM | dict(positions=None), NULL),
    (NORM | dict(k_weight=None), NULL), (dict(k_weight=FAKE), NULL), (NORM | dict(q_weight=ODD), ALIGNMENT), (NORM | dict(rope_base=1.0), SHAPE),
    (NORM | dict(rope_base=float("nan")), SHAPE), (NORM | dict(eps=-1.0), SHAPE), (dict(rope_base=0.0), LAUNCH),
    (dict(batch=64, total_kv=64 * 4096), SHAPE),                          # sizes that take the two calls: a large launch,
    (dict(batch=1, total_kv=20000), LAUNCH), (NORM | dict(batch=1, total_kv=20000), SHAPE),  # segments with norm weights
]
EXTEND = COMMON + [
    (dict(dtype=1), DTYPE), (dict(qo_indptr=None), NULL), (dict(prefix_lens=None), NULL), (dict(batch=0), SHAPE), (dict(total_q=0), SHAPE),
    (dict(total_kv=0), SHAPE), (dict(max_len_extend=0), SHAPE), (dict(window=-1), SHAPE), (dict(total_q=100, max_len_extend=60), LAUNCH),
    (dict(total_q=100, max_len_extend=60, workspace=None), WORKSPACE), (dict(total_q=4000, total_kv=6000, max_len_extend=2000), SHAPE),
    (dict(cross=1), LAUNCH), (dict(window=100), LAUNCH),
]


@pytest.mark.parametrize("change,code", DECODE)
def test_decode_step(change, code):
    assert _decode(**change) == code


@pytest.mark.parametrize("change,code", EXTEND)
def test_extend_step(change, code):
    assert _extend(**change) == code


@pytest.mark.parametrize("batch,total_kv", [(4, 2000), (1, 20000), (16, 30000)])
def test_the_size_asked_for_is_enough_and_no_more_than_needed(batch, total_kv):
    from mini_sglang_amd_kernel import _lib

    need = _lib.load().msgl_decode_step_workspace_bytes(batch, total_kv, 16, 8, 128, 0)
    assert need > 0
    assert _decode(batch=batch, total_kv=total_kv, workspace_bytes=need) == LAUNCH
    assert _decode(batch=batch, total_kv=total_kv, workspace_bytes=need - 1) == WORKSPACE
    for ext in (1, 8, 40, 100):
        need = _lib.load().msgl_extend_step_workspace_bytes(batch, batch * ext, total_kv, 16, 8, 128, ext, 0, 0)
        if need:
            sizes = dict(batch=batch, total_q=batch * ext, total_kv=total_kv, max_len_extend=ext)
            assert _extend(**sizes, workspace_bytes=need) == LAUNCH
            assert _extend(**sizes, workspace_bytes=need - 1) == WORKSPACE
