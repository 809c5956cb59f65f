"""The workspace of a launch may hold anything: shares and gang ranges over a workspace full of words that look like
their own count words as launches numbered 1, 2, 3, ... would write them, and of ordinary data.  The library is loaded a
second time, from a copy, so that its launches are the first ones of that copy."""
import ctypes
import shutil

import pytest
import torch

from _gpu_util import run_oracle
from _util import assert_close_bf16
from mini_sglang_amd.workloads import build_workload

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def fresh_library(tmp_path_factory):
    from mini_sglang_amd_kernel import _lib

    path = tmp_path_factory.mktemp("lib") / "fresh_copy.so"
    shutil.copy(_lib.LIB_PATH, path)
    lib = ctypes.CDLL(str(path))
    for name, (restype, argtypes) in _lib.SIGNATURES.items():
        fn = getattr(lib, name)
        fn.restype, fn.argtypes = restype, argtypes
    return lib


def _fills(words, first):
    """Contents for the workspace, one per launch; the launches are numbers `first`, `first` + 1, ... of the copy."""
    ids = torch.arange(words, dtype=torch.int64)
    for i, count in enumerate((0, 1, 2, 3, 0xffff)):
        yield f"words of launch {first + i}, count {count}", ((first + i) << 16 | count) + 0 * ids
    yield "token ids", 65536 + ids % 150000
    yield "offsets", ids << 12
    yield "pairs of ones", torch.ones(2 * words).view(torch.int64)
    yield "all bits set", 0 * ids - 1
    yield "zeros", 0 * ids


def _launch(lib, g, ws):
    n_kv, d, slots = g.k_cache.shape[1], g.k_cache.shape[2], g.k_cache.shape[0]
    out = torch.full_like(g.q, 7.0)
    strides = [slots, g.k_cache.stride(0), g.v_cache.stride(0), float(g.sm_scale)]
    pools = [g.q.data_ptr(), g.k_cache.data_ptr(), g.v_cache.data_ptr()]
    room = [out.data_ptr(), ws.data_ptr(), ws.numel() * 8]
    stream = torch.cuda.current_stream().cuda_stream
    if g.kind == "decode":
        rc = lib.msgl_paged_decode_attention(*pools, g.kv_indptr.data_ptr(), g.kv_indices.data_ptr(), g.num_kv_splits.data_ptr(), *room,
                                             g.q.shape[0], g.kv_indices.numel(), g.q.shape[1], n_kv, d, *strides, 32, 0, stream)
    else:
        rc = lib.msgl_paged_prefill_attention(*pools, g.qo_indptr.data_ptr(), g.kv_indptr.data_ptr(), g.kv_indices.data_ptr(),
                                              g.prefix_lens.data_ptr(), *room, g.prefix_lens.numel(), g.q.shape[0], g.kv_indices.numel(),
                                              g.q.shape[1], n_kv, d, *strides, g.max_len_extend, 0, 0, 0, stream)
    assert rc == 0
    return out


@pytest.mark.parametrize("route", ["shares", "gang ranges"])
def test_whatever_the_workspace_holds(gpu, fresh_library, route):
    from mini_sglang_amd_kernel import _lib

    lib = fresh_library
    if route == "shares":
        wl = build_workload("stale", "decode", seed=5, n_q=16, n_kv=8, kv_lens=[900, 37, 1500, 640])
        need = lib.msgl_paged_decode_workspace_bytes(4, wl.kv_indices.numel(), 16, 8, 128)
    else:
        wl = build_workload("stale", "prefill", seed=6, n_q=32, n_kv=8, kv_lens=[3000, 300, 1200], extend_lens=[256, 200, 256])
        assert lib.msgl_set_tuning(_lib.TUNE_PREFILL_GANGS, 1) == 0  # this copy's knob, small launches too
        need = lib.msgl_paged_prefill_workspace_bytes(3, wl.q.shape[0], wl.kv_indices.numel(), 32, 8, 128, 256)
    assert need > 0 and need % 8 == 0
    want = run_oracle(wl)[0]
    g = wl.to(gpu)
    for what, words in _fills(need // 8, 1):
        ws = words.to(gpu)
        print(f"{route} over {what}", flush=True)
        got = _launch(lib, g, ws)
        torch.cuda.synchronize()
        assert_close_bf16(got.cpu(), want, f"{route} over {what}")
    assert lib.msgl_set_tuning(_lib.TUNE_PREFILL_GANGS, 0) == 0
