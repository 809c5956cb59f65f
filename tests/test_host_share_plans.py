"""Which decode launches at head_dim 256 go in shares of their requests' keys: few (request, kv head) pairs, long requests, and the two
lines beyond which they go in segments.  (With norm and rotary embedding a decode step is one launch where it goes in shares.)"""
import pytest


@pytest.mark.parametrize("batch,keys,n_q,n_kv,shares", [
    (1, 51820, 16, 2, True), (2, 3814, 24, 4, True), (1, 1, 16, 2, True), (2, 45000, 24, 4, True),
    (22, 22 * 4116, 16, 4, False),      # shares long enough for one round fill less than half of it
    (22, 22 * 2900, 16, 4, True),
    (4, 717500, 16, 2, False), (4, 716000, 16, 2, True),  # 1400 MiB of keys and values
    (64, 64 * 300, 16, 4, True)])
def test_head_dim_256(batch, keys, n_q, n_kv, shares):
    from mini_sglang_amd_kernel import _lib

    lib = _lib.load()
    assert (lib.msgl_decode_step_workspace_bytes(batch, keys, n_q, n_kv, 256, 1) > 0) is shares
    assert lib.msgl_decode_step_workspace_bytes(batch, keys, n_q, n_kv, 256, 1) <= lib.msgl_paged_decode_workspace_bytes(batch, keys, n_q, n_kv, 256)


@pytest.mark.parametrize("batch,keys,n_q,n_kv,shares", [  # few pairs, one whole column tile: slower in shares between the two lines
    (1, 1500, 16, 1, True), (1, 2000, 16, 1, False), (2, 2 * 8000, 16, 1, False), (3, 3 * 16000, 16, 1, False), (3, 3 * 16500, 16, 1, True),
    (4, 4 * 8000, 16, 1, False), (4, 4 * 8100, 16, 1, True), (6, 6 * 2600, 16, 1, False), (6, 6 * 2500, 16, 1, True), (7, 7 * 4000, 16, 1, True),
    (2, 2 * 4000, 32, 2, True), (4, 4 * 4000, 12, 1, True), (1, 8000, 24, 2, False), (1, 3500, 24, 2, True), (1, 8000, 8, 1, True), (1, 8000, 64, 4, True)])
def test_few_pairs_with_many_columns(batch, keys, n_q, n_kv, shares):
    from mini_sglang_amd_kernel import _lib

    assert (_lib.load().msgl_decode_step_workspace_bytes(batch, keys, n_q, n_kv, 256, 1) > 0) is shares


@pytest.mark.parametrize("batch,heads,window,shares", [
    (1, (8, 1), 256, True), (1, (8, 1), 1024, False), (3, (8, 1), 2048, False), (4, (8, 1), 1024, True), (1, (16, 4), 4096, True)])
def test_windows_of_few_pairs(batch, heads, window, shares):
    from mini_sglang_amd_kernel import _lib

    lib, (n_q, n_kv) = _lib.load(), heads
    assert (lib.msgl_extend_step_workspace_bytes(batch, 2 * batch, 30000 * batch, n_q, n_kv, 256, 2, 0, window) > 0) is shares
