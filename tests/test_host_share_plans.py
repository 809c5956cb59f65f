"""Which decode launches at head_dim 256 go in shares of their requests' keys: few (request, kv head) pairs, long requests, and the two
lines beyond which they go in segments.  (With norm and rotary embedding a decode step is one launch where it goes in shares.)"""
import math
import random

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


def _least_cost_shares(batch, keys, n_kv, d, cols, cus=256):
    """Most shares of a launch whose lengths cost least, by the costs as they are stated: all lengths, in floating point."""
    mean, length, lowest = keys // batch, None, 0.0
    c = 512 if cols > 32 else 256 if cols > 16 and d == 128 else 128
    while c < 1 << 20:
        of_one = max(math.ceil(mean / c), 1)
        if max(batch, keys / c + 0.5 * batch + 0.43 * math.sqrt(batch), batch * of_one) * n_kv <= cus:
            cost = min(c, 1.5 * mean) + ((160 if cols > 8 else 100) if of_one > 1 else 0) + 4 * of_one + 100 * (math.ceil(of_one / 16) - 1)
            if length is None or cost < lowest:
                length, lowest = c, cost
            if c >= 2 * mean:
                break
        c = c // 3 * 4 if c & (c - 1) else c // 2 * 3
    return keys // (length or 1 << 20) + batch


def test_lengths_cost_least():
    from mini_sglang_amd_kernel import _lib

    rng, need = random.Random(3), _lib.load().msgl_decode_step_workspace_bytes
    log = lambda lo, hi: int(lo * (hi / lo) ** rng.random())  # noqa: E731
    seen = 0
    for _ in range(20000):
        d, n_kv, group = rng.choice((128, 256)), rng.choice((1, 2, 3, 4, 6, 8, 16)), rng.randint(1, 16)
        batch = log(1, 256 // n_kv + 1)
        keys = batch * log(1, 100000) + rng.randrange(batch)
        size = need(batch, keys, n_kv * group, n_kv, d, 1)
        if size == 0 or batch * n_kv > 256:
            continue
        up = lambda n: (n + 255) // 256 * 256  # noqa: E731
        rows = _least_cost_shares(batch, keys, n_kv, d, group) * n_kv * group
        assert size == up(8 * batch * n_kv) + up(rows * (d + 1) * 4), (batch, keys, n_kv, group, d)
        seen += 1
    assert seen > 5000
