"""The sizes that the ``*_workspace_bytes`` queries give are enough for the call they are asked for, whatever mask the
call then has, and launches that can do without a workspace do.  Host code only: the pointers are made up, so this runs
where no GPU is visible, and a call that passes every check ends with MSGL_ERR_LAUNCH for want of a device."""
import ctypes
import math
import os
import random
import re

import pytest
import torch

pytestmark = pytest.mark.skipif(torch.cuda.device_count() > 0, reason="made-up pointers: only where nothing can be launched")

ERR_WORKSPACE, ERR_LAUNCH = -8, -11
FAKE = ctypes.c_void_p(0x1000)
HEADS = [(16, 8, 128), (32, 8, 128), (64, 8, 128), (8, 1, 128), (128, 16, 128), (16, 2, 256), (24, 4, 256), (32, 2, 256)]


def _prefill(batch, heads, ext, kv, window=0, cross=0, workspace=True):
    from mini_sglang_amd_kernel import _lib

    lib, (n_q, n_kv, d) = _lib.load(), heads
    total_q, total_kv = batch * ext, kv
    need = lib.msgl_paged_prefill_workspace_bytes(batch, total_q, total_kv, n_q, n_kv, d, ext) if workspace else 0
    return lib.msgl_paged_prefill_attention(FAKE, FAKE, FAKE, FAKE, FAKE, FAKE, FAKE, FAKE, FAKE if need else None, need,
                                            batch, total_q, total_kv, n_q, n_kv, d, 1 << 20, n_kv * d, n_kv * d, 0.1,
                                            ext, cross, window, 0, None)


def _decode(batch, heads, kv):
    from mini_sglang_amd_kernel import _lib

    lib, (n_q, n_kv, d) = _lib.load(), heads
    need = lib.msgl_paged_decode_workspace_bytes(batch, kv, n_q, n_kv, d)
    return lib.msgl_paged_decode_attention(FAKE, FAKE, FAKE, FAKE, FAKE, FAKE, FAKE, FAKE, need, batch, kv, n_q, n_kv, d,
                                           1 << 20, n_kv * d, n_kv * d, 0.1, 32, 0, None)


@pytest.mark.parametrize("heads,ext", [((32, 8, 128), 8), ((64, 8, 128), 4), ((32, 8, 128), 4), ((16, 8, 128), 8),
                                       ((24, 4, 256), 2), ((16, 2, 256), 2)])
def test_windowed_short_blocks_of_any_batch(heads, ext):
    """Around and beyond the batch that fills the chip with one share per request."""
    for batch in (*range(1, 700, 5), 131, 256, 257, 260, 261, 512, 513, 3000):
        assert _prefill(batch, heads, ext, 4096 * batch, window=1024) == ERR_LAUNCH, batch


def test_the_size_asked_for_is_enough():
    rng = random.Random(7)
    log = lambda lo, hi: int(lo * (hi / lo) ** rng.random())  # noqa: E731
    for _ in range(20000):
        batch, heads, ext = log(1, 2000), rng.choice(HEADS), log(1, 64)
        kv = batch * (log(1, 20000) + ext) + rng.randrange(64)
        mask = dict(window=rng.choice((0, 1, 100, 128, 500, 1024, 4096, log(1, 8192))), cross=rng.random() < 0.2)
        assert _prefill(batch, heads, ext, kv, **mask) == ERR_LAUNCH, (batch, heads, ext, kv, mask)
        assert _decode(batch, heads, kv) == ERR_LAUNCH, (batch, heads, kv)


def test_launches_that_can_do_without_a_workspace_do():
    """17-48 columns under a window that most requests exceed, and longer query blocks, fall back to one pass of the tile
    kernel; short blocks of the split-K route cannot."""
    for batch in (1, 4, 32, 100, 200, 600):
        for heads, ext in (((32, 8, 128), 8), ((32, 8, 128), 5), ((64, 8, 128), 3), ((16, 8, 128), 24)):
            assert _prefill(batch, heads, ext, 4096 * batch, window=1024, workspace=False) == ERR_LAUNCH, (batch, heads, ext)
        assert _prefill(batch, (32, 8, 128), 100, 4096 * batch, workspace=False) == ERR_LAUNCH
        assert _prefill(batch, (32, 8, 128), 4, 4096 * batch, window=1024, workspace=False) == ERR_WORKSPACE
        assert _prefill(batch, (32, 8, 128), 8, 4096 * batch, workspace=False) == ERR_WORKSPACE


def test_the_builtin_scratch_holds_every_size_whose_segments_fit_8_mib():
    """Whatever route the call takes: it is refused for its size only where segments would need more."""
    from mini_sglang_amd_kernel import _lib

    lib, rng = _lib.load(), random.Random(11)
    header = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "include", "msgl_paged_attention.h")
    scratch = math.prod(map(int, re.search(r"#define MSGL_DECODE_SCRATCH_BYTES \(([\d* ]+)\)", open(header).read()).group(1).split("*")))
    log = lambda lo, hi: int(lo * (hi / lo) ** rng.random())  # noqa: E731
    sizes = [(136, 28074, 64, 8, 128), (70, 11110, 128, 16, 128)]
    while len(sizes) < 40000:
        n_kv, batch = rng.choice((1, 2, 3, 4, 5, 6, 8, 12, 16, 24, 32, 64, 128)), log(1, 2000)
        sizes.append((batch, batch * log(1, 4000) + rng.randrange(100), n_kv * rng.randint(1, 16), n_kv, rng.choice((128, 256))))
    beyond = 0
    for size in sizes:
        need = lib.msgl_paged_decode_workspace_bytes(*size)
        if need <= 8 << 20:
            continue
        _lib.set_tuning(_lib.TUNE_SHARES, -1)
        segments = lib.msgl_paged_decode_workspace_bytes(*size)
        _lib.set_tuning(_lib.TUNE_SHARES, 0)
        beyond += segments <= 8 << 20
        assert segments > 8 << 20 or need <= scratch, (size, segments, need)
    assert beyond > 2


@pytest.mark.parametrize("batch,heads,line", [  # the mean length from which the gated delta rule takes scratch memory
    (1, 32, 352), (2, 32, 384), (3, 32, 384), (4, 32, 448), (5, 32, 256), (8, 32, 256), (9, 32, 128), (64, 32, 128),
    (3, 4, 352), (4, 4, 432), (8, 4, 624), (10, 4, 704), (24, 4, 704), (5, 24, 496), (8, 16, 640), (32, 4, 768),
    (16, 16, 256), (32, 8, 384), (64, 4, 512), (64, 8, 256), (40, 8, 128), (100, 8, 128)])
def test_gated_delta_rule_from_a_mean_length_on(batch, heads, line):
    from mini_sglang_amd_kernel import _lib

    ask = _lib.load().msgl_gdn_state_workspace_bytes
    assert ask(line * batch - 1, batch, heads, 0) == 0 and ask(line * batch, batch, heads, 0) > 0
    assert ask(line * batch, batch, heads, 1) == 0


@pytest.mark.parametrize("batch,kv,heads,q,shares", [  # beyond the first lines of the shares (csrc/paged_shares.hip)
    (26, 18746, (32, 8, 128), 1, False), (32, 18048, (64, 8, 128), 1, False), (28, 18060, (32, 8, 128), 1, False),  # shares of 1536 keys
    (19, 28310, (16, 8, 128), 1, True), (39, 28509, (32, 8, 128), 1, True),
    (4, 15904, (32, 8, 128), 6, False), (5, 26780, (32, 8, 128), 6, False), (6, 26780, (32, 8, 128), 6, True), (4, 15904, (32, 8, 128), 4, True),
    # few pairs with two tiles of columns
    (5, 80000, (8, 1, 128), 3, False), (8, 90000, (8, 1, 128), 3, False), (9, 300000, (8, 1, 128), 3, True),
    # shares longer than the requests, by the mean length: up to 104 MiB twice, 128 one and a half times, 152 as long, 176 half of it; 256 MiB
    (17, 39911, (32, 8, 128), 1, False), (21, 42499, (32, 8, 128), 1, False), (17, 29900, (32, 8, 128), 1, True), (1, 60000, (32, 8, 128), 1, True),
    (1, 66000, (32, 8, 128), 1, False), (300, 300 * 436, (8, 1, 128), 4, True), (85, 66600, (16, 4, 128), 1, False), (85, 65000, (16, 4, 128), 1, True)])
def test_launches_that_go_in_shares(batch, kv, heads, q, shares):
    from mini_sglang_amd_kernel import _lib

    lib, (n_q, n_kv, d) = _lib.load(), heads
    if q == 1:  # with norm and rotary embedding a decode step is one launch where it goes in shares
        assert (lib.msgl_decode_step_workspace_bytes(batch, kv, n_q, n_kv, d, 1) > 0) is shares
    assert (lib.msgl_extend_step_workspace_bytes(batch, q * batch, kv, n_q, n_kv, d, q, 0, 0) > 0) is shares


@pytest.mark.parametrize("batch,heads,ext,kv,window", [  # partials of more than 2 GiB in all
    (17000, (32, 8, 128), 8, 240, 200), (25000, (32, 8, 128), 8, 128, 64), (40000, (64, 8, 128), 2, 1100, 1024)])
def test_windows_of_very_many_requests_are_taken(batch, heads, ext, kv, window):
    assert _prefill(batch, heads, ext, kv * batch, window=window) == ERR_LAUNCH


@pytest.mark.parametrize("length", [1, 2, 300])
def test_any_share_length_set_by_hand_is_taken(tuning, length):
    from mini_sglang_amd_kernel import _lib

    tuning(_lib.TUNE_SHARES, length | 1 << 20)
    for kv in (100, 10**5, 10**7, 10**9):
        assert _decode(1, (64, 8, 128), kv) == ERR_LAUNCH, kv
        assert _decode(3, (32, 2, 256), kv) == ERR_LAUNCH, kv
