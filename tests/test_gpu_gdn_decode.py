"""One token per request through the gated delta rule: whatever rows a lane group has and however the state is read and written
(by its size: past the caches where it is small or large, plainly between), the same bits.  One of them is checked against
the float64 oracle elsewhere; here the sizes on both sides of the lines against that one."""
import pytest
import torch

from mini_sglang_amd_kernel import _lib, gdn_state_inplace

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch,hk,hv", [(1, 1, 1), (3, 2, 6), (6, 16, 32), (7, 16, 32), (12, 16, 32), (13, 16, 32), (47, 16, 32), (48, 16, 32), (96, 16, 16)])
def test_all_ways_are_one(gpu, tuning, batch, hk, hv):
    g = torch.Generator(device=gpu)
    g.manual_seed(batch)
    rand = lambda *s: torch.randn(s, generator=g, device=gpu)  # noqa: E731
    x = [rand(batch, hk, 128).bfloat16() * 0.09, rand(batch, hk, 128).bfloat16() * 0.09, rand(batch, hv, 128).bfloat16(),
         torch.sigmoid(rand(batch, hv)).bfloat16(), torch.sigmoid(rand(batch, hv)).bfloat16()]
    start = rand(batch + 2, hv, 128, 128)
    ids = torch.randperm(batch + 2, generator=g, device=gpu)[:batch].int()

    def run(rows, kib):
        tuning(_lib.TUNE_GDN_ROWS, rows)
        tuning(_lib.TUNE_STREAM, kib)
        state = start.clone()
        print(f"gdn decode {batch} {hk}/{hv} rows {rows} kib {kib}", flush=True)
        return gdn_state_inplace(*x, state, ids, None, single_token_mode=True), state

    want_y, want_state = run(1, -1)
    rest = torch.ones(batch + 2, dtype=torch.bool, device=gpu)
    rest[ids.long()] = False
    assert torch.equal(want_state[rest], start[rest]) and not torch.equal(want_state[~rest], start[~rest])
    for rows, kib in ((0, 0), (0, 1), (1, 1), (2, -1), (2, 1), (4, -1), (4, 1)):
        y, state = run(rows, kib)
        assert torch.equal(y.view(torch.int16), want_y.view(torch.int16)) and torch.equal(state.view(torch.int32), want_state.view(torch.int32))
