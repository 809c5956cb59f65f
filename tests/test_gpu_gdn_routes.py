"""gdn_state_inplace: which requests have the same bits alone and among others, and that the longest length that a caller gives
chooses the kernel and nothing else.

Same bits: requests of one length of 9-48 tokens, whatever their number (chunks of 16, where the caller gives the longest);
a long request alone and among short ones (chunks of 64).  Not the same, to the rounding of another order of the same sums: a
request of 24-48 tokens alone and among longer ones, a window of a few tokens and as many decode steps."""
from types import SimpleNamespace

import pytest
import torch

from test_gpu_gdn_pairs import HV, _bits, _inputs

pytestmark = pytest.mark.gpu


def _run(x, lengths, longest=None, at=0):
    """-> y, state of a call on the tokens and requests from `at` tokens and no request on."""
    from mini_sglang_amd_kernel import gdn_state_inplace

    dev, total = x["q"].device, sum(lengths)
    ip = torch.tensor([0] + lengths).cumsum(0).int().to(dev)
    state = x["state"].clone()
    print(f"gdn routes {lengths[:4]} of {len(lengths)}, longest {longest}", flush=True)
    y = gdn_state_inplace(*(x[n][at:at + total] for n in ("q", "k", "v", "g", "beta")), state,
                          torch.arange(len(lengths), dtype=torch.int32, device=dev), ip, max_len_extend=longest)
    torch.cuda.synchronize()
    return y, state


def _same(a, b):
    return torch.equal(_bits(a), _bits(b))


def _close(got, want):  # fp32 throughout, each within some 1e-7 of the sum in 64 bits; y rounded to bf16 once more
    y, state = (t.float() for t in got)
    want_y, want_state = (t.float() for t in want)
    assert float((state - want_state).abs().max()) <= 2e-6 * max(1.0, float(want_state.abs().max()))
    assert bool(((y - want_y).abs() <= 2.0 ** -7 * want_y.abs() + 1e-5).all())


@pytest.mark.parametrize("length", [9, 16, 33, 48])
def test_requests_of_one_length(gpu, length):
    x = _inputs(gpu, length, 16, 1, length)
    y, state = _run(x, [length], length)
    for times in (2, 5, 17):  # 17: more than 512 heads
        many = {n: t.repeat(times, *[1] * (t.dim() - 1)) for n, t in x.items()}
        y_many, state_many = _run(many, [length] * times, length)
        assert _same(y_many, y.repeat(times, 1, 1)) and _same(state_many, state.repeat(times, 1, 1, 1))


@pytest.mark.parametrize("lengths", [[720] + [1] * 15, [2000] + [8] * 31, [1300] + [30] * 20, [211] + [1] * 5])
def test_a_long_request_among_short_ones(gpu, lengths):
    x = _inputs(gpu, sum(lengths), 16, len(lengths), sum(lengths))
    y1, state1 = _run({n: t[:1] if n == "state" else t for n, t in x.items()}, lengths[:1])
    for longest in (None, max(lengths)):
        y, state = _run(x, lengths, longest)
        assert _same(y[:lengths[0]], y1) and _same(state[0], state1[0])


@pytest.mark.parametrize("lengths", [[40, 60, 80], [24, 100, 33, 200], [48, 64] * 9])
def test_short_requests_among_longer_ones(gpu, lengths):
    x = _inputs(gpu, sum(lengths), 16, len(lengths), sum(lengths))
    y, state = _run(x, lengths, max(lengths))
    at = 0
    for r, n in enumerate(lengths[:4]):
        one = _run(dict(x, state=x["state"][r:r + 1]), [n], n, at)
        _close((y[at:at + n], state[r:r + 1]), one)
        at += n


@pytest.mark.parametrize("longest", [1, 7, 48, 100, 10**6])
def test_any_longest_gives_right_results(gpu, longest):
    lengths = [40, 3, 90, 0, 47]
    x = _inputs(gpu, sum(lengths), 16, len(lengths), 7)
    _close(_run(x, lengths, longest), _run(x, lengths))


@pytest.mark.parametrize("width,requests", [(2, 4), (4, 2), (8, 8), (8, 17)])
def test_windows_and_decode_steps(gpu, width, requests):
    from mini_sglang_amd_kernel import gdn_state_inplace

    x = _inputs(gpu, width * requests, 16, requests, width)
    got = _run(x, [width] * requests, width)
    state, steps = x["state"].clone(), []
    for t in range(width):
        steps.append(gdn_state_inplace(*(x[n][t::width].contiguous() for n in ("q", "k", "v", "g", "beta")), state,
                                       torch.arange(requests, dtype=torch.int32, device=gpu), None, single_token_mode=True))
    _close(got, (torch.stack(steps, 1).flatten(0, 1), state))


def test_the_backend_gives_the_longest(gpu):
    from mini_sglang_amd.attention import GDNBackend

    lengths = [40] * 8
    x = _inputs(gpu, sum(lengths), 16, len(lengths), 3)
    with_it, without = _run(x, lengths, 40), _run(x, lengths)
    assert not _same(with_it[1], without[1])  # two kernels
    state = x["state"].clone()
    backend = GDNBackend(SimpleNamespace(device=gpu, temporal_state=lambda layer: state))
    batch = SimpleNamespace(reqs=[SimpleNamespace(mamba_slot=r, extend_len=n) for r, n in enumerate(lengths)], is_decode=False,
                            mamba_slot_ids=None, mamba_prefill_indptr=None)
    backend.prepare_batch(batch)
    y = backend.forward(*(x[n] for n in ("q", "k", "v", "g", "beta")), 0, batch)
    assert _same(y, with_it[0]) and _same(state, with_it[1])
    # offsets of the caller's own: as without
    state.copy_(x["state"])
    batch.mamba_prefill_indptr = batch.mamba_prefill_indptr.clone()
    y = backend.forward(*(x[n] for n in ("q", "k", "v", "g", "beta")), 0, batch)
    assert _same(y, without[0]) and _same(state, without[1])
    # a window whose width the batch carries, and its replay
    batch.mamba_scratch_slots, batch.mamba_verify_indptr, batch.mamba_verify_width = batch.mamba_slot_ids, batch.mamba_prefill_indptr, 40
    batch.gdn_verify_captured = None
    state.copy_(x["state"])
    y = backend.forward_verify(*(x[n] for n in ("q", "k", "v", "g", "beta")), 0, batch)
    assert _same(y, with_it[0]) and _same(state, with_it[1])
