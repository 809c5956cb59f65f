"""The chunk kernel of the gated delta rule runs requests that the chip has room for on twice as many workgroups, state
and output waves in pairs.  Every request has the same bits either way: alone (in pairs at 32 value heads on 256 compute
units) and as one of several of its length (whole), in a launch of both kinds, and with values that are not finite, which
send the request through the token path.  The launch alone is checked against the float64 oracle elsewhere."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

HV = 32


def _inputs(gpu, tokens, hk, requests, seed):
    g = torch.Generator(device=gpu)
    g.manual_seed(seed)
    rand = lambda *s: torch.randn(s, generator=g, device=gpu)  # noqa: E731
    unit = lambda t: t / t.norm(dim=-1, keepdim=True)  # noqa: E731
    return dict(q=unit(rand(tokens, hk, 128)).bfloat16(), k=unit(rand(tokens, hk, 128)).bfloat16(), v=rand(tokens, HV, 128).bfloat16(),
                g=torch.sigmoid(3 + 3 * rand(tokens, HV)).bfloat16(), beta=torch.sigmoid(rand(tokens, HV)).bfloat16(),
                state=0.1 * rand(requests, HV, 128, 128))


def _run(x, lengths, state):
    from mini_sglang_amd_kernel import gdn_state_inplace

    ip = torch.tensor(np.cumsum([0] + lengths), dtype=torch.int32, device=state.device)
    y = gdn_state_inplace(x["q"], x["k"], x["v"], x["g"], x["beta"], state, torch.arange(len(lengths), dtype=torch.int32, device=state.device), ip)
    torch.cuda.synchronize()
    return y, state


def _bits(t):
    return torch.where(t.isnan(), torch.zeros((), dtype=t.dtype, device=t.device) + 12345, t).view(torch.int16 if t.dtype == torch.bfloat16 else torch.int32)


@pytest.mark.parametrize("what", [None, "v", "q", "k", "state"])
@pytest.mark.parametrize("length,hk", [(48, 16), (63, 32), (64, 8), (65, 16), (128, 16), (129, 4), (333, 16)])
def test_alone_and_as_one_of_many(gpu, length, hk, what):
    print(f"gdn pairs length {length} hk {hk} {what}", flush=True)
    x = _inputs(gpu, length, hk, 1, length + hk)
    if what == "state":
        x["state"][0, 3, 70, 9] = float("inf")
    elif what:
        x[what][length // 2, 1, 5] = float("nan") if what == "v" else float("inf")
    y, state = _run(x, [length], x["state"].clone())
    many = {n: t.repeat(9, *[1] * (t.dim() - 1)) for n, t in x.items()}
    y9, state9 = _run(many, [length] * 9, many["state"])
    assert what is not None or bool(y.isfinite().all())
    for r in range(9):
        assert torch.equal(_bits(y9[r * length:(r + 1) * length]), _bits(y))
        assert torch.equal(_bits(state9[r]), _bits(state[0]))


@pytest.mark.parametrize("lengths", [[24], [20, 21, 40], [100, 2900, 60, 64], [70, 0, 4000, 1, 50], [300, 300], [64, 1000, 65], [40] * 66])
def test_both_kinds_in_one_launch(gpu, lengths):
    print(f"gdn pairs lengths {lengths[:6]}", flush=True)
    x = _inputs(gpu, sum(lengths), 16, len(lengths), sum(lengths))
    y, state = _run(x, lengths, x["state"].clone())
    at = np.cumsum([0] + lengths)
    for r, n in enumerate(lengths):
        if n == 0:
            assert torch.equal(state[r], x["state"][r])
        elif r < 8:
            one = {k: t[at[r]:at[r + 1]].contiguous() for k, t in x.items() if k != "state"}
            y1, state1 = _run(one, [n], x["state"][r:r + 1].clone())
            assert n < 24 or torch.equal(_bits(y[at[r]:at[r + 1]]), _bits(y1))
            assert n < 24 or torch.equal(_bits(state[r]), _bits(state1[0]))
            assert (y[at[r]:at[r + 1]].float() - y1.float()).abs().max() <= 2.0 ** -7 * y1.float().abs().max()
