"""gdn_state_inplace on requests long enough for the chunk kernel, against the float64 oracle: lengths at
the edges of its blocks of 16 and chunks of 64, several requests of unequal length (one without tokens, more
workgroups than compute units), every ratio of value to key heads, strided inputs, decays of 0 and 1."""
import numpy as np
import pytest
import torch

from oracle import gdn_state_oracle as go

pytestmark = pytest.mark.gpu


def _inputs(rng, tokens, hk, hv, slots, decay):
    bf = lambda a: go._bf16_round(a.astype(np.float32))
    unit = lambda a: a / np.linalg.norm(a, axis=-1, keepdims=True)
    g = 1 / (1 + np.exp(-3 - 3 * rng.standard_normal((tokens, hv))))
    if decay == "zeros":
        g[rng.random((tokens, hv)) < 0.05] = 0.0
    elif decay == "ones":
        g[:] = 1.0
    d = dict(q=bf(unit(rng.standard_normal((tokens, hk, 128)))), k=bf(unit(rng.standard_normal((tokens, hk, 128)))),
             v=bf(rng.standard_normal((tokens, hv, 128))), g=bf(g), beta=bf(1 / (1 + np.exp(-rng.standard_normal((tokens, hv))))))
    return d, (0.1 * rng.standard_normal((slots, hv, 128, 128))).astype(np.float32)


@pytest.mark.parametrize("lengths,hk,hv,decay", [
    ([48], 2, 2, "some"), ([63], 2, 4, "zeros"), ([64], 2, 4, "ones"), ([65], 1, 3, "some"), ([129], 2, 4, "zeros"),
    ([193], 4, 4, "some"), ([100, 0, 1, 250, 64], 2, 6, "zeros"), ([40 + 9 * i for i in range(20)], 8, 8, "some")])
def test_against_the_oracle(gpu, lengths, hk, hv, decay):
    from mini_sglang_amd_kernel import gdn_state_inplace

    rng = np.random.default_rng(sum(lengths) + hv)
    batch, total = len(lengths), sum(lengths)
    d, state = _inputs(rng, total, hk, hv, batch + 2, decay)
    slots = rng.permutation(batch + 2)[:batch].astype(np.int32)
    indptr = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)
    want_y, want_st = go.gdn_state_inplace(d["q"], d["k"], d["v"], d["g"], d["beta"], state, slots, indptr, round_output=False)
    bf = lambda a: torch.from_numpy(a).to(torch.bfloat16).to(gpu)
    # q, k, v as views of one projection, as a model hands them over
    proj = torch.cat([bf(d["q"]).flatten(1), bf(d["k"]).flatten(1), bf(d["v"]).flatten(1)], dim=1)
    q, k, v = (t.unflatten(1, (-1, 128)) for t in proj.split([hk * 128, hk * 128, hv * 128], dim=1))
    st, ids, ip = torch.from_numpy(state.copy()).to(gpu), torch.from_numpy(slots).to(gpu), torch.from_numpy(indptr).to(gpu)
    print(f"gdn chunks {lengths[:5]} hk {hk} hv {hv} {decay}", flush=True)
    y = gdn_state_inplace(q, k, v, bf(d["g"]), bf(d["beta"]), st, ids, ip)
    torch.cuda.synchronize()
    got_y, got_st = y.float().cpu().numpy(), st.cpu().numpy()
    # the state is fp32 arithmetic, y is rounded to bf16 once
    np.testing.assert_allclose(got_st, want_st, rtol=0, atol=2e-6 * max(1.0, np.abs(want_st).max()))
    assert (np.abs(got_y - want_y) <= 2.0 ** -8 * np.abs(want_y) + 1e-5).all()
    other = np.setdiff1d(np.arange(batch + 2), slots)
    np.testing.assert_array_equal(got_st[other], state[other])
