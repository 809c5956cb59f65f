"""gdn_state_inplace on requests that go in chunks of 16 tokens, against the float64 oracle: lengths at the edges of its
chunks and groups of four, one to hundreds of heads (half a head and a whole one to a workgroup), requests without tokens,
decays of 0 and 1; and infinities and NaN, which stay where the recurrence carries them."""
import numpy as np
import pytest
import torch

from oracle import gdn_state_oracle as go

pytestmark = pytest.mark.gpu


def _run(gpu, lengths, hk, hv, decay, seed, place=None):
    """-> (y, state), the oracle's, and the state before; `place`: (name, index, value) written into the inputs."""
    from mini_sglang_amd_kernel import gdn_state_inplace

    rng = np.random.default_rng(seed)
    batch, total = len(lengths), sum(lengths)
    bf = lambda a: go._bf16_round(a.astype(np.float32))  # noqa: E731
    unit = lambda a: a / np.linalg.norm(a, axis=-1, keepdims=True)  # noqa: E731
    g = 1 / (1 + np.exp(-3 - 3 * rng.standard_normal((total, hv))))
    if decay == "zeros":
        g[rng.random((total, hv)) < 0.1] = 0.0
    elif decay == "ones":
        g[:] = 1.0
    d = dict(q=bf(unit(rng.standard_normal((total, hk, 128)))), k=bf(unit(rng.standard_normal((total, hk, 128)))),
             v=bf(rng.standard_normal((total, hv, 128))), g=bf(g), beta=bf(1 / (1 + np.exp(-rng.standard_normal((total, hv))))))
    d["state"] = (0.1 * rng.standard_normal((batch + 2, hv, 128, 128))).astype(np.float32)
    slots = rng.permutation(batch + 2)[:batch].astype(np.int32)
    if place:
        name, at, value = place
        d[name][(slots[at[0]], *at[1:]) if name == "state" else at] = value
    indptr = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)
    with np.errstate(all="ignore"):
        want = go.gdn_state_inplace(*(d[n] for n in ("q", "k", "v", "g", "beta", "state")), slots, indptr, round_output=False)
    to = lambda a: torch.from_numpy(a).to(torch.bfloat16).to(gpu)  # noqa: E731
    # q, k, v as views of one projection, as a model hands them over
    proj = torch.cat([to(d["q"]).flatten(1), to(d["k"]).flatten(1), to(d["v"]).flatten(1)], dim=1)
    q, k, v = (t.unflatten(1, (-1, 128)) for t in proj.split([hk * 128, hk * 128, hv * 128], dim=1))
    state = torch.from_numpy(d["state"].copy()).to(gpu)
    print(f"gdn short {lengths[:6]} of {batch} hk {hk} hv {hv} {decay} {place}", flush=True)
    y = gdn_state_inplace(q, k, v, to(d["g"]), to(d["beta"]), state, torch.from_numpy(slots).to(gpu), torch.from_numpy(indptr).to(gpu),
                         max_len_extend=max(lengths))
    torch.cuda.synchronize()
    return (y.float().cpu().numpy(), state.cpu().numpy()), want, d["state"], slots


@pytest.mark.parametrize("lengths,hk,hv,decay", [
    ([9], 2, 2, "some"), ([15], 1, 1, "zeros"), ([16], 2, 4, "ones"), ([17], 1, 3, "some"), ([31], 4, 4, "zeros"), ([32], 2, 6, "some"),
    ([33, 0, 16, 1, 48], 2, 4, "zeros"), ([64, 2, 3, 65, 5], 2, 8, "some"), ([1, 129, 0, 2, 7, 3], 4, 16, "zeros"),
    ([4] * 5, 16, 32, "some"), ([48, 20, 63, 17, 30], 16, 32, "ones"), ([2 + 3 * i for i in range(9)], 16, 32, "zeros"),
    ([(37 * i) % 150 for i in range(18)], 4, 32, "some"), ([16 * (i % 5 + 1) for i in range(20)], 8, 32, "zeros")])
def test_against_the_oracle(gpu, lengths, hk, hv, decay):
    (y, state), (want_y, want_state), before, slots = _run(gpu, lengths, hk, hv, decay, sum(lengths) + hv)
    # the state is fp32 arithmetic, y is rounded to bf16 once
    np.testing.assert_allclose(state, want_state, rtol=0, atol=2e-6 * max(1.0, np.abs(want_state).max()))
    assert (np.abs(y - want_y) <= 2.0 ** -8 * np.abs(want_y) + 1e-5).all()
    other = np.setdiff1d(np.arange(len(before)), slots)
    np.testing.assert_array_equal(state[other], before[other])


@pytest.mark.parametrize("lengths,hk,hv", [([30, 20, 35], 2, 4), ([18, 40, 9, 25, 31], 16, 32)])
@pytest.mark.parametrize("name,at,value", [
    ("v", (5, 1, 37), np.inf), ("v", (17, 1, 127), np.nan), ("k", (16, 0, 5), np.nan), ("k", (3, 0, 64), -np.inf), ("q", (11, 1, 99), np.inf),
    ("q", (15, 0, 0), np.nan), ("g", (9, 2), np.nan), ("g", (16, 3), np.inf), ("beta", (2, 3), np.inf), ("state", (1, 2, 17, 64), np.nan)])
def test_values_that_are_not_finite_stay_in_their_place(gpu, lengths, hk, hv, name, at, value):
    _same_places(*_run(gpu, lengths, hk, hv, "some", hv, (name, at, value))[:2])


# beyond the first four chunks of a request of nine, and behind it
@pytest.mark.parametrize("name,at,value", [
    ("v", (64, 1, 37), np.inf), ("k", (100, 0, 5), np.nan), ("k", (129, 1, 64), -np.inf), ("q", (79, 1, 99), np.inf), ("g", (127, 2), np.nan),
    ("beta", (65, 3), np.inf), ("v", (128, 0, 127), np.nan), ("v", (135, 0, 0), np.inf)])
def test_values_that_are_not_finite_in_later_groups(gpu, name, at, value):
    _same_places(*_run(gpu, [130, 10, 4, 6, 3, 2, 9, 1], 2, 4, "some", 11, (name, at, value))[:2])


def _same_places(got, want):
    for a, b, atol, rtol in zip(got, want, (1e-5, 2e-6 * 4), (2.0 ** -8, 2e-6)):
        finite = np.isfinite(b)
        np.testing.assert_array_equal(np.isfinite(a), finite)
        np.testing.assert_array_equal(a[~finite], b[~finite])  # NaN where NaN, and infinities of one sign
        assert (np.abs(a[finite] - b[finite]) <= atol + rtol * np.abs(b[finite])).all()
