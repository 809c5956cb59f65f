"""Infinities and NaN in the chunk kernel of the gated delta rule: they stay where the recurrence carries them (never to an
earlier token, another row, another head or another request), and everything else is the finite result.  Against the
float64 oracle and against the token kernel."""
import numpy as np
import pytest
import torch

from oracle import gdn_state_oracle as go

pytestmark = pytest.mark.gpu

HK, HV, LENGTHS = 2, 4, [200, 64, 97]
# where a value goes: what, token (of the first request; its chunks are 64 tokens), value
CASES = [("v", 70, np.inf), ("v", 127, -np.inf), ("v", 199, np.nan), ("v", 0, np.inf), ("k", 100, np.nan), ("k", 64, np.inf),
         ("q", 90, np.nan), ("q", 191, np.inf), ("q", 195, -np.inf), ("g", 130, np.nan), ("g", 75, np.inf), ("beta", 40, np.nan),
         ("beta", 127, np.inf), ("state", 0, np.nan), ("state", 0, np.inf)]


def _inputs(seed):
    rng = np.random.default_rng(seed)
    n = sum(LENGTHS)
    bf = lambda a: go._bf16_round(a.astype(np.float32))  # noqa: E731
    unit = lambda a: a / np.linalg.norm(a, axis=-1, keepdims=True)  # noqa: E731
    d = dict(q=bf(unit(rng.standard_normal((n, HK, 128)))), k=bf(unit(rng.standard_normal((n, HK, 128)))), v=bf(rng.standard_normal((n, HV, 128))),
             g=bf(1 / (1 + np.exp(-3 - rng.standard_normal((n, HV))))), beta=bf(1 / (1 + np.exp(-rng.standard_normal((n, HV))))))
    d["state"] = (0.1 * rng.standard_normal((len(LENGTHS) + 1, HV, 128, 128))).astype(np.float32)
    return d


def _run(d, gpu):
    from mini_sglang_amd_kernel import gdn_state_inplace

    t = {n: torch.from_numpy(a.copy()).to(gpu) for n, a in d.items()}
    x = {n: t[n].bfloat16() for n in ("q", "k", "v", "g", "beta")}
    ip = torch.tensor(np.cumsum([0] + LENGTHS), dtype=torch.int32, device=gpu)
    slots = torch.arange(1, len(LENGTHS) + 1, dtype=torch.int32, device=gpu)
    y = gdn_state_inplace(x["q"], x["k"], x["v"], x["g"], x["beta"], t["state"], slots, ip)
    torch.cuda.synchronize()
    return y.float().cpu().numpy(), t["state"].cpu().numpy()


def _same(got, want, atol, rtol, what):
    finite = np.isfinite(want)
    np.testing.assert_array_equal(np.isfinite(got), finite, err_msg=what)
    np.testing.assert_array_equal(got[~finite], want[~finite], err_msg=what)  # NaN where NaN, and infinities of one sign
    assert (np.abs(got[finite] - want[finite]) <= atol + rtol * np.abs(want[finite])).all(), what


@pytest.mark.parametrize("what,token,value", CASES)
def test_values_that_are_not_finite_stay_in_their_place(gpu, tuning, what, token, value):
    from mini_sglang_amd_kernel import _lib

    d = _inputs(token)
    where = {"v": (token, 1, 37), "k": (token, 0, 5), "q": (token, 1, 99), "g": (token, 2), "beta": (token, 3), "state": (1, 2, 17, 64)}
    d[what][where[what]] = value
    print(f"gdn chunks with {value} in {what} at token {token}", flush=True)
    y, state = _run(d, gpu)
    with np.errstate(all="ignore"):
        want_y, want_state = go.gdn_state_inplace(*(d[n] for n in ("q", "k", "v", "g", "beta", "state")), np.arange(1, 4, dtype=np.int32),
                                                  np.cumsum([0] + LENGTHS).astype(np.int32), round_output=False)
    finite = np.isfinite(want_state)
    _same(state, want_state, 2e-6 * max(1.0, np.abs(want_state[finite]).max()), 0.0, "state")
    _same(y, want_y, 1e-5, 2.0 ** -8, "y")
    if what != "state":
        assert np.isfinite(y[:token]).all() and not np.isfinite(y[token]).all()
    tuning(_lib.TUNE_GDN_ROWS, 1)  # the token kernel
    tok_y, tok_state = _run(d, gpu)
    _same(state, tok_state, 2e-6 * max(1.0, np.abs(want_state[finite]).max()), 0.0, "state, token kernel")
    _same(y, tok_y, 1e-5, 2.0 ** -7, "y, token kernel")


@pytest.mark.parametrize("scale", [30.0, 300.0])
def test_keys_so_long_that_the_recurrence_overflows(gpu, tuning, scale):
    """The inverse of a chunk's triangle overflows long before its last token; tokens before the overflow keep their
    values.  A token multiplies what came before by a few hundred or more, so rounding moves the first value that is not
    finite by one token at most."""
    from mini_sglang_amd_kernel import _lib

    d = _inputs(3)
    d["k"] = go._bf16_round(d["k"] * np.float32(scale))
    print(f"gdn chunks, keys of length {scale}", flush=True)
    y, state = _run(d, gpu)
    tuning(_lib.TUNE_GDN_ROWS, 1)
    tok_y, tok_state = _run(d, gpu)

    def first_bad(a):  # per request, head and row: tokens before the first that is not finite
        bad = ~np.isfinite(a)
        return np.array([np.where(x.any(0), x.argmax(0), len(x)) for x in np.split(bad, np.cumsum(LENGTHS)[:-1])])

    got, want = first_bad(y), first_bad(tok_y)
    assert (want < 64).any() and (np.abs(got - want) <= 1).all()
    # the first eight tokens stay far from the overflow: bf16 results of the same values
    early = np.concatenate([np.arange(s, s + 8) for s in np.cumsum([0] + LENGTHS[:-1])])
    limit = 2.0 ** -6 * np.abs(tok_y[early]).max(axis=-1, keepdims=True)
    assert (np.abs(y[early] - tok_y[early]) <= limit).all()
