"""Requests in chunks of 16 tokens on both sides of the numbers of heads and tokens between which their state comes and goes by whole lines:
half a head to a workgroup and a whole one, against the float64 oracle; a request that is not finite among them is gone through again."""
import numpy as np
import pytest

from test_gpu_gdn_short import _run, _same_places

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lengths,hk,hv", [([4] * 127, 1, 1), ([4] * 128, 1, 1), ([17, 4, 33, 9], 4, 32), ([16] * 8, 16, 32), ([17] + [16] * 8, 8, 32),
                                           ([17] * 7, 16, 32), ([17] * 8, 16, 32), ([33] * 19, 16, 32), ([33] * 20, 16, 32), ([32] * 20, 16, 32),
                                           ([33] * 40, 16, 32)])
def test_against_the_oracle(gpu, lengths, hk, hv):
    (y, state), (want_y, want_state), before, slots = _run(gpu, lengths, hk, hv, "some", len(lengths) + hv)
    # bounds as for the rest of the kernel: fp32 arithmetic in the state, y rounded to bf16 once
    np.testing.assert_allclose(state, want_state, rtol=0, atol=2e-6 * max(1.0, np.abs(want_state).max()))
    assert (np.abs(y - want_y) <= 2.0 ** -8 * np.abs(want_y) + 1e-5).all()
    other = np.setdiff1d(np.arange(len(before)), slots)
    np.testing.assert_array_equal(state[other], before[other])


@pytest.mark.parametrize("name,at,value", [("v", (5, 1, 37), np.inf), ("state", (3, 9, 17, 64), np.nan)])
def test_values_that_are_not_finite(gpu, name, at, value):
    _same_places(*_run(gpu, [18, 40, 9, 25], 16, 32, "some", 3, (name, at, value))[:2])
