"""A few tokens per request: the token kernel with 1, 2 and 4 state rows to a lane group, on both sides of where it changes over,
against the float64 oracle."""
import numpy as np
import pytest
import torch

from oracle import gdn_state_oracle as go
from test_gpu_gdn_chunk import _inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch,hk,hv", [(1, 16, 32), (1, 16, 63), (2, 16, 32), (5, 16, 32), (1, 5, 255), (8, 16, 32), (17, 16, 48)])
def test_short_requests(gpu, batch, hk, hv):
    from mini_sglang_amd_kernel import gdn_state_inplace

    hk = hk if hv % hk == 0 else 1
    lengths = [3 + (5 * i) % 7 for i in range(batch)]
    rng = np.random.default_rng(batch + hv)
    d, state = _inputs(rng, sum(lengths), hk, hv, batch, "some")
    indptr = np.cumsum([0] + lengths).astype(np.int32)
    slots = np.arange(batch, dtype=np.int32)[::-1].copy()
    want_y, want_st = go.gdn_state_inplace(d["q"], d["k"], d["v"], d["g"], d["beta"], state, slots, indptr, round_output=False)
    bf = lambda n: torch.from_numpy(d[n]).to(torch.bfloat16).to(gpu)  # noqa: E731
    st = torch.from_numpy(state.copy()).to(gpu)
    print(f"gdn rows batch {batch} hk {hk} hv {hv}", flush=True)
    y = gdn_state_inplace(bf("q"), bf("k"), bf("v"), bf("g"), bf("beta"), st, torch.from_numpy(slots).to(gpu), torch.from_numpy(indptr).to(gpu))
    torch.cuda.synchronize()
    # fp32 arithmetic in the state, y rounded to bf16 once
    np.testing.assert_allclose(st.cpu().numpy(), want_st, rtol=0, atol=2e-6 * max(1.0, np.abs(want_st).max()))
    assert (np.abs(y.float().cpu().numpy() - want_y) <= 2.0 ** -8 * np.abs(want_y) + 1e-5).all()
