"""Gated delta rule over requests of several hundred tokens: the two launches that a workspace makes possible against the one
launch, bit for bit (both make the same products in the same order), at lengths around the chunks of 64 and the steps from
halves to quarters of a head: alone, beside others, more requests than a wave has lanes, requests without tokens, strided rows, values
that are not finite.  The one launch is checked against the float64 oracle elsewhere; here one launch of each kind is too."""
import numpy as np
import pytest
import torch

from oracle import gdn_state_oracle as go
from test_gpu_gdn_chunk import _inputs

pytestmark = pytest.mark.gpu


def _launch(x, lengths, hk, hv, state, workspace, short=0):
    from mini_sglang_amd_kernel import _lib

    lib, total, batch = _lib.load(), sum(lengths), len(lengths)
    ip = torch.tensor(np.cumsum([0] + lengths), dtype=torch.int32, device=state.device)
    ids = torch.arange(batch, dtype=torch.int32, device=state.device).flip(0).contiguous()
    y = torch.full((total, hv, 128), 7.0, dtype=torch.bfloat16, device=state.device)
    need = lib.msgl_gdn_state_workspace_bytes(total, batch, hv, 0)
    assert need > 0
    need -= short
    ws = torch.full((need,), 0xff, dtype=torch.uint8, device=state.device) if workspace else None  # NaN wherever it is not written
    rc = lib.msgl_gdn_state_inplace_in(*(x[n].data_ptr() for n in ("q", "k", "v", "g", "beta")), state.data_ptr(), ids.data_ptr(),
                                       ip.data_ptr(), y.data_ptr(), total, batch, hk, hv, 128, 128, state.shape[0], state.stride(0),
                                       *(x[n].stride(0) for n in ("q", "k", "v")), 0, ws.data_ptr() if workspace else None,
                                       need if workspace else 0, torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    torch.cuda.synchronize()
    # the first request has tokens: in two launches the record of its first chunk is there, and nothing where the room is too small
    assert ws is None or bool((ws[:20480] == 0xff).all()) is (short > 0)
    assert short == 0 or bool((ws == 0xff).all())
    return y, state


def _bits(t):
    return torch.where(t.isnan(), torch.zeros((), dtype=t.dtype, device=t.device) + 12345, t).view(torch.int16 if t.dtype == torch.bfloat16 else torch.int32)


@pytest.mark.parametrize("what", [None, "v", "k", "q", "state"])
@pytest.mark.parametrize("lengths,hk,hv", [
    ([384], 16, 32), ([447], 4, 4), ([1025], 2, 6), ([500, 449], 16, 32), ([64, 1400, 1], 16, 32), ([2300, 1, 0, 640], 8, 32),
    ([700, 33, 1500, 65, 1200, 300], 16, 48), ([560] * 9, 16, 32), ([128] * 9, 16, 32),
    ([1, 1300, 60, 0, 90, 85], 16, 32), ([600] * 64 + [0, 1400, 601], 1, 2)])
def test_two_launches_are_one(gpu, lengths, hk, hv, what):
    print(f"gdn long {lengths[:6]} hk {hk} hv {hv} {what}", flush=True)
    rng = np.random.default_rng(sum(lengths) + hv)
    d, state = _inputs(rng, sum(lengths), hk, hv, len(lengths), "zeros")
    bf = lambda a: torch.from_numpy(a).to(torch.bfloat16).to(gpu)  # noqa: E731
    proj = torch.cat([bf(d[n]).flatten(1) for n in ("q", "k", "v")], dim=1)  # views of one projection
    x = dict(zip(("q", "k", "v"), (t.unflatten(1, (-1, 128)) for t in proj.split([hk * 128, hk * 128, hv * 128], dim=1))), g=bf(d["g"]), beta=bf(d["beta"]))
    start = torch.from_numpy(state).to(gpu)
    if what == "state":
        start[-1, 0, 70, 9] = float("inf")
    elif what:
        x[what][sum(lengths) // 3, 0, 5] = float("nan") if what == "v" else float("inf")
    y1, s1 = _launch(x, lengths, hk, hv, start.clone(), False)
    y2, s2 = _launch(x, lengths, hk, hv, start.clone(), True)
    assert torch.equal(_bits(y2), _bits(y1)) and torch.equal(_bits(s2), _bits(s1))
    assert what is not None or bool(y2.isfinite().all() and s2.isfinite().all())
    y3, s3 = _launch(x, lengths, hk, hv, start.clone(), True, short=1)
    assert torch.equal(_bits(y3), _bits(y1)) and torch.equal(_bits(s3), _bits(s1))


@pytest.mark.parametrize("lengths", [[385], [130, 1300, 64]])
def test_against_the_oracle(gpu, lengths):
    print(f"gdn long oracle {lengths}", flush=True)
    rng = np.random.default_rng(sum(lengths))
    d, state = _inputs(rng, sum(lengths), 2, 4, len(lengths), "some")
    x = {n: torch.from_numpy(d[n]).to(torch.bfloat16).to(gpu) for n in ("q", "k", "v", "g", "beta")}
    y, st = _launch(x, lengths, 2, 4, torch.from_numpy(state.copy()).to(gpu), True)
    slots, indptr = np.arange(len(lengths), dtype=np.int32)[::-1].copy(), np.cumsum([0] + lengths).astype(np.int32)
    want_y, want_st = go.gdn_state_inplace(d["q"], d["k"], d["v"], d["g"], d["beta"], state, slots, indptr, round_output=False)
    # bounds as for the one launch: fp32 arithmetic in the state, y rounded to bf16 once
    np.testing.assert_allclose(st.cpu().numpy(), want_st, rtol=0, atol=2e-6 * max(1.0, np.abs(want_st).max()))
    assert (np.abs(y.float().cpu().numpy() - want_y) <= 2.0 ** -8 * np.abs(want_y) + 1e-5).all()


def _operator_inputs(gpu, total, hk, hv, pad=0):
    g = torch.Generator(device=gpu)
    g.manual_seed(total)
    rand = lambda *s: torch.randn(s, generator=g, device=gpu).bfloat16()  # noqa: E731
    unit = lambda t: t / t.float().norm(dim=-1, keepdim=True).bfloat16()  # noqa: E731
    v = rand(total, hv * 128 + pad)[:, :hv * 128].unflatten(1, (hv, 128))
    return unit(rand(total, hk, 128)), unit(rand(total, hk, 128)), v, torch.rand((total, hv), generator=g, device=gpu).bfloat16(), \
        torch.rand((total, hv), generator=g, device=gpu).bfloat16(), torch.zeros((2, hv, 128, 128), device=gpu)


def _operator(x, state):
    from mini_sglang_amd_kernel import gdn_state_inplace

    ip = torch.tensor([0, x[0].shape[0]], dtype=torch.int32, device=state.device)
    return gdn_state_inplace(*x[:5], state, torch.ones(1, dtype=torch.int32, device=state.device), ip, False)


def test_without_room_for_the_systems(gpu):
    """Memory that only makes the call faster: where there is none the call goes without it, to the same bits."""
    from mini_sglang_amd_kernel import _lib

    total, hk, hv = 8192, 16, 32
    need = _lib.load().msgl_gdn_state_workspace_bytes(total, 1, hv, 0)
    x = _operator_inputs(gpu, total, hk, hv)
    s1, s2 = x[5].clone(), x[5].clone()
    y1 = _operator(x, s1)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    room, hogs = torch.empty_like(y1), []  # for the result, which then comes from the cache
    assert need > room.numel() * 2
    torch.cuda.set_per_process_memory_fraction(torch.cuda.memory_reserved() / torch.cuda.mem_get_info()[1])
    print("gdn without room", flush=True)
    try:
        with pytest.raises(torch.cuda.OutOfMemoryError):
            while True:  # what other tests left cached
                hogs.append(torch.empty(need, dtype=torch.uint8, device=gpu))
        del room
        y2 = _operator(x, s2)
        with pytest.raises(torch.cuda.OutOfMemoryError):
            torch.empty(need, dtype=torch.uint8, device=gpu)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert torch.equal(_bits(y2), _bits(y1)) and torch.equal(_bits(s2), _bits(s1))


@pytest.mark.parametrize("pad,rows", [(4, 0), (0, 1)])
def test_no_memory_where_it_is_not_used(gpu, tuning, pad, rows):
    """Rows of v that the chunked form does not take, and the token kernel set by hand."""
    from mini_sglang_amd_kernel import _lib

    x = _operator_inputs(gpu, 1024, 4, 8, pad)
    tuning(_lib.TUNE_GDN_ROWS, rows)
    state = x[5].clone()
    print(f"gdn no memory pad {pad} rows {rows}", flush=True)
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    y = _operator(x, state)
    assert torch.cuda.max_memory_allocated() - before < y.numel() * 2 + (1 << 16)
