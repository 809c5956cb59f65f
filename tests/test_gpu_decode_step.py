"""The store of a step (for decode also norm, rotary embedding and store) inside its attention launch, against the
same step as two launches, which the oracle tests pin: at the edges of a wave's 32 keys and of a share, for requests
without keys, for new tokens that are not their request's last keys, for a slot outside the pool, on strided rows,
and from a pool whose new slots hold NaN before the step."""
import pytest
import torch

from mini_sglang_amd.workloads import build_workload
from mini_sglang_amd_kernel import (_lib, decode_step, extend_step, paged_decode_attention, paged_prefill_attention,
                                    qk_norm_rope_store, store_kv_cache)

pytestmark = pytest.mark.gpu

CASES = [  # kv lengths, q heads, kv heads, head_dim, share_len, kv heads per workgroup (0: the default cut; -1: segments)
    ([1], 16, 8, 128, 0, 0),
    ([37, 128, 500, 1023], 16, 8, 128, 0, 0),
    ([31, 32, 33, 64, 65, 0, 127, 128, 129, 257], 32, 8, 128, 128, 1),
    ([2100, 5, 64], 64, 4, 128, 64, 4),
    ([1 + i % 90 for i in range(150)], 16, 8, 128, 0, 0),
    ([600, 0, 1, 255, 256, 257], 16, 2, 256, 0, 0),
    ([1500, 40, 32], 24, 4, 256, 64, 4),
    ([0, 31, 32, 33, 64, 65, 0, 127, 128, 129, 257, 0], 32, 8, 128, -1, 9),
    ([1, 1, 1], 16, 8, 128, -1, 1),
    ([0, 0], 16, 8, 128, -1, 3),
    ([1 + i % 90 for i in range(150)], 24, 3, 128, -1, 60),
    ([2100, 5, 0, 193], 16, 2, 256, -1, 20),
]


def _step(gpu, lens, n_q, n_kv, d, dtype, seed):
    """The step's tensors: q, k, v as views of one projection, and a pool with NaN in the new slots."""
    wl = build_workload("step", "decode", seed=seed, n_q=n_q, n_kv=n_kv, head_dim=d, kv_lens=lens).to(gpu)
    g = torch.Generator(device=gpu)
    g.manual_seed(seed)
    b = len(lens)
    qkv = torch.randn((b, n_q + 2 * n_kv, d), generator=g, device=gpu).to(dtype)
    slots = wl.k_cache.shape[0]
    kc, vc = (torch.cat([c.to(dtype), c.to(dtype)]) for c in (wl.k_cache, wl.v_cache))  # the upper half is nobody's
    loc = torch.arange(b, dtype=torch.int32, device=gpu) + slots
    for i, n in enumerate(lens):  # as a rule a request's last slot is the new token's
        if n > 0 and i % 5 != 4:
            loc[i] = wl.kv_indices[int(wl.kv_indptr[i + 1]) - 1]
        if n > 2 and i % 5 == 3:  # ... or stands in the middle
            loc[i] = wl.kv_indices[int(wl.kv_indptr[i]) + n // 2]
    for c in (kc, vc):
        c[loc.long()] = float("nan")
    for i, n in enumerate(lens):  # a last slot that is not the new token's holds a row
        if n > 0 and i % 5 == 4:
            for c in (kc, vc):
                c[wl.kv_indices[int(wl.kv_indptr[i + 1]) - 1].long()] = 0.5
    if b > 2:
        loc[2] = kc.shape[0] + 7  # outside the pool: nothing is stored
        at = wl.kv_indices[int(wl.kv_indptr[3]) - 1].long()
        if lens[2] > 0:
            kc[at] = vc[at] = 0.25
    parts = (qkv[:, :n_q], qkv[:, n_q:n_q + n_kv], qkv[:, n_q + n_kv:])
    return wl, parts, loc, kc, vc


@pytest.mark.parametrize("lens,n_q,n_kv,d,share,heads", CASES)
@pytest.mark.parametrize("mode", ["bf16", "f16", "norm"])
def test_one_launch_is_two(gpu, tuning, lens, n_q, n_kv, d, share, heads, mode):
    dtype = torch.float16 if mode == "f16" else torch.bfloat16
    wl, (q, k, v), loc, kc, vc = _step(gpu, lens, n_q, n_kv, d, dtype, len(lens) + d)
    norm = {}
    if mode == "norm":
        g = torch.Generator(device=gpu)
        g.manual_seed(1)
        w = (1 + 0.2 * torch.randn((2, d), generator=g, device=gpu)).to(dtype)
        pos = torch.tensor([max(n - 1, 0) + 40000 * (i % 3 == 1) for i, n in enumerate(lens)], dtype=torch.int32, device=gpu)
        norm = dict(q_weight=w[0], k_weight=w[1], positions=pos, eps=1e-6, rope_base=1e6)
    if share >= 0:
        tuning(_lib.TUNE_SHARES, share | heads << 20)
    elif mode == "norm":
        pytest.skip("norm weights: shares only")
    else:  # segments of at least 64 keys
        tuning(_lib.TUNE_SHARES, -1)
        tuning(_lib.TUNE_SEGMENTS, heads)
        tuning(_lib.TUNE_MIN_SEGMENT, 64)
    kc2, vc2 = kc.clone(), vc.clone()
    print(f"decode step {lens[:4]} {n_q}/{n_kv} d{d} {mode} cut {share} x {heads}", flush=True)
    got = decode_step(q, k, v, loc, kc, vc, wl.kv_indptr, wl.kv_indices, wl.num_kv_splits, sm_scale=wl.sm_scale, **norm)
    assert got is not None
    if mode == "norm":
        q = qk_norm_rope_store(q, k, v, w[0], w[1], pos, loc, kc2, vc2, eps=1e-6, rope_base=1e6)
    else:
        store_kv_cache(kc2, vc2, loc, k, v)
    want = paged_decode_attention(q, kc2, vc2, wl.kv_indptr, wl.kv_indices, wl.num_kv_splits, wl.sm_scale, 32)
    same = lambda a, b: torch.equal(a.view(torch.int16), b.view(torch.int16))  # noqa: E731
    assert bool(torch.isfinite(got).all())
    assert same(vc, vc2)
    assert same(kc, kc2)
    # the new key's weight and its products are fp32 where the other launch has them in 16 bits: a step of the result's
    # type, and where few keys share the weight half a 16-bit step of the new key's own
    diff = (got.float() - want.float()).abs()
    assert float(diff.max()) <= 2e-2 and float(diff.mean()) <= 1e-3, (float(diff.max()), float(diff.mean()))


def test_what_is_left_to_the_two_calls(gpu, monkeypatch):
    """None, and nothing done: rows that need a copy, a large launch, index validation on."""
    wl, (q, k, v), loc, kc, vc = _step(gpu, [40, 70], 16, 8, 128, torch.bfloat16, 3)
    before = kc.clone()
    args = lambda k=k: (q, k, v, loc, kc, vc, wl.kv_indptr, wl.kv_indices, wl.num_kv_splits)  # noqa: E731
    turned = k.transpose(1, 2).contiguous().transpose(1, 2)
    assert decode_step(*args(turned), sm_scale=0.1) is None
    monkeypatch.setenv("MSGL_DEBUG_CHECKS", "1")
    assert decode_step(*args(), sm_scale=0.1) is None
    monkeypatch.setenv("MSGL_DEBUG_CHECKS", "0")
    assert torch.equal(before.view(torch.int16), kc.view(torch.int16))
    assert decode_step(*args(), sm_scale=0.1) is not None
    need = _lib.load().msgl_decode_step_workspace_bytes
    assert need(64, 64 * 4096, 32, 8, 128, 0) == 0  # a large launch
    assert need(1, 20000, 32, 8, 128, 0) > 0 and need(1, 20000, 32, 8, 128, 1) == 0  # segments: without norm weights


# kv lengths before the step, new tokens, q heads, kv heads, head_dim, share_len, max_len_extend below the longest
ROWS = [
    ([0, 31, 32, 33, 257, 700], [8] * 6, 32, 8, 128, 0, 0),
    ([5, 64, 1000, 130, 0, 40, 300], [3, 1, 7, 0, 4, 2, 5], 16, 8, 128, 64, 0),
    ([90, 500], [48, 33], 8, 8, 128, 128, 0),
    ([90, 500, 2100], [11, 12, 5], 32, 8, 128, 512, 0),
    ([0, 1500, 77], [3, 4, 2], 16, 4, 256, 128, 0),
    ([100, 600], [9, 4], 16, 8, 128, 128, 6),
]


@pytest.mark.parametrize("cached,ext,n_q,n_kv,d,share,cap", ROWS)
@pytest.mark.parametrize("cross,window", [(False, 0), (True, 0), (False, 100), (True, 70)])
@pytest.mark.parametrize("places", ["last", "mixed"])
def test_extend_one_launch_is_two(gpu, tuning, cached, ext, n_q, n_kv, d, share, cap, cross, window, places):
    kv = [c + e for c, e in zip(cached, ext)]
    wl = build_workload("step", "prefill", seed=sum(kv), n_q=n_q, n_kv=n_kv, head_dim=d, kv_lens=kv, extend_lens=ext,
                        is_cross_attention=cross, sliding_window_size=window).to(gpu)
    g = torch.Generator(device=gpu)
    g.manual_seed(sum(kv))
    total = sum(ext)
    kvr = torch.randn((total, 2 * n_kv, d), generator=g, device=gpu).bfloat16()
    k, v = kvr[:, :n_kv], kvr[:, n_kv:]
    kc, vc = (torch.cat([c, c]) for c in (wl.k_cache, wl.v_cache))  # the upper half is nobody's
    loc, at = torch.empty(total, dtype=torch.int32, device=gpu), 0
    for b, (c, e) in enumerate(zip(cached, ext)):
        first = int(wl.kv_indptr[b])
        loc[at:at + e] = wl.kv_indices[first + c:first + c + e]
        if places == "mixed" and b % 3 == 0 and e > 1:  # one token elsewhere, its place an old key
            loc[at + 1] = wl.k_cache.shape[0] + b
        if places == "mixed" and b % 3 == 1 and c > e:  # the tokens stand in front of the last keys
            loc[at:at + e] = wl.kv_indices[first + c - e:first + c]
        at += e
    for c in (kc, vc):
        c[loc.long()] = float("nan")
    if places == "mixed" and total > 2:
        loc[total - 1] = kc.shape[0] + 3  # outside the pool: nothing is stored
        kc.nan_to_num_(0.5)
        vc.nan_to_num_(0.5)
    limit = cap or max(ext)
    tuning(_lib.TUNE_SHARES, (share or 96) | 1 << 20)
    tuning(_lib.TUNE_SMALLQ_MAXCOLS, 48)  # whatever the window
    kc2, vc2 = kc.clone(), vc.clone()
    print(f"extend step {cached[:4]} + {ext[:4]} {n_q}/{n_kv} d{d} cross={cross} window={window} {places}", flush=True)
    got = extend_step(wl.q, k, v, loc, kc, vc, wl.qo_indptr, wl.kv_indptr, wl.kv_indices, wl.prefix_lens, sm_scale=wl.sm_scale,
                      max_len_extend=limit, is_cross_attention=cross, sliding_window_size=window)
    assert got is not None
    store_kv_cache(kc2, vc2, loc, k, v)
    want = paged_prefill_attention(wl.q, kc2, vc2, wl.qo_indptr, wl.kv_indptr, wl.kv_indices, wl.prefix_lens, wl.sm_scale,
                                   limit, is_cross_attention=cross, sliding_window_size=window)
    for a, b in ((kc, kc2), (vc, vc2)):
        assert torch.equal(a.view(torch.int16), b.view(torch.int16))
    at = 0
    for e in ext:  # rows past the cap are not computed
        x, y = got[at:at + min(e, limit)].float(), want[at:at + min(e, limit)].float()
        assert bool(torch.isfinite(x).all())
        diff = (x - y).abs()
        assert e == 0 or (float(diff.max()) <= 2e-2 and float(diff.mean()) <= 1e-3), (float(diff.max()), float(diff.mean()))
        at += e


# the same for longer query blocks, whose tile kernel stores the rows of its request: trips of 32 rows (16 at head_dim 256)
# and of 4 and 8 times as many, requests beyond a wave's lanes, key splits and ragged shares, rows past the cap
TILES = [
    ([0, 0, 40], [31, 33, 0], 32, 8, 128, 0),
    ([0, 500, 64], [127, 128, 32], 16, 8, 128, 0),
    ([900], [192], 16, 8, 128, 0),
    ([1000, 200], [90, 20], 16, 4, 128, 0),
    ([100] * 70, [17 + i % 5 for i in range(70)], 8, 1, 128, 0),
    ([100] * 64, [20] * 64, 8, 1, 128, 0),
    ([0, 300], [250, 90], 32, 8, 128, 100),
    ([0, 300, 20], [17, 96, 16], 24, 4, 256, 0),
    ([79, 2000], [65, 15], 16, 2, 256, 0),
    ([30] * 66, [9] * 66, 8, 1, 256, 0),
]


@pytest.mark.parametrize("cached,ext,n_q,n_kv,d,cap", TILES)
@pytest.mark.parametrize("cross,window", [(False, 0), (True, 0), (False, 100)])
@pytest.mark.parametrize("places", ["last", "mixed"])
def test_extend_in_tiles_is_two(gpu, cached, ext, n_q, n_kv, d, cap, cross, window, places):
    if places == "last" and not cross:  # (a full mask may be shared out otherwise)
        assert _lib.load().msgl_extend_step_workspace_bytes(len(ext), sum(ext), sum(ext) + sum(cached), n_q, n_kv, d, cap or max(ext), 0, window) > 0
    test_extend_one_launch_is_two(gpu, lambda *_: None, cached, ext, n_q, n_kv, d, 0, cap, cross, window, places)


# rows that belong to no request, in front of the first and behind the last: cached, new tokens, heads, such rows, max_len_extend
NOBODYS = [
    ([90, 0, 300], [8, 8, 8], 32, 8, 128, (0, 40), 8),      # shares
    ([5, 64, 0], [3, 0, 5], 16, 8, 128, (3, 1), 8),
    ([40], [1], 16, 8, 128, (0, 2000), 1),                   # more of them than workgroups
    ([7, 9], [0, 0], 16, 8, 128, (2, 6), 3),                 # no request has rows
    ([40, 300], [5, 3], 16, 4, 256, (7, 70), 4),
    ([0, 0, 40], [31, 33, 0], 32, 8, 128, (1, 63), 33),      # tiles
    ([900], [192], 16, 8, 128, (0, 400), 192),
    ([1000, 200], [90, 20], 16, 4, 128, (5, 0), 90),
    ([7, 9], [0, 0], 32, 8, 128, (2, 300), 60),
    ([2, 700], [0, 0], 32, 8, 128, (90, 300), 100),
    ([100] * 70, [17 + i % 5 for i in range(70)], 8, 1, 128, (2, 90), 21),
    ([0, 300, 20], [17, 96, 16], 24, 4, 256, (9, 33), 96),
    ([0, 300, 20], [0, 0, 0], 24, 4, 256, (9, 33), 20),
]


@pytest.mark.parametrize("cached,ext,n_q,n_kv,d,nobodys,limit", NOBODYS)
def test_rows_of_no_request_are_stored(gpu, cached, ext, n_q, n_kv, d, nobodys, limit):
    kv = [c + e for c, e in zip(cached, ext)]
    wl = build_workload("step", "prefill", seed=sum(kv), n_q=n_q, n_kv=n_kv, head_dim=d, kv_lens=kv, extend_lens=ext).to(gpu)
    front, behind = nobodys
    total = front + sum(ext) + behind
    g = torch.Generator(device=gpu)
    g.manual_seed(total)
    q, k, v = (torch.randn((total, n, d), generator=g, device=gpu).bfloat16() for n in (n_q, n_kv, n_kv))
    spare = wl.k_cache.shape[0]
    kc, vc = (torch.cat([c, c.new_zeros((front + behind + 1, n_kv, d))]) for c in (wl.k_cache, wl.v_cache))
    own = [wl.kv_indices[int(wl.kv_indptr[b]) + c:int(wl.kv_indptr[b + 1])] for b, c in enumerate(cached)]
    rest = spare + torch.randperm(front + behind, generator=g, device=gpu).to(torch.int32)
    if behind > 1:
        rest[-1] = kc.shape[0] + 5  # outside the pool: nothing is stored
    loc = torch.cat([rest[:front], *own, rest[front:]]).contiguous()
    indptr = wl.qo_indptr + front
    sizes = (len(ext), total, sum(kv), n_q, n_kv, d, limit, 0, 0)
    assert _lib.load().msgl_extend_step_workspace_bytes(*sizes) > 0  # one launch
    kc2, vc2 = kc.clone(), vc.clone()
    print(f"rows of no request {cached[:4]} + {ext[:4]} {n_q}/{n_kv} d{d} {nobodys}", flush=True)
    got = extend_step(q, k, v, loc, kc, vc, indptr, wl.kv_indptr, wl.kv_indices, wl.prefix_lens, sm_scale=wl.sm_scale, max_len_extend=limit)
    store_kv_cache(kc2, vc2, loc, k, v)
    want = paged_prefill_attention(q, kc2, vc2, indptr, wl.kv_indptr, wl.kv_indices, wl.prefix_lens, wl.sm_scale, limit)
    for a, b in ((kc, kc2), (vc, vc2)):
        assert torch.equal(a.view(torch.int16), b.view(torch.int16))
    at = torch.cat([torch.arange(min(e, limit)) + front + sum(ext[:b]) for b, e in enumerate(ext)])  # past the limit: not computed
    diff = (got[at].float() - want[at].float()).abs()
    assert sum(ext) == 0 or (float(diff.max()) <= 2e-2 and float(diff.mean()) <= 1e-3), (float(diff.max()), float(diff.mean()))


def _turned(x):  # the same values, heads outermost
    return x.transpose(0, 1).contiguous().transpose(0, 1)


def _odd_rows(x):  # rows that start at odd multiples of 2 bytes
    wide = x.new_zeros((x.shape[0], x.numel() // x.shape[0] + 1))
    wide[:, 1:] = x.flatten(1)
    return wide[:, 1:].view(x.shape)


def _every_other(x):
    return torch.stack([x, x], dim=1).flatten()[::2]


# what one of the two operators refuses ...
REFUSED = {
    "q flat": dict(q=lambda x: x.flatten(1)), "k flat": dict(k=lambda x: x.flatten(1)), "k and v short": dict(k=lambda x: x[1:], v=lambda x: x[1:]),
    "v of another type": dict(v=lambda x: x.half()), "q float": dict(q=lambda x: x.float()), "heads that do not divide": dict(q=lambda x: x[:, :-1]),
    "slots int64": dict(loc=lambda x: x.long()), "one slot too few": dict(loc=lambda x: x[1:]), "one offset too few": dict(kv_indptr=lambda x: x[1:]),
    "ids int64": dict(kv_indices=lambda x: x.long()), "v pool shorter": dict(vc=lambda x: x[:-1]), "k pool turned": dict(kc=_turned),
    "slots in host memory": dict(loc=lambda x: x.cpu()),
}
# ... and what one of them copies, or the C ABI refuses
FORMS = REFUSED | {
    "q turned": dict(q=_turned), "k turned": dict(k=_turned), "q off by 2 bytes": dict(q=_odd_rows), "k off by 2 bytes": dict(k=_odd_rows),
    "k repeated": dict(k=lambda x: x[:1].expand(x.shape)), "slots strided": dict(loc=_every_other), "offsets strided": dict(kv_indptr=_every_other),
    "ids strided": dict(kv_indices=_every_other), "k pool off by 2 bytes": dict(kc=_odd_rows),
}


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("kind", ["decode", "norm", "extend"])
def test_forms_that_steps_leave_to_the_two_calls(gpu, kind, form):
    """None, and nothing stored; what the two calls refuse they go on to say."""
    ext = [3, 2] if kind == "extend" else [1, 1]
    kv = [40, 70]
    wl = build_workload("step", "prefill", seed=5, n_q=16, n_kv=8, head_dim=128, kv_lens=kv, extend_lens=ext).to(gpu)
    g = torch.Generator(device=gpu)
    g.manual_seed(5)
    rows = lambda n: torch.randn((sum(ext), n, 128), generator=g, device=gpu).bfloat16()  # noqa: E731
    t = dict(q=rows(16), k=rows(8), v=rows(8), kc=wl.k_cache, vc=wl.v_cache, kv_indptr=wl.kv_indptr, kv_indices=wl.kv_indices,
             loc=torch.cat([wl.kv_indices[int(wl.kv_indptr[b + 1]) - e:int(wl.kv_indptr[b + 1])] for b, e in enumerate(ext)]))
    t |= {name: change(t[name]) for name, change in FORMS[form].items()}
    kc, vc = t["kc"].clone(), t["vc"].clone()
    w, pos = torch.ones(128, dtype=torch.bfloat16, device=gpu), torch.arange(2, dtype=torch.int32, device=gpu)
    splits = torch.ones(2, dtype=torch.int32, device=gpu)

    def one_launch():
        pools = (t["loc"], t["kc"], t["vc"])
        if kind == "extend":
            return extend_step(t["q"], t["k"], t["v"], *pools, wl.qo_indptr, t["kv_indptr"], t["kv_indices"], wl.prefix_lens,
                               sm_scale=0.1, max_len_extend=max(ext))
        norm = dict(q_weight=w, k_weight=w, positions=pos, eps=1e-6, rope_base=1e6) if kind == "norm" else {}
        return decode_step(t["q"], t["k"], t["v"], *pools, t["kv_indptr"], t["kv_indices"], splits, sm_scale=0.1, **norm)

    def two_calls():
        q = t["q"]
        if kind == "norm":
            q = qk_norm_rope_store(q, t["k"], t["v"], w, w, pos, t["loc"], kc, vc, eps=1e-6, rope_base=1e6)
        else:
            store_kv_cache(kc, vc, t["loc"], t["k"], t["v"])
        if kind == "extend":
            return paged_prefill_attention(q, kc, vc, wl.qo_indptr, t["kv_indptr"], t["kv_indices"], wl.prefix_lens, 0.1, max(ext))
        return paged_decode_attention(q, kc, vc, t["kv_indptr"], t["kv_indices"], splits, 0.1, 32)

    print(f"{kind}: {form}", flush=True)
    assert one_launch() is None
    assert torch.equal(t["kc"], kc) and torch.equal(t["vc"], vc)
    if form in REFUSED:
        with pytest.raises(RuntimeError):
            two_calls()
