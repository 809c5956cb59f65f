"""Which steps may store their new rows in the launch that attends: those whose slots are their requests' own.  Host code:
the launches are replaced by a record of them."""
from types import SimpleNamespace

import pytest
import torch

from mini_sglang_amd.attention import AttnBackend, DecodeMetadata, PrefillMetadata
from mini_sglang_amd.attention import backend as backend_module
from mini_sglang_amd.kvcache import MHAKVCache

HEADS, D = 2, 128


@pytest.fixture
def calls(monkeypatch):
    """What ``forward`` launches, in order; the one-launch calls take every step."""
    log = []
    note = lambda name, result=None: lambda *a, **kw: (log.append((name, a)), result)[1]  # noqa: E731
    monkeypatch.setattr(backend_module, "_native", SimpleNamespace(decode_step=note("decode_step", "out"), extend_step=note("extend_step", "out")))
    for name in ("paged_decode_attention", "paged_prefill_attention", "qk_norm_rope_store"):
        monkeypatch.setattr(backend_module, name, note(name))
    monkeypatch.setattr(MHAKVCache, "store_kv", note("store_kv"))
    return log


def _backend():
    pool = MHAKVCache(num_kv_heads=HEADS, num_layers=1, head_dim=D, num_pages=64, dtype=torch.bfloat16, device="cpu")
    return AttnBackend(SimpleNamespace(head_dim=D), pool, torch.arange(60, dtype=torch.int32).reshape(3, 20))


def _batch(rows, is_prefill, **more):
    reqs = [SimpleNamespace(table_idx=r, extend_len=2 if is_prefill else 1, cached_len=4, device_len=6 if is_prefill else 5) for r in rows]
    return SimpleNamespace(padded_reqs=reqs, is_prefill=is_prefill, attn_metadata=None, out_loc=None, **more)


@pytest.mark.parametrize("is_prefill", [False, True])
@pytest.mark.parametrize("rows,asked,own", [((0, 2), None, True), ((1, 1), None, False), ((0, 1), False, False), ((1, 1), True, True)])
def test_the_builders_claim_it_for_distinct_rows_unless_told_otherwise(is_prefill, rows, asked, own):
    backend = _backend()
    batch = _batch(rows, is_prefill, own_slots=asked)
    backend.prepare_metadata(batch)
    assert batch.attn_metadata.own_slots is own
    build = backend.build_prefill_metadata if is_prefill else backend.build_decode_metadata
    assert build(batch.padded_reqs, own_slots=asked).own_slots is own
    if asked is None:
        plain = _batch(rows, is_prefill)
        backend.prepare_metadata(plain)
        assert plain.attn_metadata.own_slots is own


def test_metadata_made_by_hand_do_not_claim_it():
    t = torch.zeros(2, dtype=torch.int32)
    assert DecodeMetadata(t, t, t, t, 32).own_slots is False
    assert PrefillMetadata(t, t, t, t, t, 1).own_slots is False


@pytest.mark.parametrize("own", [True, False])
def test_decode_with_shared_slots_stores_first(calls, own):
    backend, batch = _backend(), _batch((0, 1), False, own_slots=own)
    backend.prepare_metadata(batch)
    backend.forward(None, None, None, 0, batch)
    assert [name for name, _ in calls] == (["decode_step"] if own else ["store_kv", "paged_decode_attention"])
    calls.clear()
    backend.forward_fused_norm_rope(None, None, None, None, None, 0, batch, rms_norm_eps=1e-6, rope_base=1e6)
    assert [name for name, _ in calls] == (["decode_step"] if own else ["qk_norm_rope_store", "paged_decode_attention"])


@pytest.mark.parametrize("own", [True, False])
def test_extends_with_shared_slots_ask_for_two_launches(calls, own):
    backend, batch = _backend(), _batch((0, 1), True, own_slots=own)
    backend.prepare_metadata(batch)
    backend.forward(None, None, None, 0, batch)
    (name, args), = calls
    assert name == "extend_step" and args[-1] is own
