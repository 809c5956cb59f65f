"""Attention backend of the path on torch-ROCm
(reference: mini_sglang_mlx/attention/backend.py:15-307).

``AttnBackend.forward`` stores the new K/V rows and attends through the slot lists
(backend.py:139-141): in one launch where the metadata say that the new slots are their
requests' own (``own_slots``) and the step's sizes make that the better way, else the store
first and then attention, which reads the new tokens back from the pool like cached ones.
Metadata are int32 CSR arrays; ``kv_indices`` holds one pool slot per token.  The builders keep
the reference's formulas and keyword overrides (virtual extend windows for speculative verify,
backend.py:205-293).
"""
from __future__ import annotations

import math
from dataclasses import dataclass
from typing import List, Optional, Sequence

import torch

from mini_sglang_amd.kvcache.mha_pool import MHAKVCache
from mini_sglang_amd_kernel import (_native, build_metadata_from_host, paged_decode_attention,
                                    paged_prefill_attention, qk_norm_rope_store)

MAX_KV_SPLITS = 32


@dataclass
class BaseAttnMetadata:
    positions: torch.Tensor

    def get_last_indices(self, bs: int) -> torch.Tensor:
        raise NotImplementedError


@dataclass
class PrefillMetadata(BaseAttnMetadata):
    """Several new query tokens per sequence on top of a cached prefix (backend.py:26-41)."""

    qo_indptr: torch.Tensor  # (batch + 1,) int32
    kv_indptr: torch.Tensor  # (batch + 1,) int32
    kv_indices: torch.Tensor  # (total_kv,) int32 pool slots
    prefix_lens: torch.Tensor  # (batch,) int32
    max_len_extend: int
    own_slots: bool = False  # see AttnBackend.forward

    def get_last_indices(self, bs: int) -> torch.Tensor:
        return self.qo_indptr[1 : 1 + bs] - 1


@dataclass
class DecodeMetadata(BaseAttnMetadata):
    """One new query token per sequence (backend.py:44-58)."""

    kv_indptr: torch.Tensor  # (batch + 1,) int32
    kv_indices: torch.Tensor  # (total_kv,) int32 pool slots
    num_kv_splits: torch.Tensor  # (batch,) int32
    max_kv_splits: int
    own_slots: bool = False  # see AttnBackend.forward

    def get_last_indices(self, bs: int) -> torch.Tensor:
        return torch.arange(bs, dtype=torch.int32, device=self.kv_indptr.device)


AttnMetadata = PrefillMetadata | DecodeMetadata


class AttnBackend:
    """Paged attention backend for MI355X using the msgl HIP kernels.

    ``config`` needs ``head_dim``; ``kvcache`` is a ``BaseKVCache``; ``page_table`` is the
    ``(max_running_req + 1, max_seq_len)`` int32 slot table the scheduler fills.
    """

    def __init__(self, config, kvcache, page_table: torch.Tensor) -> None:
        self.config = config
        self.kvcache = kvcache
        self.page_table = page_table
        self.sm_scale = 1.0 / math.sqrt(config.head_dim)

    def forward(self, q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, layer_id: int, batch, *,
                is_cross_attention: bool = False, sliding_window_size: int = 0) -> torch.Tensor:
        """Write the new K/V rows at ``batch.out_loc`` and run paged attention.

        The two flags select one of four masks on the prefill path (backend.py:112-127):
        causal, full, causal + window, bidirectional + window.  Decode rejects both.

        ``batch.attn_metadata.own_slots`` says that no slot of ``batch.out_loc`` is listed in
        ``kv_indices`` for a request that the row does not belong to, nor twice for its own.  The
        rows may then be stored by the launch that attends: a request sees its own new rows, and
        nobody waits for those of others.  Without it every row is in the pool before the
        attention starts, and requests may share new slots in any way.  Metadata made by hand do
        not claim it; of those the builders make see ``_slots_are_own``.
        """
        assert sliding_window_size >= 0, (
            f"sliding_window_size must be >= 0, got {sliding_window_size}"
        )
        metadata, cache = batch.attn_metadata, self.kvcache
        out = None
        # one native call, where this package writes the pool itself (a call of Python's own beside it costs as much as
        # all the checks in it); None: the step takes its two calls
        if type(cache) is not MHAKVCache:
            pass
        elif type(metadata) is PrefillMetadata:
            out = _native.extend_step(q, k, v, batch.out_loc, cache.k_cache(layer_id),
                                      cache.v_cache(layer_id), metadata.qo_indptr, metadata.kv_indptr,
                                      metadata.kv_indices, metadata.prefix_lens, self.sm_scale,
                                      metadata.max_len_extend, is_cross_attention, sliding_window_size,
                                      metadata.own_slots)
        elif (type(metadata) is DecodeMetadata and metadata.own_slots and not is_cross_attention
              and sliding_window_size == 0):
            out = _native.decode_step(q, k, v, None, None, None, batch.out_loc,
                                      cache.k_cache(layer_id), cache.v_cache(layer_id),
                                      metadata.kv_indptr, metadata.kv_indices,
                                      metadata.num_kv_splits, self.sm_scale, 0.0, 0.0)
        if out is not None:
            return out
        self.kvcache.store_kv(k, v, batch.out_loc, layer_id)
        k_cache = self.kvcache.k_cache(layer_id)
        v_cache = self.kvcache.v_cache(layer_id)
        return self._attend(q, k_cache, v_cache, metadata, is_cross_attention, sliding_window_size)

    def _attend(self, q, k_cache, v_cache, metadata, is_cross_attention: bool,
                sliding_window_size: int) -> torch.Tensor:
        if isinstance(metadata, PrefillMetadata):
            return paged_prefill_attention(
                q, k_cache, v_cache, metadata.qo_indptr, metadata.kv_indptr, metadata.kv_indices,
                metadata.prefix_lens, sm_scale=self.sm_scale,
                max_len_extend=metadata.max_len_extend,
                is_cross_attention=is_cross_attention, sliding_window_size=sliding_window_size)
        assert isinstance(metadata, DecodeMetadata)
        assert not is_cross_attention and sliding_window_size == 0, (
            "is_cross_attention / sliding_window_size are only "
            "supported on the prefill path."
        )
        return paged_decode_attention(
            q, k_cache, v_cache, metadata.kv_indptr, metadata.kv_indices, metadata.num_kv_splits,
            sm_scale=self.sm_scale, max_kv_splits=metadata.max_kv_splits)

    def forward_fused_norm_rope(self, q: torch.Tensor, k: torch.Tensor, v: torch.Tensor,
                                q_norm_weight: torch.Tensor, k_norm_weight: torch.Tensor,
                                layer_id: int, batch, *, rms_norm_eps: float, rope_base: float,
                                is_cross_attention: bool = False,
                                sliding_window_size: int = 0) -> torch.Tensor:
        """``forward`` for a Qwen3-style layer that hands over the raw projections: q/k RMSNorm,
        rotary embedding at ``batch.attn_metadata.positions`` and the KV-store run as one kernel
        (the reference does them as four array ops plus the store, models/qwen3.py:60-68 and
        backend.py:139), then attention runs on the pool without storing again; small decode steps
        whose slots are their requests' own (``own_slots``, see ``forward``) do it all in one."""
        assert sliding_window_size >= 0, (
            f"sliding_window_size must be >= 0, got {sliding_window_size}"
        )
        metadata = batch.attn_metadata
        cache = self.kvcache
        if (type(metadata) is DecodeMetadata and metadata.own_slots and type(cache) is MHAKVCache
                and not is_cross_attention and sliding_window_size == 0):
            out = _native.decode_step(q, k, v, q_norm_weight, k_norm_weight, metadata.positions,
                                      batch.out_loc, cache.k_cache(layer_id),
                                      cache.v_cache(layer_id), metadata.kv_indptr,
                                      metadata.kv_indices, metadata.num_kv_splits, self.sm_scale,
                                      rms_norm_eps, rope_base)
            if out is not None:
                return out
        k_cache = self.kvcache.k_cache(layer_id)
        v_cache = self.kvcache.v_cache(layer_id)
        q = qk_norm_rope_store(q, k, v, q_norm_weight, k_norm_weight, metadata.positions,
                               batch.out_loc, k_cache, v_cache, eps=rms_norm_eps,
                               rope_base=rope_base)
        return self._attend(q, k_cache, v_cache, metadata, is_cross_attention, sliding_window_size)

    def store_kv_only(self, k: torch.Tensor, v: torch.Tensor, out_loc: torch.Tensor,
                      layer_id: int) -> None:
        """Write K/V without attending (draft calibration, backend.py:174-196)."""
        self.kvcache.store_kv(k, v, out_loc, layer_id)

    def prepare_metadata(self, batch) -> None:
        """Metadata of ``batch.padded_reqs``; a batch with an attribute ``own_slots`` decides about
        theirs (``None`` and no attribute: the builders do)."""
        reqs, own_slots = batch.padded_reqs, getattr(batch, "own_slots", None)
        if batch.is_prefill:
            batch.attn_metadata = self.build_prefill_metadata(reqs, own_slots=own_slots)
        else:
            batch.attn_metadata = self.build_decode_metadata(reqs, own_slots=own_slots)

    def _gather_indices(self, reqs, kv_lens: Sequence[int]) -> torch.Tensor:
        return torch.cat([self.page_table[reqs[i].table_idx, : kv_lens[i]]
                          for i in range(len(reqs))]).to(torch.int32)

    def _device_metadata(self, reqs, kv_lens: Sequence[int],
                         extend_lens: Optional[Sequence[int]]) -> dict:
        """One kernel for every array (slot table on the GPU).  The host lists are the
        reference's own inputs (backend.py:228-238)."""
        return build_metadata_from_host(self.page_table, [req.table_idx for req in reqs], kv_lens,
                                        extend_lens, max_kv_splits=MAX_KV_SPLITS)

    def build_prefill_metadata(self, reqs: List, *, extend_lens: Optional[List[int]] = None,
                               kv_lens: Optional[List[int]] = None,
                               positions: Optional[torch.Tensor] = None,
                               own_slots: Optional[bool] = None) -> PrefillMetadata:
        device = self.page_table.device
        if own_slots is None:
            own_slots = _slots_are_own(reqs)
        if extend_lens is None:
            extend_lens = [req.extend_len for req in reqs]
        if kv_lens is None:
            kv_lens = [req.device_len for req in reqs]
        if device.type == "cuda":
            m = self._device_metadata(reqs, kv_lens, extend_lens)
            return PrefillMetadata(
                positions=m["positions"] if positions is None else positions,
                qo_indptr=m["qo_indptr"], kv_indptr=m["kv_indptr"], kv_indices=m["kv_indices"],
                prefix_lens=m["prefix_lens"], max_len_extend=max(extend_lens), own_slots=own_slots)
        # slot table in host memory (host-side tests): the same arrays with torch ops
        cached_lens = [kv_lens[i] - extend_lens[i] for i in range(len(reqs))]
        if positions is None:
            positions = torch.cat([
                torch.arange(cached_lens[i], kv_lens[i], dtype=torch.int32, device=device)
                for i in range(len(reqs))
            ])
        return PrefillMetadata(
            positions=positions,
            qo_indptr=_build_indptr(extend_lens, device),
            kv_indptr=_build_indptr(kv_lens, device),
            kv_indices=self._gather_indices(reqs, kv_lens),
            prefix_lens=torch.tensor(cached_lens, dtype=torch.int32, device=device),
            max_len_extend=max(extend_lens),
            own_slots=own_slots,
        )

    def build_decode_metadata(self, reqs: List, *, kv_lens: Optional[List[int]] = None,
                              positions: Optional[torch.Tensor] = None,
                              own_slots: Optional[bool] = None) -> DecodeMetadata:
        device = self.page_table.device
        if own_slots is None:
            own_slots = _slots_are_own(reqs)
        if kv_lens is None:
            kv_lens = [req.device_len for req in reqs]
        if device.type == "cuda":
            m = self._device_metadata(reqs, kv_lens, None)
            if positions is None:
                cached = [req.cached_len for req in reqs]
                # the new token's position is the last one, as a rule: the kernel has written it
                if (cached and min(cached) >= 0 and cached == [n - 1 for n in kv_lens]
                        and max(kv_lens) <= self.page_table.shape[1]):
                    positions = m["positions"]
                else:
                    positions = torch.tensor(cached, dtype=torch.int32, device=device)
            return DecodeMetadata(positions=positions, kv_indptr=m["kv_indptr"],
                                  kv_indices=m["kv_indices"], num_kv_splits=m["num_kv_splits"],
                                  max_kv_splits=MAX_KV_SPLITS, own_slots=own_slots)
        if positions is None:
            positions = torch.tensor([req.cached_len for req in reqs], dtype=torch.int32,
                                     device=device)
        return DecodeMetadata(
            positions=positions,
            kv_indptr=_build_indptr(kv_lens, device),
            kv_indices=self._gather_indices(reqs, kv_lens),
            num_kv_splits=_compute_num_kv_splits(kv_lens, device),
            max_kv_splits=MAX_KV_SPLITS,
            own_slots=own_slots,
        )


def _slots_are_own(reqs: Sequence) -> bool:
    """``own_slots`` of requests in the slot table, unless the caller says otherwise: the allocator
    hands a new token's slot to one request, once, and a prefix is shared when it has been computed
    (scheduler/cache.py:45-57), so it holds for distinct rows of the table, and not for a row that
    comes twice.  A caller whose rows share slots of the step's own tokens says so
    (``own_slots=False``)."""
    return len({req.table_idx for req in reqs}) == len(reqs)


def _build_indptr(lens: Sequence[int], device=None) -> torch.Tensor:
    """CSR row pointers ``cumsum([0] + lens)`` as int32 (backend.py:299-301)."""
    return torch.cumsum(torch.tensor([0] + list(lens), dtype=torch.int32), 0).to(
        dtype=torch.int32, device=device)


def _compute_num_kv_splits(kv_lens: Sequence[int], device=None) -> torch.Tensor:
    """The reference's split hint ``min(32, max(1, ceil(L / 128)))`` (backend.py:304-307)."""
    splits = [min(MAX_KV_SPLITS, max(1, (l + 127) // 128)) for l in kv_lens]
    return torch.tensor(splits, dtype=torch.int32, device=device)
