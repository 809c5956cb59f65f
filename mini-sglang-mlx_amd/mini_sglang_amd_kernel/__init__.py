"""MI355X counterpart of the reference's ``mini_sglang_mlx_kernel`` module, for the
paged-attention path only.

Same function names, positional order and keyword names as the nanobind module
(mini-sglang-mlx-kernel/csrc/bindings.cpp:27-55, mini_sglang_mlx_kernel/__init__.py:1-9);
``mx.array`` becomes ``torch.Tensor`` on a ROCm device.  Every call is an eager,
stream-ordered launch of hand-written gfx950 kernels through the C ABI of
``include/msgl_paged_attention.h``; nothing synchronises with the host and there is no
other implementation to fall back to.  The functions below carry the signatures and the
documentation; checks, allocation and the launch are native (``csrc/torch_binding.cpp``).

Argument errors raise ``RuntimeError`` with the reference's message text
(paged_decode_attention.cpp:25-62, paged_prefill_attention.cpp:31-76,
store_kv_cache.cpp:22-63).
"""
from __future__ import annotations

import os
from typing import Optional

import torch

from . import _lib

try:
    from . import _native
except ImportError as _exc:  # not built: the first call says so
    _native = _lib.MissingNative(_exc)

__all__ = ["store_kv_cache", "paged_decode_attention", "paged_prefill_attention",
           "build_attention_metadata", "build_metadata_from_host", "qk_norm_rope_store", "decode_step", "extend_step",
           "gdn_state_inplace",
           "fast_compare_key"]


def _fail(op: str, msg: str):
    raise RuntimeError(f"{op}: {msg}")


class _on_device:
    """``torch.cuda.device(dev)`` that costs nothing when ``dev`` is current already (the usual
    case: one process per GPU), and, for a call with an explicit ``stream=``, that stream made
    torch's current one for the duration of the call.  The second part is what makes a foreign
    stream safe: the output, the workspace and any ``.contiguous()`` copy of an argument are
    then allocated and produced on the stream the kernels run on, so torch's caching allocator
    never hands one of these blocks to work that is still in flight on another stream."""

    __slots__ = ("_guards",)

    def __init__(self, dev: torch.device, stream=None):
        self._guards = []
        index = dev.index
        if index is not None and index != torch.cuda.current_device():
            self._guards.append(torch.cuda.device(dev))
        if stream is not None:
            if not isinstance(stream, torch.cuda.Stream):
                stream = torch.cuda.ExternalStream(int(stream.cuda_stream), device=dev)
            self._guards.append(torch.cuda.stream(stream))

    def __enter__(self):
        for g in self._guards:
            g.__enter__()

    def __exit__(self, *exc):
        for g in reversed(self._guards):
            g.__exit__(*exc)
        return False


def _checks_on(validate: Optional[bool]) -> bool:
    """Index validation is opt-in: ``validate=True`` on the call, or ``MSGL_DEBUG_CHECKS=1`` in
    the environment for every call that does not say ``validate=False``.  It costs a few small
    device reductions and ONE host synchronisation per call, so it is off by default, and it is
    skipped while the current stream is being captured into a graph (a capture cannot sync)."""
    if validate is None:
        validate = os.environ.get("MSGL_DEBUG_CHECKS", "0") not in ("", "0")
    if not validate:
        return False
    return not (torch.cuda.is_available() and torch.cuda.is_current_stream_capturing())


def _validate_slot_ids(op: str, name: str, ids: torch.Tensor, num_slots: int,
                       unique: bool = False) -> None:
    """Every id inside ``[0, num_slots)`` and, for a store, no id twice.  The kernels read or
    write ``pool[id]`` unchecked (a stray id is a wild access: a GPU memory fault, not a wrong
    value; the writers skip such a row, the readers cannot), and two rows stored to one slot
    race (store_kv_cache.metal:24-30 has the same hole; the reference's allocator hands out
    distinct slots, scheduler/cache.py:45-57).  Works on any device: min, max and a sort there,
    then one transfer of three numbers."""
    if ids.numel() == 0:
        return
    lo, hi = torch.aminmax(ids)
    dup = torch.zeros((), dtype=torch.int64, device=ids.device)
    if unique and ids.numel() > 1:
        srt = torch.sort(ids).values
        dup = (srt[1:] == srt[:-1]).sum()
    lo, hi, dup = (int(x) for x in torch.stack([lo.long(), hi.long(), dup]).tolist())
    if lo < 0 or hi >= num_slots:
        _fail(op, f"{name} holds slot ids outside [0, {num_slots}): min {lo}, max {hi}")
    if dup:
        _fail(op, f"{name} holds {dup} duplicate slot id(s); rows stored to one slot race")


def _validate_indptr(op: str, name: str, indptr: torch.Tensor, limit: int, what: str) -> None:
    """A CSR offset array must start at >= 0, never decrease and end inside the array it
    indexes."""
    first, last = indptr[0], indptr[-1]
    down = (indptr[1:] < indptr[:-1]).sum() if indptr.numel() > 1 else torch.zeros_like(first)
    first, last, down = (int(x) for x in torch.stack([first.long(), last.long(), down.long()]).tolist())
    if first < 0 or down:
        _fail(op, f"{name} must start at >= 0 and be non-decreasing")
    if last > limit:
        _fail(op, f"{name} ends at {last}, beyond the {limit} entries of {what}")


def _run_checks(validate, op: str, *args) -> None:
    """What the native functions call when index validation is on, with the operator's index
    arrays and the tensors they point into."""
    if not _checks_on(validate):
        return
    if op == "store_kv_cache":
        indices, k_cache = args
        _validate_slot_ids(op, "indices", indices, k_cache.shape[0], unique=True)
    elif op == "qk_norm_rope_store":
        out_loc, k_cache = args
        _validate_slot_ids(op, "out_loc", out_loc, k_cache.shape[0], unique=True)
    elif op == "paged_decode_attention":
        kv_indptr, kv_indices, k_cache = args
        _validate_indptr(op, "kv_indptr", kv_indptr, kv_indices.shape[0], "kv_indices")
        _validate_slot_ids(op, "kv_indices", kv_indices, k_cache.shape[0])
    else:
        qo_indptr, kv_indptr, kv_indices, q, k_cache = args
        _validate_indptr(op, "qo_indptr", qo_indptr, q.shape[0], "q")
        _validate_indptr(op, "kv_indptr", kv_indptr, kv_indices.shape[0], "kv_indices")
        _validate_slot_ids(op, "kv_indices", kv_indices, k_cache.shape[0])


_native.set_checks(_run_checks)


def _on_stream(stream, tensor: torch.Tensor):
    """The guard of a call with an explicit ``stream=``."""
    return _on_device(tensor.device, stream if tensor.is_cuda else None)


def store_kv_cache(k_cache: torch.Tensor, v_cache: torch.Tensor, indices: torch.Tensor,
                   k: torch.Tensor, v: torch.Tensor, *, stream=None,
                   validate: Optional[bool] = None) -> None:
    """In place: ``k_cache[indices[r]] = k[r]``, ``v_cache[indices[r]] = v[r]`` (bit copy).

    Drop-in for ``mini_sglang_mlx_kernel.store_kv_cache`` (store_kv_cache.cpp:14-107).
    ``indices`` must be unique; duplicates race exactly as in the reference.  A slot id outside
    the pool stores nothing.  ``validate=True`` (or ``MSGL_DEBUG_CHECKS=1``) checks range and
    uniqueness first, at the price of one host synchronisation.
    """
    if stream is None:
        _native.store_kv_cache(k_cache, v_cache, indices, k, v, validate)
        return
    with _on_stream(stream, k_cache):
        _native.store_kv_cache(k_cache, v_cache, indices, k, v, validate)


def paged_decode_attention(q: torch.Tensor, k_cache: torch.Tensor, v_cache: torch.Tensor,
                           kv_indptr: torch.Tensor, kv_indices: torch.Tensor,
                           num_kv_splits: torch.Tensor, sm_scale: float, max_kv_splits: int,
                           *, stream=None, validate: Optional[bool] = None) -> torch.Tensor:
    """GQA paged decode: ``q (batch, n_q, d)`` against the tokens listed in ``kv_indices``.

    Drop-in for ``mini_sglang_mlx_kernel.paged_decode_attention``
    (paged_decode_attention.cpp:15-73).  Returns ``(batch, n_q, d)`` in the dtype of ``q``.
    ``validate=True`` (or ``MSGL_DEBUG_CHECKS=1``) first checks ``kv_indptr`` and that every
    entry of ``kv_indices`` names a slot of the pool (one host synchronisation).
    """
    if stream is None:
        return _native.paged_decode_attention(q, k_cache, v_cache, kv_indptr, kv_indices, num_kv_splits,
                                              sm_scale, max_kv_splits, validate)
    with _on_stream(stream, q):
        return _native.paged_decode_attention(q, k_cache, v_cache, kv_indptr, kv_indices, num_kv_splits,
                                              sm_scale, max_kv_splits, validate)


def paged_prefill_attention(q: torch.Tensor, k_cache: torch.Tensor, v_cache: torch.Tensor,
                            qo_indptr: torch.Tensor, kv_indptr: torch.Tensor,
                            kv_indices: torch.Tensor, prefix_lens: torch.Tensor,
                            sm_scale: float, max_len_extend: int, *,
                            is_cross_attention: bool = False, sliding_window_size: int = 0,
                            stream=None, validate: Optional[bool] = None) -> torch.Tensor:
    """Paged extend attention on top of a cached prefix.

    Drop-in for ``mini_sglang_mlx_kernel.paged_prefill_attention``
    (paged_prefill_attention.cpp:18-87).  Query ``i`` of request ``b`` sits at position
    ``prefix_lens[b] + i``; key ``j`` of the request is visible iff
    ``(is_cross_attention or j <= pos) and (W == 0 or j >= pos - W + 1)``.
    Returns ``(total_q, n_q, d)`` in the dtype of ``q``; rows of a request beyond
    ``max_len_extend`` are not computed.  ``validate=True`` (or ``MSGL_DEBUG_CHECKS=1``) first
    checks both offset arrays and that every entry of ``kv_indices`` names a slot of the pool
    (one host synchronisation).
    """
    if stream is None:
        return _native.paged_prefill_attention(q, k_cache, v_cache, qo_indptr, kv_indptr, kv_indices,
                                               prefix_lens, sm_scale, max_len_extend,
                                               is_cross_attention, sliding_window_size, validate)
    with _on_stream(stream, q):
        return _native.paged_prefill_attention(q, k_cache, v_cache, qo_indptr, kv_indptr, kv_indices,
                                               prefix_lens, sm_scale, max_len_extend,
                                               is_cross_attention, sliding_window_size, validate)


def build_attention_metadata(page_table: torch.Tensor, table_rows: torch.Tensor,
                             kv_lens: torch.Tensor, extend_lens: Optional[torch.Tensor] = None, *,
                             total_kv: int, total_q: Optional[int] = None,
                             max_kv_splits: int = 32, stream=None) -> dict:
    """CSR metadata of one step from the slot table, in one launch on the device.

    Device counterpart of ``AttnBackend.build_prefill_metadata`` / ``build_decode_metadata``
    (mini_sglang_mlx/attention/backend.py:205-307), which slice the table per request in
    Python.  ``page_table`` is the ``(rows, max_seq_len)`` int32 slot table, ``table_rows`` /
    ``kv_lens`` / ``extend_lens`` are int32 ``[batch]`` device tensors; ``extend_lens=None``
    builds decode metadata (one query per request).  ``total_kv`` / ``total_q`` are the sums
    of the lengths, which the scheduler knows on the host; they size the outputs.  Returns a
    dict with ``kv_indptr``, ``kv_indices``, ``qo_indptr``, ``prefix_lens``, ``positions``,
    ``num_kv_splits``.
    """
    if stream is None:
        return _native.build_attention_metadata(page_table, table_rows, kv_lens, extend_lens, total_kv,
                                                total_q, max_kv_splits)
    with _on_stream(stream, page_table):
        return _native.build_attention_metadata(page_table, table_rows, kv_lens, extend_lens, total_kv,
                                                total_q, max_kv_splits)


def build_metadata_from_host(page_table: torch.Tensor, table_rows, kv_lens, extend_lens=None, *,
                             max_kv_splits: int = 32) -> dict:
    """``build_attention_metadata`` from the scheduler's own lists of ints (same arrays, same
    clamping): up to 128 requests they travel as arguments of the one kernel, more through one
    pinned buffer; nothing waits either way."""
    return _native.build_metadata_from_host(page_table, table_rows, kv_lens, extend_lens, max_kv_splits)


def qk_norm_rope_store(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, q_weight: torch.Tensor,
                       k_weight: torch.Tensor, positions: torch.Tensor, out_loc: torch.Tensor,
                       k_cache: torch.Tensor, v_cache: torch.Tensor, *, eps: float,
                       rope_base: float, stream=None,
                       validate: Optional[bool] = None) -> torch.Tensor:
    """Per-head RMSNorm of q and k, rotary embedding of both at ``positions``, and the store of
    the new k and v rows at ``out_loc``, in one pass; returns the rotated q.

    One call for ``q_norm`` / ``k_norm`` / ``rope`` / ``rope`` of the reference's Qwen3 attention
    layer (mini_sglang_mlx/models/qwen3.py:60-68) plus the store that ``AttnBackend.forward``
    does first (attention/backend.py:139).  Attention then runs on the result with no further
    store.  q / k / v may be strided views (tokens, heads, head_dim) of a fused projection.
    """
    if stream is None:
        return _native.qk_norm_rope_store(q, k, v, q_weight, k_weight, positions, out_loc, k_cache,
                                          v_cache, eps, rope_base, validate)
    with _on_stream(stream, q):
        return _native.qk_norm_rope_store(q, k, v, q_weight, k_weight, positions, out_loc, k_cache,
                                          v_cache, eps, rope_base, validate)


def decode_step(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, out_loc: torch.Tensor,
                k_cache: torch.Tensor, v_cache: torch.Tensor, kv_indptr: torch.Tensor,
                kv_indices: torch.Tensor, num_kv_splits: torch.Tensor, *, sm_scale: float,
                q_weight: Optional[torch.Tensor] = None, k_weight: Optional[torch.Tensor] = None,
                positions: Optional[torch.Tensor] = None, eps: float = 0.0,
                rope_base: float = 0.0) -> Optional[torch.Tensor]:
    """``paged_decode_attention`` of a decode step with ``store_kv_cache`` inside or, with norm weights,
    ``qk_norm_rope_store``: the attention output, or ``None`` (nothing done) where the two calls are
    the way: large launches, forms that need a copy, arguments that they refuse, index
    validation on.

    One new token per request, row ``b`` at slot ``out_loc[b]``.  No slot of ``out_loc`` may be listed in
    ``kv_indices`` for another request, nor twice for its own: the launch that reads it writes it.  A
    step with such slots is the two calls.
    """
    return _native.decode_step(q, k, v, q_weight, k_weight, positions, out_loc, k_cache, v_cache,
                               kv_indptr, kv_indices, num_kv_splits, sm_scale, eps, rope_base)


def extend_step(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, out_loc: torch.Tensor,
                k_cache: torch.Tensor, v_cache: torch.Tensor, qo_indptr: torch.Tensor,
                kv_indptr: torch.Tensor, kv_indices: torch.Tensor, prefix_lens: torch.Tensor, *,
                sm_scale: float, max_len_extend: int, is_cross_attention: bool = False,
                sliding_window_size: int = 0, own_slots: bool = True) -> Optional[torch.Tensor]:
    """``store_kv_cache`` of the queries' own rows of k and v and ``paged_prefill_attention`` as one call: in one
    launch where the query blocks are short, the launch is small, or at head_dim 128 its requests are prompts with nothing
    cached that fill the chip (keys and values are then taken from the new rows, which are stored on the way, where
    their slots are the listed ones), else as the two calls.  Returns the
    attention output, or ``None`` (nothing done) where the two calls have to be made by themselves: forms
    that need a copy, arguments that they refuse, index validation on.

    As with ``decode_step`` no slot of ``out_loc`` may be listed in ``kv_indices`` for a request that its row does not
    belong to, nor twice for its own; ``own_slots=False`` is for such batches: the two launches, whatever the size.
    """
    return _native.extend_step(q, k, v, out_loc, k_cache, v_cache, qo_indptr, kv_indptr, kv_indices,
                               prefix_lens, sm_scale, max_len_extend, is_cross_attention,
                               sliding_window_size, own_slots)


def gdn_state_inplace(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, g: torch.Tensor,
                      beta: torch.Tensor, state: torch.Tensor, slot_ids: torch.Tensor,
                      qo_indptr: torch.Tensor, single_token_mode: bool = False, *,
                      stream=None, max_len_extend: Optional[int] = None) -> torch.Tensor:
    """Gated delta-rule recurrence over each request's tokens with the fp32 state of slot
    ``slot_ids[b]`` updated in place; returns ``y`` ``(tokens, hv, dv)`` bf16.

    Drop-in for ``mini_sglang_mlx_kernel.gdn_state_inplace`` (bindings.cpp:56-65,
    gdn_state.cpp:87-135): same argument order, ``single_token_mode`` (decode: one token per
    request, ``qo_indptr`` ignored) and error texts (gdn_state.cpp:26-84, 107-126).

    ``max_len_extend``, most tokens of a request, is for callers that have the lengths on the host:
    requests of a few dozen tokens are faster with it where none of them is long.  It chooses the
    kernel and nothing else; any value gives right results.
    """
    if stream is None:
        return _native.gdn_state_inplace(q, k, v, g, beta, state, slot_ids, qo_indptr,
                                         single_token_mode, max_len_extend)
    with _on_stream(stream, q):
        return _native.gdn_state_inplace(q, k, v, g, beta, state, slot_ids, qo_indptr,
                                         single_token_mode, max_len_extend)


def fast_compare_key(a: torch.Tensor, b: torch.Tensor) -> int:
    """Length of the common prefix of two 1-D integer arrays (host tensors).

    Drop-in for ``mini_sglang_mlx_kernel.fast_compare_key`` (fast_compare_key.cpp:9-45): the
    radix tree's key comparison.  Pure host code; device tensors are refused instead of being
    copied behind the caller's back.
    """
    op = "fast_compare_key"
    if a.dim() != 1 or b.dim() != 1:
        _fail(op, "Both arrays must be 1D.")
    if not a.is_contiguous() or not b.is_contiguous():
        _fail(op, "Both arrays must be contiguous.")
    if a.dtype != b.dtype:
        _fail(op, "Both arrays must have the same dtype.")
    if a.dtype not in (torch.int32, torch.int64):
        _fail(op, "Arrays must be int32 or int64.")
    if a.device.type != "cpu" or b.device.type != "cpu":
        _fail(op, "Both arrays must live in host memory.")
    return int(_lib.load().msgl_fast_compare_key(a.data_ptr(), a.numel(), b.data_ptr(), b.numel(),
                                                 a.element_size(), None))
