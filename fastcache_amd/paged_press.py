"""Score -> select -> compact over a paged KV pool, all layers and sequences per launch.

This is the fused counterpart of the reference's per-sequence loop
``_extract_kv_cache_fast`` -> press -> ``_write_compressed_kv_cache_fast``
(nanovllm/engine/llava_model_runner.py:712-793): K is scored where it lies in its pages, the kept
indices are selected per (layer, sequence, kv head) and the kept K/V rows are moved to the front
of the same pages in place.  Three launches per pass, nothing leaves the device.
"""
from __future__ import annotations

import math
from collections import namedtuple
from dataclasses import dataclass
from typing import List, Optional, Sequence

import torch

from . import _lib, ops


@dataclass
class PressResult:
    indices: torch.Tensor          # int32 [L, B, Hkv (or 1), n_kept] ascending token positions (-1 past a row's count)
    n_kept: int                    # kept tokens per sequence (the largest count when the sequences differ)
    scores: Optional[torch.Tensor]  # fp32 [L, B, Hkv, S] (None for index-only presses)
    kept_per_seq: Optional[List[int]] = None    # set when the sequences have different lengths


def n_kept_for(seq_len: int, compression_ratio: float) -> int:
    """kvpress ``ScorerPress.compress``: ``int(q_len * (1 - compression_ratio))``, in double."""
    return int(seq_len * (1 - compression_ratio))


def _views(kv_cache: torch.Tensor, block_tables: torch.Tensor, seq_lens: torch.Tensor, max_seq_len: int):
    if kv_cache.dim() != 6 or kv_cache.shape[0] != 2:
        raise _lib.FastcacheError("kv_cache must be [2, L, num_blocks, block_size, Hkv, D]")
    return (_lib.paged_view(kv_cache[0], block_tables, seq_lens, max_seq_len),
            _lib.paged_view(kv_cache[1], block_tables, seq_lens, max_seq_len))


# what ops.snapkv_press_fits reads of a key view
_Geometry = namedtuple("_Geometry", "block_tables block_size max_seq_len stride_token num_kv_heads")


def _press_rows(kv_cache, block_tables, seq_lens, seq_len, width, counts=None, order=None, snapkv=None) -> bool:
    """The host module's call for callers that want the moved rows alone; False: not of the plain form, nothing done."""
    if counts is not None:
        _lib.refuse_capture()
    if _lib.host().press_rows(kv_cache, block_tables, seq_lens, seq_len, width, counts, order, snapkv) is None:
        return False
    _lib.note_enqueued()
    return True


def _select_and_compact(kview, vview, scores, seq_lens, kept: List[int], compact: bool, heads: int) -> PressResult:
    """Top-k per (layer, sequence, head) row and in-place compaction; one launch each whether or not the
    sequences keep the same number of tokens.  (Both in one launch, ``ops.select_compact``, has half the workgroups for
    the compaction: 288 columns of 12000 keys 294 us against 237, 576 of 16384 1228 against 1181, 2304 of 4096 536 against
    525.)"""
    width = max(kept)
    if len(set(kept)) == 1:
        idx = ops.topk_select(scores, width)
        if compact and width > 0:
            ops.compact(kview, vview, kview, vview, idx)
        return PressResult(idx, width, scores)
    n_kept = _lib.upload_ints(kept, scores)
    idx = ops.topk_select(scores, width, row_lens=seq_lens, n_kept=n_kept, rows_per_len=heads)
    if compact and width > 0:
        ops.compact(kview, vview, kview, vview, idx, n_kept=n_kept)
    return PressResult(idx, width, scores, list(kept))


def knorm_compress_paged(kv_cache: torch.Tensor, block_tables: torch.Tensor, seq_lens: torch.Tensor,
                         seq_len: int, compression_ratio: float, compact: bool = True,
                         host_lens: Optional[Sequence[int]] = None, rows_only: bool = False) -> Optional[PressResult]:
    """KnormPress over sequences that all hold ``seq_len`` tokens, or, with ``host_lens`` (the lengths as
    Python ints, ``seq_len`` their maximum), over sequences of different lengths in the same launches: each keeps
    ``int(its length * (1 - compression_ratio))`` tokens.  ``rows_only``: the caller wants the pages compacted and
    nothing else (scores and indices stay scratch)."""
    lens = list(host_lens) if host_lens is not None else [seq_len] * block_tables.shape[0]
    kept = [n_kept_for(n, compression_ratio) for n in lens]
    width = max(kept)
    # One launch (every (layer, sequence, head) column is scored, selected and compacted by one workgroup) or norms,
    # selection and compaction each over the whole chip.  One workgroup per column leaves part of the chip idle below about
    # one and a half columns per compute unit, which long columns feel and short ones do not (us per pass, 60 % dropped, one
    # launch against three, bf16: 112 columns of 300 keys 47 48, of 1000 55 62, of 3000 87 91, of 9000 219 202; 224 of 1000 64
    # 73, of 3000 112 124, of 9000 343 332; 288 of 300 52 53, of 1000 81 80, of 3000 175 160, of 9000 516 446; from there on
    # one launch wins: 448 of 3000 227 229, 576 of 1000 102 116, 1024 of 3000 443 492).
    columns = kv_cache.shape[1] * block_tables.shape[0] * kv_cache.shape[-2] if kv_cache.is_cuda else 0
    cus = _lib.compute_units(kv_cache.device) if columns else 1
    one_launch = (compact and 0 < width and ops.press_column_fits(seq_len, width) and
                  seq_len <= (5000 if columns <= cus else 1000 if 2 * columns <= 3 * cus else seq_len))
    if (rows_only and compact and 0 < width and columns and
            _press_rows(kv_cache, block_tables, seq_lens, seq_len, width, None if len(set(kept)) == 1 else kept,
                        snapkv=None if one_launch else False)):
        return None
    kview, vview = _views(kv_cache, block_tables, seq_lens, seq_len)
    if one_launch:
        if len(set(kept)) == 1:
            scores, idx = ops.knorm_press(kview, vview, width, kv_cache.device)
            return PressResult(idx, width, scores)
        n_kept = _lib.upload_ints(kept, kv_cache)
        scores, idx = ops.knorm_press(kview, vview, width, kv_cache.device, n_kept=n_kept, rows_only=rows_only)
        return PressResult(idx, width, scores, list(kept))
    scores = ops.knorm_score(kview, kv_cache.device)
    return _select_and_compact(kview, vview, scores, seq_lens, kept, compact, kv_cache.shape[4])


def snapkv_compress_paged(kv_cache: torch.Tensor, block_tables: torch.Tensor, seq_lens: torch.Tensor,
                          seq_len: int, queries: torch.Tensor, compression_ratio: float, window_size: int = 64,
                          kernel_size: int = 5, causal_window: bool = True, reduction: str = "mean",
                          window_in_budget: bool = True, compact: bool = True,
                          host_lens: Optional[Sequence[int]] = None, rows_only: bool = False) -> Optional[PressResult]:
    """SnapKVPress over sequences that all hold ``seq_len`` tokens, or (``host_lens``) of different lengths in
    the same launches.  ``queries`` are the rotated window queries ``[L, B, Hq, W, D]`` (the last W positions of
    every sequence).  With ``window_in_budget`` (kvpress) the observation window counts towards ``n_kept``;
    otherwise it is kept on top of it.  ``rows_only``: the caller wants the pages compacted and nothing else."""
    lens = list(host_lens) if host_lens is not None else [seq_len] * block_tables.shape[0]
    kept = [n_kept_for(n, compression_ratio) for n in lens]
    if not window_in_budget:
        kept = [min(n, k + window_size) for n, k in zip(lens, kept)]
    width = max(kept)
    # Without the filled scores: every row keeps more than the window (sequences no longer than the window keep their
    # first positions either way), the window positions rank above every scored key and only the others are ranked.
    # After the window fill they TIE with scored keys that equal the layer's largest score; the two selections differ
    # only when more such keys than a row has places outside the window tie exactly, which needs equal scores at the
    # very top: rows with fewer scored keys than the pooling kernel is wide (every pooled score the same) take the
    # filled scores.
    window_apart = (compact and all(k > window_size or n <= window_size for n, k in zip(lens, kept)) and
                    width > window_size and all(n <= window_size or n - window_size > kernel_size for n in lens))
    # One launch (the workgroup that scored a column also selects and compacts it) or key ranges: with the scores wanted
    # by the rule of snapkv_press_preferred; without them the selection needs no pooled scores in memory and the
    # compaction has a workgroup per plane, and ranges win wherever cutting the columns does (us per pass, a third kept:
    # 112 columns of 4096 keys 295 -> 193, of 1000 94 -> 73, 320 of 12000 1721 -> 1341, 288 of 8192 623 -> 583; whole columns
    # 576 of 2000 281 against 306, 896 of 4096 736 against 812).
    hq = queries.shape[-3]
    H = kv_cache.shape[-2]
    if (rows_only and window_apart and queries.dim() == 5 and kv_cache.dim() == 6 and reduction in ("mean", "sum") and
            window_size > 0 and H > 0 and hq % H == 0 and hq > 0):
        shape = _Geometry(True, kv_cache.shape[3], seq_len, kv_cache.stride(3), H)
        same = len(set(kept)) == 1 and len(set(lens)) == 1
        order = sorted(range(len(lens)), key=lambda b: -lens[b]) if len(set(lens)) > 1 else None   # longest first
        if _press_rows(kv_cache, block_tables, seq_lens, seq_len, width, None if same else kept, order,
                       (queries, window_size, kernel_size, int(causal_window), 1.0 / math.sqrt(kv_cache.shape[5]),
                        1.0 / (window_size * (hq // H)) if reduction == "mean" else 1.0,
                        int(ops.snapkv_press_fits(shape, hq, window_size, width)), sum(lens) // len(lens))):
            return None
    kview, vview = _views(kv_cache, block_tables, seq_lens, seq_len)
    fits = window_apart and ops.snapkv_press_fits(kview, hq, window_size, width)
    once = False      # one pass over the keys, selection and compaction: every kept position is written (window_apart)
    if rows_only and window_apart:
        route = ops.snapkv_rows_route(kview, hq, window_size, fits, sum(lens) // len(lens))
        once = ops.snapkv_rows_once_pays(kview, hq, window_size, sum(lens) // len(lens), width, route)
    else:
        route = 0 if fits and ops.snapkv_press_preferred(kview, hq, window_size, _lib.compute_units(kv_cache.device)) else -1
    if route == 0 and not once:
        same = len(set(kept)) == 1 and len(set(lens)) == 1
        res = ops.snapkv_press(kview, vview, queries, window_size, kernel_size, width, causal_window, reduction,
                               seq_lens=seq_lens, n_kept=None if same else kept, host_lens=lens, rows_only=rows_only)
        if rows_only:
            return None
        scores, idx = res
        return PressResult(idx, width, scores, None if same else list(kept))
    if once or route > 0:
        n_kept = None if len(set(kept)) == 1 and len(set(lens)) == 1 else _lib.upload_ints(kept, kv_cache)
        idx = ops.snapkv_select(kview, queries, window_size, kernel_size, width, causal_window, reduction, n_kept=n_kept,
                                **({"workgroups": 0} if once else {"splits": route}))
        ops.compact(kview, vview, kview, vview, idx, n_kept=n_kept)
        return None
    scores = ops.snapkv_score(kview, queries, window_size, kernel_size, causal_window, reduction,
                              seq_lens=seq_lens)
    return _select_and_compact(kview, vview, scores, seq_lens, kept, compact, kv_cache.shape[4])
