"""Sparse absorbed-MLA (DeepSeek sparse attention) on the dense MLA kernels: the reference's
``python/sgl_jax/srt/kernels/dsa/sparse_mla.py`` re-indexes the page table (or gathers rows) and
hands the result to its dense kernel; here ``rpa_mla_sparse_attention`` writes one page table per query
token and runs the dense kernel over it, two launches in all.  All index work stays
on the device (no host reads), so a call can sit inside a captured step.

* ``compute_topk_pages``     sparse_mla.py:35-60   unique pages a top-k list touches
* ``sparse_mla_page_level``  sparse_mla.py:63-203  decode: dense kernel over the touched pages
* ``sparse_mla_via_dense``   sparse_mla.py:206-297 any T: gather the k rows, dense kernel over them
"""

from __future__ import annotations

import torch

from . import _lib
from .ragged_paged_attention import _i32, _require_gpu


def _first_hits(mask: torch.Tensor, count: int) -> torch.Tensor:
    """Indices of the first ``count`` True entries of each row, ascending (what jax.lax.top_k
    returns for a 0/1 row: equal values keep index order); rows with fewer hits continue with
    the lowest unset indices, as top_k does."""
    n = mask.shape[1]
    pos = torch.arange(n, device=mask.device, dtype=torch.int64)
    key = torch.where(mask, pos, pos + n)
    return torch.sort(key, dim=1).values[:, :count] % n


def compute_topk_pages(topk_indices, *, page_size: int, pages_per_seq: int, k_pages_max: int) -> torch.Tensor:
    """i32[T, k_pages_max]: the sequence-local pages touched by each row of ``topk_indices``
    (i32[T, k], -1 = unused), ascending, padded with -1 (sparse_mla.py:35-60)."""
    idx = topk_indices.to(torch.int64)
    T = idx.shape[0]
    valid = idx >= 0
    page_local = torch.where(valid, idx // page_size, torch.full_like(idx, pages_per_seq))
    mask = torch.zeros((T, pages_per_seq + 1), dtype=torch.bool, device=idx.device)
    mask.scatter_(1, page_local, torch.ones_like(page_local, dtype=torch.bool))
    mask = mask[:, :pages_per_seq]
    n_hit = mask.sum(dim=1)
    k_eff = min(k_pages_max, pages_per_seq)
    hit = _first_hits(mask, k_eff)
    if k_eff < k_pages_max:
        hit = torch.nn.functional.pad(hit, (0, k_pages_max - k_eff))
    col = torch.arange(k_pages_max, device=idx.device)[None, :]
    return torch.where(col < n_hit[:, None], hit, torch.full_like(hit, -1)).to(torch.int32)


def _sparse(ql_nope, q_pe, new_kv_c, new_k_pe, cache_kv, kv_lens, topk, topk_is_pages, page_indices, cu_q_lens,
            cu_kv_lens, sm_scale, page_size, pages_per_seq, k_pages_max):
    """The table of every query token's selection and the dense kernel over it (csrc/rpa_dsa.h, rpa_mla.hip)."""
    native = _lib.load_torch().sparse_mla
    rest = (sm_scale, page_size, pages_per_seq, k_pages_max)
    o = native(ql_nope, q_pe, new_kv_c, new_k_pe, cache_kv, kv_lens, topk, topk_is_pages, page_indices, cu_q_lens,
               cu_kv_lens, *rest)
    if o is None:  # host metadata, wide indices, strided rows: brought into the common form
        _require_gpu(ql_nope, "ql_nope")
        _require_gpu(cache_kv, "cache_kv")
        dev = ql_nope.device
        o = native(ql_nope.contiguous(), q_pe.contiguous(), new_kv_c, new_k_pe, cache_kv, _i32(kv_lens, dev),
                   topk.to(dev).to(torch.int32).contiguous(), topk_is_pages, _i32(page_indices, dev).reshape(-1),
                   _i32(cu_q_lens, dev), _i32(cu_kv_lens, dev), *rest)
        if o is None:
            raise ValueError(f"Expected bfloat16 queries [T, heads, lkv] and [T, heads, rope], a contiguous bfloat16 or float8_e4m3fn "
                             f"cache of pages of {page_size} rows of lkv + rope elements (or each rounded up to 128), new rows of the "
                             f"cache's dtype and one row of indices per query token; got {tuple(ql_nope.shape)} {ql_nope.dtype}, "
                             f"{tuple(q_pe.shape)} {q_pe.dtype}, {tuple(cache_kv.shape)} {cache_kv.dtype}, {tuple(topk.shape)}")
    if type(o) is int:
        _lib.check(o)
    return o


def sparse_mla_page_level(ql_nope, q_pe, new_kv_c, new_k_pe, cache_kv, kv_lens, topk_indices, page_indices,
                          cu_q_lens, cu_kv_lens, distribution, topk_pages=None, *, sm_scale: float, page_size: int,
                          pages_per_seq: int, kv_lora_rank: int, k_pages_max: int = 64, **_tile_hints):
    """Decode (one query token per sequence): attends the whole pages that ``topk_indices``
    touches (or ``topk_pages`` names) plus the page of the new token, which goes last so that the new row
    lands in the true slot (sparse_mla.py:63-203).  Returns ``(o_latent, cache_kv)``; the last
    page of the cache is the padding target, as in the reference."""
    pre = topk_pages is not None
    o = _sparse(ql_nope, q_pe, new_kv_c, new_k_pe, cache_kv, kv_lens, topk_pages if pre else topk_indices, pre, page_indices,
                cu_q_lens, cu_kv_lens, sm_scale, page_size, pages_per_seq, k_pages_max)
    cache_out = cache_kv if cache_kv.dim() == 3 else cache_kv.view(cache_kv.shape[0], -1, cache_kv.shape[3])
    return o if o.shape[-1] == kv_lora_rank else o[..., :kv_lora_rank], cache_out


def sparse_mla_via_dense(ql_nope, q_pe, new_kv_c, new_k_pe, cache_kv, kv_lens, topk_indices, page_indices,
                         cu_q_lens, cu_kv_lens, distribution, *, sm_scale: float, page_size: int,
                         pages_per_seq: int, kv_lora_rank: int, **_tile_hints) -> torch.Tensor:
    """Token-level sparse attention for any T: the k selected rows of every query token are one short
    "sequence" of pages of a single row, ``kv_len`` = number of valid entries; the new token's row
    stands for the last valid entry, where the dense kernel's cache write puts it in the reference
    (sparse_mla.py:206-297; the reference gathers the rows first).  Valid entries must come first in each row."""
    o = _sparse(ql_nope, q_pe, new_kv_c, new_k_pe, cache_kv, kv_lens, topk_indices, False, page_indices, cu_q_lens, cu_kv_lens,
                sm_scale, page_size, pages_per_seq, 0)
    return o if o.shape[-1] == kv_lora_rank else o[..., :kv_lora_rank]
