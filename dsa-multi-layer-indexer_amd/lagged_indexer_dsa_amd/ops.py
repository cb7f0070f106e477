"""torch-tensor entry points onto the C ABI (one launch sequence each).

Every op requires device (HIP) tensors and runs on torch's current stream;
there is no CPU path.  Shapes/dtypes are checked here; the library re-checks
its own contract and raises :class:`DsaError` (a RuntimeError) on violation.
"""

from __future__ import annotations

import torch

from . import _lib
from ._lib import (
    DSA_TOPK_POSITION_ORDER,
    DSA_TOPK_SORTED,
    INDEX_DIM,
    INDEX_PAGE_BYTES,
    LATENT_DIM,
    LATENT_ROW_BYTES,
    PAGE_TOKENS,
    QK_DIM,
)


def _dev(*tensors: torch.Tensor) -> None:
    for t in tensors:
        if not isinstance(t, torch.Tensor) or not t.is_cuda:
            raise RuntimeError("lagged_indexer_dsa_amd ops need GPU (HIP) tensors; there is no CPU path")
        if not t.is_contiguous():
            raise RuntimeError("lagged_indexer_dsa_amd ops need contiguous tensors")


def _stream() -> int:
    return torch.cuda.current_stream().cuda_stream


def _ptr(t: torch.Tensor | None) -> int | None:
    return None if t is None else t.data_ptr()


def _nbytes(t: torch.Tensor) -> int:
    return t.numel() * t.element_size()


def _need_bytes(name: str, t: torch.Tensor, nbytes: int) -> None:
    """The C ABI takes raw pointers: a caller buffer smaller than the
    library's size function says would be overrun on the device."""
    if _nbytes(t) < nbytes:
        raise RuntimeError(f"{name} holds {_nbytes(t)} bytes, the call needs {nbytes}")


def _need_shape(name: str, t: torch.Tensor, shape: tuple, dtype) -> None:
    if tuple(t.shape) != tuple(shape) or t.dtype != dtype or not t.is_contiguous():
        raise RuntimeError(f"{name} must be contiguous {dtype} {tuple(shape)}, got {t.dtype} {tuple(t.shape)}")


def indexer_scan(q_fp8: torch.Tensor, w: torch.Tensor, index_k: torch.Tensor,
                 page_table: torch.Tensor, seq_lens: torch.Tensor, slab_stride: int,
                 out: torch.Tensor | None = None) -> torch.Tensor:
    """fp8 lightning-indexer scores over the paged index-K cache.

    q_fp8 [B,Hidx,128] uint8 (e4m3 codes) or float8_e4m3fn; w [B,Hidx] f32
    (q-scale folded in); index_k [P,8448] uint8; page_table [B,pt] int32;
    seq_lens [B] int32  ->  scores [B, slab_stride] f32 (-inf past seq_len).
    Reference: K:2990-2992 ref_indexer_logits_fp8; attention_core.py:27-49.
    """
    q_fp8 = q_fp8.view(torch.uint8) if q_fp8.dtype == torch.float8_e4m3fn else q_fp8
    _dev(q_fp8, w, index_k, page_table, seq_lens)
    B, Hidx, D = q_fp8.shape
    if D != INDEX_DIM or q_fp8.dtype != torch.uint8:
        raise RuntimeError("q_fp8 must be [B, Hidx, 128] e4m3 bytes")
    if w.shape != (B, Hidx) or w.dtype != torch.float32:
        raise RuntimeError("w must be [B, Hidx] float32")
    if index_k.dim() != 2 or index_k.shape[1] != INDEX_PAGE_BYTES or index_k.dtype != torch.uint8:
        raise RuntimeError("index_k must be [pages, 8448] uint8")
    if page_table.dim() != 2 or page_table.shape[0] != B or page_table.dtype != torch.int32:
        raise RuntimeError("page_table must be [B, pt_stride] int32")
    if seq_lens.shape != (B,) or seq_lens.dtype != torch.int32:
        raise RuntimeError("seq_lens must be [B] int32")
    if out is None:
        out = torch.empty(B, slab_stride, dtype=torch.float32, device=q_fp8.device)
    _dev(out)
    if out.shape != (B, slab_stride) or out.dtype != torch.float32:
        raise RuntimeError("out must be [B, slab_stride] float32")
    _lib.call("dsa_indexer_scan", q_fp8.data_ptr(), w.data_ptr(), index_k.data_ptr(),
              index_k.shape[0], page_table.data_ptr(), seq_lens.data_ptr(), out.data_ptr(),
              B, Hidx, page_table.shape[1], slab_stride, _stream())
    return out


def topk_scratch(B: int, slab: int, device) -> torch.Tensor:
    """Zero-filled scratch for :func:`topk` (each call leaves it zeroed)."""
    nbytes = _lib.load().dsa_topk_scratch_bytes(B, slab)
    if nbytes == 0:
        raise RuntimeError(f"bad top-k scratch shape B={B} slab={slab}")
    return torch.zeros(nbytes // 4, dtype=torch.int32, device=device)


def topk(scores: torch.Tensor, seq_lens: torch.Tensor, k: int, sorted: bool = False,
         pad_value: int = -1, page_table: torch.Tensor | None = None,
         out: torch.Tensor | None = None, scratch: torch.Tensor | None = None) -> torch.Tensor:
    """Exact top-k per row (score desc, ties -> lower index), int32 [B, k].

    sorted=False: ascending positions (or KV slots through page_table), pads
    last.  sorted=True: torch.topk order with the lower-index tie rule.
    Non-finite selections and missing slots are ``pad_value``.
    Reference: attention_core.py:66-91 select_topk.
    """
    _dev(scores, seq_lens)
    if scores.dim() != 2 or scores.dtype != torch.float32:
        raise RuntimeError("scores must be [B, slab] float32")
    B, slab = scores.shape
    if seq_lens.shape != (B,) or seq_lens.dtype != torch.int32:
        raise RuntimeError("seq_lens must be [B] int32")
    if page_table is not None:
        _dev(page_table)
    if out is None:
        out = torch.empty(B, k, dtype=torch.int32, device=scores.device)
    if scratch is None:
        scratch = topk_scratch(B, slab, scores.device)
    _dev(out, scratch)
    _need_shape("out", out, (B, k), torch.int32)
    _need_bytes("top-k scratch", scratch, _lib.load().dsa_topk_scratch_bytes(B, slab))
    _lib.call("dsa_topk", scores.data_ptr(), seq_lens.data_ptr(), _ptr(page_table),
              0 if page_table is None else page_table.shape[1], scratch.data_ptr(),
              out.data_ptr(), B, slab, k,
              DSA_TOPK_SORTED if sorted else DSA_TOPK_POSITION_ORDER, pad_value, _stream())
    return out


def select_rows(scores: torch.Tensor, k: int, pad_value: int) -> torch.Tensor | None:
    """:func:`topk` with sorted=True over whole rows, as int64 and in one
    launch; None for the shapes the row kernel does not take."""
    _dev(scores)
    shape = scores.shape
    if len(shape) != 2 or scores.dtype != torch.float32:
        raise RuntimeError("scores must be [B, slab] float32")
    B, slab = shape
    if not _lib.load().dsa_select_rows_supported(B, slab, k):
        return None
    out = torch.empty(B, k, dtype=torch.int64, device=scores.device)
    _lib.call("dsa_select_rows", scores.data_ptr(), None, out.data_ptr(), B, slab, k, pad_value, _stream())
    return out


def sparse_mla_workspace(B: int, H: int, nsplit: int, device) -> torch.Tensor:
    """Zero-filled workspace (split partials + the splits' barriers; every
    call leaves the barriers ready).  nsplit=0 sizes it for any split count."""
    nbytes = _lib.load().dsa_sparse_mla_workspace_bytes(B, H, nsplit)
    if nbytes == 0:
        raise RuntimeError(f"bad sparse MLA workspace shape B={B} H={H} nsplit={nsplit}")
    return torch.zeros(nbytes // 4, dtype=torch.float32, device=device)


def _call_workspace(B: int, H: int, nsplit: int, device) -> torch.Tensor:
    """Workspace of one call at a known split count: the barriers zeroed, the
    partials (overwritten before they are read) not.  Many unsplit rows read
    neither."""
    lib = _lib.load()
    nbytes = lib.dsa_sparse_mla_workspace_bytes(B, H, nsplit)
    if nbytes == 0:
        raise RuntimeError(f"bad sparse MLA workspace shape B={B} H={H} nsplit={nsplit}")
    barriers = lib.dsa_sparse_mla_barrier_bytes(B, H, nsplit)
    ws = torch.empty(nbytes // 4 if barriers else 4, dtype=torch.float32, device=device)
    ws[:barriers // 4].zero_()
    return ws


def _resolve_nsplit(nsplit: int, B: int, H: int, keys: int) -> int:
    """The split count a call takes (nsplit = 0: the library's choice)."""
    return nsplit or max(1, _lib.load().dsa_sparse_mla_auto_nsplit(B, H, keys))


def sparse_mla_decode(q: torch.Tensor, kv_pool: torch.Tensor, idx: torch.Tensor,
                      sm_scale: float | None = None, nsplit: int = 0,
                      workspace: torch.Tensor | None = None,
                      out: torch.Tensor | None = None) -> torch.Tensor:
    """Split-K sparse MLA over the fp8 656-byte latent pool.

    q [B,H,576] bf16; kv_pool [rows,656] uint8; idx [B,topk] int32 KV slots
    (out-of-range = masked)  ->  out [B,H,512] bf16.
    Reference: attention_core.py:121-146 sparse_mla_core; K:2950-2966.
    """
    _dev(q, kv_pool, idx)
    if q.dim() != 3 or q.shape[2] != QK_DIM or q.dtype != torch.bfloat16:
        raise RuntimeError("q must be [B, H, 576] bfloat16")
    B, H, _ = q.shape
    if kv_pool.dim() != 2 or kv_pool.shape[1] != LATENT_ROW_BYTES or kv_pool.dtype != torch.uint8:
        raise RuntimeError("kv_pool must be [rows, 656] uint8")
    if idx.dim() != 2 or idx.shape[0] != B or idx.dtype != torch.int32:
        raise RuntimeError("idx must be [B, topk] int32")
    if sm_scale is None:
        sm_scale = QK_DIM ** -0.5
    if workspace is None:
        nsplit = _resolve_nsplit(nsplit, B, H, idx.shape[1])
        workspace = _call_workspace(B, H, nsplit, q.device)
    else:  # sized for this nsplit (nsplit=0, the library's choice: the largest size)
        _dev(workspace)
        _need_bytes("sparse MLA workspace", workspace, _lib.load().dsa_sparse_mla_workspace_bytes(B, H, nsplit))
    if out is None:
        out = torch.empty(B, H, LATENT_DIM, dtype=torch.bfloat16, device=q.device)
    _dev(out)
    _need_shape("out", out, (B, H, LATENT_DIM), torch.bfloat16)
    _lib.call("dsa_sparse_mla_decode", q.data_ptr(), kv_pool.data_ptr(), kv_pool.shape[0],
              idx.data_ptr(), workspace.data_ptr(), out.data_ptr(), B, H, idx.shape[1], nsplit,
              float(sm_scale), _stream())
    return out


def dense_mla_decode(q: torch.Tensor, kv_pool: torch.Tensor, page_table: torch.Tensor, seq_lens: torch.Tensor,
                     sm_scale: float | None = None, nsplit: int = 0,
                     workspace: torch.Tensor | None = None,
                     out: torch.Tensor | None = None) -> torch.Tensor:
    """Dense MLA of each decode row over its first seq_lens[b] tokens, their
    latent rows found through the page table (64-token pages).

    q [B,H,576] bf16; kv_pool [rows,656] uint8; page_table [B,pt] int32;
    seq_lens [B] int32  ->  out [B,H,512] bf16.
    Reference: attention_core.py:142-160 dense_mla_core; model.py:104-114.
    """
    _dev(q, kv_pool, page_table, seq_lens)
    if q.dim() != 3 or q.shape[2] != QK_DIM or q.dtype != torch.bfloat16:
        raise RuntimeError("q must be [B, H, 576] bfloat16")
    B, H, _ = q.shape
    if kv_pool.dim() != 2 or kv_pool.shape[1] != LATENT_ROW_BYTES or kv_pool.dtype != torch.uint8:
        raise RuntimeError("kv_pool must be [rows, 656] uint8")
    if page_table.dim() != 2 or page_table.shape[0] != B or page_table.dtype != torch.int32:
        raise RuntimeError("page_table must be [B, pt_stride] int32")
    _need_shape("seq_lens", seq_lens, (B,), torch.int32)
    if sm_scale is None:
        sm_scale = QK_DIM ** -0.5
    if workspace is None:
        nsplit = _resolve_nsplit(nsplit, B, H, page_table.shape[1] * PAGE_TOKENS)
        workspace = _call_workspace(B, H, nsplit, q.device)
    else:  # sized for this nsplit (nsplit=0, the library's choice: the largest size)
        _dev(workspace)
        _need_bytes("sparse MLA workspace", workspace, _lib.load().dsa_sparse_mla_workspace_bytes(B, H, nsplit))
    if out is None:
        out = torch.empty(B, H, LATENT_DIM, dtype=torch.bfloat16, device=q.device)
    _dev(out)
    _need_shape("out", out, (B, H, LATENT_DIM), torch.bfloat16)
    _lib.call("dsa_dense_mla_decode", q.data_ptr(), kv_pool.data_ptr(), kv_pool.shape[0], page_table.data_ptr(),
              page_table.shape[1], seq_lens.data_ptr(), workspace.data_ptr(), out.data_ptr(), B, H, nsplit,
              float(sm_scale), _stream())
    return out


# ---- prefill attention (many query rows against the same keys) ----

_PACK_DTYPES = {torch.float32: 0, torch.bfloat16: 1, torch.float16: 2}


def _kernel_input(x: torch.Tensor) -> torch.Tensor:
    """x as the prefill kernels read it: fp32, bf16 or fp16, contiguous,
    16-byte aligned."""
    x = (x if x.dtype in _PACK_DTYPES else x.float()).contiguous()
    return x if x.data_ptr() % 16 == 0 else x.clone()


def _need_kv(kv: torch.Tensor) -> None:
    shape = kv.shape
    if len(shape) != 3 or shape[2] != QK_DIM:
        raise RuntimeError(f"kv must be [B, T, 576], got {tuple(shape)}")


def _pack_source(kv: torch.Tensor) -> torch.Tensor:
    """kv [B, T, 576] as the pack kernels read it (rope rounded to bf16 once)."""
    if kv.dtype not in _PACK_DTYPES:
        x = kv.float()
        x[..., LATENT_DIM:] = kv[..., LATENT_DIM:].to(torch.bfloat16)
        kv = x
    return _kernel_input(kv)


def prefill_logits(q: torch.Tensor, k: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """Indexer scores [B, S, T] fp32 of q [B, S, H, 128] and w [B, S, H] over
    k [B, T, 128], quantised per row inside.  Reference: attention_core.py:27-49."""
    q, k, w = _kernel_input(q), _kernel_input(k), _kernel_input(w)
    _dev(q, k, w)
    qs, ks = q.shape, k.shape  # (each read of a shape builds it anew)
    if len(qs) != 4 or qs[3] != INDEX_DIM:
        raise RuntimeError(f"q must be [B, S, H, 128], got {tuple(qs)}")
    B, S, H, _ = qs
    if len(ks) != 3 or ks[0] != B or ks[2] != INDEX_DIM:
        raise RuntimeError(f"k must be [{B}, T, 128], got {tuple(ks)}")
    if w.shape != qs[:3]:
        raise RuntimeError(f"w must be {(B, S, H)}, got {tuple(w.shape)}")
    T = ks[1]
    ws = torch.empty(_lib.load().dsa_prefill_logits_workspace_bytes(B, S, H, T), dtype=torch.uint8, device=q.device)
    out = torch.empty(B, S, T, dtype=torch.float32, device=q.device)
    _lib.call("dsa_prefill_logits", q.data_ptr(), _PACK_DTYPES[q.dtype], k.data_ptr(), _PACK_DTYPES[k.dtype],
              w.data_ptr(), _PACK_DTYPES[w.dtype], ws.data_ptr(), out.data_ptr(), B, S, H, T, _stream())
    return out


def pack_latent_rows(kv: torch.Tensor, row_stride: int) -> torch.Tensor:
    """kv [B, T, 576] -> 656-byte fp8 rows [B * row_stride, 656] (rows past T
    of a request zero)."""
    _need_kv(kv)
    kv = _pack_source(kv)
    _dev(kv)
    B, T, _ = kv.shape
    if row_stride < T:
        raise RuntimeError(f"row_stride {row_stride} below the {T} rows of a request")
    rows = torch.empty(B * row_stride, LATENT_ROW_BYTES, dtype=torch.uint8, device=kv.device)
    _lib.call("dsa_pack_latent_rows", kv.data_ptr(), _PACK_DTYPES[kv.dtype], B, T, row_stride, rows.data_ptr(),
              _stream())
    return rows


def selection_set(idx: torch.Tensor, T: int, as_bits: bool) -> torch.Tensor:
    """Selections idx [B, S, n] (int32 or int64 positions) as sets over the
    row's causal keys (query row s of S sees keys 0 .. T - S + s): a bitmap per
    row, or the KV slots b * T + position ascending, then -1 [B * S, n]."""
    idx = idx.contiguous()
    _dev(idx)
    shape = idx.shape
    if len(shape) != 3 or idx.dtype not in (torch.int32, torch.int64):
        raise RuntimeError(f"idx must be [B, S, n] int32 or int64, got {idx.dtype} {tuple(shape)}")
    B, S, n = shape
    lib = _lib.load()
    if as_bits:
        out = torch.empty(lib.dsa_selection_bits_bytes(B * S, T) // 4, dtype=torch.int32, device=idx.device)
    else:
        out = torch.empty(B * S, n, dtype=torch.int32, device=idx.device)
    _lib.call("dsa_selection_set", idx.data_ptr(), idx.element_size(), B, S, n, T,
              out.data_ptr() if as_bits else None, None if as_bits else out.data_ptr(), _stream())
    return out


def prefill_attention(q: torch.Tensor, kv: torch.Tensor, bits: torch.Tensor | None = None,
                      sm_scale: float | None = None) -> torch.Tensor:
    """q [B, S, H, 576] bf16 over kv [B, T, 576]: query row s of S attends keys
    0 .. T - S + s, or those of its bitmap (:func:`selection_set`) ->
    [B, S, H, 512] bf16.  Reference: attention_core.py:121-160."""
    _need_kv(kv)
    kv = _pack_source(kv)
    _dev(q, kv)
    qs = q.shape
    if len(qs) != 4 or qs[3] != QK_DIM or q.dtype != torch.bfloat16:
        raise RuntimeError("q must be [B, S, H, 576] bfloat16")
    B, S, H, _ = qs
    requests, T, _ = kv.shape
    if requests != B:
        raise RuntimeError(f"kv holds {requests} requests, q {B}")
    lib = _lib.load()
    keys = torch.empty(lib.dsa_prefill_keys_bytes(B, T), dtype=torch.uint8, device=q.device)
    ws = torch.empty(lib.dsa_prefill_workspace_bytes(B, S, H, T), dtype=torch.uint8, device=q.device)
    out = torch.empty(B, S, H, LATENT_DIM, dtype=torch.bfloat16, device=q.device)
    if bits is not None:
        _dev(bits)
        if bits.dtype != torch.int32:
            raise RuntimeError("bits must be int32")
        _need_bytes("bits", bits, lib.dsa_selection_bits_bytes(B * S, T))
    st = _stream()
    _lib.call("dsa_pack_prefill_keys", kv.data_ptr(), _PACK_DTYPES[kv.dtype], B, T, keys.data_ptr(), st)
    _lib.call("dsa_prefill_attention", q.data_ptr(), keys.data_ptr(), _ptr(bits), ws.data_ptr(), out.data_ptr(),
              B, S, H, T, float(QK_DIM ** -0.5 if sm_scale is None else sm_scale), st)
    return out


# ---- decode-step operand preparation (the inputs the decode layer reads) ----

def quantize_index_query(q: torch.Tensor, w: torch.Tensor, out_q: torch.Tensor | None = None,
                         out_w: torch.Tensor | None = None) -> tuple[torch.Tensor, torch.Tensor]:
    """Indexer query [B, Hidx, 128] bf16 and head weights [B, Hidx] fp32 ->
    (e4m3 codes uint8 [B, Hidx, 128], folded weights w * scale fp32).
    Per (token, head): scale = max(amax, 1e-6) / 448 (K:2969-2974, K:2984-2985)."""
    _dev(q, w)
    if q.dim() != 3 or q.shape[2] != INDEX_DIM or q.dtype != torch.bfloat16:
        raise RuntimeError("q must be [B, Hidx, 128] bfloat16")
    B, H, _ = q.shape
    _need_shape("w", w, (B, H), torch.float32)
    if out_q is None:
        out_q = torch.empty(B, H, INDEX_DIM, dtype=torch.uint8, device=q.device)
    if out_w is None:
        out_w = torch.empty(B, H, dtype=torch.float32, device=q.device)
    _dev(out_q, out_w)
    _need_shape("out_q", out_q, (B, H, INDEX_DIM), torch.uint8)
    _need_shape("out_w", out_w, (B, H), torch.float32)
    _lib.call("dsa_quantize_index_query", q.data_ptr(), w.data_ptr(), out_q.data_ptr(), out_w.data_ptr(),
              B, H, _stream())
    return out_q, out_w


def append_index_keys(index_k: torch.Tensor, page_table: torch.Tensor, rows: torch.Tensor,
                      pos: torch.Tensor, keys: torch.Tensor) -> None:
    """Quantize keys [n, 128] bf16 (per token, e4m3 + fp32 scale) into the
    paged index cache at token positions pos[i] of rows rows[i] (P:339-342)."""
    _dev(index_k, page_table, rows, pos, keys)
    n = keys.shape[0]
    if keys.dim() != 2 or keys.shape[1] != INDEX_DIM or keys.dtype != torch.bfloat16:
        raise RuntimeError("keys must be [n, 128] bfloat16")
    if index_k.dim() != 2 or index_k.shape[1] != INDEX_PAGE_BYTES or index_k.dtype != torch.uint8:
        raise RuntimeError("index_k must be [pages, 8448] uint8")
    if page_table.dim() != 2 or page_table.dtype != torch.int32:
        raise RuntimeError("page_table must be [B, pt_stride] int32")
    _need_shape("rows", rows, (n,), torch.int32)
    _need_shape("pos", pos, (n,), torch.int32)
    _lib.call("dsa_append_index_keys", keys.data_ptr(), rows.data_ptr(), pos.data_ptr(), n,
              page_table.data_ptr(), page_table.shape[1], index_k.data_ptr(), index_k.shape[0], _stream())


def append_latent_rows(kv_pool: torch.Tensor, slots: torch.Tensor, latent: torch.Tensor) -> None:
    """Pack latent [n, 576] bf16 (512 latent | 64 rope) into 656-byte fp8 rows
    at KV slots slots[i] (per-128 e4m3 + fp32 scales, bf16 rope; K:1114)."""
    _dev(kv_pool, slots, latent)
    n = latent.shape[0]
    if latent.dim() != 2 or latent.shape[1] != QK_DIM or latent.dtype != torch.bfloat16:
        raise RuntimeError("latent must be [n, 576] bfloat16")
    if kv_pool.dim() != 2 or kv_pool.shape[1] != LATENT_ROW_BYTES or kv_pool.dtype != torch.uint8:
        raise RuntimeError("kv_pool must be [rows, 656] uint8")
    _need_shape("slots", slots, (n,), torch.int32)
    _lib.call("dsa_append_latent_rows", latent.data_ptr(), slots.data_ptr(), n, kv_pool.data_ptr(),
              kv_pool.shape[0], _stream())
