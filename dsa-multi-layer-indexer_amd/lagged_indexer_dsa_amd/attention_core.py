"""Drop-in for the reference's core DSA ops on the MI355X path.

Same names, argument shapes, return shapes and argument errors (ValueError)
as the reference's plain-PyTorch ops (src/lagged_indexer_dsa/
attention_core.py:23-160), so ``DSALayer`` and ``DSAModel`` (dsa_layer.py,
model.py) can call them unchanged -- see :func:`install`.  Every op takes
GPU (HIP) tensors and runs the hand-written kernels of this package; there is
no CPU path (a CPU tensor raises).

Numerics are those of the reference's GPU decode path, which the HIP kernels
implement:

* :func:`indexer_logits` quantises the keys per token and the queries per
  head to OCP e4m3 (scale = amax / 448, the query scale folded into the head
  weight; K:2969-2974, K:2984-2985) and contracts them on fp8 MFMA:
  ``I[g] = s_k[g] * sum_h w'[h] * ReLU(q8[h] . k8[g])`` (K:2990-2992).
* :func:`select_topk` is exact on the fp32 logits it is given: rank by
  value (-0.0 == +0.0, NaN above +inf), ties to the LOWER index (the tie
  order torch.topk leaves open), non-finite selections and missing slots
  -> the sentinel ``S_kv`` (attention_core.py:66-91).
* :func:`sparse_mla_core` quantises the latent rows to the 656-byte fp8
  format (512 e4m3 + 4 fp32 per-128 scales + 64 bf16 rope; K:1181-1197)
  and the queries to bf16, and runs the split-K sparse MLA kernel over each
  row's gathered keys, or the prefill kernel over all keys with the others
  masked (the same values either way).  A row
  with no admissible key returns 0 (the GPU kernels' rule, K:1038-1042;
  the dense CPU op would return NaN there).

Causality follows the GPU kernels' convention: query row s of S sits at
position ``S_kv - S + s`` (K:245).  For S == S_kv (aligned prefill) that is
the reference CPU ops' rule; for a decode row (S == 1) it admits the whole
prefix, which is what the reference's decode kernels do.
"""

from __future__ import annotations

import torch

from . import ops
from ._lib import INDEX_DIM, LATENT_DIM, QK_DIM, SELECTION_MAX_CTX, TOPK_MAX_CTX

def _gpu(*ts: torch.Tensor) -> None:
    for t in ts:
        if not t.is_cuda:
            raise RuntimeError("lagged_indexer_dsa_amd.attention_core runs on GPU (HIP) tensors only")


def _need_rows(rows: int) -> None:
    if not 1 <= rows <= 65535:
        raise RuntimeError(f"B * S must be in [1, 65535] (got {rows})")


def pad_index(seq_len_kv: int) -> int:
    """The out-of-range index sentinel: ``S_kv`` (attention_core.py:21-23)."""
    return seq_len_kv


def _q_pos(S: int, Skv: int, device) -> torch.Tensor:
    return torch.arange(Skv - S, Skv, device=device)


def indexer_logits(index_q: torch.Tensor, index_k: torch.Tensor, weights: torch.Tensor) -> torch.Tensor:
    """Lightning-indexer scores ``[B, S, S_kv]`` (attention_core.py:27-49).

    index_q ``[B, S, H_idx, 128]``, index_k ``[B, S_kv, 128]``, weights
    ``[B, S, H_idx]``; H_idx one of 16, 32, 48, 64.  No causal masking
    (apply it with :func:`apply_causal_mask`, as the reference does).
    """
    qs, ks = index_q.shape, index_k.shape
    if len(qs) != 4:
        raise ValueError(f"index_q must be [B,S,H,D], got {tuple(qs)}")
    if len(ks) != 3:
        raise ValueError(f"index_k must be [B,S_kv,D], got {tuple(ks)}")
    B, S, H, D = qs
    if ks[0] != B or ks[2] != D or weights.shape != qs[:3]:
        raise ValueError("index_q, index_k and weights disagree in B, S, H or D")
    if D != INDEX_DIM:
        raise ValueError(f"the fp8 indexer contracts D = {INDEX_DIM}, got {D}")
    _gpu(index_q, index_k, weights)
    if ks[1] == 0:  # no key: nothing to launch, the other limits hold
        _need_rows(B * S)
        if H not in (16, 32, 48, 64):
            raise RuntimeError(f"index_n_heads must be 16, 32, 48 or 64 (got {H})")
        return torch.empty(B, S, 0, dtype=torch.float32, device=index_q.device)
    return ops.prefill_logits(index_q, index_k, weights)


def apply_causal_mask(logits: torch.Tensor) -> torch.Tensor:
    """Scores of keys after each query's position -> -inf
    (attention_core.py:52-63; query row s is at position S_kv - S + s)."""
    _gpu(logits)
    S, Skv = logits.shape[1], logits.shape[2]
    k_pos = torch.arange(Skv, device=logits.device)[None, :]
    causal = k_pos <= _q_pos(S, Skv, logits.device)[:, None]
    return logits.masked_fill(~causal.unsqueeze(0), float("-inf"))


def select_topk(logits: torch.Tensor, topk: int) -> torch.Tensor:
    """Top-``topk`` key indices per query, int64 ``[B, S, topk]``, ordered by
    score (attention_core.py:66-91); non-finite or missing -> ``S_kv``."""
    if logits.dim() != 3:
        raise ValueError(f"logits must be [B,S,S_kv], got {tuple(logits.shape)}")
    _gpu(logits)
    B, S, Skv = logits.shape
    if Skv > TOPK_MAX_CTX:
        raise ValueError(f"S_kv {Skv} above the select's limit {TOPK_MAX_CTX}")
    rows = logits.reshape(B * S, Skv).float().contiguous()
    idx = ops.select_rows(rows, topk, pad_index(Skv))
    if idx is not None:
        return idx.reshape(B, S, topk)
    seq = torch.full((B * S,), Skv, dtype=torch.int32, device=logits.device)
    idx = ops.topk(rows, seq, topk, sorted=True, pad_value=pad_index(Skv))
    return idx.to(torch.int64).reshape(B, S, topk)


def _pool_rows(kv: torch.Tensor) -> torch.Tensor:
    """[B, S_kv, 576] -> the 656-byte fp8 latent rows, batch-major slots."""
    return ops.pack_latent_rows(kv, kv.shape[1])


def _attend_by_tiles(B: int, S: int, H: int, Skv: int, n: int) -> bool:
    """Whether selections of n entries are attended by the prefill kernel,
    which reads every key once per 128 (query, head) rows and masks the
    others, or gathered row by row.

    With the chip full (4096 rows and more) a gathered key costs about what
    2.5 streamed ones do (1024 queries x 16 heads, top-2048: 4096 tokens
    189 us against 236, 5120 tokens 224 against 236, 6144 tokens 261 against
    234, 8192 tokens 325 against 230; 2048 queries, 6144 tokens 411 against
    424); with fewer rows the gather spreads over the idle CUs and the line
    lies near 2 (100 queries, top-2048: 2048 tokens 45 against 52, 4096 equal,
    8192 69 against 57; 200 queries, 4096 equal); with a handful of queries both are a few launches
    and splitting the stream over the CUs is as quick up to a few thousand
    tokens (4 queries: 4096 tokens 33 against 43 us, 12000 tokens 44 against
    43; 16 queries: 2048 tokens 37 against 43, 4096 tokens 45 against 43)."""
    rows = B * S * H
    visible = Skv - (S - 1) / 2
    if rows <= 64:
        return visible <= 8192
    if rows <= 256:
        return visible <= 4096
    return visible <= (2.5 if rows >= 4096 else 2.0) * n


def _attend_rows(q: torch.Tensor, kv: torch.Tensor, idx: torch.Tensor, sm_scale: float) -> torch.Tensor:
    """q [B,S,H,576], kv [B,S_kv,576], idx [B,S,n] int64 (admissible key
    positions or -1) -> [B,S,H,512] in q's dtype."""
    B, S, H, _ = q.shape
    Skv = kv.shape[1]
    # a selection is a set: a repeated index counts once (the reference's
    # scatter mask, attention_core.py:94-103)
    srt, _ = torch.sort(idx, dim=-1)
    dup = torch.zeros_like(srt, dtype=torch.bool)
    dup[..., 1:] = (srt[..., 1:] == srt[..., :-1]) & (srt[..., 1:] >= 0)
    srt = srt.masked_fill(dup, -1)
    base = (torch.arange(B, device=q.device) * Skv)[:, None, None]
    slots = torch.where(srt >= 0, srt + base, torch.full_like(srt, -1))
    n = slots.shape[-1]
    qb = q.reshape(B * S, H, QK_DIM).to(torch.bfloat16).contiguous()
    out = ops.sparse_mla_decode(qb, _pool_rows(kv), slots.reshape(B * S, n).to(torch.int32).contiguous(),
                                sm_scale=sm_scale)
    return out.reshape(B, S, H, LATENT_DIM).to(q.dtype)


def _check_mla(q: torch.Tensor, kv: torch.Tensor, value_dim: int) -> None:
    if q.dim() != 4 or kv.dim() != 3:
        raise ValueError(f"q must be [B,S,H,D] and kv [B,S_kv,D], got {tuple(q.shape)}, {tuple(kv.shape)}")
    if q.shape[0] != kv.shape[0] or q.shape[3] != kv.shape[2]:
        raise ValueError("q and kv disagree in B or D")
    if q.shape[3] != QK_DIM or value_dim != LATENT_DIM:
        raise ValueError(f"the fp8 latent format is D_qk = {QK_DIM}, value_dim = {LATENT_DIM}")
    if q.shape[2] % 16:
        raise ValueError("the head count must be a multiple of 16")
    _gpu(q, kv)


def sparse_mla_core(q: torch.Tensor, kv: torch.Tensor, indices: torch.Tensor, value_dim: int,
                    sm_scale: float | None = None) -> torch.Tensor:
    """Sparse MLA over the selected and causal keys, ``[B, S, H, value_dim]``
    (attention_core.py:121-139).  indices ``[B, S, topk]``; out-of-range
    entries (the sentinel ``S_kv``, negatives) and keys after the query's
    position are not attended."""
    _check_mla(q, kv, value_dim)
    if indices.dim() != 3 or indices.shape[:2] != q.shape[:2]:
        raise ValueError(f"indices must be [B,S,topk], got {tuple(indices.shape)}")
    _gpu(indices)
    B, S, H, _ = q.shape
    Skv, n = kv.shape[1], indices.shape[2]
    if sm_scale is None:
        sm_scale = q.shape[-1] ** -0.5
    idx = indices if indices.dtype in (torch.int32, torch.int64) else indices.long()
    if 1 <= Skv <= SELECTION_MAX_CTX and B * Skv < 1 << 31 and B * S >= 1 and n >= 1:
        if B * S <= 65535 and _attend_by_tiles(B, S, H, Skv, n):
            out = ops.prefill_attention(q.to(torch.bfloat16).contiguous(), kv, ops.selection_set(idx, Skv, True),
                                        float(sm_scale))
        else:
            qb = q.reshape(B * S, H, QK_DIM).to(torch.bfloat16).contiguous()
            out = ops.sparse_mla_decode(qb, _pool_rows(kv), ops.selection_set(idx, Skv, False),
                                        sm_scale=float(sm_scale))
        return out.reshape(B, S, H, LATENT_DIM).to(q.dtype)
    idx = idx.long()
    q_pos = _q_pos(S, Skv, q.device)[None, :, None]
    ok = (idx >= 0) & (idx < Skv) & (idx <= q_pos)
    return _attend_rows(q, kv, torch.where(ok, idx, torch.full_like(idx, -1)), float(sm_scale))


def dense_mla_core(q: torch.Tensor, kv: torch.Tensor, value_dim: int,
                   sm_scale: float | None = None) -> torch.Tensor:
    """Dense causal MLA (full-attention layers and the DENSE cold start,
    attention_core.py:142-160): query row s attends keys 0 .. S_kv - S + s,
    on the prefill kernel (no limit on S_kv), at every number of rows: down to
    one query of 16 heads it reads and converts the keys once for all of
    them (measured against a decode row per query: 1 query over 8192 keys 33
    against 144 us, 8 over 1000 31 against 111, 1000 over 1000 74 against
    194)."""
    _check_mla(q, kv, value_dim)
    B, S, H, _ = q.shape
    if sm_scale is None:
        sm_scale = q.shape[-1] ** -0.5
    if kv.shape[1] == 0:  # no key: every row is empty, the other limits hold
        _need_rows(B * S)
        if not 16 <= H <= 1024:
            raise RuntimeError(f"the head count must be 16 to 1024 (got {H})")
        return torch.zeros(B, S, H, LATENT_DIM, dtype=q.dtype, device=q.device)
    out = ops.prefill_attention(q.to(torch.bfloat16).contiguous(), kv, sm_scale=float(sm_scale))
    return out.to(q.dtype)


_NAMES = ("pad_index", "indexer_logits", "apply_causal_mask", "select_topk", "sparse_mla_core",
          "dense_mla_core")


def install(module) -> None:
    """Rebind the core-op names a reference module imported (for instance
    ``lagged_indexer_dsa.dsa_layer``, which binds them at import time,
    dsa_layer.py:21-27) to these GPU ops."""
    for name in _NAMES:
        if hasattr(module, name):
            setattr(module, name, globals()[name])
