"""GPU: the prefill attention kernel (attention_core.dense_mla_core, and
sparse_mla_core where it streams and masks) and its pack and selection-set
kernels, at the edges of their tiles.

Reference: softmax attention in float64 over the values the 656-byte row
format holds (oracle: quantise per 128 dims, dequantise to bf16) with bf16
queries.  Bound per output, from the two roundings the path has: the
probabilities are rounded to bf16 (each off by at most 2^-9 of itself, and
so is their sum, which normalises them) and so is the output:
  |got - ref| <= 2 * 2^-9 * sum_j w_j |v_j| + 2^-9 |ref|, plus 1% of it for
the fp32 sums.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import dsa_oracle as O

pytestmark = pytest.mark.gpu


def _values(kv: torch.Tensor) -> torch.Tensor:
    """[B, T, 576] -> what the row format holds, float64 (oracle pack and dequantisation)."""
    x = kv.float().cpu().numpy().reshape(-1, 576)
    vals = O.dequant_latent_rows(O.pack_latent_rows(x[:, :512], x[:, 512:]))
    return torch.from_numpy(np.asarray(vals, dtype=np.float64)).reshape(*kv.shape)


def _reference(q, kv, mask, sm):
    """-> (out, bound) float64 [B, S, H, 512]; mask [B, S, T] bool."""
    keys, qd = _values(kv).to(q.device), q.to(torch.bfloat16).double()
    s = torch.matmul(qd, keys[:, None].transpose(-1, -2).contiguous()) * sm
    w = torch.softmax(s.masked_fill(~mask[:, :, None], float("-inf")), -1).nan_to_num(0.0)
    v = keys[:, None, :, :512].contiguous()
    out = torch.matmul(w, v)
    return out, 1.01 * (2 * 2.0 ** -9 * torch.matmul(w, v.abs()) + 2.0 ** -9 * out.abs())


def _causal(S, T, dev):
    return torch.arange(T, device=dev)[None, :] <= torch.arange(T - S, T, device=dev)[:, None]


def _check(got, q, kv, mask, sm=576 ** -0.5, rows=None):
    ref, bound = _reference(q, kv, mask, sm)
    bad = (got.double() - ref).abs() > bound + 1e-30
    if got.dtype == torch.float16:  # fp16 outputs: bf16 values are exact unless subnormal
        bad &= ref.abs() > 1e-4
    if rows is not None:
        bad = bad[:, rows]
    assert not bad.any(), f"{int(bad.sum())} outputs off, worst {((got.double() - ref).abs() - bound).max():.2e}"


# (B, S, H, T, dtype): row tiles of 128 (S*H = 16, 112, 128, 144, ...), key
# tiles of 32 (T = 1, 31, 32, 33), fewer keys than queries (rows without any
# key), key splits (few rows over many keys) and none (many rows)
DENSE = [
    (1, 1, 16, 1, torch.bfloat16), (2, 7, 16, 31, torch.float32), (1, 8, 16, 32, torch.float16),
    (2, 9, 16, 33, torch.bfloat16), (1, 3, 48, 65, torch.float32), (1, 40, 16, 10, torch.bfloat16),
    (1, 2, 128, 700, torch.bfloat16), (2, 5, 32, 4097, torch.float32), (1, 520, 64, 530, torch.bfloat16),
    (1, 1, 16, 20000, torch.bfloat16),
]


@pytest.mark.parametrize("B,S,H,T,dt", DENSE)
def test_dense_rows(dev, B, S, H, T, dt):
    from lagged_indexer_dsa_amd import attention_core as ac

    print(f"[prefill] dense B={B} S={S} H={H} T={T} {dt}", flush=True)
    g = torch.Generator(device=dev).manual_seed(T)
    q = torch.randn(B, S, H, 576, generator=g, device=dev).to(dt)
    kv = torch.randn(B, T, 576, generator=g, device=dev).to(dt)
    got = ac.dense_mla_core(q, kv, 512)
    assert got.shape == (B, S, H, 512) and got.dtype == dt
    _check(got, q, kv, _causal(S, T, dev)[None].expand(B, -1, -1))


def test_scores_that_rise_far_above_the_first_tile(dev):
    """Rows whose scores climb by hundreds (log2) after the first key tile are
    redone from their true maximum; rows that do not stay in the same tile."""
    from lagged_indexer_dsa_amd import attention_core as ac

    print("[prefill] rising scores", flush=True)
    g = torch.Generator(device=dev).manual_seed(5)
    S, H, T = 6, 32, 300
    q = torch.randn(1, S, H, 576, generator=g, device=dev)
    kv = torch.randn(1, T, 576, generator=g, device=dev) * 0.1
    kv[0, 200:] += q[0, 3, 7] * 2.0       # query (3, 7) meets keys along itself at the end
    kv[0, 20] -= q[0, 1, 1] * 3.0         # and (1, 1) one far below its others
    got = ac.dense_mla_core(q, kv, 512)
    _check(got, q, kv, _causal(S, T, dev)[None])


def test_non_finite_keys_reach_only_the_rows_that_attend_them(dev):
    from lagged_indexer_dsa_amd import attention_core as ac

    print("[prefill] NaN keys", flush=True)
    g = torch.Generator(device=dev).manual_seed(6)
    S, H, T = 20, 16, 90
    q = torch.randn(1, S, H, 576, generator=g, device=dev)
    kv = torch.randn(1, T, 576, generator=g, device=dev)
    bad = kv.clone()
    bad[0, T - 5, 3] = float("nan")     # seen by queries S-5 ..
    bad[0, T - 2, 400] = float("inf")   # seen by queries S-2 ..
    got, ref = ac.dense_mla_core(q, bad, 512), ac.dense_mla_core(q, kv, 512)
    assert torch.isnan(got[0, S - 5:]).all()
    assert torch.equal(got[0, :S - 5], ref[0, :S - 5])
    # selections that leave the bad keys out, streamed or gathered
    for sel in (torch.arange(T - 5, device=dev), torch.arange(0, T - 5, 7, device=dev)):
        idx = sel.expand(1, S, -1).contiguous()
        assert torch.equal(ac.sparse_mla_core(q, bad, idx, 512), ac.sparse_mla_core(q, kv, idx, 512))


@pytest.mark.parametrize("B,S,H,T,n", [(2, 3, 16, 70, 40), (1, 9, 64, 1000, 300), (2, 300, 16, 600, 256),
                                       (1, 300, 16, 3000, 128), (1, 30, 16, 33, 100)])
@pytest.mark.parametrize("itype", [torch.int64, torch.int32])
def test_selections(dev, B, S, H, T, n, itype):
    """Sets with repeats, the sentinel, negatives and keys after the query,
    through the streamed and the gathered form (the shapes lie on both
    sides of the rule)."""
    from lagged_indexer_dsa_amd import attention_core as ac
    from lagged_indexer_dsa_amd import ops

    print(f"[prefill] sparse B={B} S={S} H={H} T={T} n={n} {itype}", flush=True)
    g = torch.Generator(device=dev).manual_seed(n)
    q = torch.randn(B, S, H, 576, generator=g, device=dev).to(torch.bfloat16)
    kv = torch.randn(B, T, 576, generator=g, device=dev).to(torch.bfloat16)
    idx = torch.randint(0, T, (B, S, n), generator=g, device=dev)
    idx[:, :, 1::9] = T
    idx[:, :, 2::11] = -3
    idx[:, :, 3] = idx[:, :, 4]
    idx[0, 0] = -1                       # a row without a key
    idx = idx.to(itype)
    ok = (idx >= 0) & (idx < T)
    mask = torch.zeros(B, S, T + 1, dtype=torch.bool, device=dev)
    mask.scatter_(2, torch.where(ok, idx, torch.full_like(idx, T)).long(), True)
    mask = mask[..., :T] & _causal(S, T, dev)
    _check(ac.sparse_mla_core(q, kv, idx, 512), q, kv, mask)
    _check(ops.prefill_attention(q, kv, ops.selection_set(idx, T, True)), q, kv, mask)
    slots = ops.selection_set(idx, T, False).cpu().numpy().reshape(B, S, n)
    for b in range(B):
        for s in range(0, S, 17):
            want = np.flatnonzero(mask[b, s].cpu().numpy()) + b * T
            assert np.array_equal(slots[b, s, :want.size], want) and (slots[b, s, want.size:] == -1).all()


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16, torch.float16, torch.float64])
def test_pack_latent_rows_bytes(dev, dt):
    """The packed rows are the fixture quantiser's, byte for byte; rows past
    T are zero; an input off a 16-byte boundary and a strided one are taken."""
    from lagged_indexer_dsa_amd import formats as F
    from lagged_indexer_dsa_amd import ops

    g = torch.Generator(device=dev).manual_seed(9)
    x = torch.randn(2, 37, 576, generator=g, device=dev, dtype=torch.float64)
    x[0, 1, :128] = 0.0
    x[1, 2] *= 300.0
    x = x.to(dt)
    flat = x.reshape(-1, 576)
    want = F.pack_latent_rows(flat[:, :512], flat[:, 512:]).reshape(2, 37, 656)
    off = torch.empty(x.numel() + 1, dtype=dt, device=dev)[1:].view(x.shape)
    off.copy_(x)
    wide = torch.zeros(2, 37, 600, dtype=dt, device=dev)
    wide[..., 7:583] = x
    for src in (x, off, wide[..., 7:583]):
        got = ops.pack_latent_rows(src, 40).reshape(2, 40, 656)
        assert torch.equal(got[:, :37], want) and not got[:, 37:].any()


@pytest.mark.parametrize("S,T,n,scale", [(1000, 1000, 0, 1.0), (2999, 2999, 0, 1.0), (64, 2999, 0, 1.0),
                                         (512, 4096, 0, 1.0), (700, 700, 0, 3.0), (600, 1200, 512, 1.0),
                                         (512, 4096, 2048, 1.0)])
def test_error_is_that_of_a_softmax_about_the_maximum(dev, S, T, n, scale):
    """The error against 64 bits is no larger than that of one bf16 term a
    probability about the row's true maximum (1 exactly for the largest),
    normalised by the sum of the rounded ones, and the rounding of the output."""
    from lagged_indexer_dsa_amd import attention_core as ac

    print(f"[prefill] error S={S} T={T} n={n}", flush=True)
    H = 16
    g = torch.Generator(device=dev).manual_seed(T + S)
    q = (scale * torch.randn(1, S, H, 576, generator=g, device=dev)).to(torch.bfloat16)
    kv = torch.randn(1, T, 576, generator=g, device=dev).to(torch.bfloat16)
    mask = _causal(S, T, dev)
    if n:
        idx = torch.rand(1, S, T, generator=g, device=dev).masked_fill(~mask, -1.0).topk(n, -1).indices
        got = ac.sparse_mla_core(q, kv, idx, 512)
        mask = mask & torch.zeros(1, S, T, dtype=torch.bool, device=dev).scatter_(2, idx, True)[0]
    else:
        got = ac.dense_mla_core(q, kv, 512)
    keys = _values(kv).to(dev)[0]
    err, about_max, size = 0.0, 0.0, 0.0
    for s0 in range(0, S, 128):
        s = torch.matmul(q[0, s0:s0 + 128].double(), keys.t().contiguous()) * 576 ** -0.5
        s = s.masked_fill(~mask[s0:s0 + 128, None], float("-inf"))
        p = torch.exp(s - s.amax(-1, keepdim=True))
        ref = torch.matmul(p, keys[:, :512].contiguous()) / p.sum(-1, keepdim=True)
        p = p.to(torch.bfloat16).double()
        one = (torch.matmul(p, keys[:, :512].contiguous()) / p.sum(-1, keepdim=True)).to(torch.bfloat16).double()
        err += float((got[0, s0:s0 + 128].double() - ref).square().sum())
        about_max += float((one - ref).square().sum())
        size += float(ref.square().sum())
    print(f"[prefill] error {(err / size) ** 0.5:.6f}, about the maximum {(about_max / size) ** 0.5:.6f}", flush=True)
    assert err <= about_max


@pytest.mark.parametrize("T", [524288, 524287, 523264])
@pytest.mark.parametrize("itype", [torch.int64, torch.int32])
def test_selection_set_at_the_longest_context(dev, T, itype):
    """The bitmap fills 64 KB of LDS: first, last and middle positions, and
    those the row does not see."""
    from lagged_indexer_dsa_amd import ops

    S = 3
    idx = torch.tensor([0, T - 1, T - 2, T - 3, T - 4, T // 2, T, -1, 31, 32, T - 1], device=dev).to(itype)
    idx = idx.expand(1, S, -1).contiguous()
    bits = ops.selection_set(idx, T, True).cpu().numpy().view(np.uint32).reshape(S, -1)
    slots = ops.selection_set(idx, T, False).cpu().numpy()
    for s in range(S):
        want = sorted(v for v in {0, T - 1, T - 2, T - 3, T - 4, T // 2, 31, 32} if v < T - S + s + 1)
        assert np.flatnonzero(np.unpackbits(bits[s].view(np.uint8), bitorder="little")).tolist() == want
        assert slots[s].tolist() == want + [-1] * (idx.shape[2] - len(want))


@pytest.mark.parametrize("T", [575, 576, 577, 900])
@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("rising", [False, True])
def test_second_terms_by_rule_and_by_need(dev, T, masked, rising):
    """130 row tiles, one split: on both sides of the 512 keys from which the
    probabilities' second terms are taken by need; also with rows that are
    redone from their true maximum."""
    from lagged_indexer_dsa_amd import ops

    print(f"[prefill] second terms T={T} masked={masked} rising={rising}", flush=True)
    S, H = 130, 128
    g = torch.Generator(device=dev).manual_seed(T)
    q = torch.randn(1, S, H, 576, generator=g, device=dev).to(torch.bfloat16)
    kv = torch.randn(1, T, 576, generator=g, device=dev).to(torch.bfloat16)
    if rising:
        kv *= 0.1
        kv[0, T - 40:T - 30] += q[0, S - 9, 7] * 2.0
        kv[0, 300] += q[0, 5, 100]
    mask, bits = _causal(S, T, dev), None
    if masked:
        idx = torch.randint(0, T, (1, S, 700), generator=g, device=dev)
        bits = ops.selection_set(idx, T, True)
        mask = mask & torch.zeros(1, S, T, dtype=torch.bool, device=dev).scatter_(2, idx, True)[0]
    _check(ops.prefill_attention(q, kv, bits), q, kv, mask[None])
