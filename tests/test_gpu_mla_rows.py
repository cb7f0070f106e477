"""GPU: MLA decode of many unsplit rows (one workgroup a row and head group:
sparse_mla_decode and dense_mla_decode from 129 such groups on), at the edges
of its 16-key steps and 128-key rounds.

Reference: softmax attention in float64 over the pool rows' values (oracle:
dequantised to bf16).  Bound per output: the probabilities enter in two bf16
terms (off by at most 2^-17 of themselves) from fp32 scores, each off by at
most 2^-24 a term over its 576 terms (and as much again for the scale and the
exponential), and the output is rounded to bf16:
  |got - ref| <= (2^-17 + 2 * 2^-24 * 576 * max_j sum_d |q_d k_jd| sm)
                 * 2 * sum_j w_j |v_j| + 2^-8 |ref|, plus 1% for the sums.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import dsa_oracle as O

pytestmark = pytest.mark.gpu
SM = 576 ** -0.5


def _pool(rows, dev, seed, scale=1.0):
    rng = np.random.default_rng(seed)
    x = rng.standard_normal((rows, 576)).astype(np.float32) * scale
    packed = O.pack_latent_rows(x[:, :512], x[:, 512:])
    vals = torch.from_numpy(np.asarray(O.dequant_latent_rows(packed), dtype=np.float64)).to(dev)
    return torch.from_numpy(np.ascontiguousarray(packed).view(np.uint8).reshape(rows, 656)).to(dev), vals


def _check(got, q, vals, slots):
    """slots [B, n] int64, -1: no key."""
    for b in range(q.shape[0]):
        k = vals[slots[b][slots[b] >= 0]]
        if not len(k):
            assert not got[b].any()
            continue
        qd = q[b].double()
        w = torch.softmax(qd @ k.t().contiguous() * SM, -1)
        mag = (qd.abs() @ k.abs().t().contiguous()).amax(-1, keepdim=True) * SM
        ref = w @ k[:, :512].contiguous()
        bound = 1.01 * ((2.0 ** -17 + 2 * 2.0 ** -24 * 576 * mag) * 2 * (w @ k[:, :512].abs()) + 2.0 ** -8 * ref.abs())
        bad = (got[b].double() - ref).abs() > bound + 1e-30
        assert not bad.any(), f"row {b}: {int(bad.sum())} off"


@pytest.mark.parametrize("n", [1, 15, 16, 17, 127, 128, 129, 145, 300])
@pytest.mark.parametrize("B,H", [(129, 16), (33, 64)])
def test_sparse_rows(dev, B, H, n):
    from lagged_indexer_dsa_amd import _lib, ops

    R = 411
    pool, vals = _pool(R, dev, n)
    q = torch.randn(B, H, 576, device=dev, generator=torch.Generator(dev).manual_seed(n)).to(torch.bfloat16)
    g = torch.Generator().manual_seed(n)
    idx = torch.stack([torch.randperm(R, generator=g)[:n] for _ in range(B)]).int()
    idx[1, : n // 2] = -1            # masked entries, before and after the others
    idx[2, n // 2:] = R + 5
    idx[3] = -7                      # no key at all
    idx[4, ::2] = 2 ** 31 - 1
    idx = idx.to(dev)
    out = ops.sparse_mla_decode(q, pool, idx, SM, nsplit=1)
    _check(out, q, vals, torch.where((idx >= 0) & (idx < R), idx, -1).long())
    same = torch.empty_like(out)
    _lib.call("dsa_sparse_mla_decode_noalloc", q.data_ptr(), pool.data_ptr(), R, idx.data_ptr(), same.data_ptr(), B, H,
              n, 1, SM, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert torch.equal(same.view(torch.int16), out.view(torch.int16))


def test_rising_scores_start_over(dev):
    """Scores that rise by far more than 2^32 after a wave's first step."""
    from lagged_indexer_dsa_amd import ops

    R, B, H, n = 1024, 132, 16, 512
    pool, vals = _pool(R, dev, 3, scale=6.0)
    q = (torch.randn(B, H, 576, device=dev, generator=torch.Generator(dev).manual_seed(5)) * 6).to(torch.bfloat16)
    score = torch.matmul(q[:, 0].double(), vals.t().contiguous())
    idx = score.argsort(-1)[:, ::2].int().contiguous()  # head 0's scores ascend
    spread = score.amax(-1) - score.amin(-1)
    assert (spread * SM > 64).all()
    _check(ops.sparse_mla_decode(q, pool, idx, SM, nsplit=1), q, vals, idx.long())


def test_dense_rows(dev):
    from lagged_indexer_dsa_amd import ops

    B, H, pt = 130, 16, 5
    lens = ([0, 1, 15, 16, 17, 63, 64, 65, 127, 128, 129, 255, 257, 319, 320, 400] * 9)[:B]
    pool, vals = _pool(64 * 40, dev, 11)
    g = torch.Generator().manual_seed(2)
    table = torch.randint(0, 40, (B, pt), generator=g, dtype=torch.int32)
    table[7, 0] = -1                 # a page that is not there
    table = table.to(dev)
    q = torch.randn(B, H, 576, device=dev, generator=torch.Generator(dev).manual_seed(8)).to(torch.bfloat16)
    out = ops.dense_mla_decode(q, pool, table, torch.tensor(lens, dtype=torch.int32, device=dev), SM, nsplit=1)
    pos = torch.arange(64 * pt, device=dev)
    slots = table.long()[:, pos // 64] * 64 + pos % 64
    ok = (pos[None] < torch.tensor(lens, device=dev)[:, None]) & (slots >= 0)
    _check(out, q, vals, torch.where(ok, slots, -1))
