"""GPU: indexer_logits' kernel at the edges of its key tiles (64 keys a wave,
512 a workgroup) and query stages (4 rows), for each head count and element
type, against float64 over the oracle-quantised operands, and against the
decode scan over the same operands, bit for bit (the same products in the
same order).

Bound against float64: 1e-4 of the largest |logit| (the matrix unit's sums of
128 products; the same bound as the decode scan's tests)."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import dsa_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,S,H,T,dt", [
    (1, 1, 16, 1, torch.float32), (2, 3, 32, 63, torch.bfloat16), (1, 4, 48, 64, torch.float16),
    (2, 5, 64, 65, torch.float32), (1, 9, 64, 512, torch.bfloat16), (2, 8, 16, 513, torch.bfloat16),
    (1, 700, 64, 1500, torch.bfloat16), (1, 2, 64, 40001, torch.float32),
])
def test_against_quantised_operands(dev, B, S, H, T, dt):
    from lagged_indexer_dsa_amd import attention_core as ac
    from lagged_indexer_dsa_amd import ops

    print(f"[logits] B={B} S={S} H={H} T={T} {dt}", flush=True)
    g = torch.Generator(device=dev).manual_seed(T + S)
    q = torch.randn(B, S, H, 128, generator=g, device=dev).to(dt)
    k = torch.randn(B, T, 128, generator=g, device=dev).to(dt)
    w = (torch.randn(B, S, H, generator=g, device=dev) * H ** -0.5).to(dt)
    k[0, T // 2] = 0.0
    got = ac.indexer_logits(q, k, w)
    assert got.shape == (B, S, T) and got.dtype == torch.float32
    qc, qs = O.quantize_rowwise(q.float().cpu().numpy())
    kc, ks = O.quantize_rowwise(k.float().cpu().numpy())
    wf = (w.float().cpu().numpy() * qs).astype(np.float32)
    qd, kd = (torch.from_numpy(O.e4m3_decode(c)).double().to(dev) for c in (qc, kc))
    wd, sd = torch.from_numpy(wf).double().to(dev), torch.from_numpy(ks).double().to(dev)
    for b in range(B):
        ref = sum(wd[b, :, h, None] * torch.relu(qd[b, :, h] @ kd[b].T) for h in range(H)) * sd[b]
        assert (got[b].double() - ref).abs().max() <= 1e-4 * ref.abs().max()
        # the decode scan over the same codes (identity paging)
        npg = (T + 63) // 64
        pages = torch.from_numpy(O.pack_index_pages(kc[b], ks[b], np.arange(npg), npg)).to(dev)
        rows = list(range(S))[:: max(1, S // 8)]
        scan = ops.indexer_scan(torch.from_numpy(qc[b, rows]).to(dev), torch.from_numpy(wf[b, rows]).to(dev), pages,
                                torch.arange(npg, dtype=torch.int32, device=dev).repeat(len(rows), 1),
                                torch.full((len(rows),), T, dtype=torch.int32, device=dev), npg * 64)
        assert torch.equal(scan[:, :T].view(torch.int32), got[b, rows].view(torch.int32))


def test_strided_misaligned_and_other_types(dev):
    from lagged_indexer_dsa_amd import attention_core as ac

    g = torch.Generator(device=dev).manual_seed(3)
    q, k, w = (torch.randn(*s, generator=g, device=dev) for s in ((1, 3, 32, 128), (1, 100, 128), (1, 3, 32)))
    want = ac.indexer_logits(q, k, w)
    off = torch.empty(k.numel() + 1, device=dev)[1:].view(k.shape).copy_(k)
    wide = torch.zeros(1, 3, 32, 130, device=dev)
    wide[..., 1:129] = q
    assert torch.equal(ac.indexer_logits(wide[..., 1:129], off, w), want)
    assert torch.equal(ac.indexer_logits(q.double(), k.double(), w.double()), want)
    assert torch.equal(ac.indexer_logits(q, k, w.t() if w.dim() == 2 else w.transpose(1, 2).contiguous().transpose(1, 2)),
                       want)


def test_non_finite_rows(dev):
    """A NaN or infinity in a key or a query row makes that row's or that
    key's scores NaN and no other's."""
    from lagged_indexer_dsa_amd import attention_core as ac

    g = torch.Generator(device=dev).manual_seed(4)
    q, k, w = (torch.randn(*s, generator=g, device=dev) for s in ((1, 6, 16, 128), (1, 70, 128), (1, 6, 16)))
    want = ac.indexer_logits(q, k, w)
    kn, qn = k.clone(), q.clone()
    kn[0, 7, 5] = float("nan")
    kn[0, 66, 0] = float("inf")
    qn[0, 2, 3, 9] = float("nan")
    got = ac.indexer_logits(q, kn, w)
    keep = [i for i in range(70) if i not in (7, 66)]
    assert torch.isnan(got[0, :, [7, 66]]).all() and torch.equal(got[..., keep], want[..., keep])
    got = ac.indexer_logits(qn, k, w)
    assert torch.isnan(got[0, 2]).all() and torch.equal(got[0, [0, 1, 3, 4, 5]], want[0, [0, 1, 3, 4, 5]])
