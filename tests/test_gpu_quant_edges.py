"""GPU: the operand-preparation kernels off their 16-byte boundaries, at row
counts around a workgroup's, and on quotients that sit on or next to an e4m3
rounding boundary (scales of every significand), bit-exact against the
oracle's quantiser (numpy's IEEE division)."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import dsa_oracle as O

pytestmark = pytest.mark.gpu


def _rows(n: int, seed: int) -> np.ndarray:
    """Rows whose amax spans all bf16 significands and many exponents, the
    rest at or beside midpoints of the code grid times that row's scale."""
    rng = np.random.default_rng(seed)
    amax = O.bf16_rn((rng.uniform(1, 2, n) * np.exp2(rng.integers(-30, 30, n))).astype(np.float32))
    pos = O.e4m3_decode(np.arange(0x7F, dtype=np.uint8))
    mid = ((pos[:-1] + pos[1:]) / 2).astype(np.float32)
    x = mid[rng.integers(0, mid.size, (n, 128))] * (amax[:, None] / 448.0) * rng.choice([-1, 1], (n, 128))
    x[:, 0] = amax
    x[:, 1] = -0.0
    x[:, 2] = 1e-38
    return O.bf16_rn(x.astype(np.float32))


def _dev(x: np.ndarray, dev, shift: int) -> torch.Tensor:
    """bf16 tensor of x's values, `shift` elements past a 16-byte boundary."""
    t = torch.from_numpy(O.bf16_bits(x).view(np.int16)).view(torch.bfloat16)
    out = torch.empty(x.size + 8, dtype=torch.bfloat16, device=dev)[shift:shift + x.size].view(x.shape)
    return out.copy_(t)


@pytest.mark.parametrize("shift", [0, 1, 4])
@pytest.mark.parametrize("B,H", [(1, 1), (1, 15), (1, 17), (64, 64)])
def test_query(dev, shift, B, H):
    from lagged_indexer_dsa_amd import ops

    x = _rows(B * H, B + H).reshape(B, H, 128)
    w = np.random.default_rng(1).standard_normal((B, H)).astype(np.float32)
    out_q = torch.empty(B * H * 128 + 8, dtype=torch.uint8, device=dev)[shift:shift + B * H * 128].view(B, H, 128)
    codes, wf = ops.quantize_index_query(_dev(x, dev, shift), torch.from_numpy(w).to(dev), out_q=out_q)
    ref_c, ref_s = O.quantize_rowwise(x)
    assert np.array_equal(codes.cpu().numpy(), ref_c)
    assert np.array_equal(wf.cpu().numpy(), (w * ref_s).astype(np.float32))


@pytest.mark.parametrize("shift", [0, 2])
def test_keys_and_latent_rows(dev, shift):
    from lagged_indexer_dsa_amd import ops

    n = 131
    keys, lat = _rows(n, 7), np.concatenate([_rows(n, 8 + g) for g in range(4)] + [_rows(n, 12)[:, :64]], axis=1)
    pt = torch.tensor([[2, 0, 1]], dtype=torch.int32, device=dev)
    pos = torch.arange(n, dtype=torch.int32, device=dev)
    pages = torch.zeros(3 * 8448 + 8, dtype=torch.uint8, device=dev)[2 * shift:2 * shift + 3 * 8448].view(3, 8448)
    ops.append_index_keys(pages, pt, torch.zeros_like(pos), pos, _dev(keys, dev, shift))
    codes, scale = O.quantize_rowwise(keys)
    want = O.pack_index_pages(codes, scale, np.array([2, 0, 1]), 3)
    assert np.array_equal(pages.cpu().numpy(), want)
    pool = torch.zeros(n * 656 + 16, dtype=torch.uint8, device=dev)[4 * shift:4 * shift + n * 656].view(n, 656)
    ops.append_latent_rows(pool, pos, _dev(lat, dev, shift))
    assert np.array_equal(pool.cpu().numpy(), O.pack_latent_rows(lat[:, :512], lat[:, 512:]))
