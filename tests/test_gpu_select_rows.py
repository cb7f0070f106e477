"""GPU: the sorted select of one workgroup a row (ops.select_rows, ops.topk
with sorted=True, attention_core.select_topk) against the oracle, bit-exact:
register sizes and their edges (2048, 4096, 8192, 16384 scores and one more
or less), the re-read form of longer rows, top-k from 1 to 4096 (above,
equal to and below the row), and the score patterns of each branch: spread
scores (the bins), masked tails, NaN and infinities, ties, one outlier that
leaves every other score in one bin, and all equal (the radix and bitonic
form)."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import dsa_oracle as O

pytestmark = pytest.mark.gpu


def _rows(kind: str, n_rows: int, n: int, seed: int) -> np.ndarray:
    rng = np.random.default_rng(seed)
    x = rng.standard_normal((n_rows, n)).astype(np.float32)
    if kind == "masked":
        for r in range(n_rows):
            x[r, (r * n) // n_rows + 1:] = -np.inf
    elif kind == "special":
        x[:, ::5] = -np.inf
        x[:, 1::97] = np.nan
        x[:, 2::89] = np.inf
        x[:, 3::7] = 0.0
        x[:, 4::7] = -0.0
    elif kind == "ties":
        x = np.round(x * 4) / 4
    elif kind == "outlier":
        x[:, n // 2] = 3e38
        x[:, n // 3] = -3e38 if n_rows > 1 else x[:, n // 3]
    elif kind == "equal":
        x[:] = 1.5
        x[0, :] = -np.inf
    elif kind == "exponents":
        x = (np.sign(x) * np.exp2(rng.uniform(-140, 120, x.shape))).astype(np.float32)
    return x


@pytest.mark.parametrize("kind", ["normal", "masked", "special", "ties", "outlier", "equal", "exponents"])
@pytest.mark.parametrize("n,k", [(1, 3), (500, 64), (2048, 2048), (2049, 300), (4096, 7), (8191, 2048), (8193, 4096),
                                 (16384, 2048)])
def test_rows(dev, kind, n, k):
    from lagged_indexer_dsa_amd import ops

    x = _rows(kind, 5, n, n + k)
    lens = np.array([n, max(0, n - 1), n // 2, 0, n], dtype=np.int32)
    got = ops.topk(torch.from_numpy(x).to(dev), torch.from_numpy(lens).to(dev), k, sorted=True, pad_value=-7)
    ref = O.topk_select(x, lens, k, sorted_=True, pad=-7)
    assert np.array_equal(got.cpu().numpy(), ref)
    whole = ops.select_rows(torch.from_numpy(x).to(dev), k, n)
    ref = O.topk_select(x, np.full(5, n, dtype=np.int32), k, sorted_=True, pad=n)
    assert whole.dtype == torch.int64 and np.array_equal(whole.cpu().numpy(), ref)


@pytest.mark.parametrize("kind", ["normal", "masked", "special", "ties", "outlier"])
@pytest.mark.parametrize("rows,n", [(3, 16385), (2, 20001), (24, 131073)])
def test_longer_rows(dev, kind, rows, n):
    from lagged_indexer_dsa_amd import ops

    k = 2048
    x = _rows(kind, 2, n, 3)
    got = ops.select_rows(torch.from_numpy(x).to(dev).repeat(rows, 1)[:rows], k, n).cpu().numpy()
    ref = O.topk_select(x, np.full(2, n, dtype=np.int32), k, sorted_=True, pad=n)
    assert all(np.array_equal(got[r], ref[r % 2]) for r in range(rows))


def test_few_very_long_rows_take_the_slice_kernels(dev):
    from lagged_indexer_dsa_amd import attention_core as ac
    from lagged_indexer_dsa_amd import ops

    n = 131073
    x = _rows("normal", 2, n, 4)
    assert ops.select_rows(torch.from_numpy(x).to(dev), 2048, n) is None
    ref = O.topk_select(x, np.full(2, n, dtype=np.int32), 2048, sorted_=True, pad=n)
    assert np.array_equal(ac.select_topk(torch.from_numpy(x).to(dev)[None], 2048)[0].cpu().numpy(), ref)


@pytest.mark.parametrize("n,k,finite", [(2048, 64, 2), (2049, 300, 100), (8192, 2048, 128), (8193, 2048, 129),
                                        (16384, 2048, 16384), (20000, 512, 120), (20000, 512, 20000)])
def test_rows_whose_range_overflows(dev, n, k, finite):
    """Finite scores further apart than the largest float: one bin, of few
    members (ranked) and of many (the radix form)."""
    from lagged_indexer_dsa_amd import ops

    rng = np.random.default_rng(n + finite)
    x = np.full((3, n), -np.inf, dtype=np.float32)
    for r in range(3):
        p = rng.permutation(n)[:finite]
        x[r, p] = rng.uniform(-3e38, 3e38, finite)
        x[r, p[0]], x[r, p[1]] = 3.4e38, -3.4e38
    got = ops.select_rows(torch.from_numpy(x).to(dev), k, n)
    ref = O.topk_select(x, np.full(3, n, dtype=np.int32), k, sorted_=True, pad=n)
    assert np.array_equal(got.cpu().numpy(), ref)
