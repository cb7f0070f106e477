"""GPU: dense MLA decode of 2 to 64 rows, whose splits follow the rows' lengths.

Reference: softmax attention in float64 over the pool rows' values (oracle:
dequantised to bf16).  Bound per output: the probabilities are rounded to bf16
(off by at most 2^-8 of themselves; their sum, which normalises them, is not)
and so is the output: |got - ref| <= 2^-8 (sum_j w_j |v_j| + |ref|), plus 1%
for the fp32 sums.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import dsa_oracle as O

pytestmark = pytest.mark.gpu
SM = 576 ** -0.5

# (lens, heads, table entries beyond the longest row, nsplit): rows without a
# key beside long ones, one longer than all others together, a split of its
# last key, no key at all, equal rows, tables far wider than the rows, 64 and
# 65 rows, given split counts
CASES = [
    ([0, 5000], 16, 0, 0), ([1, 63, 64, 65, 3000], 64, 3, 0), ([0, 0, 0], 32, 4, 0), ([9000, 1], 128, 0, 0),
    ([700] * 4, 16, 0, 0), ([130, 4097, 257], 48, 400, 0), ([5, 900, 0, 129] * 16, 16, 0, 0),
    ([5, 900, 0, 129] * 16 + [700], 16, 0, 0), ([2000, 31, 640], 16, 2, 7), ([300, 8191], 16, 0, 128),
]


@pytest.mark.parametrize("lens,H,extra,nsplit", CASES)
def test_dense_rows_by_length(dev, lens, H, extra, nsplit):
    from lagged_indexer_dsa_amd import _lib, ops

    B, pt, pages = len(lens), max(1, -(-max(lens) // 64)) + extra, 160
    rng = np.random.default_rng(B + H)
    x = rng.standard_normal((64 * pages, 576)).astype(np.float32)
    packed = O.pack_latent_rows(x[:, :512], x[:, 512:])
    vals = torch.from_numpy(np.asarray(O.dequant_latent_rows(packed), dtype=np.float64)).to(dev)
    pool = torch.from_numpy(np.ascontiguousarray(packed).view(np.uint8).reshape(-1, 656)).to(dev)
    table = torch.from_numpy(rng.integers(0, pages, (B, pt)).astype(np.int32)).to(dev)
    q = torch.randn(B, H, 576, device=dev, generator=torch.Generator(dev).manual_seed(7)).to(torch.bfloat16)
    seq = torch.tensor(lens, dtype=torch.int32, device=dev)
    _lib.sync_timeouts(reset=True)
    ws = ops.sparse_mla_workspace(B, H, nsplit, dev)
    outs = [ops.dense_mla_decode(q, pool, table, seq, SM, nsplit=nsplit, workspace=ws) for _ in range(3)]
    torch.cuda.synchronize()
    assert _lib.sync_timeouts() == 0
    assert all(torch.equal(o.view(torch.int16), outs[0].view(torch.int16)) for o in outs[1:])
    for b, n in enumerate(lens):
        if not n:
            assert not outs[0][b].any()
            continue
        pos = torch.arange(n, device=dev)
        k = vals[table[b].long()[pos // 64] * 64 + pos % 64]
        w = torch.softmax(q[b].double() @ k.t().contiguous() * SM, -1)
        ref = w @ k[:, :512].contiguous()
        bound = 1.01 * 2.0 ** -8 * (w @ k[:, :512].abs() + ref.abs())
        bad = (outs[0][b].double() - ref).abs() > bound + 1e-30
        assert not bad.any(), f"row {b}: {int(bad.sum())} off"


@pytest.mark.parametrize("lens,H,extra", [([2000], 16, 2016), ([2000], 64, 2016), ([1], 16, 2047), ([0], 16, 2048),
                                          ([2000, 2000], 16, 2016), ([65, 1, 4000], 64, 1985)])
def test_rows_in_a_table_of_131072_keys(dev, lens, H, extra):
    """One row keeps the even division of the table, whose later splits hold
    no key; several share the splits by length."""
    test_dense_rows_by_length(dev, lens, H, extra, 0)
