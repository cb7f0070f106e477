"""GPU: the cooperative select on rows of a few times top-k, where the
workgroups' lists hold every key and the union's threshold bin is split
again (once, twice, down to one value with ties), in position order against
the oracle, bit-exact; one row and ragged rows, with and without a page
table, and through the decode layer's fused launch."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import dsa_oracle as O

pytestmark = pytest.mark.gpu


def _scores(kind: str, rows: int, n: int, seed: int) -> np.ndarray:
    rng = np.random.default_rng(seed)
    x = rng.standard_normal((rows, n)).astype(np.float32)
    if kind == "rounded":        # bins of many equal scores on both sides of the threshold
        x = np.round(x * 16) / 16
    elif kind == "close":        # scores that differ in their last ten bits
        x = (1.0 + rng.integers(0, 1024, (rows, n)) * 2.0 ** -23).astype(np.float32)
    elif kind == "close_cluster":  # a crowded cluster at the threshold among spread scores
        x[:, ::2] = (0.01 + rng.integers(0, 50, x[:, ::2].shape) * 1e-9).astype(np.float32)
    elif kind == "tiny":         # subnormal to huge
        x = (np.sign(x) * np.exp2(rng.uniform(-148, 100, x.shape))).astype(np.float32)
    elif kind == "special":
        x[:, ::3] = -np.inf
        x[:, 1::50] = np.nan
        x[:, 2::60] = np.inf
        x[:, 4::5] = -0.0
        x[:, 5::10] = 0.0
    return x


@pytest.mark.parametrize("kind", ["normal", "rounded", "close", "close_cluster", "tiny", "special"])
@pytest.mark.parametrize("lens,k", [([2049], 2048), ([2600], 2048), ([4133], 2048), ([6000], 2048), ([8192], 512),
                                    ([1030], 1024), ([4133, 2100, 70, 6000], 2048), ([3000] * 9, 1024)])
def test_short_rows(dev, kind, lens, k):
    from lagged_indexer_dsa_amd import _lib, ops

    _lib.sync_timeouts(reset=True)
    slab = max(lens) + 3
    x = _scores(kind, len(lens), slab, slab + k)
    seq = torch.tensor(lens, dtype=torch.int32, device=dev)
    pt = np.random.default_rng(1).permutation(len(lens) * (slab // 64 + 1)).astype(np.int32).reshape(len(lens), -1)
    scratch = ops.topk_scratch(len(lens), slab, dev)
    for table in (None, pt):
        for _ in range(2):  # the scratch re-arms itself
            got = ops.topk(torch.from_numpy(x).to(dev), seq, k, scratch=scratch,
                           page_table=None if table is None else torch.from_numpy(table).to(dev))
            assert np.array_equal(got.cpu().numpy(), O.topk_select(x, np.array(lens), k, page_table=table))
    assert _lib.sync_timeouts() == 0


@pytest.mark.parametrize("lens", [[2049], [3000], [4133], [7777], [4133, 2500]])
def test_short_layers(dev, lens):
    from lagged_indexer_dsa_amd import _lib
    from lagged_indexer_dsa_amd import synthetic as S

    _lib.sync_timeouts(reset=True)
    pt, num_pages = S.make_page_table(lens, seed=61, device=dev)
    L = S.make_decode_layer(lens, seed=62, device=dev, page_table=pt, num_pages=num_pages)
    att = S.random_selection(lens, 2048, pt, seed=63, device=dev)
    for attend in (att, None):
        L.next_idx.fill_(-7)
        L.run(attend_idx=attend)
        torch.cuda.synchronize()
        ref = O.topk_select(L.scores.cpu().numpy(), np.array(lens), L.topk, page_table=pt.cpu().numpy())
        assert np.array_equal(L.next_idx.cpu().numpy(), ref)
    assert _lib.sync_timeouts() == 0
