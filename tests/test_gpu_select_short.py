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


# Rows whose K-th key is NaN (ranked above +inf): nothing finite is selected,
# the row is all pads.  The threshold bin is then the topmost one, next to
# 2^32, and the lists' zero padding must not count in it.
@pytest.mark.parametrize("nans", ["many", "k", "k-1"])
@pytest.mark.parametrize("lens,k", [([2600], 2048), ([3000], 2048), ([4133], 2048), ([8192], 512), ([1030], 1024),
                                    ([20000], 2048), ([131072], 2048), ([4133, 2100, 70, 6000], 2048)])
def test_rows_of_nans(dev, lens, k, nans):
    from lagged_indexer_dsa_amd import _lib, ops

    _lib.sync_timeouts(reset=True)
    rng = np.random.default_rng(k + sum(lens))
    x = rng.standard_normal((len(lens), max(lens))).astype(np.float32)
    for r, n in enumerate(lens):
        count = {"many": k + (n - k) // 3, "k": k, "k-1": k - 1}[nans] if n > k else n // 2
        x[r, rng.permutation(n)[:count]] = np.nan
    seq = torch.tensor(lens, dtype=torch.int32, device=dev)
    pt = rng.permutation(len(lens) * (max(lens) // 64 + 1)).astype(np.int32).reshape(len(lens), -1)
    for table in (None, pt):
        got = ops.topk(torch.from_numpy(x).to(dev), seq, k,
                       page_table=None if table is None else torch.from_numpy(table).to(dev))
        assert np.array_equal(got.cpu().numpy(), O.topk_select(x, np.array(lens), k, page_table=table))
    assert _lib.sync_timeouts() == 0


@pytest.mark.parametrize("lens,k", [([4133], 2048), ([8192], 512), ([3000, 6000], 1024), ([4133] * 9, 2048)])
def test_layers_of_nan_scores(dev, lens, k):
    from lagged_indexer_dsa_amd import _lib
    from lagged_indexer_dsa_amd import synthetic as S

    _lib.sync_timeouts(reset=True)
    pt, num_pages = S.make_page_table(lens, seed=71, device=dev)
    L = S.make_decode_layer(lens, seed=72, device=dev, page_table=pt, num_pages=num_pages, topk=k)
    scales = L.index_k[:, 8192:].view(torch.float32)  # a NaN key scale: a NaN score
    g = torch.Generator().manual_seed(73)
    for b, n in enumerate(lens):
        p = torch.randperm(n, generator=g)[:k + (n - k) // 2].to(dev)
        scales[pt[b].long()[p // 64], p % 64] = float("nan")
    att = S.random_selection(lens, k, pt, seed=74, device=dev)
    for attend in (att, None):  # the fused launch; scan + select, then an attention over no key
        L.next_idx.fill_(-7)
        L.run(attend_idx=attend)
        torch.cuda.synchronize()
        assert bool((L.next_idx == -1).all())
        if attend is None:
            assert bool((L.out == 0).all())
    assert _lib.sync_timeouts() == 0


# A threshold bin of more than a wave's equal scores: the split ends at one
# key value, whose entries are taken lowest position first.
@pytest.mark.parametrize("ties", [63, 64, 65, 130, 1024, 1500])
@pytest.mark.parametrize("lens,k", [([2600], 2048), ([4133], 1024), ([6000], 2048), ([20000], 2048), ([131072], 2048),
                                    ([4133, 2600, 3000], 2048)])
def test_ties_at_the_threshold(dev, lens, k, ties):
    from lagged_indexer_dsa_amd import _lib, ops

    _lib.sync_timeouts(reset=True)
    rng = np.random.default_rng(ties + k + sum(lens))
    x = rng.standard_normal((len(lens), max(lens))).astype(np.float32)
    for r, n in enumerate(lens):
        # k - ties // 3 scores above the tied ones, the others below
        order = np.argsort(-x[r, :n], kind="stable")
        top = k - ties // 3
        tied = rng.permutation(order[top:])[:ties]
        v = x[r, order[top]]
        x[r, order[top:]] = np.minimum(x[r, order[top:]], np.nextafter(v, np.float32(-np.inf)))
        x[r, tied] = v
    seq = torch.tensor(lens, dtype=torch.int32, device=dev)
    pt = rng.permutation(len(lens) * (max(lens) // 64 + 1)).astype(np.int32).reshape(len(lens), -1)
    for table in (None, pt):
        got = ops.topk(torch.from_numpy(x).to(dev), seq, k,
                       page_table=None if table is None else torch.from_numpy(table).to(dev))
        assert np.array_equal(got.cpu().numpy(), O.topk_select(x, np.array(lens), k, page_table=table))
    assert _lib.sync_timeouts() == 0
