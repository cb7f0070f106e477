"""GPU: the prefill ops (ops.select_rows, prefill_logits, pack_latent_rows,
selection_set, prefill_attention) refuse tensors of other shapes, types or
devices before anything is launched."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


def _make(dev, B=2, S=3, H=16, T=40, n=8):
    return dict(q=torch.zeros(B, S, H, 576, dtype=torch.bfloat16, device=dev),
                kv=torch.zeros(B, T, 576, dtype=torch.bfloat16, device=dev),
                iq=torch.zeros(B, S, H, 128, device=dev), ik=torch.zeros(B, T, 128, device=dev),
                iw=torch.zeros(B, S, H, device=dev), idx=torch.zeros(B, S, n, dtype=torch.int64, device=dev),
                scores=torch.zeros(B * S, T, device=dev))


@pytest.mark.parametrize("name,args,message", [
    ("select_rows", lambda a: (a["scores"].to(torch.bfloat16), 4, 40), "float32"),
    ("select_rows", lambda a: (a["scores"].double(), 4, 40), "float32"),
    ("select_rows", lambda a: (a["scores"][None], 4, 40), "slab"),
    ("select_rows", lambda a: (a["scores"].cpu(), 4, 40), "GPU"),
    ("prefill_logits", lambda a: (a["iq"][0], a["ik"], a["iw"]), "q must"),
    ("prefill_logits", lambda a: (a["iq"][..., :64], a["ik"], a["iw"]), "q must"),
    ("prefill_logits", lambda a: (a["iq"], a["ik"][:1], a["iw"]), "k must"),
    ("prefill_logits", lambda a: (a["iq"], a["ik"][..., :64], a["iw"]), "k must"),
    ("prefill_logits", lambda a: (a["iq"], a["ik"], a["iw"][:, :2]), "w must"),
    ("prefill_logits", lambda a: (a["iq"], a["ik"], a["iw"][..., None]), "w must"),
    ("prefill_logits", lambda a: (a["iq"], a["ik"], a["iw"].cpu()), "GPU"),
    ("pack_latent_rows", lambda a: (a["kv"][0], 40), "kv must"),
    ("pack_latent_rows", lambda a: (a["kv"][..., :512], 40), "kv must"),
    ("pack_latent_rows", lambda a: (a["kv"], 39), "row_stride"),
    ("pack_latent_rows", lambda a: (a["kv"], -1), "row_stride"),
    ("selection_set", lambda a: (a["idx"].float(), 40, True), "int32 or int64"),
    ("selection_set", lambda a: (a["idx"].to(torch.int16), 40, False), "int32 or int64"),
    ("selection_set", lambda a: (a["idx"][0], 40, True), "idx must"),
    ("selection_set", lambda a: (a["idx"].cpu(), 40, True), "GPU"),
    ("prefill_attention", lambda a: (a["q"].float(), a["kv"]), "bfloat16"),
    ("prefill_attention", lambda a: (a["q"][0], a["kv"]), "q must"),
    ("prefill_attention", lambda a: (a["q"][..., :512].contiguous(), a["kv"]), "q must"),
    ("prefill_attention", lambda a: (a["q"], a["kv"][:1]), "requests"),
    ("prefill_attention", lambda a: (a["q"], a["kv"][..., :512]), "kv must"),
    ("prefill_attention", lambda a: (a["q"], a["kv"][0]), "kv must"),
    ("prefill_attention", lambda a: (a["q"], a["kv"], torch.zeros(6, 2, dtype=torch.int32)), "GPU"),
    ("prefill_attention", lambda a: (a["q"], a["kv"], torch.zeros(6, 2, device=a["q"].device)), "int32"),
    ("prefill_attention", lambda a: (a["q"], a["kv"], torch.zeros(6, 1, dtype=torch.int32, device=a["q"].device)),
     "bits holds"),
])
def test_refused(dev, name, args, message):
    from lagged_indexer_dsa_amd import ops

    with pytest.raises(RuntimeError, match=message):
        getattr(ops, name)(*args(_make(dev)))


def test_accepted(dev):
    from lagged_indexer_dsa_amd import ops

    a = _make(dev)
    assert ops.select_rows(a["scores"], 4, 40).shape == (6, 4)
    assert ops.prefill_logits(a["iq"], a["ik"], a["iw"]).shape == (2, 3, 40)
    assert ops.pack_latent_rows(a["kv"], 40).shape == (80, 656)
    bits = ops.selection_set(a["idx"], 40, True)
    assert ops.selection_set(a["idx"].int(), 40, False).shape == (6, 8)
    assert ops.prefill_attention(a["q"], a["kv"], bits).shape == (2, 3, 16, 512)


def test_empty_contexts(dev):
    """No key: empty scores and zero rows, for the shapes that a context of
    one key is taken with, and refused like it for the others."""
    from lagged_indexer_dsa_amd import attention_core as ac

    for T in (0, 1):
        def logits(B, S, H):
            return ac.indexer_logits(torch.zeros(B, S, H, 128, device=dev), torch.zeros(B, T, 128, device=dev),
                                     torch.zeros(B, S, H, device=dev))

        def dense(B, S, H):
            return ac.dense_mla_core(torch.ones(B, S, H, 576, dtype=torch.bfloat16, device=dev),
                                     torch.zeros(B, T, 576, dtype=torch.bfloat16, device=dev), 512)

        assert logits(2, 3, 32).shape == (2, 3, T)
        assert dense(2, 3, 32).shape == (2, 3, 32, 512) and not dense(2, 3, 32).any()
        for shape in ((2, 3, 24), (2, 3, 80), (2, 0, 32), (1, 65536, 16)):
            with pytest.raises(RuntimeError):
                logits(*shape)
        for shape in ((1, 1, 1040), (1, 2, 0), (2, 0, 32), (1, 65536, 16)):
            with pytest.raises(RuntimeError):
                dense(*shape)
