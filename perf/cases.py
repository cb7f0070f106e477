"""Performance cases: the calls a program that serves with this package makes.

Each case is one of these kinds:

* ``prep``    -- the operand step of new tokens: quantise their indexer
  queries, append their index keys and latent rows to the paged caches
  (``ops.quantize_index_query``, ``append_index_keys``,
  ``append_latent_rows``).  One token per request in decode, a whole prompt
  chunk in prefill.
* ``step``    -- a decode step of a stack of layers under the lag schedule,
  replayed as its captured graph (``MLISchedule.replay``): every
  ``indexer_every``-th layer runs its indexer, the others reuse.
* ``own``     -- decode layers that attend their own fresh selection (no
  lag), launched eagerly (``DecodeLayer.run``).
* ``dense``   -- the decode attention of a full-attention layer
  (``ops.dense_mla_decode``).
* ``logits``, ``select``, ``attend``, ``full`` -- the four core ops a prefill
  or a chunk of one goes through (``attention_core.indexer_logits``,
  ``select_topk``, ``sparse_mla_core``, ``dense_mla_core``): ``q_len`` query
  rows at the end of a context of ``ctx`` tokens.

Ranges: 1-64 requests of 64-196608 tokens, 1-16 layers; 16-128 attention
heads, 16-64 indexer heads, top-512 to top-2048; prefill chunks of 1-3000 (all
of a short prompt) to 1024 rows over contexts of up to 16384 tokens, float32
and bfloat16.
"""

from __future__ import annotations

import sys
from pathlib import Path

import torch

_PKG = Path(__file__).resolve().parent.parent / "dsa-multi-layer-indexer_amd"
if str(_PKG) not in sys.path:
    sys.path.insert(0, str(_PKG))

from lagged_indexer_dsa_amd import attention_core, ops, synthetic  # noqa: E402
from lagged_indexer_dsa_amd.decode import MLISchedule  # noqa: E402

PAGE = 64
DTYPES = {"float32": torch.float32, "bfloat16": torch.bfloat16}


# ---------------------------------------------------------------- the cases

def listed() -> list[dict]:
    return [
        # one new token of one request: three tiny launches
        dict(name="prep_token", kind="prep", rows=1, tokens=1, hidx=64),
        # a prompt chunk's tokens written to the caches (odd length)
        dict(name="prep_prompt", kind="prep", rows=1, tokens=8191, hidx=64),
        # a short chat turn: everything fits a few pages' worth of work
        dict(name="step_short", kind="step", rows=1, lo=4133, hi=4133, layers=2, indexer_every=1, heads=16,
             hidx=64, topk=2048, window=False),
        # the benchmark's workload: long context, batch 1, two layers under the lag
        dict(name="step_128k", kind="step", rows=1, lo=131072, hi=131072, layers=2, indexer_every=1, heads=16,
             hidx=64, topk=2048, window=False),
        # batched serving of ragged requests
        dict(name="step_ragged32", kind="step", rows=32, lo=16384, hi=131072, layers=2, indexer_every=1, heads=16,
             hidx=64, topk=2048, window=False),
        # a stage of a deep stack at the longest context, a fresh selection in one layer of four
        dict(name="step_stack196k", kind="step", rows=1, lo=196608, hi=196608, layers=16, indexer_every=4, heads=16,
             hidx=64, topk=2048, window=False),
        # unsharded heads (64 heads, 32 indexer heads), no lag, a few requests
        dict(name="own_64heads", kind="own", rows=4, lo=8000, hi=65536, layers=1, indexer_every=1, heads=64,
             hidx=32, topk=2048, window=False),
        # a full-attention layer of a few requests
        dict(name="dense_32k", kind="dense", rows=3, lo=777, hi=32768, heads=64),
        # a prompt's chunk of 1024 queries: its four core ops
        dict(name="prefill_logits", kind="logits", rows=1, q_len=1024, ctx=8192, hidx=64, dtype="bfloat16"),
        dict(name="prefill_select", kind="select", rows=1, q_len=1024, ctx=8192, topk=2048),
        dict(name="prefill_attend", kind="attend", rows=1, q_len=1024, ctx=8192, heads=16, topk=2048,
             dtype="bfloat16"),
        # a whole prompt through a full-attention layer (odd length)
        dict(name="prefill_full", kind="full", rows=1, q_len=2999, ctx=2999, heads=16, dtype="bfloat16"),
    ]


def _log(rng, lo: int, hi: int) -> int:
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng) -> dict:
    kind = rng.choice(["prep", "step", "step", "step", "own", "dense", "logits", "select", "attend", "full"])
    hidx = rng.choice([16, 32, 48, 64, 64, 64])
    if kind == "prep":
        rows = _log(rng, 1, 64)
        tokens = 1 if rng.random() < 0.4 else _log(rng, 2, max(2, 8191 // rows))
        return dict(kind="prep", rows=rows, tokens=tokens, hidx=hidx)
    if kind in ("step", "own"):
        rows = _log(rng, 1, 64)
        layers = rng.randint(1, 2) if rows > 8 else rng.randint(1, 4)
        # tokens of all rows and layers: at most those of step_ragged32
        hi = _log(rng, 64, min(196608, 4_000_000 // (rows * layers)))
        lo = max(1, int(hi * rng.random()))
        return dict(kind=kind, rows=rows, lo=lo, hi=hi, layers=layers,
                    indexer_every=rng.choice([1, 1, 2, 4]) if kind == "step" else 1,
                    heads=rng.choice([16, 16, 32, 64, 128]) if rows <= 8 else 16, hidx=hidx,
                    topk=rng.choice([512, 1024, 2048, 2048]), window=rng.random() < 0.25)
    if kind == "dense":
        rows = _log(rng, 1, 16)
        hi = _log(rng, 64, min(131072, 200_000 // rows))
        heads = rng.choice([16, 32, 64, 128]) if rows * hi <= 60_000 else 16
        return dict(kind="dense", rows=rows, lo=max(1, int(hi * rng.random())), hi=hi, heads=heads)
    if kind == "full":
        rows = rng.choice([1, 1, 2])
        ctx = _log(rng, 64, 2999 // rows)
        q_len = ctx if rng.random() < 0.6 else _log(rng, 1, ctx)
        return dict(kind="full", rows=rows, q_len=q_len, ctx=ctx, heads=rng.choice([16, 32]) if ctx <= 2000 else 16,
                    dtype=rng.choice(["float32", "bfloat16"]))
    rows = rng.choice([1, 1, 2])
    ctx = _log(rng, 256, 16384)
    q_len = min(ctx, _log(rng, 1, min(1024, 8_000_000 // ctx) // rows))
    case = dict(kind=kind, rows=rows, q_len=q_len, ctx=ctx)
    if kind == "logits":
        return dict(case, hidx=hidx, dtype=rng.choice(["float32", "bfloat16"]))
    case["topk"] = rng.choice([512, 1024, 2048, 2048])
    if kind == "select":
        return case
    heads = rng.choice([16, 16, 32, 64]) if q_len <= 256 else 16
    return dict(case, heads=heads, dtype=rng.choice(["float32", "bfloat16"]))


def _lens(case: dict) -> list[int]:
    """The requests' lengths: spread over [lo, hi], the longest hi (a function
    of the case, so that every seed has the same work)."""
    n, lo, hi = case["rows"], case["lo"], case["hi"]
    g = torch.Generator().manual_seed(4000 + n)
    u = torch.rand(n, generator=g).tolist()
    u[n // 2] = 1.0
    return [lo + int(round((hi - lo) * x)) for x in u]


# ------------------------------------------------------------ inputs

def prepare(case: dict, seed: int) -> dict:
    dev = torch.device("cuda:0")
    kind = case["kind"]
    g = torch.Generator(device=dev).manual_seed(1_000_003 * seed + 17)

    def randn(*shape, dtype=torch.float32):
        return torch.randn(*shape, generator=g, device=dev).to(dtype)

    if kind == "prep":
        B, T, H = case["rows"], case["tokens"], case["hidx"]
        npg = -(-(T + 100) // PAGE)
        n = B * T
        pt = torch.randperm(B * npg, generator=torch.Generator().manual_seed(seed)).to(torch.int32)
        pt = pt.reshape(B, npg).to(dev)
        rows = torch.arange(B, dtype=torch.int32, device=dev).repeat_interleave(T)
        pos = (torch.arange(T, dtype=torch.int32, device=dev) + 37).repeat(B)  # after a 37-token prefix
        slots = pt[rows.long(), (pos // PAGE).long()] * PAGE + pos % PAGE
        return dict(kind=kind, q=randn(n, H, 128, dtype=torch.bfloat16), w=randn(n, H) * H ** -0.5,
                    keys=randn(n, 128, dtype=torch.bfloat16), latent=randn(n, 576, dtype=torch.bfloat16),
                    rows=rows, pos=pos, pt=pt, slots=slots.to(torch.int32).contiguous(),
                    out_q=torch.empty(n, H, 128, dtype=torch.uint8, device=dev),
                    out_w=torch.empty(n, H, dtype=torch.float32, device=dev),
                    index_k=torch.zeros(B * npg, 8448, dtype=torch.uint8, device=dev),
                    kv_pool=torch.zeros(B * npg * PAGE, 656, dtype=torch.uint8, device=dev))
    if kind in ("step", "own", "dense"):
        lens = _lens(case)
        pt, num_pages = synthetic.make_page_table(lens, seed=seed, device=dev)
        n_layers = case.get("layers", 1)
        layers = [synthetic.make_decode_layer(
            lens, seed=1_000_003 * seed + i, device=dev, page_table=pt, num_pages=num_pages, heads=case["heads"],
            hidx=case.get("hidx", 64), topk=case.get("topk", 2048),
            indexer=kind != "dense" and i % case["indexer_every"] == 0) for i in range(n_layers)]
        if case.get("window"):
            # the scores of a 3000-token window of each row 50 times the rest
            # (the selection is packed in a few positions)
            for L in layers:
                if L.has_indexer:
                    scales = L.index_k[:, 8192:].view(torch.float32)
                    for b, n in enumerate(lens):
                        p = torch.arange(n // 3, min(n, n // 3 + 3000), device=dev)
                        scales[pt[b].long()[p // PAGE], p % PAGE] *= 50.0
        if kind == "dense":
            return dict(kind=kind, layer=layers[0])
        if kind == "own":
            return dict(kind=kind, layers=layers)
        first = synthetic.random_selection(lens, case["topk"], pt, seed=seed, device=dev)
        sched = MLISchedule(layers, first)
        sched.capture()
        return dict(kind=kind, layers=layers, first=first, sched=sched)
    B, S, T = case["rows"], case["q_len"], case["ctx"]
    dt = DTYPES[case.get("dtype", "float32")]
    if kind == "logits":
        H = case["hidx"]
        return dict(kind=kind, q=randn(B, S, H, 128, dtype=dt), k=randn(B, T, 128, dtype=dt),
                    w=(randn(B, S, H) * H ** -0.5).to(dt))
    causal = torch.arange(T, device=dev)[None, :] <= torch.arange(T - S, T, device=dev)[:, None]
    if kind == "select":
        return dict(kind=kind, logits=randn(B, S, T).masked_fill(~causal, float("-inf")), topk=case["topk"])
    state = dict(kind=kind, q=randn(B, S, case["heads"], 576, dtype=dt), kv=randn(B, T, 576, dtype=dt))
    if kind == "attend":
        # a selection as select_topk returns it: score order, the sentinel
        # ctx where the causal prefix is shorter than top-k
        K = case["topk"]
        score = torch.rand(B, S, T, generator=g, device=dev).masked_fill(~causal, -1.0)
        val, idx = torch.topk(score, min(K, T), dim=-1)
        idx = torch.where(val >= 0, idx, torch.full_like(idx, T))
        if K > T:
            idx = torch.cat([idx, torch.full((B, S, K - T), T, dtype=idx.dtype, device=dev)], dim=-1)
        state["idx"] = idx.contiguous()
    return state


# ------------------------------------------------------------ one pass

def run(s: dict):
    kind = s["kind"]
    if kind == "prep":
        ops.quantize_index_query(s["q"], s["w"], out_q=s["out_q"], out_w=s["out_w"])
        ops.append_index_keys(s["index_k"], s["pt"], s["rows"], s["pos"], s["keys"])
        ops.append_latent_rows(s["kv_pool"], s["slots"], s["latent"])
        return dict(q=s["out_q"], w=s["out_w"], index_k=s["index_k"], kv=s["kv_pool"])
    if kind == "step":
        s["sched"].replay()
        return _layer_outputs(s["layers"])
    if kind == "own":
        for L in s["layers"]:
            L.run()
        return _layer_outputs(s["layers"])
    if kind == "dense":
        L = s["layer"]
        return ops.dense_mla_decode(L.q_bf16, L.kv_pool, L.page_table, L.seq_lens, workspace=L.workspace, out=L.out)
    if kind == "logits":
        return attention_core.indexer_logits(s["q"], s["k"], s["w"])
    if kind == "select":
        return attention_core.select_topk(s["logits"], s["topk"])
    if kind == "attend":
        return attention_core.sparse_mla_core(s["q"], s["kv"], s["idx"], 512)
    return attention_core.dense_mla_core(s["q"], s["kv"], 512)


def _layer_outputs(layers) -> list:
    return [dict(out=L.out, scores=L.scores, sel=L.next_idx) if L.has_indexer else dict(out=L.out) for L in layers]


# ------------------------------------------------------------ what it cannot do without

def work(case: dict) -> dict:
    kind = case["kind"]
    if kind == "prep":
        n, H = case["rows"] * case["tokens"], case["hidx"]
        return dict(bytes=n * (H * (256 + 4 + 128 + 4) + 256 + 132 + 1152 + 656 + 12), flops=n * 3 * (H + 5) * 128)
    if kind in ("step", "own", "dense"):
        lens, H = _lens(case), case["heads"]
        qo = case["rows"] * H * (1152 + 1024)
        if kind == "dense":
            return dict(bytes=sum(lens) * 656 + qo, flops=sum(lens) * H * 1088 * 2)
        tok, hidx, K = sum(lens), case["hidx"], case["topk"]
        sel = sum(min(K, n) for n in lens)
        n_idx = -(-case["layers"] // case["indexer_every"])
        return dict(bytes=n_idx * (tok * 136 + case["rows"] * (hidx * 132 + 4 * K)) + case["layers"] * (sel * 656 + qo),
                    flops=n_idx * tok * hidx * 256 + case["layers"] * sel * H * 1088 * 2)
    B, S, T = case["rows"], case["q_len"], case["ctx"]
    es = 2 if case.get("dtype") == "bfloat16" else 4
    if kind == "logits":
        H = case["hidx"]
        return dict(bytes=B * (S * H * 129 * es + T * 128 * es + 4 * S * T), flops=B * S * T * H * 256)
    if kind == "select":
        return dict(bytes=B * S * (4 * T + 8 * case["topk"]), flops=0)
    H = case["heads"]
    pairs = B * sum(min(T - S + s + 1, case.get("topk", T)) for s in range(S))
    nbytes = B * (T * 576 + S * H * 1088) * es + (B * S * case["topk"] * 8 if kind == "attend" else 0)
    return dict(bytes=nbytes, flops=pairs * H * 1088 * 2)


def tolerance(case: dict):
    kind = case["kind"]
    if kind in ("prep", "select"):
        return "exact"  # codes, scales and selections: IEEE fp32 and integer work
    if kind == "logits":
        # the matrix unit's sum of 128 exact fp8 products, in its own order
        # and width: 1.3e-5 from the 64-bit sums
        return dict(rel=5e-5)
    # bf16 probabilities and outputs: 1.7e-3 to 2.1e-3 from 64 bits
    return dict(rel=1e-2, max=0.1)


# ------------------------------------------------------------ the same in 64 bits

def _e4m3_rows(x: torch.Tensor):
    """Per-row e4m3 codes (as float64 values) and scales of the last dim:
    scale = max(amax, 1e-6) / 448 in fp32, codes rounded to nearest even."""
    x = x.float()
    scale = (x.abs().amax(-1, keepdim=True).clamp_min(1e-6).double() / 448.0).float()
    y = (x.double() / scale.double()).float().clamp(-448.0, 448.0)
    return y.to(torch.float8_e4m3fn).double(), scale.double()


def _latent_values(x: torch.Tensor) -> torch.Tensor:
    """[..., 576] -> the values the 656-byte row format holds, float64."""
    codes, scale = _e4m3_rows(x[..., :512].unflatten(-1, (4, 128)))
    nope = (codes * scale).float().to(torch.bfloat16).flatten(-2)
    return torch.cat([nope, x[..., 512:].to(torch.bfloat16)], -1).double()


def _pool_values(rows: torch.Tensor) -> torch.Tensor:
    """[n, 656] bytes -> [n, 576] float64."""
    rows = rows.contiguous()
    n = rows.shape[0]
    codes = rows[:, :512].contiguous().view(torch.float8_e4m3fn).float().reshape(n, 4, 128)
    scale = rows[:, 512:528].contiguous().view(torch.float32)
    nope = (codes * scale[:, :, None]).to(torch.bfloat16).reshape(n, 512)
    return torch.cat([nope, rows[:, 528:].contiguous().view(torch.bfloat16)], -1).double()


def _attend(q: torch.Tensor, keys: torch.Tensor, mask: torch.Tensor | None = None) -> torch.Tensor:
    """softmax(q keys^T / 24) keys[:, :512] in float64; rows without a key give 0."""
    s = q @ keys.transpose(-1, -2) * 576 ** -0.5
    if mask is not None:
        s = s.masked_fill(~mask, float("-inf"))
    return torch.softmax(s, -1).nan_to_num(0.0) @ keys[..., :512]


def exact(case: dict, seed: int):
    kind = case["kind"]
    s = prepare(case, seed)
    if kind == "prep":
        _, scale = _e4m3_rows(s["q"])
        return dict(q=None, w=s["w"].double() * scale.squeeze(-1), index_k=None, kv=None)
    if kind == "select":
        return None  # whole numbers
    if kind in ("step", "own", "dense"):
        lens = _lens(case)
        if kind == "dense":
            L = s["layer"]
            out = torch.zeros(L.out.shape, dtype=torch.float64, device=L.out.device)
            for b, n in enumerate(lens):
                p = torch.arange(n, device=out.device)
                slots = L.page_table[b].long()[p // PAGE] * PAGE + p % PAGE
                out[b] = _attend(L.q_bf16[b].double(), _pool_values(L.kv_pool[slots]))
            return out
        carried, got = s.get("first"), []
        for L in s["layers"]:
            res = {}
            if L.has_indexer:
                res["scores"], fresh = _exact_selection(L, lens)
                res["sel"] = None
            att = fresh if kind == "own" else carried
            out = torch.zeros(L.out.shape, dtype=torch.float64, device=L.out.device)
            for b in range(len(lens)):
                slots = att[b].long()
                out[b] = _attend(L.q_bf16[b].double(), _pool_values(L.kv_pool[slots[slots >= 0]]))
            if L.has_indexer:
                carried = fresh
            got.append(dict(res, out=out))
        return got
    B, S, T = case["rows"], case["q_len"], case["ctx"]
    if kind == "logits":
        qv, sq = _e4m3_rows(s["q"])
        kv, sk = _e4m3_rows(s["k"])
        w = (s["w"].float() * sq.squeeze(-1).float()).double()
        out = torch.zeros(B, S, T, dtype=torch.float64, device=qv.device)
        for b in range(B):
            for h in range(case["hidx"]):
                out[b] += w[b, :, h, None] * torch.relu(qv[b, :, h] @ kv[b].T)
            out[b] *= sk[b].T
        return out
    keys, q = _latent_values(s["kv"]), s["q"].to(torch.bfloat16).double()
    out = torch.zeros(B, S, case["heads"], 512, dtype=torch.float64, device=q.device)
    if kind == "full":
        mask = torch.arange(T, device=q.device)[None, :] <= torch.arange(T - S, T, device=q.device)[:, None]
        for b in range(B):
            for h in range(case["heads"]):
                out[b, :, h] = _attend(q[b, :, h], keys[b], mask)
        return out
    for b in range(B):
        for i in range(0, S, 16):
            idx = s["idx"][b, i:i + 16]
            sel = keys[b][idx.clamp(max=T - 1)]
            out[b, i:i + 16] = _attend(q[b, i:i + 16], sel, (idx < T)[:, None, :])
    return out


def _exact_selection(L, lens: list[int]):
    """A layer's scores [B, slab] in float64 and the KV slots of its top-k."""
    pages = L.index_k
    keys = pages[:, :8192].contiguous().view(torch.float8_e4m3fn).reshape(-1, PAGE, 128)
    scales = pages[:, 8192:].contiguous().view(torch.float32)
    q = L.q_fp8.view(torch.float8_e4m3fn).double()
    scores = torch.full((len(lens), L.slab_stride), float("-inf"), dtype=torch.float64, device=pages.device)
    sel = torch.full((len(lens), L.topk), -1, dtype=torch.int64, device=pages.device)
    for b, n in enumerate(lens):
        pt = L.page_table[b].long()[: -(-n // PAGE)]
        k = keys[pt].double().reshape(-1, 128)[:n]
        v = torch.relu(k @ q[b].T) @ L.w[b].double() * scales[pt].double().reshape(-1)[:n]
        scores[b, :n] = v
        pos = torch.topk(v, min(L.topk, n)).indices
        sel[b, :pos.shape[0]] = pt[pos // PAGE] * PAGE + pos % PAGE
    return scores, sel
