"""The work a user of this framework has it do, as cases that can be timed and compared.

Seven kinds of pass, each through public entry points:

- prefill: causal GQA attention of one prompt (row_kernels.prefill_attention);
- attend: decode attention over selected pool rows (row_kernels.attend_batched);
- select: Quest scoring, page selection and row resolution of a batch
  (row_kernels.quest_batched + select_resolve_batched);
- step: one layer's whole sparse decode step, host-row gather included
  (batch_step.SparseDecodeBatch);
- dense: the dense half of one decode layer (add + RMSNorm, q/k/v with RoPE,
  output projection, add + RMSNorm, gate/up with SiLU, down);
- model-prefill: a prompt through Model.prefill into a cache;
- model-decode: one token for a batch of requests through Model.decode_batch.

Head shapes, widths, page sizes and budgets are those of bench.py and tests/:
32/8 and 28/4 heads of 128 (hidden 4096 and 3584), 4/2 heads of 64, pages of
16, 32 and 64, and fp32, fp16 and bf16 KV.
"""

import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "nano-hisparse_amd"))

from nano_hisparse import CacheConfig, HotConfig, HybridKVCache  # noqa: E402
from nano_hisparse import row_kernels as rk  # noqa: E402
from nano_hisparse.batch_step import BatchTables, SparseDecodeBatch  # noqa: E402
from nano_hisparse.model import Model, ModelConfig  # noqa: E402

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
SIZE = {"bf16": 2, "fp16": 2, "fp32": 4}
EPS, THETA = 1e-6, 10000.0


def listed():
    return [
        # the longest prompt the benchmark's contexts reach: one layer's prompt attention
        _prefill("prefill-32k", 32768, 32, 8, 128, "bf16"),
        # an ordinary prompt of a length that is no multiple of anything, group of seven
        _prefill("prefill-2k", 1999, 28, 4, 128, "bf16"),
        # a short prompt of a small model: few workgroups, launch latency counts
        _prefill("prefill-short", 333, 4, 2, 64, "fp16"),
        # one decode layer's attention, 16 requests x 2048 rows (the benchmark's default)
        _attend("attend-b16", 16, 32, 8, 128, 64, 32, 9, "bf16"),
        # many requests, group of seven, pages of 32 (the resolver-stress heads)
        _attend("attend-b64", 64, 28, 4, 128, 32, 32, 0, "bf16"),
        # one request of a small fp32 model: the smallest call
        _attend("attend-one-fp32", 1, 4, 2, 64, 16, 8, 5, "fp32"),
        # selection and resolution for 64 requests with ragged histories up to 64K tokens
        _select("select-b64", 64, 28, 4, 128, 32, 2048, 32, "bf16"),
        # a whole layer step of 16 requests, about a quarter of its rows from host memory
        _step("step-b16", 16, 32, 8, 128, 64, 256, 32, "bf16"),
        # the dense half of a decode layer at a serving batch
        _dense("dense-b8", 8, 4096, 32, 8, 14336, "bf16"),
        # one request alone on a smaller model
        _dense("dense-one", 1, 2048, 16, 4, 4096, "fp16"),
        # a prompt through two full-width layers into the cache, page by page
        _model("model-prefill", "model-prefill", 1, 2, 4096, 32, 8, 14336, 4000, 32),
        # one token for eight requests, replayed from the step's graph
        _model("model-decode", "model-decode", 8, 2, 4096, 32, 8, 14336, 4000, 16),
    ]


def draw(rng):
    """One more case of the ranges the listed ones stand for."""

    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["prefill"] * 4 + ["attend"] * 4 + ["select"] * 2 + ["step"] * 2 + ["dense"] * 3 + ["model"])
    heads, kv, dim = rng.choice([(32, 8, 128), (28, 4, 128), (16, 4, 128), (4, 2, 64), (14, 2, 64)])
    half = rng.choice(["bf16", "bf16", "fp16"])
    page = rng.choice([16, 32, 64])
    if kind == "prefill":
        return _prefill(None, size(1, 24000), heads, kv, dim, half)
    if kind == "attend":
        pages = size(2, 4096 // page)
        return _attend(None, size(1, 64), heads, kv, dim, page, pages, rng.randrange(page), rng.choice([half, half, "fp32"]))
    if kind == "select":
        n_pages = size(8, 2048)
        return _select(None, size(1, 64), heads, kv, dim, page, n_pages, size(1, min(n_pages, 2048 // page)), half)
    if kind == "step":
        n_pages = size(16, 256)
        return _step(None, size(1, 16), 32, 8, 128, page, n_pages, size(2, min(n_pages, 32)), half)
    if kind == "dense":
        hidden, h, k, inter = rng.choice([(4096, 32, 8, 14336), (2048, 16, 4, 4096), (2048, 16, 4, 6144)])
        return _dense(None, size(1, 16), hidden, h, k, inter, half)
    if rng.random() < 0.5:
        return _model(None, "model-prefill", 1, 2, 2048, 16, 4, 4096, size(100, 5000), 16)
    return _model(None, "model-decode", size(2, 12), 2, 2048, 16, 4, 4096, size(500, 4000), 8)


def _case(name, **values):
    return dict(values, name=name) if name else values


def _prefill(name, seq, heads, kv, dim, dtype):
    return _case(name, kind="prefill", seq=seq, heads=heads, kv=kv, dim=dim, dtype=dtype)


def _attend(name, batch, heads, kv, dim, page, pages, pad, dtype):
    # pages * page selected rows per request, the last `pad` of them past the request's end (-1)
    return _case(name, kind="attend", batch=batch, heads=heads, kv=kv, dim=dim, page=page, pages=pages, pad=pad,
                 dtype=dtype)


def _select(name, batch, heads, kv, dim, page, n_pages, top, dtype):
    return _case(name, kind="select", batch=batch, heads=heads, kv=kv, dim=dim, page=page, n_pages=n_pages, top=top,
                 dtype=dtype)


def _step(name, batch, heads, kv, dim, page, n_pages, top, dtype):
    return _case(name, kind="step", batch=batch, heads=heads, kv=kv, dim=dim, page=page, n_pages=n_pages, top=top,
                 dtype=dtype)


def _dense(name, batch, hidden, heads, kv, inter, dtype):
    return _case(name, kind="dense", batch=batch, hidden=hidden, heads=heads, kv=kv, inter=inter, dtype=dtype)


def _model(name, kind, batch, layers, hidden, heads, kv, inter, context, top):
    return _case(name, kind=kind, batch=batch, layers=layers, hidden=hidden, heads=heads, kv=kv, inter=inter,
                 context=context, top=top, vocab=32000, page=64, dtype="bf16")


# ---- inputs ---------------------------------------------------------------------------------


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    return _PREPARE[case["kind"]](case, gen, seed)


def _randn(gen, *shape, dtype=torch.float32, scale=1.0):
    return (torch.randn(*shape, generator=gen, device="cuda") * scale).to(dtype)


def _prepare_prefill(c, gen, seed):
    t, n = DTYPES[c["dtype"]], c["seq"]
    return {"kind": "prefill", "q": _randn(gen, n, c["heads"], c["dim"], dtype=t),
            "k": _randn(gen, n, c["kv"], c["dim"], dtype=t), "v": _randn(gen, n, c["kv"], c["dim"], dtype=t)}


def _prepare_attend(c, gen, seed):
    t, B, P, n = DTYPES[c["dtype"]], c["batch"], c["page"], c["pages"]
    blocks = B * n + 3
    pool = rk.padded_pool(blocks, P, c["kv"], c["dim"], t, "cuda")
    for at in range(0, blocks, 512):
        part = pool[at:at + 512]
        part.copy_(_randn(gen, *part.shape, dtype=t))
    order = torch.randperm(blocks, generator=gen, device="cuda")[: B * n].view(B, n, 1)
    rows = (order * P + torch.arange(P, device="cuda")).view(B, n * P)
    if c["pad"]:
        rows[:, n * P - c["pad"]:] = -1
    return {"kind": "attend", "q": _randn(gen, B, c["heads"], c["dim"], dtype=t), "pool": pool, "rows": rows, "page": P}


def _tables(c, gen):
    """Residency of B requests' pages: half resident in the pool (the last two
    always), a quarter's rows in a full hot buffer at random slots and LRU
    order, the rest in host memory only. Histories end at ragged lengths."""
    B, P, n = c["batch"], c["page"], c["n_pages"]
    H = 2 * c["top"] * P
    dev = "cuda"
    hot_blocks = H // P
    n_res = max(2, n // 2)
    per = hot_blocks + n_res
    if c["kind"] == "step":
        lengths = n * P - torch.randint(0, P, (B,), generator=gen, device=dev)
    else:
        lengths = (torch.rand(B, generator=gen, device=dev) * (n * P * 15 // 16)).long() + max(1, n * P // 16)
    score = torch.rand(B, n, generator=gen, device=dev)
    last = (lengths - 1) // P
    index = torch.arange(n, device=dev)
    score[(index >= last[:, None] - 1) & (index <= last[:, None])] = -1.0  # the tail pages come first
    order = score.argsort(1)
    base = torch.arange(B, device=dev)[:, None] * per
    resident = torch.full((B, n), -1, dtype=torch.int32, device=dev)
    resident.scatter_(1, order[:, :n_res], (base + hot_blocks + torch.arange(n_res, device=dev)).int())
    source = torch.arange(B * n, dtype=torch.int32, device=dev).view(B, n)
    hot = (base + torch.arange(hot_blocks, device=dev)).int()
    pages = order[:, n_res:n_res + hot_blocks][:, : max(0, n // 4)]
    rows = ((source.long().gather(1, pages)[:, :, None] * P) + torch.arange(P, device=dev)).view(B, -1)
    slots = torch.rand(B, H, generator=gen, device=dev).argsort(1)[:, : rows.shape[1]]
    tags = torch.full((B, H), -1, dtype=torch.int32, device=dev)
    tags.scatter_(1, slots, rows.int())
    lru = torch.rand(B, H, generator=gen, device=dev).argsort(1)
    return {"source": source, "resident": resident, "hot": hot, "tags0": tags, "lru0": lru, "lengths": lengths,
            "slots": slots, "rows": rows, "order": order, "n_res": n_res, "per": per}


def _prepare_select(c, gen, seed):
    t = DTYPES[c["dtype"]]
    s = _tables(c, gen)
    a = _randn(gen, c["batch"], c["n_pages"], c["kv"], c["dim"])
    width = torch.rand(a.shape, generator=gen, device="cuda") * 2 + 1
    s.update(kind="select", q=_randn(gen, c["batch"], c["heads"], c["dim"], dtype=t), minimum=(a - width).to(t),
             maximum=(a + width).to(t), page=c["page"], top=c["top"], tags=s["tags0"].clone(), lru=s["lru0"].clone())
    return s


def _prepare_step(c, gen, seed):
    t, B, P, n, Hkv, D = DTYPES[c["dtype"]], c["batch"], c["page"], c["n_pages"], c["kv"], c["dim"]
    s = _tables(c, gen)
    data = torch.empty(B * n, 2, P, Hkv, D, dtype=t, device="cuda")
    for at in range(0, B * n, 512):
        part = data[at:at + 512]
        noise = _randn(gen, part.shape[0], 1, 1, Hkv, D, scale=0.3)
        part.copy_(torch.randn(part.shape, generator=gen, device="cuda") + noise)
    host = torch.empty(data.shape, dtype=t, pin_memory=True)
    host.copy_(data)
    pool = rk.padded_pool(B * s["per"], P, Hkv, D, t, "cuda")
    at = torch.arange(B, device="cuda")[:, None]
    res_pages = s["source"].long().gather(1, s["order"][:, : s["n_res"]])
    pool[s["resident"].long().gather(1, s["order"][:, : s["n_res"]]).flatten()] = data[res_pages.flatten()]
    block = s["hot"].long()[at, s["slots"] // P].flatten()
    rows = s["rows"].flatten()
    pool[block, :, (s["slots"] % P).flatten()] = data[rows // P, :, rows % P]
    lo = data[:, 0].amin(1).view(B, n, Hkv, D)
    hi = data[:, 0].amax(1).view(B, n, Hkv, D)
    tables = BatchTables(s["source"], s["resident"], s["hot"], s["tags0"].clone(), s["lru0"].clone(), lo, hi,
                         s["lengths"])
    s.update(kind="step", q=_randn(gen, B, c["heads"], D, dtype=t), tables=tables, host=host,
             step=SparseDecodeBatch(pool, host, tables, P, c["top"]))
    return s


def _prepare_dense(c, gen, seed):
    t, B, w, D = DTYPES[c["dtype"]], c["batch"], c["hidden"], c["hidden"] // c["heads"]
    n = (c["heads"] + 2 * c["kv"]) * D

    def weight(rows, cols):
        return _randn(gen, rows, cols, dtype=t, scale=cols ** -0.5)

    angle = torch.randint(0, 32768, (B, 1), generator=gen, device="cuda") * _inv_freq(D)
    return {"kind": "dense", "x": _randn(gen, B, w, dtype=t), "delta": _randn(gen, B, w, dtype=t),
            "attention": _randn(gen, B, w, dtype=t, scale=0.1), "norm1": 1 + _randn(gen, w, dtype=t, scale=0.1),
            "norm2": 1 + _randn(gen, w, dtype=t, scale=0.1), "qkv": weight(n, w), "bias": _randn(gen, n, dtype=t),
            "o": weight(w, w), "gate_up": weight(2 * c["inter"], w), "down": weight(w, c["inter"]),
            "cos": angle.cos().to(t), "sin": angle.sin().to(t), "rotated": c["heads"] + c["kv"], "dim": D}


def _inv_freq(dim, dtype=torch.float32):
    return THETA ** (-torch.arange(0, dim, 2, device="cuda").to(dtype) / dim)


def _prepare_model(c, gen, seed):
    B, L, P, D = c["batch"], c["layers"], c["page"], c["hidden"] // c["heads"]
    cfg = ModelConfig(vocab_size=c["vocab"], hidden_size=c["hidden"], intermediate_size=c["inter"],
                      num_hidden_layers=L, num_attention_heads=c["heads"], num_key_value_heads=c["kv"],
                      rope_theta=THETA)
    torch.manual_seed(seed)
    default = torch.get_default_dtype()
    torch.set_default_dtype(torch.bfloat16)
    try:
        with torch.device("cuda"):
            model = Model(cfg).eval()
    finally:
        torch.set_default_dtype(default)
    decode = c["kind"] == "model-decode"
    # decoding: room for the tokens of a long answer
    length = c["context"] + (8192 if decode else 64)
    pages = -(-length // P)
    hot = HotConfig(c["top"] * P, c["top"] * P)
    used = B * L * -(-c["context"] // P)
    kv = CacheConfig(gpu_pages=(B + 1) * hot.admission_blocks(P, L) + int(0.3 * used),
                     host_pages=(B * pages + 2) * L, page_size=P, kv_heads=c["kv"],
                     head_dim=D, dtype=torch.bfloat16, device="cuda:0", index_budget_bytes=1 << 30)
    cache = HybridKVCache(kv, hot)
    s = {"kind": c["kind"], "model": model, "cache": cache, "top": c["top"], "length": length, "layers": L}
    host_rng = torch.Generator().manual_seed(seed)
    if not decode:
        s["tokens"] = torch.randint(0, c["vocab"], (c["context"],), generator=host_rng).tolist()
        return s
    s["tokens"] = torch.randint(0, c["vocab"], (B,), generator=host_rng).tolist()
    s["ids"] = [f"r{b}" for b in range(B)]
    # a short request warms the model up eagerly (its projections are fused then, before any graph is captured)
    cache.reserve("warm", 2 * P, L)
    for layer in range(L):
        rows = _randn(gen, 2, 5, c["kv"], D, dtype=torch.bfloat16)
        cache.write("warm", layer, rows[0], rows[1])
    model.decode_batch([0], ["warm"], cache, c["top"])
    cache.release_request("warm")
    for b, rid in enumerate(s["ids"]):
        cache.reserve(rid, length, L)
        for layer in range(L):
            kv_rows = _history(c, seed, b, layer)
            cache.write(rid, layer, kv_rows[0], kv_rows[1])
    return s


def _history(c, seed, b, layer):
    """K/V [2, tokens, kv_heads, head_dim] of request b's history in one
    layer; the requests' histories differ by 37 tokens each."""
    gen = torch.Generator(device="cuda").manual_seed((seed * 64 + b) * 64 + layer)
    n = max(c["page"] + 1, c["context"] - 37 * b)
    return _randn(gen, 2, n, c["kv"], c["hidden"] // c["heads"], dtype=torch.bfloat16)


_PREPARE = {"prefill": _prepare_prefill, "attend": _prepare_attend, "select": _prepare_select, "step": _prepare_step,
            "dense": _prepare_dense, "model-prefill": _prepare_model, "model-decode": _prepare_model}


# ---- one pass -------------------------------------------------------------------------------


def run(s):
    return _RUN[s["kind"]](s)


def _run_prefill(s):
    return rk.prefill_attention(s["q"], s["k"], s["v"])


def _run_attend(s):
    return rk.attend_batched(s["q"], s["pool"], s["rows"], s["page"])


def _run_select(s):
    # every pass starts from the same hot-buffer state, so that it finds the same misses
    tags, lru = s["tags"].copy_(s["tags0"]), s["lru"].copy_(s["lru0"])
    P, top = s["page"], s["top"]
    _, _, scores = rk.quest_batched(s["q"], s["minimum"], s["maximum"], s["lengths"], P, top, select=False)
    pages, positions, physical, miss_host, miss_device, counts = rk.select_resolve_batched(
        scores, s["source"], s["resident"], s["hot"], tags, lru, s["lengths"], P, top)
    # (the scores of pages past a request's end are never written, so they are no output)
    return {"pages": pages, "positions": positions, "physical": physical, "miss_host": miss_host,
            "miss_device": miss_device, "counts": counts, "tags": tags, "lru": lru}


def _run_step(s):
    t = s["tables"]
    t.tags.copy_(s["tags0"])
    t.lru.copy_(s["lru0"])
    out, result = s["step"].step(s["q"])
    return {"out": out, "positions": result.positions, "physical": result.physical, "counts": result.counts,
            "tags": t.tags, "lru": t.lru}


def _run_dense(s):
    x = s["x"].clone()  # the residual stream is updated in place
    h = rk.add_rmsnorm(x, s["delta"], s["norm1"], EPS)
    qkv = rk.linear_rope(h, s["qkv"], s["bias"], s["rotated"], s["dim"], s["cos"], s["sin"])
    o = rk.linear_small_m(s["attention"], s["o"])
    h = rk.add_rmsnorm(x, o, s["norm2"], EPS)
    act = rk.linear_silu_mul(h, s["gate_up"])
    return {"qkv": qkv, "x": x, "act": act, "down": rk.linear_small_m(act, s["down"])}


def _run_model_prefill(s):
    cache = s["cache"]
    cache.reserve("prompt", s["length"], s["layers"])
    request = cache.storage.requests["prompt"]
    logits = s["model"].prefill(s["tokens"], cache, "prompt")
    used = -(-len(s["tokens"]) // cache.config.page_size)
    bounds = {name: getattr(request, name)[:, :used] for name in ("minimum", "maximum", "summaries")}
    cache.release_request("prompt")
    return dict(bounds, logits=logits)


def _run_model_decode(s):
    s["cache"].collect()
    return s["model"].decode_batch(s["tokens"], s["ids"], s["cache"], s["top"], graph=True)


_RUN = {"prefill": _run_prefill, "attend": _run_attend, "select": _run_select, "step": _run_step,
        "dense": _run_dense, "model-prefill": _run_model_prefill, "model-decode": _run_model_decode}


# ---- what a pass cannot do without ----------------------------------------------------------


def work(c):
    e, kind = SIZE[c["dtype"]], c["kind"]
    if kind == "prefill":
        n, H, G, D = c["seq"], c["heads"], c["kv"], c["dim"]
        return {"bytes": (2 * n * H * D + 2 * n * G * D) * e, "flops": 2.0 * n * (n + 1) * H * D}
    if kind == "attend":
        N, B, H, D = c["pages"] * c["page"], c["batch"], c["heads"], c["dim"]
        valid = N - c["pad"]
        return {"bytes": B * (valid * 2 * c["kv"] * D * e + 2 * H * D * e + 8 * N), "flops": 4.0 * B * valid * H * D}
    if kind in ("select", "step"):
        B, n, K, H = c["batch"], c["n_pages"], c["top"] * c["page"], c["heads"]
        row = c["kv"] * c["dim"] * e
        mean_pages = n if kind == "step" else n * 17 // 32
        state = B * (4 * K * 8 + 2 * 2 * K * 24)  # positions and plan written; tags and LRU read and written
        w = {"bytes": B * mean_pages * 2 * row + state, "flops": 4.0 * B * mean_pages * H * c["dim"]}
        if kind == "step":  # the selected rows are read, about a quarter of them written from host memory
            w["bytes"] += B * K * 2 * row * 5 // 4
            w["flops"] += 4.0 * B * K * H * c["dim"]
        return w
    D = c["hidden"] // c["heads"]
    weights = c["hidden"] * ((c["heads"] + 2 * c["kv"]) * D + c["hidden"] + 3 * c["inter"])
    if kind == "dense":
        return {"bytes": weights * e, "flops": 2.0 * c["batch"] * weights}
    L, B, n = c["layers"], c["batch"], c["context"]
    row = 2 * c["kv"] * D * e
    head = c["vocab"] * c["hidden"]
    if kind == "model-prefill":  # K/V go to the pool and to host memory
        return {"bytes": (L * weights + head) * e + L * n * (2 * row + 4 * c["hidden"] * e),
                "flops": 2.0 * n * L * weights + 2.0 * head + 2.0 * L * n * n * c["hidden"]}
    rows = c["top"] * c["page"]
    return {"bytes": (L * weights + head) * e + L * B * row * (rows + n // c["page"]),
            "flops": 2.0 * B * (L * weights + head) + 4.0 * L * B * rows * c["hidden"]}


def tolerance(c):
    # whole values (positions, rows, plans, tags, LRU) stay the same everywhere
    if c["kind"] == "select":
        return "exact"
    if c["kind"] in ("model-prefill", "model-decode"):
        return {"rel": 2e-2, "max": 0.3}  # 16-bit rounding through two layers
    if c["dtype"] == "fp32":
        return {"rel": 4e-6, "max": 2e-5}
    eps = {"bf16": 2.0 ** -8, "fp16": 2.0 ** -11}[c["dtype"]]
    # one rounding of the output for attention over rows; weights rounded to
    # the input type before P.V for prompts; three roundings in a row for the dense half
    return {"rel": {"attend": 1.0, "step": 1.0, "prefill": 2.0, "dense": 2.0}[c["kind"]] * eps, "max": 16 * eps}


# ---- the same in 64 bits ----------------------------------------------------------------------


def exact(case, seed):
    if case["kind"] == "select":  # whole values only
        return None
    return _EXACT[case["kind"]](case, prepare(case, seed), seed)


def _causal(q, k, v):
    """Causal GQA attention, q [S, Hq, D] and k/v [S, Hkv, D] in float64."""
    n, H, D = q.shape
    group = H // k.shape[1]
    out = torch.empty_like(q)
    for h in range(H):
        kh, vh = k[:, h // group].contiguous(), v[:, h // group].contiguous()
        kt = kh.t().contiguous()
        for a in range(0, n, 2048):
            b = min(n, a + 2048)
            scores = (q[a:b, h].contiguous() @ kt[:, :b]) * D ** -0.5
            scores.masked_fill_(torch.arange(b, device="cuda") > torch.arange(a, b, device="cuda")[:, None], -math.inf)
            out[a:b, h] = torch.softmax(scores, -1) @ vh[:b]
    return out


def _one_query(q, k, v):
    """q [Hq, D] over k/v [N, Hkv, D] in float64."""
    group = q.shape[0] // k.shape[1]
    k, v = k.repeat_interleave(group, 1), v.repeat_interleave(group, 1)
    p = torch.softmax((q[None] * k).sum(-1) * q.shape[1] ** -0.5, 0)
    return (p[:, :, None] * v).sum(0)


def _quest_scores(q, lo, hi):
    """Quest page scores of q [Hq, D] over bounds [pages, Hkv, D] in float64."""
    heads = q.shape[0]
    total = torch.zeros(lo.shape[0], dtype=torch.float64, device="cuda")
    for h in range(heads):
        g = h // (heads // lo.shape[1])
        total += torch.maximum(q[h] * lo[:, g], q[h] * hi[:, g]).sum(-1)
    return total / heads


def _quest_positions(scores, length, page, top):
    """The chosen pages' token positions: the last page, the first with a
    budget above one, and the best of the rest."""
    count = -(-length // page)
    scores = scores[:count].clone()
    scores[count - 1] = math.inf
    if top > 1:
        scores[0] = math.inf
    chosen = scores.topk(min(top, count)).indices.sort().values
    positions = (chosen[:, None] * page + torch.arange(page, device="cuda")).flatten()
    return positions[positions < length]


def _exact_prefill(c, s, seed):
    return _causal(s["q"].double(), s["k"].double(), s["v"].double())


def _exact_attend(c, s, seed):
    out, P = [], s["page"]
    for b in range(c["batch"]):
        rows = s["rows"][b]
        rows = rows[rows >= 0]
        kv = s["pool"][rows // P, :, rows % P].double()
        out.append(_one_query(s["q"][b].double(), kv[:, 0], kv[:, 1]))
    return torch.stack(out)


def _exact_step(c, s, seed):
    out, P, n = [], c["page"], c["n_pages"]
    t = s["tables"]
    for b in range(c["batch"]):
        q = s["q"][b].double()
        scores = _quest_scores(q, t.minimum[b].double(), t.maximum[b].double())
        pos = _quest_positions(scores, int(t.lengths[b]), P, c["top"])
        kv = s["host"][b * n:(b + 1) * n].to("cuda")[pos // P, :, pos % P].double()
        out.append(_one_query(q, kv[:, 0], kv[:, 1]))
    return {"out": torch.stack(out), "positions": None, "physical": None, "counts": None, "tags": None, "lru": None}


def _norm(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()


def _rope(t, cos, sin):
    """t [rows, heads, D] in float64; cos/sin [rows, D/2]."""
    lo, hi = t.chunk(2, -1)
    cos, sin = cos.double()[:, None], sin.double()[:, None]
    return torch.cat((lo * cos - hi * sin, hi * cos + lo * sin), -1)


def _mm(x, w):
    return x @ w.double().t().contiguous()


def _exact_dense(c, s, seed):
    x = s["x"].double() + s["delta"].double()
    qkv = _mm(_norm(x, s["norm1"]), s["qkv"]) + s["bias"].double()
    qkv = qkv.view(len(x), -1, s["dim"])
    qkv = torch.cat((_rope(qkv[:, : s["rotated"]], s["cos"], s["sin"]), qkv[:, s["rotated"]:]), 1).flatten(1)
    x = x + _mm(s["attention"].double(), s["o"])
    gate, up = _mm(_norm(x, s["norm2"]), s["gate_up"]).chunk(2, -1)
    act = torch.nn.functional.silu(gate) * up
    return {"qkv": qkv, "x": x, "act": act, "down": _mm(act, s["down"])}


def _layer_qkv(c, layer, x, positions):
    D, a = c["hidden"] // c["heads"], layer.self_attn
    h = _norm(x, layer.input_layernorm.weight)
    q, k, v = ((_mm(h, p.weight) + p.bias.double()).view(len(x), -1, D) for p in (a.q_proj, a.k_proj, a.v_proj))
    angle = positions.double()[:, None] * _inv_freq(D, torch.float64)
    return _rope(q, angle.cos(), angle.sin()), _rope(k, angle.cos(), angle.sin()), v


def _layer_rest(layer, x, attention):
    x = x + _mm(attention.flatten(1), layer.self_attn.o_proj.weight)
    h = _norm(x, layer.post_attention_layernorm.weight)
    act = torch.nn.functional.silu(_mm(h, layer.mlp.gate_proj.weight)) * _mm(h, layer.mlp.up_proj.weight)
    return x + _mm(act, layer.mlp.down_proj.weight)


@torch.no_grad()
def _exact_model_prefill(c, s, seed):
    m, P, n = s["model"], c["page"], c["context"]
    x = m.model.embed_tokens.weight[torch.tensor(s["tokens"], device="cuda")].double()
    bounds = {"minimum": [], "maximum": [], "summaries": []}
    for layer in m.model.layers:
        q, k, v = _layer_qkv(c, layer, x, torch.arange(n, device="cuda"))
        pages = k.split(P)
        bounds["minimum"].append(torch.stack([p.amin(0) for p in pages]))
        bounds["maximum"].append(torch.stack([p.amax(0) for p in pages]))
        bounds["summaries"].append(torch.stack([p.mean(0) for p in pages]))
        x = _layer_rest(layer, x, _causal(q, k, v))
    logits = _mm(_norm(x[-1:], m.model.norm.weight), m.lm_head.weight)[0]
    return dict({name: torch.stack(v) for name, v in bounds.items()}, logits=logits)


@torch.no_grad()
def _exact_model_decode(c, s, seed):
    m, P, B = s["model"], c["page"], c["batch"]
    x = m.model.embed_tokens.weight[torch.tensor(s["tokens"], device="cuda")].double()
    for index, layer in enumerate(m.model.layers):
        past = [_history(c, seed, b, index).double() for b in range(B)]
        at = torch.tensor([p.shape[1] for p in past], device="cuda")
        q, k, v = _layer_qkv(c, layer, x, at)
        out = []
        for b in range(B):
            kv = torch.cat((past[b], torch.stack((k[b:b + 1], v[b:b + 1]))), 1)
            pages = kv[0].split(P)
            lo, hi = torch.stack([p.amin(0) for p in pages]), torch.stack([p.amax(0) for p in pages])
            pos = _quest_positions(_quest_scores(q[b], lo, hi), kv.shape[1], P, c["top"])
            out.append(_one_query(q[b], kv[0, pos], kv[1, pos]))
        x = _layer_rest(layer, x, torch.stack(out))
    return _mm(_norm(x, m.model.norm.weight), m.lm_head.weight)


_EXACT = {"prefill": _exact_prefill, "attend": _exact_attend, "step": _exact_step,
          "dense": _exact_dense, "model-prefill": _exact_model_prefill, "model-decode": _exact_model_decode}
