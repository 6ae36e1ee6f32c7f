"""The work a user of this package has it do, as measurable cases through its public entry points.

``listed()`` names the cases, ``draw(rng)`` gives further ones from the same ranges,
``prepare(case, seed)`` makes what a caller holds before the call (caches, donors, weights,
positions, one request's attention plan), ``run(state)`` is one pass, ``work(case)`` the bytes
and operations that pass cannot do without, ``tolerance(case)`` how far a correct
implementation of the same precision may differ, and ``exact(case, seed)`` the same result in
64 bits from plain torch.

Sizes: the Qwen2.5-7B (28 query / 4 KV heads x 128, hidden 3584, 28 layers), Qwen2.5-0.5B
(14 / 2 x 64, hidden 896) and Llama-3-8B (32 / 8 x 128, hidden 4096) shapes of the tests and
the benchmark, pages of 16 tokens, contexts of some hundred to 32K tokens, 5-40% of them
recomputed.
"""

from __future__ import annotations

import math

import torch

from semblend_amd import rope_correction as rc
from semblend_amd import triton_kernels as tk

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
CHUNK = 256  # tokens of a donor chunk: one RoPE delta per chunk

# (query heads, KV heads, head_dim, hidden, RoPE base) of the model shapes.
QWEN7B = {"hq": 28, "hkv": 4, "d": 128, "hidden": 3584, "base": 1e6}
QWEN05B = {"hq": 14, "hkv": 2, "d": 64, "hidden": 896, "base": 1e6}
LLAMA8B = {"hq": 32, "hkv": 8, "d": 128, "hidden": 4096, "base": 5e5}
SHAPES = (QWEN7B, QWEN05B, LLAMA8B)


def listed() -> list[dict]:
    return [
        # The smallest call: one layer's K rotated in place by one delta at the positions that
        # share it (the per-delta caller pattern after a load; fp32 as the 0.5B pipeline).
        {"name": "rope_delta_8_positions", "kind": "rope_delta", "dtype": "fp32", "bs": 16,
         "ctx": 1024, "positions": 8, **QWEN05B},
        # One layer's donor K/V scattered into its paged cache with K rotated: the per-layer
        # call an engine's layer loop makes.
        {"name": "scatter_rope_1_layer_4k", "kind": "scatter_rope", "dtype": "fp16", "bs": 16,
         "layers": 1, "ctx": 4096, "frac": 0.15, **LLAMA8B},
        # The same for every layer of a 16K request in one call.
        {"name": "scatter_rope_28_layers_16k", "kind": "scatter_rope", "dtype": "bf16",
         "bs": 16, "layers": 28, "ctx": 16384, "frac": 0.15, **QWEN7B},
        # A donor's whole K corrected out of place before it is handed on.
        {"name": "rope_k_28_layers_8k", "kind": "rope_k", "dtype": "bf16", "layers": 28,
         "ctx": 8192, **QWEN7B},
        # The post-load hook: every layer's vLLM-layout cache permuted and rotated, the pairs
        # as the host list the connector holds.
        {"name": "permute_28_layers_8k", "kind": "permute", "dtype": "bf16", "bs": 16,
         "layers": 28, "ctx": 8192, **QWEN7B},
        # Almost everything reused: a few rows attend over a 4K context.
        {"name": "attn_40_rows_4k", "kind": "attn", "dtype": "bf16", "bs": 16, "ctx": 4096,
         "rows": 40, **LLAMA8B},
        # fp32 attention of the 0.5B pipeline (15% of 1024 tokens).
        {"name": "attn_fp32_154_rows_1k", "kind": "attn", "dtype": "fp32", "bs": 16,
         "ctx": 1024, "rows": 154, **QWEN05B},
        # The dense drop-in: heads-major Q/K/V and a device mask of the rows to compute.
        {"name": "attn_dense_28_heads_4k", "kind": "attn_dense", "dtype": "fp16", "ctx": 4096,
         "frac": 0.15, **QWEN7B},
        # One layer of a serving batch: four requests of 8K-32K tokens, 10-30% recomputed.
        {"name": "attn_batch_8k_to_32k", "kind": "attn_batch", "dtype": "bf16", "bs": 16,
         "requests": 4, "ctx": 32768, "frac": 0.30, **LLAMA8B},
        # QKV projection of few recomputed rows, new K/V written into the pages.
        {"name": "projection_64_rows", "kind": "projection", "dtype": "bf16", "bs": 16,
         "ctx": 4096, "rows": 64, **QWEN7B},
        # One attention layer of a 16K request: projection with RoPE, attention over the pages
        # (with the request's plan), output projection.
        {"name": "layer_16k", "kind": "layer", "dtype": "bf16", "bs": 16, "ctx": 16384,
         "frac": 0.15, **QWEN7B},
        # The single-layer orchestrator (multi-head attention, contiguous caches, 24 layers of
        # donor K/V assembled).
        {"name": "prefill_1k", "kind": "prefill", "dtype": "bf16", "layers": 24, "ctx": 1024,
         "frac": 0.3, **dict(QWEN05B, hkv=14)},
    ]


def _log(rng, lo: int, hi: int) -> int:
    """An integer spread over the logarithm of [lo, hi]."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng) -> dict:
    kind = rng.choice(("rope_delta", "scatter_rope", "rope_k", "permute", "attn", "attn_fp32",
                       "attn_dense", "attn_batch", "projection", "layer", "prefill"))
    shape = dict(rng.choice(SHAPES))
    half = rng.choice(("bf16", "bf16", "fp16"))
    bs = rng.choice((16, 16, 32))
    frac = round(rng.uniform(0.05, 0.4), 3)
    if kind == "rope_delta":
        ctx = _log(rng, 300, 16000)
        return {"kind": kind, "dtype": rng.choice(("fp32", half)), "bs": bs, "ctx": ctx,
                "positions": min(_log(rng, 1, 2000), ctx), **shape}
    if kind == "scatter_rope":
        return {"kind": kind, "dtype": rng.choice(("bf16", "fp16", "fp32")), "bs": bs,
                "layers": rng.choice((1, 1, 7, 24)), "ctx": _log(rng, 500, 12000),
                "frac": frac, **shape}
    if kind == "rope_k":
        return {"kind": kind, "dtype": rng.choice(("bf16", "fp16", "fp32")),
                "layers": rng.choice((1, 4, 13)), "ctx": _log(rng, 250, 8000), **shape}
    if kind == "permute":
        return {"kind": kind, "dtype": half, "bs": bs, "layers": rng.choice((1, 8, 24)),
                "ctx": _log(rng, 300, 6000), **shape}
    if kind == "attn":
        ctx = _log(rng, 300, 16000)
        return {"kind": kind, "dtype": half, "bs": bs, "ctx": ctx,
                "rows": min(_log(rng, 1, 3000), ctx // 2), **shape}
    if kind == "attn_fp32":
        ctx = _log(rng, 200, 4000)
        return {"kind": "attn", "dtype": "fp32", "bs": bs, "ctx": ctx,
                "rows": max(1, int(ctx * frac)), **shape}
    if kind == "attn_dense":
        return {"kind": kind, "dtype": rng.choice(("bf16", "fp16", "fp32")),
                "ctx": _log(rng, 200, 5000), "frac": frac, **shape}
    if kind == "attn_batch":
        return {"kind": kind, "dtype": half, "bs": bs, "requests": rng.randint(2, 6),
                "ctx": _log(rng, 1000, 16000), "frac": frac, **shape}
    if kind == "projection":
        ctx = _log(rng, 500, 8000)
        return {"kind": kind, "dtype": half, "bs": bs, "ctx": ctx,
                "rows": min(_log(rng, 1, 4000), ctx), **shape}
    if kind == "layer":
        return {"kind": kind, "dtype": half, "bs": bs, "ctx": _log(rng, 500, 14000),
                "frac": frac, **shape}
    heads = rng.choice((4, 8, 14))
    d = rng.choice((64, 128))
    return {"kind": "prefill", "dtype": rng.choice(("bf16", "fp16", "fp32")),
            "layers": rng.choice((1, 8, 24)), "ctx": _log(rng, 100, 2000), "frac": frac,
            "hq": heads, "hkv": heads, "d": d, "hidden": heads * d, "base": 1e6}


# ---- inputs ------------------------------------------------------------------------------

def _recompute(g: torch.Generator, ctx: int, n: int) -> torch.Tensor:
    """n ascending positions: the first tokens, one whole chunk and a uniform scatter, as a
    reuse plan leaves them (host, int32)."""
    mask = torch.zeros(ctx, dtype=torch.bool)
    mask[:min(CHUNK, n // 4)] = True
    if ctx > 4 * CHUNK and n > 2 * CHUNK:
        c = int(torch.randint(1, ctx // CHUNK, (1,), generator=g))
        mask[c * CHUNK:(c + 1) * CHUNK] = True
    rest = (~mask).nonzero().flatten()
    mask[rest[torch.randperm(rest.numel(), generator=g)[:n - int(mask.sum())]]] = True
    return mask.nonzero().flatten().to(torch.int32)


def _rows(case) -> int:
    return max(1, int(round(case["ctx"] * case["frac"])))


def _batch_sizes(case) -> list[tuple[int, int]]:
    """(context, recomputed rows) of each request: contexts and shares rise to the largest."""
    n = case["requests"]
    ctx = [max(64, case["ctx"] * (i + 1) // n) for i in range(n)]
    return [(c, max(1, int(round(c * case["frac"] * (i + 2) / (n + 1)))))
            for i, c in enumerate(ctx)]


class _Maker:
    """Seeded inputs: small index data from a host generator, values on the GPU."""

    def __init__(self, case, seed: int):
        self.host = torch.Generator("cpu").manual_seed(seed)
        self.gpu = torch.Generator("cuda").manual_seed(seed)
        self.dtype = DTYPES[case["dtype"]]
        self.case = case

    def randn(self, *shape, scale: float = 1.0) -> torch.Tensor:
        t = torch.randn(shape, generator=self.gpu, device="cuda", dtype=self.dtype)
        return t if scale == 1.0 else t.mul_(scale)

    def table(self, ctx: int, spare: int = 0) -> tuple[torch.Tensor, int]:
        """(block table, blocks in the pool): the request's pages lie scattered in a pool with
        a quarter more."""
        n = -(-ctx // self.case["bs"])
        pool = n + n // 4 + 4 + spare
        return torch.randperm(pool, generator=self.host)[:n].to(torch.int32).cuda(), pool

    def pairs(self, ctx: int, skip: torch.Tensor | None) -> tuple[torch.Tensor, torch.Tensor]:
        """Chunks of the donor moved to other places of the target, recomputed rows left out."""
        n = ctx // CHUNK
        t = torch.arange(ctx)
        perm = torch.randperm(n, generator=self.host) if n else torch.zeros(0, dtype=torch.long)
        d = t.clone()
        d[:n * CHUNK] = perm.repeat_interleave(CHUNK) * CHUNK + t[:n * CHUNK] % CHUNK
        if skip is not None:
            keep = torch.ones(ctx, dtype=torch.bool)
            keep[skip.long()] = False
            d, t = d[keep], t[keep]
        return d.to(torch.int32), t.to(torch.int32)


def _inputs(case, seed: int) -> dict:
    m, c = _Maker(case, seed), case
    k, ctx, d, hkv, hq = c["kind"], c["ctx"], c["d"], c["hkv"], c["hq"]
    s = {"case": dict(c)}
    if k == "rope_delta":
        s["bt"], nb = m.table(ctx)
        s["cache"] = m.randn(nb, 2, hkv, c["bs"], d)
        pick = torch.randperm(ctx, generator=m.host)[:c["positions"]].sort().values
        s["positions"] = pick.tolist()
        s["delta"] = int(torch.randint(1, 2048, (1,), generator=m.host))
    elif k == "scatter_rope":
        skip = _recompute(m.host, ctx, _rows(c))
        dp, tp = m.pairs(ctx, skip)
        s["bt"], nb = m.table(ctx)
        s["cache"] = m.randn(c["layers"], nb, 2, hkv, c["bs"], d)
        s["donor"] = m.randn(c["layers"], 2, hkv, ctx, d)
        s["dpos"], s["tpos"] = dp.cuda(), tp.cuda()
    elif k == "rope_k":
        delta = torch.randint(-2048, 2049, (ctx // CHUNK + 1,), generator=m.host)
        p = torch.arange(ctx)
        s["k"] = m.randn(c["layers"], hkv, ctx, d)
        s["dpos"] = p.to(torch.int32).cuda()
        s["tpos"] = (p + delta[p // CHUNK]).to(torch.int32).cuda()
    elif k == "permute":
        sp, tp = m.pairs(ctx, None)
        s["bt"], nb = m.table(ctx)
        s["cache"] = m.randn(c["layers"], 2, nb, c["bs"], hkv, d)
        s["pairs"] = list(zip(sp.tolist(), tp.tolist()))
    elif k == "attn":
        pos = _recompute(m.host, ctx, c["rows"])
        s["bt"], nb = m.table(ctx)
        s["cache"] = m.randn(nb, 2, hkv, c["bs"], d)
        s["q"] = m.randn(c["rows"], hq, d, scale=1.5)
        s["pos"] = pos.cuda()
    elif k == "attn_dense":
        mask = torch.zeros(ctx, dtype=torch.bool)
        mask[_recompute(m.host, ctx, _rows(c)).long()] = True
        s["q"] = m.randn(hq, ctx, d, scale=1.5)
        s["k"], s["v"] = m.randn(hq, ctx, d), m.randn(hq, ctx, d)
        s["mask"] = mask.cuda()
    elif k == "attn_batch":
        sizes = _batch_sizes(c)
        s["rows"] = [r for _, r in sizes]
        s["blocks"] = [-(-x // c["bs"]) for x, _ in sizes]
        pool = sum(s["blocks"]) + 8
        perm = torch.randperm(pool, generator=m.host).to(torch.int32)
        tables = torch.full((len(sizes), max(s["blocks"])), -1, dtype=torch.int32)
        at = 0
        for i, b in enumerate(s["blocks"]):
            tables[i, :b] = perm[at:at + b]
            at += b
        s["bt"] = tables.cuda()
        s["cache"] = m.randn(pool, 2, hkv, c["bs"], d)
        s["pos"] = torch.cat([_recompute(m.host, x, r) for x, r in sizes]).cuda()
        s["q"] = m.randn(sum(s["rows"]), hq, d, scale=1.5)
    elif k in ("projection", "layer"):
        rows = c["rows"] if k == "projection" else _rows(c)
        pos = _recompute(m.host, ctx, rows)
        feats = (hq + 2 * hkv) * d
        s["bt"], nb = m.table(ctx)
        s["cache"] = m.randn(nb, 2, hkv, c["bs"], d)
        s["x"] = m.randn(ctx, c["hidden"])
        s["w"] = m.randn(feats, c["hidden"], scale=c["hidden"] ** -0.5)
        s["b"] = m.randn(feats, scale=0.1)
        s["pos"], s["pos_host"] = pos.cuda(), pos
        if k == "layer":
            s["wo"] = m.randn(c["hidden"], hq * d, scale=(hq * d) ** -0.5)
    else:
        f = hq * d
        skip = _recompute(m.host, ctx, _rows(c))
        dp, tp = m.pairs(ctx, skip)
        mask = torch.zeros(ctx, dtype=torch.bool)
        mask[skip.long()] = True
        s["x"] = m.randn(ctx, c["hidden"])
        s["donor"] = m.randn(c["layers"], 2, hq, ctx, d)
        s["w"] = m.randn(3 * f, c["hidden"], scale=c["hidden"] ** -0.5)
        s["b"] = m.randn(3 * f, scale=0.1)
        s["wo"] = m.randn(c["hidden"], f, scale=f ** -0.5)
        s["dpos"], s["tpos"], s["mask"] = dp.cuda(), tp.cuda(), mask.cuda()
    return s


def prepare(case, seed: int) -> dict:
    s = _inputs(case, seed)
    c = s["case"]
    if c["kind"] == "scatter_rope":
        s["caches"], s["donors"] = list(s["cache"]), list(s["donor"])
    elif c["kind"] == "permute":
        s["caches"] = list(s["cache"])
    elif c["kind"] == "layer":
        # made once per request, used by every layer of it
        s["plan"] = tk.plan_partial_attention_paged(
            s["pos_host"], c["hq"], c["hkv"], c["d"], c["bs"], s["bt"].shape[0],
            DTYPES[c["dtype"]], torch.device("cuda", torch.cuda.current_device()))
    return s


def run(s):
    c = s["case"]
    k = c["kind"]
    if k == "rope_delta":
        n = rc.apply_rope_delta_inplace(s["cache"], s["bt"], s["positions"], s["delta"],
                                        rope_base=c["base"])
        return {"cache": s["cache"], "count": n}
    if k == "scatter_rope":
        if c["layers"] == 1:
            rc.rope_correct_scatter_paged(s["caches"][0], s["donors"][0], s["bt"], s["dpos"],
                                          s["tpos"], rope_base=c["base"])
        else:
            rc.rope_correct_scatter_paged_layers(s["caches"], s["donors"], s["bt"], s["dpos"],
                                                 s["tpos"], rope_base=c["base"])
        return s["cache"]
    if k == "rope_k":
        return rc.rope_correct_k(s["k"], s["dpos"], s["tpos"], head_dim=c["d"],
                                 rope_base=c["base"])
    if k == "permute":
        rc.permute_paged_kv_with_rope_layers(s["caches"], s["bt"], s["pairs"],
                                             rope_base=c["base"], layout="vllm")
        return s["cache"]
    if k == "attn":
        return tk.partial_prefill_attention_paged(s["q"], s["cache"], s["bt"], s["pos"])
    if k == "attn_dense":
        return tk.partial_prefill_attention(s["q"], s["k"], s["v"], s["mask"])
    if k == "attn_batch":
        return tk.partial_prefill_attention_paged_varlen(
            s["q"], s["cache"], s["bt"], s["pos"], s["rows"], s["blocks"])
    if k == "projection":
        q = tk.qkv_projection_paged(s["x"], s["w"], s["pos"], s["cache"], s["bt"], c["hq"],
                                    c["hkv"], c["d"], qkv_bias=s["b"], rope_base=c["base"])
        return {"q": q, "cache": s["cache"]}
    if k == "layer":
        r = tk.partial_prefill_layer_paged(
            s["x"], s["w"], s["wo"], s["pos"], s["cache"], s["bt"], c["hq"], c["hkv"], c["d"],
            qkv_bias=s["b"], rope_base=c["base"], plan=s["plan"])
        return {"output": r.output, "query": r.query, "attention": r.attention,
                "cache": s["cache"]}
    r = tk.partial_prefill(s["x"], s["donor"], s["w"], s["wo"], s["dpos"], s["tpos"],
                           s["mask"], c["hq"], c["d"], qkv_bias=s["b"])
    return {"output": r.output, "cache": r.kv_cache, "computed": r.positions_computed}


# ---- work --------------------------------------------------------------------------------

def _keys(case, ctx: int, rows: int) -> float:
    """Keys that `rows` recomputed positions of a `ctx`-token request attend to, about: the
    first quarter of them (up to a chunk) are the first tokens, the rest uniform."""
    head = min(CHUNK, rows // 4)
    return head * (head + 1) / 2 + (rows - head) * (head + ctx) / 2


def work(case) -> dict:
    c = case
    k, ctx, d, hkv, hq = c["kind"], c["ctx"], c["d"], c["hkv"], c["hq"]
    es = 4 if c["dtype"] == "fp32" else 2
    row = d * es
    if k == "rope_delta":
        return {"bytes": 2 * c["positions"] * hkv * row, "flops": 3 * c["positions"] * hkv * d}
    if k == "scatter_rope":
        n = (ctx - _rows(c)) * c["layers"] * hkv
        return {"bytes": 2 * 2 * n * row, "flops": 3 * n * d}
    if k == "rope_k":
        n = c["layers"] * hkv * ctx
        return {"bytes": 2 * n * row, "flops": 3 * n * d}
    if k == "permute":
        n = c["layers"] * hkv * ctx
        return {"bytes": 2 * 2 * n * row, "flops": 3 * n * d}
    if k == "attn":
        return {"bytes": 2 * c["rows"] * hq * row + 2 * ctx * hkv * row,
                "flops": 4 * d * hq * _keys(c, ctx, c["rows"])}
    if k == "attn_dense":
        r = _rows(c)
        return {"bytes": hq * row * (r + 2 * ctx + ctx), "flops": 4 * d * hq * _keys(c, ctx, r)}
    if k == "attn_batch":
        z = _batch_sizes(c)
        return {"bytes": sum(2 * r * hq * row + 2 * x * hkv * row for x, r in z),
                "flops": sum(4 * d * hq * _keys(c, x, r) for x, r in z)}
    feats = (hq + 2 * hkv) * d
    if k == "projection":
        r = c["rows"]
        return {"bytes": es * (r * c["hidden"] + feats * c["hidden"] + r * feats),
                "flops": 2 * r * feats * c["hidden"]}
    if k == "layer":
        r, f = _rows(c), hq * d
        return {"bytes": es * (r * c["hidden"] + feats * c["hidden"] + r * feats
                               + 2 * ctx * hkv * d + r * f + f * c["hidden"]
                               + r * c["hidden"]),
                "flops": 2 * r * feats * c["hidden"] + 4 * d * hq * _keys(c, ctx, r)
                + 2 * r * f * c["hidden"]}
    r, f = _rows(c), hq * d
    donor = c["layers"] * 2 * (ctx - r) * f        # donor rows read
    cache = c["layers"] * 2 * ctx * f              # assembled cache written
    return {"bytes": es * (r * c["hidden"] + 4 * f * c["hidden"] + donor + cache
                           + ctx * c["hidden"]),
            "flops": 8 * r * f * c["hidden"] + 4 * d * hq * _keys(c, ctx, r)}


def tolerance(case):
    """About four times the difference seen between the path and 64 bits (which for 16-bit
    outputs is the final rounding, and for attention also the 16-bit weights of P)."""
    k, t = case["kind"], case["dtype"]
    if k in ("rope_delta", "scatter_rope", "rope_k", "permute"):
        # rotated values are rounded once; moved ones are the same bits
        return {"fp32": {"rel": 1e-6, "max": 1e-5}, "fp16": {"rel": 1e-3, "max": 2e-3},
                "bf16": {"rel": 7e-3, "max": 1.6e-2}}[t]
    if k == "projection":
        return {"fp16": {"rel": 1e-3, "max": 2e-3}, "bf16": {"rel": 7e-3, "max": 1.6e-2}}[t]
    if t == "fp32":  # sums in another order; the orchestrator chains three of them
        return {"rel": 5e-6 if k == "prefill" else 2e-6, "max": 1e-4}
    return {"fp16": {"rel": 1.5e-3, "max": 1e-2}, "bf16": {"rel": 1e-2, "max": 5e-2}}[t]


# ---- the same in 64 bits -------------------------------------------------------------------

def _rotate(x: torch.Tensor, delta: torch.Tensor, base: float) -> torch.Tensor:
    """Interleaved pairs of x [..., P, D] (64 bits) rotated by delta [P] positions. The angle is
    the path's definition, the fp32 product of the delta and the fp32 inverse frequency."""
    d = x.shape[-1]
    inv = (1.0 / (base ** (torch.arange(0, d, 2, dtype=torch.float32) / d))).to(x.device)
    th = (delta.to(torch.float32)[:, None] * inv).double()
    c, sn = th.cos(), th.sin()
    e, o = x[..., 0::2], x[..., 1::2]
    return torch.stack([e * c - o * sn, e * sn + o * c], dim=-1).flatten(-2)


def _slots(bt: torch.Tensor, pos: torch.Tensor, bs: int):
    p = pos.long()
    return bt.long()[p // bs], p % bs


def _paged(cache64: torch.Tensor, bt: torch.Tensor, ctx: int) -> torch.Tensor:
    """[2, H, ctx, D] of one request from a [NB, 2, H, bs, D] cache."""
    x = cache64[bt.long()].permute(1, 2, 0, 3, 4)
    return x.reshape(2, x.shape[1], -1, x.shape[-1])[:, :, :ctx]


def _attend(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, pos: torch.Tensor) -> torch.Tensor:
    """q [R, Hq, D], k / v [Hkv, S, D], all 64 bits; row r attends to keys 0..pos[r]."""
    r, hq, d = q.shape
    group = hq // k.shape[0]
    out = torch.empty_like(q)
    step = max(1, int(2e8) // k.shape[1])  # at most 1.6 GB of scores at a time
    keys = torch.arange(k.shape[1], device=q.device)
    for h in range(hq):
        kt, vv = k[h // group].t().contiguous(), v[h // group]
        for a in range(0, r, step):
            sc = (q[a:a + step, h] @ kt) / math.sqrt(d)
            sc.masked_fill_(keys[None] > pos[a:a + step, None].long(), -math.inf)
            out[a:a + step, h] = torch.softmax(sc, dim=-1) @ vv
    return out


def exact(case, seed: int):
    s = _inputs(case, seed)
    c = s["case"]
    k, bs, ctx, d, hq, hkv = c["kind"], c.get("bs"), c["ctx"], c["d"], c["hq"], c["hkv"]
    dt = DTYPES[c["dtype"]]
    if k == "rope_delta":
        cache = s["cache"].double()
        p = torch.tensor(s["positions"], device="cuda")
        b, o = _slots(s["bt"], p, bs)
        rows = cache[b, 0, :, o].transpose(0, 1)
        turn = torch.full((p.numel(),), s["delta"], device="cuda")
        cache[b, 0, :, o] = _rotate(rows, turn, c["base"]).transpose(0, 1)
        return {"cache": cache, "count": p.numel()}
    if k == "scatter_rope":
        cache = s["cache"].double()
        b, o = _slots(s["bt"], s["tpos"], bs)
        dl, turn = s["dpos"].long(), s["tpos"] - s["dpos"]
        for i in range(c["layers"]):
            kv = s["donor"][i][:, :, dl].double()
            cache[i][b, 0, :, o] = _rotate(kv[0], turn, c["base"]).transpose(0, 1)
            cache[i][b, 1, :, o] = kv[1].transpose(0, 1)
        return cache
    if k == "rope_k":
        return _rotate(s["k"].double(), s["tpos"] - s["dpos"], c["base"])
    if k == "permute":
        cache = s["cache"].double()
        pr = torch.tensor(s["pairs"], device="cuda")
        (sb, so), (tb, to) = _slots(s["bt"], pr[:, 0], bs), _slots(s["bt"], pr[:, 1], bs)
        for i in range(c["layers"]):
            kv = cache[i][:, sb, so]  # [2, P, H, D]
            turned = _rotate(kv[0].transpose(0, 1), pr[:, 1] - pr[:, 0], c["base"])
            cache[i][0, tb, to] = turned.transpose(0, 1)
            cache[i][1, tb, to] = kv[1]
        return cache
    if k == "attn":
        kk, vv = _paged(s["cache"].double(), s["bt"], ctx)
        return _attend(s["q"].double(), kk, vv, s["pos"])
    if k == "attn_dense":
        pos = s["mask"].nonzero().flatten()
        out = torch.zeros(s["q"].shape, dtype=torch.float64, device="cuda")
        q = s["q"][:, pos].double().transpose(0, 1).contiguous()
        out[:, pos] = _attend(q, s["k"].double(), s["v"].double(), pos).transpose(0, 1)
        return out
    if k == "attn_batch":
        out, at = [], 0
        cache = s["cache"].double()
        for i, (x, r) in enumerate(_batch_sizes(c)):
            kk, vv = _paged(cache, s["bt"][i, :s["blocks"][i]], x)
            out.append(_attend(s["q"][at:at + r].double(), kk, vv, s["pos"][at:at + r]))
            at += r
        return torch.cat(out)
    if k in ("projection", "layer"):
        pos = s["pos"].long()
        y = s["x"][pos].double() @ s["w"].double().t().contiguous() + s["b"].double()
        r, kf = pos.numel(), hq * d
        q = _rotate(y[:, :kf].view(r, hq, d).transpose(0, 1), pos, c["base"]).transpose(0, 1)
        nk = _rotate(y[:, kf:kf + hkv * d].view(r, hkv, d).transpose(0, 1), pos,
                     c["base"]).transpose(0, 1)
        nv = y[:, kf + hkv * d:].view(r, hkv, d)
        cache = s["cache"].double()
        b, o = _slots(s["bt"], pos, bs)
        cache[b, 0, :, o], cache[b, 1, :, o] = nk, nv
        if k == "projection":
            return {"q": q.contiguous(), "cache": cache}
        # the attention reads Q, K and V as stored, in the cache's type
        kk, vv = _paged(cache.to(dt).double(), s["bt"], ctx)
        at = _attend(q.to(dt).double().contiguous(), kk, vv, s["pos"])
        out = at.to(dt).double().reshape(r, kf) @ s["wo"].double().t().contiguous()
        return {"output": out, "query": q.contiguous(), "attention": at, "cache": cache}
    f = hq * d
    pos = s["mask"].nonzero().flatten()
    y = s["x"][pos].double() @ s["w"].double().t().contiguous() + s["b"].double()
    qkv = y.to(dt).double().view(-1, 3, hq, d).permute(1, 2, 0, 3)  # stored in the input type
    cache = torch.zeros(s["donor"].shape, dtype=torch.float64, device="cuda")
    cache[:, :, :, s["tpos"].long()] = s["donor"][:, :, :, s["dpos"].long()].double()
    cache[:, 0][:, :, pos] = qkv[1][None]
    cache[:, 1][:, :, pos] = qkv[2][None]
    at = _attend(qkv[0].transpose(0, 1).contiguous(), cache[0, 0], cache[0, 1], pos)
    out = torch.zeros((ctx, c["hidden"]), dtype=torch.float64, device="cuda")
    out[pos] = at.reshape(-1, f) @ s["wo"].double().t().contiguous()
    return {"output": out, "cache": cache, "computed": int(pos.numel())}
