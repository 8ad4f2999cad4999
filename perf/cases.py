"""Performance cases of the KV-cache path: what a serving or prefill program asks of it.

Each case names an operation (``op``) and plain sizes.  ``listed()`` holds the fixed ones,
``draw()`` more of the same ranges.  ``prepare`` makes a program's state on the GPU (inputs of
the seed, caches, block tables, output buffers), ``run`` is one pass through the package's public
functions, ``exact`` the same outputs in 64-bit torch.

The operations and their ranges:

* ``quant``: quant_to_paged_cache, one decode step (a token per sequence, random slots, some
  padding) up to a 32768-token prefill chunk (runs of consecutive slots); int8 and
  float8_e4m3fn pages, head sizes 64 to 256, K/V contiguous or views into a fused qkv tensor.
* ``smooth``: moe_quantize, dense activations or rows gathered by a top-2 expert choice with one
  smooth row per expert; hidden sizes 1024 to 16384.
* ``rope``: fused_rmsnorm_rope_store_paged_cache / fused_rope (layernorm) into int8 or
  unquantised pages, decode steps and prefill chunks.
* ``dequant``: dequant_from_paged_cache of every sequence's context.
* ``attn``: single_query_cached_kv_attn, one query token per sequence (decode) or a ragged chunk
  of them (cu_seq_q), over int8, float8_e4m3fn, int4 or unquantised pages, grouped heads or one
  latent KV head whose rows hold keys and values.
* ``linear``: quant_to_linear_cache of packed prompts, then dequant_from_linear_cache.
"""
import math

import torch

import domesticated_torch_mlu_ops_amd as tmo

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
CACHES = {"int8": torch.int8, "fp8": torch.float8_e4m3fn}
TOP_K = 2                      # experts per token of the gathered smooth quantisation


def listed():
    return [
        # one decode step of 16 sequences: the smallest call, launch and host latency
        quant("quant_decode_step", tokens=16, runs=0, heads=8, dim=128, block=16),
        # a 32768-token prefill chunk of 8 sequences, 8 KV heads x 128: the headline workload
        quant("quant_prefill", tokens=32768, runs=8, heads=8, dim=128, block=16),
        # an odd chunk with head size 96 read in place from the projection's fused qkv output
        quant("quant_qkv_view_d96", tokens=9973, runs=5, heads=8, dim=96, block=16, dtype="f16",
              cache="fp8", fused=True),
        # activations in front of an int8 GEMM, hidden size 4096
        smooth("smooth_dense", rows=8192, channels=4096),
        # mixture-of-experts dispatch: 4099 tokens, each to 2 of 64 experts, hidden size 7168
        smooth("smooth_moe_7168", rows=4099, channels=7168, experts=64),
        # prefill of 8 x 4096 tokens, 32 query and 8 KV heads: norm, rotation, int8 store
        rope("rope_prefill", batch=8, seq=4096, heads=32, kv_heads=8, dim=128),
        # gathering 64 contexts of 1K..32K tokens back to bf16
        dequant("dequant_64_seqs", batch=64, ctx_lo=1024, ctx_hi=32768, heads=8, dim=128),
        # decode over the same 64 contexts in int8 pages, 32 query heads
        attn("attn_decode_int8", batch=64, ctx_lo=1024, ctx_hi=32768, heads=32, kv_heads=8,
             dim=128, kv="int8"),
        # an interactive decode step: 8 short contexts in bf16 pages
        attn("attn_decode_small", batch=8, ctx_lo=128, ctx_hi=4096, heads=32, kv_heads=8,
             dim=128, kv="same"),
        # latent-attention decode: one KV head of 576 channels, values its first 512
        attn("attn_decode_latent", batch=32, ctx_lo=512, ctx_hi=8192, heads=16, kv_heads=1,
             dim=576, dim_v=512, kv="same", lse=True),
        # chunked prefill: up to 512 new tokens of each of 8 sequences over int8 pages
        attn("attn_chunk_int8", batch=8, q_tokens=512, ctx_lo=512, ctx_hi=8192, heads=32,
             kv_heads=8, dim=128, kv="int8"),
        # prompts into linear int8 caches and back, head size 80
        linear("linear_d80", batch=12, seq=1531, heads=8, dim=80, dtype="f16"),
    ]


# ------------------------------------------------------------------------------ case makers


def quant(name=None, tokens=16, runs=0, heads=8, dim=128, block=16, dtype="bf16", cache="int8",
          fused=False):
    """`runs` 0: a decode step (random slots, a tenth of them padding); else the number of
    sequences whose consecutive slots the tokens fill."""
    return _named(name, op="quant", tokens=tokens, runs=runs, heads=heads, dim=dim, block=block,
                  dtype=dtype, cache=cache, fused=fused)


def smooth(name=None, rows=8192, channels=4096, experts=0, dtype="bf16"):
    return _named(name, op="smooth", rows=rows, channels=channels, experts=experts, dtype=dtype)


def rope(name=None, batch=8, seq=4096, heads=32, kv_heads=8, dim=128, dtype="bf16",
         store="int8", norm="rmsnorm"):
    return _named(name, op="rope", batch=batch, seq=seq, heads=heads, kv_heads=kv_heads, dim=dim,
                  dtype=dtype, store=store, norm=norm)


def dequant(name=None, batch=64, ctx_lo=1024, ctx_hi=32768, heads=8, dim=128, block=16,
            dtype="bf16", cache="int8"):
    return _named(name, op="dequant", batch=batch, ctx_lo=ctx_lo, ctx_hi=ctx_hi, heads=heads,
                  dim=dim, block=block, dtype=dtype, cache=cache)


def attn(name=None, batch=64, q_tokens=1, ctx_lo=1024, ctx_hi=32768, heads=32, kv_heads=8,
         dim=128, dim_v=0, block=16, dtype="bf16", kv="int8", lse=False):
    """`dim_v` 0: separate K and V caches of `dim`; else one cache whose rows hold both."""
    return _named(name, op="attn", batch=batch, q_tokens=q_tokens, ctx_lo=ctx_lo, ctx_hi=ctx_hi,
                  heads=heads, kv_heads=kv_heads, dim=dim, dim_v=dim_v, block=block, dtype=dtype,
                  kv=kv, lse=lse)


def linear(name=None, batch=12, seq=1531, heads=8, dim=80, dtype="f16", bits=8):
    return _named(name, op="linear", batch=batch, seq=seq, heads=heads, dim=dim, dtype=dtype,
                  bits=bits)


def _named(name, **case):
    return case if name is None else dict(case, name=name)


def _spread(rng, lo, hi):
    """A whole number in [lo, hi], uniform in its logarithm."""
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    op = rng.choice(["quant", "quant", "smooth", "smooth", "rope", "dequant", "attn", "attn",
                     "attn", "attn", "linear"])
    dtype = rng.choice(["bf16", "bf16", "f16"])
    dim = rng.choice([64, 80, 96, 128, 128, 128, 256])
    if op == "quant":
        decode = rng.random() < 0.5
        tokens = _spread(rng, 1, 512) if decode else _spread(rng, 256, 32768)
        return quant(tokens=tokens, runs=0 if decode else rng.randint(1, 8),
                     heads=rng.choice([1, 2, 4, 8]), dim=dim, block=rng.choice([16, 16, 32, 64]),
                     dtype=dtype, cache=rng.choice(["int8", "int8", "fp8"]),
                     fused=rng.random() < 0.5)
    if op == "smooth":
        return smooth(rows=_spread(rng, 1, 8192),
                      channels=rng.choice([1024, 2048, 3584, 4096, 5120, 7168, 8192, 14336, 16384]),
                      experts=rng.choice([0, 0, 8, 64]), dtype=dtype)
    if op == "rope":
        decode = rng.random() < 0.5
        kv_heads = rng.choice([1, 2, 4, 8])
        return rope(batch=_spread(rng, 1, 256) if decode else rng.randint(1, 4),
                    seq=1 if decode else _spread(rng, 64, 4096),
                    heads=kv_heads * rng.choice([1, 4, 8]), kv_heads=kv_heads, dim=dim,
                    dtype=dtype, store=rng.choice(["int8", "int8", "same"]),
                    norm=rng.choice(["rmsnorm", "rmsnorm", "layernorm"]))
    if op == "dequant":
        hi = _spread(rng, 128, 8192 if dim > 128 else 16384)
        return dequant(batch=_spread(rng, 1, 64), ctx_lo=max(1, hi // 8), ctx_hi=hi,
                       heads=rng.choice([1, 2, 4, 8]), dim=dim, block=rng.choice([16, 16, 32, 64]),
                       dtype=dtype, cache=rng.choice(["int8", "int8", "fp8"]))
    if op == "linear":
        return linear(batch=_spread(rng, 1, 32), seq=_spread(rng, 16, 4096),
                      heads=rng.choice([1, 2, 4, 8]), dim=dim, dtype=dtype,
                      bits=rng.choice([8, 8, 4]))
    lse = rng.random() < 0.3
    form = rng.choice(["decode", "decode", "latent", "chunk"])
    if form == "latent":
        hi = _spread(rng, 256, 8192)
        return attn(batch=_spread(rng, 1, 32), ctx_lo=max(1, hi // 8), ctx_hi=hi,
                    heads=rng.choice([16, 16, 32, 64]), kv_heads=1, dim=576, dim_v=512,
                    block=rng.choice([16, 16, 64]), dtype=dtype, kv="same", lse=lse)
    kv = rng.choice(["same", "int8", "int8", "fp8", "int4"])
    kv_heads = rng.choice([1, 2, 4, 8])
    heads = kv_heads * rng.choice([1, 4, 8])
    block = rng.choice([16, 16, 32, 64])
    if form == "decode":
        hi = _spread(rng, 128, 16384)
        return attn(batch=_spread(rng, 1, 64), ctx_lo=max(1, hi // 8), ctx_hi=hi, heads=heads,
                    kv_heads=kv_heads, dim=dim, block=block, dtype=dtype, kv=kv, lse=lse)
    hi = _spread(rng, 128, 4096)
    return attn(batch=_spread(rng, 1, 8), q_tokens=_spread(rng, 2, min(256, hi // 2)),
                ctx_lo=max(1, hi // 8), ctx_hi=hi, heads=heads, kv_heads=kv_heads, dim=dim,
                block=block, dtype=dtype, kv=kv, lse=lse)


# ------------------------------------------------------------------------------ inputs


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _contexts(case):
    """Context lengths in [ctx_lo, ctx_hi], the longest present: the case's own, so that outputs
    of every seed have one shape."""
    g = torch.Generator().manual_seed(case["batch"] + case["ctx_hi"])
    ctx = torch.randint(case["ctx_lo"], case["ctx_hi"] + 1, (case["batch"],), generator=g)
    ctx[0] = case["ctx_hi"]
    return ctx.to(torch.int32)


def _counts(case, ctx):
    """New query tokens per sequence: up to q_tokens, never more than its context."""
    g = torch.Generator().manual_seed(case["batch"] + case["q_tokens"])
    n = torch.randint(max(1, case["q_tokens"] // 2), case["q_tokens"] + 1, (case["batch"],),
                      generator=g).to(torch.int32)
    n[0] = case["q_tokens"]
    return torch.minimum(n, ctx.to(torch.int32))


def _pages(ctx, block, seed):
    """A pool with a quarter more pages than the contexts need, each sequence's pages a random
    choice of them: (block_tables, pages in the pool)."""
    per = (int(ctx.max()) + block - 1) // block
    need = int(((ctx + block - 1) // block).sum())
    pool = need + need // 4 + 1
    g = torch.Generator().manual_seed(seed + 2)
    order = torch.randperm(pool, generator=g).to(torch.int32)
    table = torch.zeros(len(ctx), per, dtype=torch.int32)
    at = 0
    for i, n in enumerate(((ctx + block - 1) // block).tolist()):
        table[i, :n] = order[at:at + n]
        at += n
    return table.cuda(), pool


def _outlier_rows(shape, g, dtype):
    """Rows as projections give them: N(0, 1) with one channel per head twenty times larger."""
    x = torch.randn(shape, generator=g, device="cuda")
    ch = torch.randint(0, shape[-1], (shape[-2],), generator=g, device="cuda")
    x[:, torch.arange(shape[-2], device="cuda"), ch] *= 20.0
    return x.to(dtype)


def _codes(pages, heads, block, dim, kv, g):
    """Quantised pages and per-token scales: rows quantised as quant_to_paged_cache does, a base
    of at most 2048 pages repeated over the pool."""
    base = min(pages, 2048)
    x = _outlier_rows((base * block, heads, dim), g, torch.bfloat16).float()
    x = x.view(base, block, heads, dim).transpose(1, 2).contiguous()
    top = {"int8": 127.0, "fp8": 448.0, "int4": 7.0}[kv]
    scale = x.abs().amax(-1) / top
    q = x / scale[..., None]
    c = q.clamp(-448, 448).to(torch.float8_e4m3fn).view(torch.int8) if kv == "fp8" \
        else q.round().clamp(-top - 1, top).to(torch.int8)
    reps = (pages + base - 1) // base
    c = c.repeat(reps, 1, 1, 1)[:pages]
    return (c.view(torch.float8_e4m3fn) if kv == "fp8" else c), scale.repeat(reps, 1, 1)[:pages].contiguous()


def _pack4(c, dim):
    """int4 codes to bytes of pairs along `dim`, the even element in the high nibble."""
    hi, lo = c.unflatten(dim, (-1, 2)).unbind(dim + 1)
    return ((hi << 4) | (lo & 15)).contiguous()


def prepare(case, seed):
    return globals()["_prepare_" + case["op"]](case, seed)


def _prepare_quant(case, seed):
    g, T, H, D = _gen(seed), case["tokens"], case["heads"], case["dim"]
    dtype, BS = DTYPES[case["dtype"]], case["block"]
    if case["fused"]:  # [T, 4 H query + H key + H value heads, D]
        qkv = _outlier_rows((T, 6 * H, D), g, dtype)
        k, v = qkv[:, 4 * H:5 * H], qkv[:, 5 * H:]
    else:
        k, v = _outlier_rows((T, H, D), g, dtype), _outlier_rows((T, H, D), g, dtype)
    hg = torch.Generator().manual_seed(seed)
    if case["runs"]:
        per = (T + case["runs"] - 1) // case["runs"]
        blocks = (per + BS - 1) // BS
        pool = 2 * case["runs"]
        start = torch.randperm(pool, generator=hg)[:case["runs"]] * blocks * BS
        slot = (start[:, None] + torch.arange(per)).reshape(-1)[:T]
        pool *= blocks
    else:
        pool = max(64, 2 * T)
        slot = torch.randperm(pool * BS, generator=hg)[:T]
        slot[torch.randperm(T, generator=hg)[:T // 10]] = -1
    cache = torch.zeros(2, pool, H, BS, D, dtype=torch.int8, device="cuda")
    cache = cache.view(CACHES[case["cache"]])
    scale = torch.zeros(2, pool, H, BS, device="cuda")
    return dict(op="quant", k=k, v=v, kc=cache[0], vc=cache[1], ks=scale[0], vs=scale[1],
                slot=slot.to(torch.int32).cuda())


def _prepare_smooth(case, seed):
    g, T, C, E = _gen(seed), case["rows"], case["channels"], case["experts"]
    x = torch.randn(T, C, generator=g, device="cuda")
    ch = torch.randperm(C, generator=g, device="cuda")[:C // 100]
    x[:, ch] = torch.randn(T, len(ch), generator=g, device="cuda") / torch.sqrt(
        torch.randn(T, len(ch), 3, generator=g, device="cuda").pow(2).mean(-1))  # Student t, 3
    s = dict(op="smooth", x=x.to(DTYPES[case["dtype"]]), count=None, gather=None)
    s["smooth"] = 0.5 + 1.5 * torch.rand((E, C) if E else (C,), generator=g, device="cuda")
    if E:
        chosen = torch.randn(T, E, generator=g, device="cuda").topk(TOP_K, dim=-1).indices.reshape(-1)
        s["gather"] = (torch.sort(chosen, stable=True).indices // TOP_K).to(torch.int32)
        s["count"] = torch.bincount(chosen, minlength=E).to(torch.int32)
    return s


def _prepare_rope(case, seed):
    g, B, S, D = _gen(seed), case["batch"], case["seq"], case["dim"]
    Hq, Hk, dtype, BS = case["heads"], case["kv_heads"], DTYPES[case["dtype"]], 16
    qkv = torch.randn(B, S, Hq + 2 * Hk, D, generator=g, device="cuda").to(dtype)
    rows = 8192
    freq = 10000.0 ** (-torch.arange(0, D, 2, device="cuda") / D)
    ang = torch.arange(rows, device="cuda")[:, None] * torch.cat([freq, freq])[None]
    hg = torch.Generator().manual_seed(seed)
    pos = torch.randint(0, rows - S + 1, (B,), generator=hg).to(torch.int32).cuda()
    per = (S + BS - 1) // BS
    first = torch.randperm(2 * B, generator=hg)[:B] * per * BS
    slot = (first[:, None] + torch.arange(S)).reshape(-1).to(torch.int32).cuda()
    int8 = case["store"] == "int8"
    kc = torch.zeros(2 * B * per, Hk, BS, D, dtype=torch.int8 if int8 else dtype, device="cuda")
    ks = torch.zeros(kc.shape[:3], device="cuda") if int8 else None
    gamma = (0.5 + torch.rand(3, D, generator=g, device="cuda")).to(dtype)
    return dict(op="rope", qkv=qkv, kc=kc, vc=kc.clone(), ks=ks,
                vs=ks.clone() if int8 else None, sin=ang.sin().to(dtype), cos=ang.cos().to(dtype),
                pos=pos, slot=slot, gamma=gamma, norm=case["norm"])


def _prepare_dequant(case, seed):
    g, H, D = _gen(seed), case["heads"], case["dim"]
    ctx = _contexts(case)
    table, pool = _pages(ctx, case["block"], seed)
    kc, ks = _codes(pool, H, case["block"], D, case["cache"], g)
    vc, vs = _codes(pool, H, case["block"], D, case["cache"], g)
    out = torch.empty(2, int(ctx.sum()), H, D, dtype=DTYPES[case["dtype"]], device="cuda")
    return dict(op="dequant", kc=kc, vc=vc, ks=ks, vs=vs, table=table, ctx=ctx.cuda(),
                longest=int(ctx.max()), key=out[0], value=out[1])


def _prepare_attn(case, seed):
    g, D, Hkv, BS = _gen(seed), case["dim"], case["kv_heads"], case["block"]
    dtype, kv = DTYPES[case["dtype"]], case["kv"]
    ctx = _contexts(case)
    table, pool = _pages(ctx, BS, seed)
    s = dict(op="attn", table=table, ctx=ctx.cuda(), longest=int(ctx.max()), ks=None, vs=None,
             vc=None, cu=None, bits={"same": -1, "int8": 8, "fp8": 8, "int4": 4}[kv],
             lse=case["lse"], max_q=case["q_tokens"], scale=D ** -0.5)
    if kv == "same":
        s["kc"] = torch.randn(pool, Hkv, BS, D, generator=g, device="cuda", dtype=dtype)
        if not case["dim_v"]:
            s["vc"] = torch.randn(pool, Hkv, BS, D, generator=g, device="cuda", dtype=dtype)
    else:
        s["kc"], s["ks"] = _codes(pool, Hkv, BS, D, kv, g)
        s["vc"], s["vs"] = _codes(pool, Hkv, BS, D, kv, g)
        if kv == "int4":
            s["kc"], s["vc"] = _pack4(s["kc"], 3), _pack4(s["vc"], 2)
    if case["q_tokens"] == 1:
        shape = (case["batch"], 1, case["heads"], D)
    else:
        n = _counts(case, ctx)
        s["cu"] = torch.cat([torch.zeros(1, dtype=torch.int32), n.cumsum(0).to(torch.int32)]).cuda()
        shape = (int(n.sum()), case["heads"], D)
    s["q"] = torch.randn(shape, generator=g, device="cuda").to(dtype)
    s["out"] = torch.empty(shape[:-1] + (case["dim_v"] or D,), dtype=dtype, device="cuda")
    return s


def _lengths(case):
    """Prompt lengths, the case's own as the context lengths are."""
    g = torch.Generator().manual_seed(case["batch"] + case["seq"])
    n = torch.randint(max(1, case["seq"] // 2), case["seq"] + 1, (case["batch"],), generator=g)
    n[0] = case["seq"]
    return n.to(torch.int32)


def _prepare_linear(case, seed):
    g, B, H, D = _gen(seed), case["batch"], case["heads"], case["dim"]
    n = _lengths(case)
    T, L, dtype = int(n.sum()), (case["seq"] + 63) // 64 * 64, DTYPES[case["dtype"]]
    four = case["bits"] == 4
    kc = torch.zeros(B, H, L, D // 2 if four else D, dtype=torch.int8, device="cuda")
    vc = torch.zeros(B, H, L // 2 if four else L, D, dtype=torch.int8, device="cuda")
    ks = torch.zeros(B, H, L, device="cuda")
    cu = torch.cat([torch.zeros(1, dtype=torch.int32), n.cumsum(0).to(torch.int32)])
    return dict(op="linear", k=_outlier_rows((T, H, D), g, dtype), v=_outlier_rows((T, H, D), g, dtype),
                kc=kc, vc=vc, ks=ks, vs=ks.clone(), cu=cu.cuda(), n=n.cuda(), longest=case["seq"],
                bits=case["bits"], key=torch.empty(T, H, D, dtype=dtype, device="cuda"),
                value=torch.empty(T, H, D, dtype=dtype, device="cuda"))


# ------------------------------------------------------------------------------ one pass


def run(s):
    op = s["op"]
    if op == "quant":
        return tmo.quant_to_paged_cache(s["k"], s["v"], s["kc"], s["vc"], s["ks"], s["vs"], s["slot"])
    if op == "smooth":
        return tmo.moe_quantize(s["x"], s["smooth"], None, s["count"], s["gather"])
    if op == "rope":
        g = s["gamma"]
        if s["norm"] == "layernorm":
            tmo.fused_rope(s["qkv"], s["kc"], s["vc"], s["sin"], s["cos"], s["pos"], g[0], g[2],
                           k_scale_hp=s["ks"], v_scale_hp=s["vs"], slot_mapping_hp=s["slot"],
                           norm_type="layernorm")
        else:
            tmo.fused_rmsnorm_rope_store_paged_cache(
                s["qkv"], s["kc"], s["vc"], s["sin"], s["cos"], s["pos"], g[0], g[1], s["slot"],
                s["ks"], s["vs"])
        return s["qkv"], s["kc"], s["vc"], s["ks"], s["vs"]
    if op == "dequant":
        tmo.dequant_from_paged_cache(s["key"], s["value"], s["kc"], s["vc"], s["ks"], s["vs"],
                                     s["ctx"], s["longest"], None, s["table"], 1, 8)
        return s["key"], s["value"]
    if op == "attn":
        return tmo.single_query_cached_kv_attn(
            s["q"], s["kc"], s["vc"], s["out"], s["table"], s["ctx"], s["ks"], s["vs"], None,
            s["longest"], -1, -1, s["scale"], s["lse"], s["bits"], cu_seq_q=s["cu"],
            max_seq_q=s["max_q"])
    tmo.quant_to_linear_cache(s["k"], s["v"], s["kc"], s["vc"], s["ks"], s["vs"], s["cu"],
                              s["longest"], True, None, None, None, s["bits"])
    tmo.dequant_from_linear_cache(s["key"], s["value"], s["kc"], s["vc"], s["ks"], s["vs"], s["n"],
                                  s["longest"], None, None, None, 1, s["bits"])
    return s["kc"], s["vc"], s["ks"], s["vs"], s["key"], s["value"]


# ------------------------------------------------------------------------------ work


def _bytes(dtype):
    return 4 if dtype == "f32" else 2


def work(case):
    """Every input once in, every output once out."""
    op, es = case["op"], _bytes(case["dtype"])
    flops = 0.0
    if op == "quant":
        n = 2 * case["tokens"] * case["heads"]
        valid = 1.0 if case["runs"] else (case["tokens"] - case["tokens"] // 10) / case["tokens"]
        bytes_ = n * valid * (case["dim"] * (es + 1) + 4) + 4 * case["tokens"]
        flops = n * valid * case["dim"] * 4
    elif op == "smooth":
        C, E = case["channels"], case["experts"]
        rows = case["rows"] * (TOP_K if E else 1)
        bytes_ = case["rows"] * C * es + rows * (C + 4) + 4 * C * max(1, E) + (4 * rows if E else 0)
        flops = rows * C * 5
    elif op == "rope":
        T, D, Hq, Hk = case["batch"] * case["seq"], case["dim"], case["heads"], case["kv_heads"]
        store = D + 4 if case["store"] == "int8" else D * es
        bytes_ = T * ((2 * Hq + 2 * Hk) * D * es + 2 * Hk * store + 2 * D * es + 4)
        flops = T * (Hq + 2 * Hk) * D * 8
    elif op == "dequant":
        T = int(_contexts(case).sum())
        bytes_ = 2 * T * case["heads"] * (case["dim"] * (es + 1) + 4)
        flops = 2 * T * case["heads"] * case["dim"]
    elif op == "attn":
        D, Dv = case["dim"], case["dim_v"] or case["dim"]
        ctx = _contexts(case).double()
        nq = _counts(case, ctx).double() if case["q_tokens"] > 1 else torch.ones_like(ctx)
        row = {"same": D * es, "int8": D + 4, "fp8": D + 4, "int4": D / 2 + 4}[case["kv"]]
        rows = int(ctx.sum()) * case["kv_heads"] * (1 if case["dim_v"] else 2)
        cols = int(nq.sum()) * case["heads"]
        bytes_ = rows * row + cols * (D + Dv) * es + (4 * cols if case["lse"] else 0)
        flops = 2 * case["heads"] * float((nq * (ctx - (nq - 1) / 2)).sum()) * (D + Dv)
    else:
        n = 2 * int(_lengths(case).sum()) * case["heads"]
        code = case["dim"] * case["bits"] / 8 + 4
        bytes_ = n * (2 * case["dim"] * es + 2 * code)
        flops = n * case["dim"] * 6
    return {"bytes": float(bytes_), "flops": float(flops)}


def tolerance(case):
    """The quantisers and their inverses round as IEEE arithmetic does, element by element, and
    have one right answer.  The rotation sums squares in fp32 and rounds once to 16 bits, the
    attention rounds a fp32 sum to 16 bits: another order of the sums flips last bits of a few
    outputs and moves a code now and then."""
    if case["op"] == "rope":
        return {"rel": 5e-4, "max": 0.02, "differ": 1e-3}
    if case["op"] == "attn":
        return {"rel": 3e-3 if case["dtype"] == "bf16" else 4e-4, "max": 0.05}
    return "exact"


# ------------------------------------------------------------------------------ 64-bit answers


def exact(case, seed):
    s = prepare(case, seed)
    return globals()["_exact_" + case["op"]](case, s)


def _exact_quant(case, s):
    top = 127.0 if case["cache"] == "int8" else 448.0
    got = []
    for x in (s["k"], s["v"]):
        scale = torch.zeros(s["ks"].shape, dtype=torch.float64, device="cuda")
        live = s["slot"] >= 0
        slot = s["slot"][live].long()
        BS = case["block"]
        scale[slot // BS, :, slot % BS] = x[live].double().abs().amax(-1) / top
        got.append(scale)
    return [None, None, got[0], got[1]]


def _exact_smooth(case, s):
    if s["gather"] is None:
        return None, (s["x"].double() * s["smooth"].double()).abs().amax(-1) / 127.0
    expert = torch.repeat_interleave(torch.arange(case["experts"], device="cuda"), s["count"].long())
    scale = torch.empty(len(s["gather"]), dtype=torch.float64, device="cuda")
    for at in range(0, len(scale), 2048):
        rows = slice(at, at + 2048)
        scale[rows] = (s["x"][s["gather"][rows].long()].double()
                       * s["smooth"][expert[rows]].double()).abs().amax(-1) / 127.0
    return None, scale


def _exact_rope(case, s):
    Hq, Hk, D, BS = case["heads"], case["kv_heads"], case["dim"], 16
    pos = (s["pos"][:, None] + torch.arange(case["seq"], device="cuda")).long()
    sin, cos = (s[n][pos].double()[:, :, None] for n in ("sin", "cos"))
    gamma = s["gamma"].double()

    def rotate(x):
        half = D // 2
        return x * cos + torch.cat([-x[..., half:], x[..., :half]], -1) * sin

    def rms(x, g):
        return x / torch.sqrt(x.pow(2).mean(-1, keepdim=True) + 1e-5) * g

    x = s["qkv"].double()
    q, k, v = x[:, :, :Hq], x[:, :, Hq:Hq + Hk], x[:, :, Hq + Hk:]
    if case["norm"] == "rmsnorm":
        q, k = rotate(rms(q, gamma[1])), rotate(rms(k, gamma[0]))
    else:
        q, k = rotate(q), rotate(k)
        mean = k.mean(-1, keepdim=True)
        var = (k - mean).pow(2).mean(-1, keepdim=True)
        k = (k - mean) / torch.sqrt(var + 1e-5) * gamma[0] + gamma[2]
    slot = s["slot"].long()
    caches, scales = [], []
    for rows in (k, v):
        rows = rows.reshape(-1, Hk, D)
        if case["store"] == "int8":
            caches.append(None)
            scale = torch.zeros(s["ks"].shape, dtype=torch.float64, device="cuda")
            scale[slot // BS, :, slot % BS] = rows.abs().amax(-1) / 127.0
            scales.append(scale)
        else:
            cache = torch.zeros(s["kc"].shape, dtype=torch.float64, device="cuda")
            cache[slot // BS, :, slot % BS] = rows
            caches.append(cache)
            scales.append(None)
    return [torch.cat([q, x[:, :, Hq:]], 2)] + caches + scales


def _tokens_of(s, i, n, cache, scale, BS):
    """The first n context rows of sequence i as [n, heads, dim] doubles."""
    page = s["table"][i, :(n + BS - 1) // BS].long()
    x = cache[page].double()
    if scale is not None:
        x = x * scale[page].double()[..., None]
    return x.transpose(1, 2).reshape(-1, x.shape[1], x.shape[3])[:n]


def _exact_dequant(case, s):
    got = torch.empty((2,) + tuple(s["key"].shape), dtype=torch.float64, device="cuda")
    at = 0
    for i, n in enumerate(s["ctx"].tolist()):
        got[0, at:at + n] = _tokens_of(s, i, n, s["kc"], s["ks"], case["block"])
        got[1, at:at + n] = _tokens_of(s, i, n, s["vc"], s["vs"], case["block"])
        at += n
    return [got[0], got[1]]


def _unpack4(b, dim):
    return torch.stack([b >> 4, (b << 4) >> 4], dim + 1).flatten(dim, dim + 1)


def _exact_attn(case, s):
    Hq, Hkv, BS = case["heads"], case["kv_heads"], case["block"]
    kc, vc = s["kc"], s["vc"]
    if case["kv"] == "int4":
        kc, vc = _unpack4(kc, 3), _unpack4(vc, 2)
    q = s["q"].reshape(-1, Hq, case["dim"])
    out = torch.empty(q.shape[:2] + s["out"].shape[-1:], dtype=torch.float64, device="cuda")
    lse = torch.empty(q.shape[:2], dtype=torch.float64, device="cuda")
    cu = s["cu"].tolist() if s["cu"] is not None else list(range(case["batch"] + 1))
    for i, L in enumerate(s["ctx"].tolist()):
        k = _tokens_of(s, i, L, kc, s["ks"], BS)
        v = k[..., :case["dim_v"]] if case["dim_v"] else _tokens_of(s, i, L, vc, s["vs"], BS)
        n = cu[i + 1] - cu[i]
        pos = torch.arange(L - n, L, device="cuda")
        hidden = torch.arange(L, device="cuda")[None] > pos[:, None]
        for h in range(Hkv):  # [tokens * group, L]
            g = Hq // Hkv
            qi = q[cu[i]:cu[i + 1], h * g:(h + 1) * g].reshape(n * g, -1).double()
            sc = (qi @ k[:, h].T.contiguous()) * s["scale"]
            sc = sc.view(n, g, L).masked_fill(hidden[:, None], -math.inf).view(n * g, L)
            lse[cu[i]:cu[i + 1], h * g:(h + 1) * g] = sc.logsumexp(-1).view(n, g)
            out[cu[i]:cu[i + 1], h * g:(h + 1) * g] = (sc.softmax(-1) @ v[:, h].contiguous()).view(n, g, -1)
    out = out.view(s["out"].shape)
    if not case["lse"]:
        return out
    if s["cu"] is not None:
        return out, lse.T.contiguous()                     # [heads, total_q]
    return out, lse.view(case["batch"], 1, Hq).transpose(1, 2).contiguous()  # [batch, heads, 1]


def _exact_linear(case, s):
    top = 127.0 if case["bits"] == 8 else 7.0
    scales, rows = [], []
    ends = s["n"].cumsum(0).tolist()
    for x in (s["k"], s["v"]):
        x = x.double()
        amax = x.abs().amax(-1) / top
        scale = torch.zeros(s["ks"].shape, dtype=torch.float64, device="cuda")
        for i, n in enumerate(s["n"].tolist()):
            scale[i, :, :n] = amax[ends[i] - n:ends[i]].T
        scales.append(scale)
        a = amax[..., None]
        rows.append((x / a).round().clamp(-top - 1, top) * a)
    return [None, None] + scales + rows
