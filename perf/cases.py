"""The work that users of flashspec_amd have it do, as measurable cases.

Each case goes through the package's public entry points: decode attention over a quantized KV cache
(paged and contiguous), tree verification, building a paged cache from dense K/V, reading one back,
admitting a request into a page pool, and a whole serving round (admit, decode steps with append,
release).  Sizes come from the repository's configurations, benchmark and command lines, or are
ragged neighbours of those.
"""

from __future__ import annotations

import math

import torch

import flashspec_amd as fa
from flashspec_amd.serving import DecodeBatch

_DTYPES = {"float16": torch.float16, "bfloat16": torch.bfloat16}
_DEVICE = "cuda"


# ---- the cases -----------------------------------------------------------------------------------

def listed():
    return [
        # one short request on the package's default heads and head_dim: launch and host latency
        {"name": "paged_tiny", "kind": "paged", "batch": 1, "heads": 8, "seq": 128, "dim": 64, "page": 16,
         "kv": "affine_block", "dtype": "float16", "layout": "contiguous", "lengths": "full"},
        # the headline decode step: paged INT8, eight requests of 4096 tokens
        {"name": "paged_headline", "kind": "paged", "batch": 8, "heads": 32, "seq": 4096, "dim": 128, "page": 16,
         "kv": "affine_block", "dtype": "float16", "layout": "contiguous", "lengths": "full"},
        # one long context over an FP8 cache with bf16 queries: split rows and their merge
        {"name": "paged_long_fp8", "kind": "paged", "batch": 1, "heads": 32, "seq": 16384, "dim": 128, "page": 16,
         "kv": "fp8_block", "dtype": "bfloat16", "layout": "shuffled", "lengths": "full"},
        # the contiguous kernel on the per-token symmetric format
        {"name": "fused_token", "kind": "fused", "batch": 4, "heads": 32, "seq": 2048, "dim": 128, "page": 16,
         "kv": "symmetric_token", "dtype": "float16", "lengths": "full"},
        # the attention of a serving step at scale: 64 ragged requests in a fragmented pool
        {"name": "pool_64_ragged", "kind": "pool", "batch": 64, "heads": 32, "shortest": 128, "longest": 16384,
         "dim": 128, "page": 16, "dtype": "float16"},
        # speculative decoding, a small draft tree
        {"name": "tree_16", "kind": "tree", "batch": 4, "nodes": 16, "heads": 32, "seq": 4096, "dim": 128, "page": 16,
         "kv": "affine_block", "dtype": "float16", "layout": "contiguous", "lengths": "full"},
        # speculative decoding, a wide draft tree, in the type that models run in
        {"name": "tree_64_bf16", "kind": "tree", "batch": 8, "nodes": 64, "heads": 32, "seq": 4096, "dim": 128,
         "page": 16, "kv": "affine_block", "dtype": "bfloat16", "layout": "contiguous", "lengths": "full"},
        # a prefilled batch quantized into a paged cache
        {"name": "build_i8", "kind": "build", "batch": 8, "heads": 32, "seq": 4096, "dim": 128, "page": 16,
         "kv": "affine_block", "dtype": "float16", "layout": "contiguous"},
        # the same into FP8 pages, a ragged length and shuffled pages
        {"name": "build_fp8_ragged", "kind": "build", "batch": 4, "heads": 32, "seq": 2039, "dim": 128, "page": 16,
         "kv": "fp8_block", "dtype": "bfloat16", "layout": "shuffled"},
        # the cache read back as dense K/V (a prefix handed to a dense attention)
        {"name": "read_dense", "kind": "dense", "batch": 4, "heads": 32, "seq": 2039, "dim": 128, "page": 16,
         "kv": "affine_block", "dtype": "float16", "layout": "shuffled"},
        # one prompt admitted to a pool that other requests live in, and its pages given back
        {"name": "admit_prompt", "kind": "admit", "length": 3001, "before": 700, "gap": 333, "after": 1200,
         "heads": 32, "dim": 128, "page": 16, "dtype": "float16"},
        # a whole serving round on the package's default model size: admit, 16 decode steps, release
        {"name": "serving_round", "kind": "round", "requests": 8, "prompt_a": 512, "prompt_b": 2048, "steps": 16,
         "heads": 8, "dim": 64, "page": 16, "dtype": "float16"},
    ]


def _log(rng, low, high):
    """A whole number spread over the logarithm of [low, high]."""
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


_HEADS = (8, 12, 16, 32, 40)
_DIMS = (64, 80, 96, 128, 128, 128, 256)
_KV = ("affine_block", "affine_block", "fp8_block", "symmetric_token", "affine_channel")
_LAYOUTS = ("contiguous", "shuffled", "interleaved")


def draw(rng):
    kind = rng.choice(("paged", "paged", "fused", "pool", "tree", "tree", "build", "build", "dense", "admit", "admit",
                       "round"))
    dtype = rng.choice(("float16", "bfloat16"))
    if kind == "pool":
        longest = _log(rng, 512, 8192)
        return {"kind": kind, "batch": rng.randint(9, 48), "heads": rng.choice((8, 16, 32)),
                "shortest": rng.randint(1, 128), "longest": longest, "dim": rng.choice((64, 128)), "page": 16,
                "dtype": dtype}
    if kind == "admit":
        return {"kind": kind, "length": _log(rng, 333, 16000), "before": rng.randint(1, 2000),
                "gap": rng.randint(1, 333), "after": rng.randint(1, 2000), "heads": rng.choice(_HEADS),
                "dim": rng.choice((64, 80, 96, 128, 128)), "page": rng.choice((16, 16, 32)), "dtype": dtype}
    if kind == "round":
        return {"kind": kind, "requests": rng.randint(2, 12), "prompt_a": rng.randint(20, 700),
                "prompt_b": rng.randint(700, 2048), "steps": rng.randint(8, 20), "heads": rng.choice((8, 16)),
                "dim": rng.choice((64, 128)), "page": 16, "dtype": dtype}
    dim, heads = rng.choice(_DIMS), rng.choice(_HEADS)
    case = {"kind": kind, "heads": heads, "dim": dim, "page": rng.choice((16, 16, 16, 32)), "dtype": dtype}
    # elements of K: at most a quarter of the largest listed attention, at most half of the largest build
    most = {"paged": 2 ** 28, "fused": 2 ** 28, "tree": 2 ** 26, "build": 2 ** 26, "dense": 2 ** 25}[kind]
    case["batch"] = _log(rng, 1, 16 if kind in ("paged", "fused") else 8)
    case["seq"] = _log(rng, 64, max(65, min(16384, most // (case["batch"] * heads * dim))))
    if kind == "tree":
        case["nodes"] = rng.randint(1, 64)
        case["dim"] = rng.choice((64, 128, 128))
        case["kv"] = rng.choice(("affine_block", "affine_block", "fp8_block", "symmetric_token"))
    elif kind == "dense":
        case["kv"] = rng.choice(("affine_block", "fp8_block"))
    else:
        case["kv"] = rng.choice(_KV)
    if kind != "fused":
        case["layout"] = rng.choice(_LAYOUTS)
    if kind in ("paged", "fused", "tree"):
        case["lengths"] = rng.choice(("full", "descending", "ragged"))
    return case


# ---- inputs ----------------------------------------------------------------------------------------

def _generator(seed):
    g = torch.Generator(device=_DEVICE)
    g.manual_seed(int(seed))
    return g


def _normal(g, case, *shape):
    return torch.randn(shape, generator=g, device=_DEVICE, dtype=_DTYPES[case["dtype"]])


def _lengths(case):
    """Valid tokens of each request, as a list (None: every request is full); sizes, so part of the case."""
    b, s = case["batch"], case["seq"]
    if case["lengths"] == "full":
        return None
    if case["lengths"] == "descending":
        return [max(1, s - (s * i * 15) // (16 * max(1, b - 1))) for i in range(b)]
    g = torch.Generator().manual_seed(s)
    return torch.randint(1, s + 1, (b,), generator=g).tolist()


def _dense_kv(case, seed):
    shape = (case["batch"], case["heads"], case["seq"], case["dim"])
    g = _generator(seed)
    return _normal(g, case, *shape), _normal(g, case, *shape), g


def _pool_lengths(case):
    g = torch.Generator().manual_seed(case["batch"])
    rest = torch.randint(case["shortest"], case["longest"] + 1, (case["batch"] - 1,), generator=g).tolist()
    return [case["longest"]] + rest


def _parents(case, seed):
    """A random forest in topological order, on the host as a drafter builds it."""
    g = torch.Generator().manual_seed(int(seed) + 7)
    n = case["nodes"]
    at = torch.rand((case["batch"], n), generator=g) * (torch.arange(n) + 1)
    return at.floor().to(torch.int64) - 1


def _pages(case, tokens):
    return -(-tokens // case["page"])


def _prompts(case):
    return [case["prompt_a"] if i % 2 == 0 else case["prompt_b"] for i in range(case["requests"])]


def _allocator(case, pages):
    return fa.PagedKVAllocator(capacity_blocks=pages, heads=case["heads"], head_dim=case["dim"],
                               block_size=case["page"], device=_DEVICE, dtype=_DTYPES[case["dtype"]])


def _contiguous(case, x):
    if case["kv"] == "symmetric_token":
        return fa.quantize_int8_symmetric_per_token(x)
    quantize = {"affine_block": fa.quantize_int8_per_block, "fp8_block": fa.quantize_fp8_per_block,
                "affine_channel": fa.quantize_int8_per_channel}[case["kv"]]
    return quantize(x, case["page"])


def _admit_inputs(case, seed):
    """K/V of the requests in the order they arrive: before, gap (released again), after, the prompt."""
    g = _generator(seed)
    got = []
    for length in (case["before"], case["gap"], case["after"], case["length"]):
        shape = (1, case["heads"], length, case["dim"])
        got.append((_normal(g, case, *shape), _normal(g, case, *shape)))
    return got


def _admit_pages(case):
    return sum(_pages(case, case[n]) for n in ("before", "gap", "after", "length"))


def _round_inputs(case, seed):
    g = _generator(seed)
    h, d, n = case["heads"], case["dim"], case["requests"]
    prompts = [(_normal(g, case, 1, h, length, d), _normal(g, case, 1, h, length, d)) for length in _prompts(case)]
    tokens = [(_normal(g, case, n, h, d), _normal(g, case, n, h, 1, d), _normal(g, case, n, h, 1, d))
              for _ in range(case["steps"])]
    return prompts, tokens


def _round_pages(case):
    return sum(_pages(case, length + case["steps"]) for length in _prompts(case))


def prepare(case, seed):
    kind = case["kind"]
    if kind == "pool":
        lengths = _pool_lengths(case)
        pool = _allocator(case, sum(_pages(case, length + 16) for length in lengths))
        pool.shuffle_free_blocks(int(seed))
        g = _generator(seed)
        for rid, length in enumerate(lengths):
            shape = (1, case["heads"], length, case["dim"])
            pool.add_request(rid, _normal(g, case, *shape), _normal(g, case, *shape))
        q = _normal(g, case, case["batch"], case["heads"], case["dim"])
        return {"kind": kind, "q": q, "decode": DecodeBatch(pool, list(range(case["batch"])), max_new_tokens=16)}
    if kind == "admit":
        *others, prompt = _admit_inputs(case, seed)
        pool = _allocator(case, _admit_pages(case))
        for rid, (k, v) in enumerate(others):
            pool.add_request(rid, k, v)
        pool.release_request(1)
        return {"kind": kind, "pool": pool, "k": prompt[0], "v": prompt[1]}
    if kind == "round":
        prompts, tokens = _round_inputs(case, seed)
        return {"kind": kind, "pool": _allocator(case, _round_pages(case)), "prompts": prompts, "tokens": tokens}
    k, v, g = _dense_kv(case, seed)
    if kind == "build":
        return {"kind": kind, "k": k, "v": v, "page": case["page"], "layout": case["layout"], "kv": case["kv"],
                "seed": int(seed)}
    state = {"kind": kind}
    if kind == "tree":
        shape = (case["batch"], case["nodes"], case["heads"], case["dim"])
        state.update(q=_normal(g, case, *shape), draft_k=_normal(g, case, *shape), draft_v=_normal(g, case, *shape),
                     parents=_parents(case, seed))
    elif kind != "dense":
        state["q"] = _normal(g, case, case["batch"], case["heads"], case["dim"])
    lengths = None if kind == "dense" else _lengths(case)
    lengths = None if lengths is None else torch.tensor(lengths, dtype=torch.int64, device=_DEVICE)
    if kind == "fused":
        state.update(k=_contiguous(case, k), v=_contiguous(case, v), lengths=lengths)
    else:
        state["cache"] = fa.PagedKVCache.from_dense(k, v, case["page"], lengths=lengths,
                                                    block_table_pattern=case["layout"], layout_seed=int(seed),
                                                    kv_format=case["kv"])
    return state


# ---- one pass ----------------------------------------------------------------------------------------

def _store(prefix, quant):
    values = quant.values if quant.values.dtype == torch.int8 else quant.values.view(torch.uint8)
    return {prefix + "_values": values, prefix + "_scale": quant.scale, prefix + "_zero": quant.zero_point}


def run(state):
    kind = state["kind"]
    if kind == "paged":
        return fa.paged_quant_attention_triton(state["q"], state["cache"])
    if kind == "fused":
        return fa.fused_dequant_attention_triton(state["q"], state["k"], state["v"], state["lengths"])
    if kind == "pool":
        return state["decode"].attend(state["q"])
    if kind == "tree":
        return fa.tree_verify_attention(state["q"], state["cache"], state["draft_k"], state["draft_v"],
                                        state["parents"])
    if kind == "build":
        cache = fa.PagedKVCache.from_dense(state["k"], state["v"], state["page"],
                                           block_table_pattern=state["layout"], layout_seed=state["seed"],
                                           kv_format=state["kv"])
        return {**_store("k", cache.k_quant), **_store("v", cache.v_quant), "table": cache.block_table,
                "lengths": cache.lengths}
    if kind == "dense":
        return state["cache"].to_dense()
    pool = state["pool"]
    if kind == "admit":
        pool.add_request(3, state["k"], state["v"])
        pool.release_request(3)
        return {**_store("k", pool.k_quant), **_store("v", pool.v_quant)}
    ids = list(range(len(state["prompts"])))
    for rid, (k, v) in zip(ids, state["prompts"]):
        pool.add_request(rid, k, v)
    batch = DecodeBatch(pool, ids, max_new_tokens=len(state["tokens"]))
    outs = [batch.step(q, k, v) for q, k, v in state["tokens"]]
    batch.close()
    for rid in ids:
        pool.release_request(rid)
    return {"outs": outs, **_store("k", pool.k_quant), **_store("v", pool.v_quant)}


# ---- what a pass cannot do without -----------------------------------------------------------------------

def _kv_bytes(case, tokens):
    """Codes and parameters of one head's `tokens` K (or V) rows."""
    d = case["dim"]
    kv = case.get("kv", "affine_block")
    per_page = {"affine_block": 6, "fp8_block": 4, "affine_channel": 6 * d, "symmetric_token": 0}[kv]
    per_token = 6 if kv == "symmetric_token" else 0
    return tokens * (d + per_token) + _pages(case, tokens) * per_page


def work(case):
    kind, h, d, page = case["kind"], case["heads"], case["dim"], case["page"]
    if kind == "admit":
        n = case["length"]
        return {"bytes": 2 * h * (n * d * 2 + _kv_bytes(case, n)), "flops": 4 * 2 * h * n * d}
    if kind == "round":
        b = f = 0
        for n in _prompts(case):
            b += 2 * h * (n * d * 2 + _kv_bytes(case, n))
            for step in range(case["steps"]):
                # the prefix read, one page rewritten, the token, the query and the output
                b += 2 * h * (_kv_bytes(case, n + step + 1) + page * d + 6) + 4 * h * d * 2
                f += 4 * h * (n + step + 1) * d
        return {"bytes": b, "flops": f}
    if kind == "pool":
        lengths = _pool_lengths(case)
    elif kind in ("build", "dense"):
        lengths = [case["seq"]] * case["batch"]
    else:
        lengths = _lengths(case) or [case["seq"]] * case["batch"]
    kv = sum(2 * h * _kv_bytes(case, n) for n in lengths)
    table = 0 if kind == "fused" else sum(8 * _pages(case, n) for n in lengths)
    tokens = sum(lengths)
    if kind == "build":
        return {"bytes": 2 * h * tokens * d * 2 + kv + table, "flops": 4 * 2 * h * tokens * d}
    if kind == "dense":
        return {"bytes": kv + table + 2 * h * tokens * d * 4, "flops": 2 * 2 * h * tokens * d}
    nodes = case.get("nodes", 1)
    rows = case["batch"] * nodes * h * d * 2
    flops = 4 * h * d * nodes * tokens
    return {"bytes": kv + table + rows * (4 if kind == "tree" else 2), "flops": flops}


def tolerance(case):
    # quantized pages are defined bit by bit, and reading them back is one product per value
    if case["kind"] in ("build", "dense", "admit"):
        return "exact"
    # attention rounds its result once to the query's type; pages stay exact (no "differ")
    if case["dtype"] == "float16":
        return {"rel": 1.0e-3, "max": 4.0e-3}
    return {"rel": 8.0e-3, "max": 3.0e-2}


# ---- the same results in 64 bits, in plain torch -------------------------------------------------------------

def _over(x, number):
    """x / number, correctly rounded (a plain number would be multiplied by its reciprocal on the GPU)."""
    return x / torch.full((1,), number, dtype=x.dtype, device=x.device)


def _affine(x, dims):
    """Codes, scale and zero point of groups over `dims`: float32, step by step as the format is defined."""
    lo, hi = x.amin(dim=dims, keepdim=True), x.amax(dim=dims, keepdim=True)
    scale = _over(hi - lo, 255.0).clamp_min(1.0e-8)
    zero = torch.round(-lo / scale).clamp(0, 255)
    return torch.round(x / scale + zero).clamp(0, 255), scale, zero


def _grouped(case, x):
    """[..., tokens, dim] -> float32 [..., pages, page, dim], zeros past the last token."""
    page = case["page"]
    x = x.to(torch.float32)
    pad = -x.shape[-2] % page
    if pad:
        x = torch.cat([x, x.new_zeros((*x.shape[:-2], pad, x.shape[-1]))], dim=-2)
    return x.reshape(*x.shape[:-2], x.shape[-2] // page, page, x.shape[-1])


def _dequantized(case, x):
    """What the cache holds for [..., tokens, dim], in 64 bits."""
    kv = case.get("kv", "affine_block")
    if kv == "symmetric_token":
        x = x.to(torch.float32)
        scale = _over(x.abs().amax(dim=-1, keepdim=True), 127.0).clamp_min(1.0e-8)
        return torch.round(x / scale).clamp(-127, 127).double() * scale.double()
    g = _grouped(case, x)
    if kv == "fp8_block":
        scale = _over(g.abs().amax(dim=(-2, -1), keepdim=True), 448.0).clamp_min(1.0e-8)
        got = (g / scale).clamp(-448.0, 448.0).to(torch.float8_e4m3fn).double() * scale.double()
    else:
        codes, scale, zero = _affine(g, (-2,) if kv == "affine_channel" else (-2, -1))
        got = (codes.double() - zero.double()) * scale.double()
    return got.reshape(*x.shape[:-2], -1, x.shape[-1])[..., : x.shape[-2], :]


def _scales(case, x):
    """The scale of every group of [..., tokens, dim], in 64 bits."""
    kv = case.get("kv", "affine_block")
    if kv == "symmetric_token":
        x = _grouped(case, x)
        return (x.double().abs().amax(dim=-1, keepdim=True) / 127.0).clamp_min(1.0e-8)[..., None]
    g = _grouped(case, x).double()
    if kv == "fp8_block":
        return (g.abs().amax(dim=(-2, -1), keepdim=True) / 448.0).clamp_min(1.0e-8)
    dims = (-2,) if kv == "affine_channel" else (-2, -1)
    return ((g.amax(dim=dims, keepdim=True) - g.amin(dim=dims, keepdim=True)) / 255.0).clamp_min(1.0e-8)


def _attend(q, k, v):
    """One request in 64 bits: q [rows, heads, dim] over k, v [heads, tokens, dim]."""
    scores = torch.matmul(k, q.double().permute(1, 2, 0).contiguous()) / math.sqrt(q.shape[-1])  # [h, tokens, rows]
    p = torch.softmax(scores, dim=1)
    return torch.matmul(p.transpose(1, 2).contiguous(), v).permute(1, 0, 2)


def _physical(case, x, seed):
    """[batch, heads, pages, ...] groups -> [physical pages, heads, ...], as the cache's layout places them."""
    b, n = x.shape[0], x.shape[2]
    x = x.transpose(1, 2).reshape(b * n, x.shape[1], *x.shape[3:])
    if case["layout"] == "shuffled":
        return x[torch.randperm(b * n, generator=_generator(seed), device=_DEVICE)]
    if case["layout"] == "interleaved":
        return x[torch.arange(b * n, device=_DEVICE).reshape(b, n).t().reshape(-1)]
    return x


def _exact_build(case, seed):
    k, v, _ = _dense_kv(case, seed)
    out = {n: None for n in ("k_values", "k_zero", "v_values", "v_zero", "table", "lengths")}
    for name, x in (("k_scale", k), ("v_scale", v)):
        scale = _physical(case, _scales(case, x), seed)  # [pages, heads, (page,) 1, 1 or dim]
        shape = scale.shape[:2]
        if case["kv"] == "symmetric_token":
            out[name] = scale.reshape(*shape, case["page"], 1, 1)
        else:
            out[name] = scale.reshape(*shape, 1, 1, -1)
    return out


def _exact_admit(case, seed):
    requests = _admit_inputs(case, seed)
    n = [_pages(case, x[0].shape[2]) for x in requests]
    out = {name: None for name in ("k_values", "k_zero", "v_values", "v_zero")}
    for name, which in (("k_scale", 0), ("v_scale", 1)):
        before, gap, after, new = (_scales(case, x[which])[0].transpose(0, 1) for x in requests)
        # the gap's pages are taken first, then the ones past the last request; what the gap's
        # request left in pages that nobody took stays
        took = min(n[1], n[3])
        rest = gap.new_full((n[1] - took, *gap.shape[1:]), 0.0)
        rest[:] = gap[took:]
        free = gap.new_full((_admit_pages(case) - sum(n[:3]) - (n[3] - took), *gap.shape[1:]), 1.0e-8)
        out[name] = torch.cat([before, new[:took], rest, after, new[took:], free]).reshape(-1, case["heads"], 1, 1, 1)
    return out


class _Pages:
    """One request's K or V pages as they are requantized token by token: float32, [heads, pages, page, dim]."""

    def __init__(self, case, x, tokens):
        self.codes, self.scale, self.zero = _affine(_grouped(case, x[0]), (-2, -1))
        more = _pages(case, tokens) - self.codes.shape[1]
        if more:  # pages of a pool that nobody wrote: zeros
            h, _, page, d = self.codes.shape
            self.codes = torch.cat([self.codes, self.codes.new_zeros((h, more, page, d))], dim=1)
            self.scale = torch.cat([self.scale, self.scale.new_full((h, more, 1, 1), 1.0e-8)], dim=1)
            self.zero = torch.cat([self.zero, self.zero.new_zeros((h, more, 1, 1))], dim=1)

    def append(self, at, row):
        page = self.codes.shape[2]
        j = at // page
        block = (self.codes[:, j] - self.zero[:, j]) * self.scale[:, j]
        block[:, at % page] = row.to(torch.float32)
        self.codes[:, j], self.scale[:, j], self.zero[:, j] = _affine(block, (-2, -1))

    def tokens(self, n):
        x = (self.codes.double() - self.zero.double()) * self.scale.double()
        return x.reshape(x.shape[0], -1, x.shape[-1])[:, :n]


def _exact_round(case, seed):
    prompts, tokens = _round_inputs(case, seed)
    outs = [[] for _ in tokens]
    for i, (k, v) in enumerate(prompts):
        n = k.shape[2]
        ks, vs = _Pages(case, k, n + len(tokens)), _Pages(case, v, n + len(tokens))
        for t, (q, k_new, v_new) in enumerate(tokens):
            ks.append(n + t, k_new[i, :, 0])
            vs.append(n + t, v_new[i, :, 0])
            outs[t].append(_attend(q[i: i + 1], ks.tokens(n + t + 1), vs.tokens(n + t + 1)))
    pages = {name: None for name in ("k_values", "k_scale", "k_zero", "v_values", "v_scale", "v_zero")}
    return {"outs": [torch.cat(o) for o in outs], **pages}


def exact(case, seed):
    kind = case["kind"]
    if kind == "build":
        return _exact_build(case, seed)
    if kind == "admit":
        return _exact_admit(case, seed)
    if kind == "round":
        return _exact_round(case, seed)
    if kind == "pool":
        g, kv = _generator(seed), []
        for length in _pool_lengths(case):
            shape = (1, case["heads"], length, case["dim"])
            kv.append((_normal(g, case, *shape), _normal(g, case, *shape)))
        q = _normal(g, case, case["batch"], case["heads"], case["dim"])
        return torch.cat([_attend(q[i: i + 1], _dequantized(case, k)[0], _dequantized(case, v)[0])
                          for i, (k, v) in enumerate(kv)])
    k, v, g = _dense_kv(case, seed)
    if kind == "dense":
        return _dequantized(case, k), _dequantized(case, v)
    lengths = _lengths(case) or [case["seq"]] * case["batch"]
    outs = []
    if kind == "tree":
        shape = (case["batch"], case["nodes"], case["heads"], case["dim"])
        q, dk, dv = _normal(g, case, *shape), _normal(g, case, *shape), _normal(g, case, *shape)
        parents = _parents(case, seed).tolist()
    else:
        q = _normal(g, case, case["batch"], case["heads"], case["dim"])
    for b, n in enumerate(lengths):
        kb, vb = _dequantized(case, k[b])[:, :n], _dequantized(case, v[b])[:, :n]
        if kind != "tree":
            outs.append(_attend(q[b: b + 1], kb, vb))
            continue
        path = torch.zeros((case["nodes"], case["nodes"]), dtype=torch.bool)
        for node, parent in enumerate(parents[b]):
            if parent >= 0:
                path[node] = path[parent]
            path[node, node] = True
        kb = torch.cat([kb, dk[b].double().transpose(0, 1)], dim=1)
        vb = torch.cat([vb, dv[b].double().transpose(0, 1)], dim=1)
        scores = torch.matmul(kb, q[b].double().permute(1, 2, 0).contiguous()) / math.sqrt(case["dim"])
        scores[:, n:].masked_fill_(~path.t().to(_DEVICE), -math.inf)
        p = torch.softmax(scores, dim=1)
        outs.append(torch.matmul(p.transpose(1, 2).contiguous(), vb).permute(1, 0, 2)[None])
    return torch.cat(outs)
