"""The decode calls whose time counts on this path: listed ones, and a draw of more from the same ranges.

A case is one decode step of one attention layer (or one score call) through the public entry points of
`flash_recontruction` and `flash_decoding`, at the shapes of this repository's benchmark and tests: batch 1 at up to 256K
tokens, batches of tens at some thousands, ragged batches, and short contexts where launches and latency count."""
import math
import random

import torch

import kernel_collections_amd.flash_recontruction as fr
from kernel_collections_amd.flash_decoding import deepseek_mla, gqa, mla2

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
D = 128   # head width of every path but MLA and the prefix + tail form


def listed():
    return [
        # Fused decode with RoPE over factorised keys and values.  A Llama-shaped layer at batch 16, 32K tokens, one basis shared
        # by keys and values: the serving workload the framework is quoted on, and its heaviest call.
        dict(name="rope_decode_batch16_32k", kind="rope_decode", batch=16, heads=32, kv_heads=8, tokens=32768, rank=512,
             v_rank=512, shared=True, splits=2, theta=5e5, std=1.0, scale=D ** -0.5, dtype="bf16"),
        # One user, short context, bases of their own: the smallest call of the path, all launches and latency.
        dict(name="rope_decode_batch1_4k", kind="rope_decode", batch=1, heads=32, kv_heads=8, tokens=4096, rank=256,
             v_rank=256, shared=False, splits=8, theta=5e5, std=1.0, scale=D ** -0.5, dtype="bf16"),
        # One user with a long document: key rank 384, value rank 512 over 128K tokens.
        dict(name="rope_decode_batch1_128k", kind="rope_decode", batch=1, heads=32, kv_heads=8, tokens=131072, rank=384,
             v_rank=512, shared=False, splits=32, theta=5e5, std=1.0, scale=D ** -0.5, dtype="bf16"),
        # Scores of rotated reconstructed keys (for callers with their own softmax), at the rank of the sweep over lengths.
        dict(name="rope_scores_rank192_128k", kind="rope_scores", batch=1, heads=32, kv_heads=8, tokens=131072, rank=192,
             theta=1e7, std=0.2, scale=1.0, dtype="fp16", out="fp16"),
        # Scores without positional encoding, a batch at 16K tokens, fp32 out.
        dict(name="scores_batch8_16k", kind="scores", batch=8, heads=32, kv_heads=8, tokens=16384, rank=512, std=1.0,
             scale=D ** -0.5, dtype="bf16", out="fp32"),
        # Fused decode without positional encoding, one user at 256K tokens, ranks 256 / 384, 128 splits.
        dict(name="decode_batch1_256k", kind="decode", batch=1, heads=32, kv_heads=8, tokens=262144, rank=256, v_rank=384,
             splits=128, std=1 / 3, scale=1.0, dtype="fp16"),
        # Plain keys and values, a ragged batch of 32 sequences of 1K .. 128K tokens in 4096-token splits: the uncompressed layers
        # of a serving batch, and the largest call by bytes.
        dict(name="gqa_ragged_batch32", kind="gqa", batch=32, heads=32, kv_heads=8, tokens=131072, least=1024, lengths=0,
             split_tokens=4096, std=1.0, scale=D ** -0.5, dtype="bf16"),
        # Plain keys and values, a small batch of a model with few kv heads and an odd length.
        dict(name="gqa_batch3_2kv_4099", kind="gqa", batch=3, heads=16, kv_heads=2, tokens=4099, least=4099, lengths=0,
             split_tokens=1024, std=1.0, scale=D ** -0.5, dtype="fp16"),
        # Plain keys, factorised values, an ordinary ragged batch of short and middling sequences.
        dict(name="gqa_v_factorized_ragged_batch8", kind="gqa_v_factorized", batch=8, heads=32, kv_heads=8, tokens=16384, least=1024,
             lengths=1, v_rank=512, split_tokens=4096, std=1.0, scale=D ** -0.5, dtype="bf16"),
        # Absorbed MLA over the latent cache: batch 64 at 8K tokens.
        dict(name="mla_batch64_8k", kind="mla", batch=64, heads=16, tokens=8192, std=0.3, scale=192 ** -0.5, dtype="bf16"),
        # MLA whose latent is itself factorised at rank 256: batch 8 at 64K tokens.
        dict(name="mla_xkv_batch8_64k", kind="mla_xkv", batch=8, heads=16, tokens=65536, rank=256, std=1 / 3, scale=512 ** -0.5,
             dtype="fp16"),
        # A factorised 256K-token prefix and the tail of tokens decoded since.
        dict(name="prefix_tail_256k", kind="prefix_tail", batch=1, heads=32, tokens=262144, tail=128, rank=512, width=512, std=1.0,
             scale=512 ** -0.5, dtype="fp16"),
    ]


MOST_FLOPS, MOST_BYTES = 5.7e11, 3.0e9   # a drawn case stays below the heaviest listed ones


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_any(rng):
    kind = rng.choice(["rope_decode", "rope_decode", "rope_scores", "scores", "decode", "gqa", "gqa", "gqa_v_factorized", "mla",
                       "mla_xkv", "prefix_tail"])
    c = dict(kind=kind, batch=_log_int(rng, 1, 64), dtype=rng.choice(["bf16", "fp16"]))
    heads, kv_heads = rng.choice([(32, 8), (32, 8), (32, 8), (16, 2), (24, 8), (16, 4), (64, 8)])
    if kind.startswith("gqa"):
        heads, kv_heads = rng.choice([(32, 8), (32, 8), (16, 2), (8, 8), (16, 4)])
    if kind == "rope_decode":
        rank, shared = rng.choice([192, 256, 384, 512]), rng.random() < 0.5
        c.update(batch=_log_int(rng, 1, 32), heads=heads, kv_heads=kv_heads, tokens=_log_int(rng, 512, 262144), rank=rank,
                 v_rank=rank if shared else rng.choice([256, 384, 512]), shared=shared, splits=rng.choice([2, 4, 8, 16, 32, 128]),
                 theta=rng.choice([1e4, 5e5, 1e7]), std=1.0, scale=D ** -0.5)
    elif kind == "rope_scores":
        c.update(batch=_log_int(rng, 1, 8), heads=heads, kv_heads=kv_heads, tokens=_log_int(rng, 2048, 262144),
                 rank=rng.choice([128, 192, 192, 256, 384, 512]), theta=rng.choice([1e4, 5e5, 1e7]), std=0.2, scale=1.0,
                 out=rng.choice([c["dtype"], "fp32"]))
    elif kind == "scores":
        c.update(heads=heads, kv_heads=kv_heads, tokens=_log_int(rng, 512, 131072), rank=rng.choice([192, 256, 384, 512]), std=1.0,
                 scale=D ** -0.5, out=rng.choice([c["dtype"], "fp32"]))
    elif kind == "decode":
        c.update(heads=heads, kv_heads=kv_heads, tokens=_log_int(rng, 512, 262144), rank=rng.choice([192, 256, 384, 512]),
                 v_rank=rng.choice([256, 384, 512]), splits=rng.choice([4, 8, 16, 32, 128]), std=1 / 3, scale=1.0)
    elif kind in ("gqa", "gqa_v_factorized"):
        tokens = _log_int(rng, 256, 131072)
        c.update(heads=heads, kv_heads=kv_heads, tokens=tokens, least=rng.choice([tokens, max(1, tokens // 16)]),
                 lengths=rng.randrange(1 << 20), split_tokens=rng.choice([512, 1024, 4096]), std=1.0, scale=D ** -0.5)
        if kind == "gqa_v_factorized":
            c["v_rank"] = rng.choice([256, 384, 512])
    elif kind == "mla":
        c.update(batch=_log_int(rng, 1, 128), heads=rng.choice([16, 16, 32, 128]), tokens=_log_int(rng, 512, 131072), std=0.3,
                 scale=192 ** -0.5)
    elif kind == "mla_xkv":
        c.update(heads=rng.choice([16, 16, 32]), tokens=_log_int(rng, 512, 131072), rank=rng.choice([256, 384, 512]), std=1 / 3,
                 scale=512 ** -0.5)
    else:
        c.update(batch=_log_int(rng, 1, 4), heads=rng.choice([8, 16, 32]), tokens=_log_int(rng, 2048, 262144),
                 tail=_log_int(rng, 1, 2048), rank=rng.choice([256, 384, 512]), width=rng.choice([128, 512]), std=1.0)
        c["scale"] = c["width"] ** -0.5
    return c


def draw(rng):
    while True:   # sizes independent of each other; combinations beyond the heaviest listed calls are drawn again
        c = _draw_any(rng)
        w = work(c)
        padded = c["batch"] * c["tokens"] * _token_bytes(c)
        if w["flops"] <= MOST_FLOPS and w["bytes"] <= MOST_BYTES and padded <= 2 * MOST_BYTES:
            return c


def _lengths(c):
    """Lengths of a batch of plain-cache sequences: all equal, or log-uniform between `least` and `tokens`."""
    if c["least"] >= c["tokens"]:
        return [c["tokens"]] * c["batch"]
    rng = random.Random(c["lengths"])
    lo, hi = math.log(c["least"]), math.log(c["tokens"])
    lens = [int(math.exp(rng.uniform(lo, hi))) for _ in range(c["batch"])]
    lens[rng.randrange(c["batch"])] = c["tokens"]
    return lens


def _token_bytes(c):
    """Bytes of cache per token of a sequence."""
    k = c["kind"]
    if k == "rope_decode":
        return 2 * (c["rank"] + (0 if c["shared"] else c["v_rank"]))
    if k in ("rope_scores", "scores"):
        return 2 * c["rank"]
    if k == "decode":
        return 2 * (c["rank"] + c["v_rank"])
    if k == "gqa":
        return 4 * c["kv_heads"] * D
    if k == "gqa_v_factorized":
        return 2 * (c["kv_heads"] * D + c["v_rank"])
    if k == "mla":
        return 2 * (512 + 64)
    if k == "mla_xkv":
        return 2 * (c["rank"] + 64)
    return 4 * c["rank"]


def work(c):
    """Bytes and operations one pass cannot do without: the cache of every token once, the factors and queries once, the outputs
    once; keys rebuilt where they are rotated, dot products in the absorbed form where they are not."""
    k, b, h = c["kind"], c["batch"], c["heads"]
    n = sum(_lengths(c)) if k.startswith("gqa") else b * c["tokens"]
    bytes_ = n * _token_bytes(c)
    if k in ("rope_decode", "rope_scores", "scores", "decode"):
        hk, r = c["kv_heads"], c["rank"]
        bytes_ += 2 * hk * r * D + 2 * b * h * D
        flops = n * 2 * h * r + b * 2 * h * r * D if k in ("scores", "decode") else n * (2 * r * hk * D + 2 * h * D)
        if k in ("rope_decode", "decode"):
            bytes_ += 2 * hk * c["v_rank"] * D + 2 * b * h * D
            flops += n * 2 * h * c["v_rank"] + b * 2 * h * c["v_rank"] * D
        else:
            bytes_ += n * h * (4 if c["out"] == "fp32" else 2)
    elif k == "gqa":
        bytes_ += 4 * b * h * D
        flops = n * 4 * h * D
    elif k == "gqa_v_factorized":
        bytes_ += 4 * b * h * D + 2 * b * c["kv_heads"] * c["v_rank"] * D
        flops = n * 2 * h * (D + c["v_rank"]) + b * 2 * h * c["v_rank"] * D
    elif k == "mla":
        bytes_ += 2 * b * h * (512 + 64 + 512)
        flops = n * 2 * h * (512 + 64 + 512)
    elif k == "mla_xkv":
        r = c["rank"]
        bytes_ += 2 * b * h * (512 + 64 + 512) + 2 * b * r * 512
        flops = n * 2 * h * (r + 64 + r) + b * 4 * h * r * 512
    else:
        r, w, t = c["rank"], c["width"], b * c["tail"]
        bytes_ += 4 * t * w + 4 * b * h * w + 4 * b * r * w
        flops = n * 4 * h * r + t * 4 * h * w + b * 4 * h * r * w
    return {"bytes": int(bytes_), "flops": int(flops)}


def tolerance(c):
    """About four times the relative error against float64 evaluations of the same inputs (700 and 9000 tokens of every listed
    case): 2.0e-3 .. 2.4e-3 with 16-bit results in bf16 and 2.3e-4 .. 5.3e-4 in fp16 (the larger ones where keys are rebuilt
    and rotated; their fp32 angles differ by a few 1e-3 radians beyond position 100000).  fp32 scores: keys that were rebuilt are
    16 bits wide on the way (3e-4); absorbed queries are a high and a low 16-bit part (2.5e-6)."""
    if c.get("out") == "fp32":
        return {"rel": 2e-3 if c["kind"] == "rope_scores" else 1e-5}
    return {"rel": 1e-2 if c["dtype"] == "bf16" else 2e-3}


def _randn(g, shape, std, dtype):
    out = torch.empty(shape, dtype=dtype, device="cuda")
    flat = out.view(-1)
    for i in range(0, flat.numel(), 1 << 28):   # fp32 slabs of at most 1 GiB
        n = min(1 << 28, flat.numel() - i)
        flat[i:i + n] = torch.randn(n, device="cuda", dtype=torch.float32, generator=g) * std
    return out


def prepare(c, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    dt, std, k, b, h, n = DTYPES[c["dtype"]], c["std"], c["kind"], c["batch"], c["heads"], c["tokens"]
    s = {"case": c}

    def splits(counts):
        s["splits"] = torch.tensor(counts, dtype=torch.int32, device="cuda")
        s["max_splits"] = max(counts)

    def factor(rank, heads=1, width=D):   # one matrix per kv head for the whole batch, as [batch, kv_heads, rank, width]
        return _randn(g, (rank, heads, width), rank ** -0.5, dt).permute(1, 0, 2).unsqueeze(0).expand(b, heads, rank, width)

    if k in ("rope_decode", "decode"):
        s["q"] = _randn(g, (b, h, D), std, dt)
        s["k_a"], s["k_b"] = _randn(g, (b, n, c["rank"]), std, dt), factor(c["rank"], c["kv_heads"])
        s["v_a"] = s["k_a"] if c.get("shared") else _randn(g, (b, n, c["v_rank"]), std, dt)
        s["v_b"] = factor(c["v_rank"], c["kv_heads"])
        splits([c["splits"]] * b)
        s["o"] = torch.empty_like(s["q"])
    elif k in ("rope_scores", "scores"):
        s["q"] = _randn(g, (b, h, 1, D), std, dt)
        s["k_a"], s["k_b"] = _randn(g, (b, n, c["rank"]), std, dt), factor(c["rank"], c["kv_heads"])
    elif k in ("gqa", "gqa_v_factorized"):
        lens = _lengths(c)
        s["lens"] = None if c["least"] >= n else torch.tensor(lens, dtype=torch.int32, device="cuda")
        splits([-(-m // c["split_tokens"]) for m in lens])
        s["q"] = _randn(g, (b, h, D), std, dt)
        s["k"] = _randn(g, (b, n, c["kv_heads"], D), std, dt)
        if k == "gqa":
            s["v"] = _randn(g, (b, n, c["kv_heads"], D), std, dt)
        else:
            s["v_a"] = _randn(g, (b, n, c["v_rank"]), std, dt)
            s["v_b"] = _randn(g, (b, c["kv_heads"], c["v_rank"], D), c["v_rank"] ** -0.5, dt)
        s["o"] = torch.empty_like(s["q"])
    elif k in ("mla", "mla_xkv"):
        s["q_nope"], s["q_rope"] = _randn(g, (b, h, 512), std, dt), _randn(g, (b, h, 64), std, dt)
        s["latent"] = _randn(g, (b, n, 1, c.get("rank", 512)), std, dt)
        s["k_rope"] = _randn(g, (b, n, 1, 64), std, dt)
        if k == "mla_xkv":
            s["factor"] = _randn(g, (b, 1, c["rank"], 512), c["rank"] ** -0.5, dt)
    else:
        r, w = c["rank"], c["width"]
        s["q"] = _randn(g, (b, h, w), std, dt)
        s["k_a"], s["v_a"] = _randn(g, (b, n, r), std, dt), _randn(g, (b, n, r), std, dt)
        s["k_b"], s["v_b"] = factor(r, width=w), factor(r, width=w)
        s["k_tail"], s["v_tail"] = _randn(g, (b, c["tail"], 1, w), std, dt), _randn(g, (b, c["tail"], 1, w), std, dt)
    return s


def run(s):
    c = s["case"]
    k, scale = c["kind"], c["scale"]
    if k == "rope_decode":
        return fr.gqa_xKV_rope(s["q"], s["k_a"], s["k_b"], s["v_a"], s["v_b"], s["o"], s["splits"], s["max_splits"], scale, c["theta"])
    if k == "decode":
        return fr.gqa_xKV_no_pe(s["q"], s["k_a"], s["k_b"], s["v_a"], s["v_b"], s["o"], s["splits"], s["max_splits"], scale)
    if k == "rope_scores":
        return fr.qAB_rope_v1(s["q"], s["k_a"], s["k_b"], c["theta"], out_dtype=DTYPES[c["out"]])
    if k == "scores":
        return fr.qAB_no_pe_v1(s["q"], s["k_a"], s["k_b"], sm_scale=scale, out_dtype=DTYPES[c["out"]])
    if k == "gqa":
        return gqa.decode_attention_fwd(s["q"], s["k"], s["v"], s["o"], s["splits"], s["max_splits"], scale, kv_lens=s["lens"])
    if k == "gqa_v_factorized":
        return gqa.decode_attention_fwd_v_factorized(s["q"], s["k"], s["v_a"], s["v_b"], s["o"], s["splits"], s["max_splits"], scale,
                                                     kv_lens=s["lens"])
    if k == "mla":
        return mla2.mla_decode_attention_fwd(s["q_nope"], s["q_rope"], s["latent"], s["k_rope"], scale)
    if k == "mla_xkv":
        return mla2.mla_decode_attention_xKV(s["q_nope"], s["q_rope"], s["latent"], s["factor"], s["k_rope"], scale)
    return deepseek_mla.mla_decode_attention_fwd_pd_sep_xKV(s["q"], s["k_a"], s["k_b"], s["v_a"], s["v_b"], s["k_tail"], s["v_tail"], scale)
