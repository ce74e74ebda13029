"""The measured cases: what a rollout engine has this library do, call by call.

Every case goes through the public entry points as a serving loop uses them:
decode steps through the plans (``DecodeStep``, ``GraphDecodeStep``,
``MLADecodeStep``), prompts through ``prefill_gqa``, the step's tokens through
``sample`` and prefix-cache reads through ``PagedKVCache.gather``. Sizes are
the model layouts, batches and context ranges of this repository's benchmark
and tests; block tables are dealt from a shuffled pool, as a running engine's
are. ``draw`` gives further cases of the same ranges.

Every input is made from the seed by torch's own generators, and ``exact``
restates each result in float64 from those inputs.
"""

from __future__ import annotations

import math

import torch

# layout: query heads, KV heads, head dim, layers
MODELS = {
    "qwen2.5-0.5b": (14, 2, 64, 24),
    "qwen3-0.6b": (16, 8, 128, 28),
    "qwen3-4b": (32, 8, 128, 36),
    "qwen2.5-7b": (28, 4, 128, 28),
    "qwen3-30b-a3b": (32, 4, 128, 48),
}
MLA_RANK, MLA_ROPE = 512, 64  # DeepSeek-V3's latent row
QWEN_VOCAB = 151936


def listed() -> list[dict]:
    return [
        # One sequence of a small model, the engine's default captured step: every layer's launch
        # is a few microseconds of fixed cost (an interactive request, a rollout's last straggler).
        dict(name="decode_one", kind="decode", model="qwen2.5-0.5b", kv="bf16", batch=1, lo=700, hi=700, block=16,
             layers=24, graph=True, group=0, prefix=0),
        # A rollout batch of the small model over mixed lengths.
        dict(name="decode_small_model", kind="decode", model="qwen2.5-0.5b", kv="bf16", batch=128, lo=256, hi=2048,
             block=16, layers=12, graph=False, group=0, prefix=0),
        # The headline decode step: 64 sequences of 4,096 tokens, bf16 KV.
        dict(name="decode_headline", kind="decode", model="qwen3-4b", kv="bf16", batch=64, lo=4096, hi=4096, block=16,
             layers=2, graph=False, group=0, prefix=0),
        # Few long sequences (agentic rollouts, the tail of a batch), ragged.
        dict(name="decode_long_few", kind="decode", model="qwen3-4b", kv="bf16", batch=3, lo=9001, hi=32001, block=16,
             layers=4, graph=False, group=0, prefix=0),
        # GRPO groups of eight samples over a shared 1,024-token prompt, fp8 KV.
        dict(name="decode_groups_fp8", kind="decode", model="qwen2.5-7b", kv="fp8_e4m3", batch=256, lo=1025, hi=4096,
             block=16, layers=2, graph=False, group=8, prefix=1024),
        # Weight-absorbed MLA decode, all 128 heads on one GPU.
        dict(name="mla_128_heads", kind="mla", heads=128, batch=32, lo=4096, hi=4096, block=64, layers=4),
        # One rank's 16 heads of an eight-way tensor-parallel MLA decode, mixed lengths.
        dict(name="mla_16_heads", kind="mla", heads=16, batch=16, lo=1000, hi=8000, block=64, layers=4),
        # A prompt step: eight whole prompts of 2,048 tokens.
        dict(name="prefill_prompts", kind="prefill", model="qwen3-4b", kv="bf16", batch=8, new_lo=2048, new_hi=2048,
             ctx_lo=0, ctx_hi=0, block=16),
        # Short continuations of long cached contexts (prefix-cache hits, a multi-turn rollout's
        # next turn), fp8 KV, seven query heads per KV head.
        dict(name="prefill_turns_fp8", kind="prefill", model="qwen2.5-7b", kv="fp8_e4m3", batch=4, new_lo=37,
             new_hi=250, ctx_lo=5000, ctx_hi=15000, block=16),
        # The rollout batch's tokens under top_k and top_p, bf16 logits, with the sampling mask.
        dict(name="sample_batch", kind="sample", rows=256, vocab=QWEN_VOCAB, dtype="bf16", mode="topk_topp"),
        # A few requests' tokens at the RL defaults (temperature 1, nothing cut), fp32 logits.
        dict(name="sample_few", kind="sample", rows=4, vocab=QWEN_VOCAB, dtype="fp32", mode="default"),
        # A contiguous copy of cached contexts (prefix-cache read, cache migration).
        dict(name="gather", kind="gather", model="qwen3-4b", kv="bf16", batch=8, lo=500, hi=4000, block=16,
             dequant=False),
    ]


# The largest drawn decode, prefill, sampler and gather cost no more than the largest listed one.
_MAX_DECODE_BYTES = 2.0e9
_MAX_PREFILL_FLOPS = 2.5e11


def _log_int(rng, lo: int, hi: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng) -> dict:
    kind = rng.choice(["decode", "decode", "decode", "mla", "prefill", "prefill", "sample", "sample", "gather"])
    if kind == "decode":
        group = rng.choice([0, 0, 0, 8])
        case = dict(kind=kind, model=rng.choice(sorted(MODELS)), kv=rng.choice(["bf16", "bf16", "fp8_e4m3"]),
                    batch=_log_int(rng, 1, 256), block=rng.choice([16, 16, 32, 64]), layers=1,
                    graph=bool(rng.random() < 0.3) and group == 0, group=group, prefix=0)
        if group:
            case["batch"] = max(1, case["batch"] // group) * group
            case["prefix"] = case["block"] * _log_int(rng, 4, 64)
            case["lo"] = case["prefix"] + 1
            case["hi"] = case["lo"] + _log_int(rng, 16, 4096)
        else:
            hi = _log_int(rng, 64, 32768)
            case["hi"] = hi
            case["lo"] = rng.choice([hi, max(1, hi // 4), max(1, hi // 8)])
        while _decode_bytes(case) > _MAX_DECODE_BYTES:
            if case["hi"] // 2 > case["lo"]:
                case["hi"] //= 2
            elif case["batch"] > 2 * max(1, group):
                case["batch"] = max(1, case["batch"] // 2 // max(1, group)) * max(1, group)
            else:
                case["lo"] = case["hi"] = case["hi"] // 2
        case["layers"] = max(1, min(12, MODELS[case["model"]][3], int(_MAX_DECODE_BYTES / _decode_bytes(case))))
        return case
    if kind == "mla":
        hi = _log_int(rng, 128, 8192)
        case = dict(kind=kind, heads=rng.choice([16, 32, 64, 128]), batch=_log_int(rng, 1, 64),
                    lo=rng.choice([hi, max(1, hi // 4)]), hi=hi, block=64, layers=2)
        while case["batch"] * case["hi"] > 32 * 4096:
            case["batch"] = max(1, case["batch"] // 2)
        return case
    if kind == "prefill":
        new = _log_int(rng, 16, 2048)
        ctx = rng.choice([0, 0, _log_int(rng, 64, 16384)])
        case = dict(kind=kind, model=rng.choice(sorted(MODELS)), kv=rng.choice(["bf16", "bf16", "fp8_e4m3"]),
                    batch=_log_int(rng, 1, 16), new_lo=rng.choice([new, max(1, new // 3)]), new_hi=new,
                    ctx_lo=ctx // 3, ctx_hi=ctx, block=rng.choice([16, 16, 32]))
        while work(case)["flops"] > _MAX_PREFILL_FLOPS:
            if case["batch"] > 1:
                case["batch"] //= 2
            else:
                case["new_hi"] //= 2
                case["new_lo"] = min(case["new_lo"], case["new_hi"])
        return case
    if kind == "sample":
        vocab = rng.choice([QWEN_VOCAB, QWEN_VOCAB, 129280, 32001, _log_int(rng, 8000, 256000)])
        return dict(kind=kind, rows=max(1, min(_log_int(rng, 1, 256), 256 * QWEN_VOCAB // vocab)), vocab=vocab,
                    dtype=rng.choice(["bf16", "fp32"]),
                    mode=rng.choice(["default", "topk_topp", "topp", "minp", "greedy", "penalty"]))
    hi = _log_int(rng, 64, 8192)
    case = dict(kind=kind, model=rng.choice(sorted(MODELS)), kv=rng.choice(["bf16", "fp8_e4m3"]),
                batch=_log_int(rng, 1, 16), lo=rng.choice([hi, max(1, hi // 4)]), hi=hi,
                block=rng.choice([16, 16, 32, 64]), dequant=False)
    case["dequant"] = case["kv"] != "bf16" and bool(rng.random() < 0.7)
    return case


# --------------------------------------------------------------------------- sizes

def _spread(lo: int, hi: int, n: int) -> list[int]:
    """n lengths spread evenly over [lo, hi]: the same for every seed (which sequence has which is not)."""
    return [lo + (hi - lo) * i // (n - 1) if n > 1 else hi for i in range(n)]


def _decode_tokens(case: dict) -> int:
    """Cached tokens one layer's step reads, a group's shared prompt once."""
    lens = _spread(case["lo"], case["hi"], case["batch"])
    total = sum(lens)
    if case["group"]:
        total -= case["prefix"] * (case["batch"] - case["batch"] // case["group"])
    return total


def _decode_bytes(case: dict) -> int:
    """Bytes one layer's decode step reads and writes."""
    hq, hkv, d, _ = MODELS[case["model"]]
    esz = 2 if case["kv"] == "bf16" else 1
    return (_decode_tokens(case) + case["batch"]) * hkv * d * 2 * esz + case["batch"] * (2 * hq + 2 * hkv) * d * 2


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind == "decode":
        hq, _, d, _ = MODELS[case["model"]]
        attended = sum(_spread(case["lo"], case["hi"], case["batch"]))
        return {"bytes": case["layers"] * _decode_bytes(case), "flops": case["layers"] * 4 * attended * hq * d}
    if kind == "mla":
        total, h, row = sum(_spread(case["lo"], case["hi"], case["batch"])), case["heads"], MLA_RANK + MLA_ROPE
        return {"bytes": case["layers"] * 2 * (total * row + case["batch"] * (h * (row + MLA_RANK) + 2 * row)),
                "flops": case["layers"] * 2 * total * h * (row + MLA_RANK)}
    if kind == "prefill":
        hq, hkv, d, _ = MODELS[case["model"]]
        esz = 2 if case["kv"] == "bf16" else 1
        new = _spread(case["new_lo"], case["new_hi"], case["batch"])
        ctx = _spread(case["ctx_lo"], case["ctx_hi"], case["batch"])
        t = sum(new)
        pairs = sum(n * c + n * (n + 1) // 2 for n, c in zip(new, ctx))
        return {"bytes": t * (2 * hq * d * 2 + 2 * hkv * d * (2 + esz)) + sum(ctx) * 2 * hkv * d * esz,
                "flops": 4 * pairs * hq * d}
    if kind == "sample":
        esz = 2 if case["dtype"] == "bf16" else 4
        return {"bytes": case["rows"] * (case["vocab"] * esz + case["vocab"] // 8 + 16), "flops": 0}
    _, hkv, d, _ = MODELS[case["model"]]
    esz = 2 if case["kv"] == "bf16" else 1
    osz = 2 if case["dequant"] else esz
    return {"bytes": sum(_spread(case["lo"], case["hi"], case["batch"])) * 2 * hkv * d * (esz + osz), "flops": 0}


def tolerance(case: dict):
    """Measured against ``exact`` (the errors in parentheses) and stated at about four times that."""
    kind = case["kind"]
    if kind == "decode":
        return {"rel": 1e-2, "max": 0.08}  # bf16 probabilities and outputs (0.0023)
    if kind == "mla":
        return {"rel": 1e-2, "max": 0.08}  # the same, with bf16 partials (0.0024)
    if kind == "prefill":
        return {"rel": 1e-2, "max": 0.1}  # (0.0023)
    if kind == "sample":
        # fp32 sums of up to 151,936 weights (4.4e-6); tokens, masks and counts are whole
        return {"rel": 2e-5, "max": 1e-4, "differ": 0.0}
    return "exact"


# --------------------------------------------------------------------------- inputs (no code of the library)

def _device() -> torch.device:
    return torch.device("cuda", torch.cuda.current_device())


def _gen(seed: int) -> torch.Generator:
    g = torch.Generator(device=_device())
    g.manual_seed(seed)
    return g


def _normal(gen, shape, dtype=torch.bfloat16, std: float = 1.0) -> torch.Tensor:
    x = torch.empty(shape, dtype=dtype, device=_device()).normal_(generator=gen)
    return x if std == 1.0 else x.mul_(std)


def _tables(lens: list[int], block: int, seed: int, group: int = 0, prefix: int = 0):
    """Lengths in a shuffled order, and a block table dealt from a shuffled pool (a group's leading blocks shared)."""
    g = torch.Generator()
    g.manual_seed(seed)
    order = torch.randperm(len(lens), generator=g).tolist()
    lens = [lens[i] for i in order]
    need = [-(-n // block) for n in lens]
    pb = prefix // block if group else 0
    n_groups = len(lens) // group if group else 0
    total = sum(need) - pb * (len(lens) - n_groups)
    perm = torch.randperm(total, generator=g, dtype=torch.int64).to(torch.int32)
    table = torch.full((len(lens), max(need)), -1, dtype=torch.int32)
    at = 0
    for i, n in enumerate(need):
        if group:
            if i % group == 0:
                shared = perm[at:at + pb]
                at += pb
            table[i, :pb] = shared
        table[i, pb:n] = perm[at:at + n - pb]
        at += n - pb
    return lens, table, total


def _slots(table: torch.Tensor, row: int, lo: int, hi: int, block: int) -> torch.Tensor:
    pos = torch.arange(lo, hi, dtype=torch.int64)
    return table[row, pos // block].to(torch.int64) * block + pos % block


def _pow2_scale(amax: torch.Tensor) -> torch.Tensor:
    """The smallest power of two at or above max(amax, 1e-10) / 448."""
    m, e = torch.frexp(amax.float().clamp_min(1e-10) / 448.0)
    return torch.ldexp(torch.ones_like(m), torch.where(m == 0.5, e - 1, e))


def _fill_kv(gen, blocks: int, hkv: int, d: int, block: int, kv: str):
    """One layer's cache contents in the library's documented layout: K [N, H, D/x, B, x], V [N, H, D, B], scales."""
    if kv == "bf16":
        return _normal(gen, (blocks, hkv, d // 8, block, 8)), _normal(gen, (blocks, hkv, d, block)), None, None
    out = []
    for shape in ((blocks, hkv, d // 16, block, 16), (blocks, hkv, d, block)):
        x = _normal(gen, shape)
        s = _pow2_scale(x.abs().flatten(2).amax(2))
        x.div_(s.view(blocks, hkv, *([1] * (len(shape) - 2))).to(torch.bfloat16))
        out.append((x.to(torch.float8_e4m3fn).view(torch.uint8), s))
    return out[0][0], out[1][0], out[0][1], out[1][1]


def _decode_inputs(case: dict, seed: int) -> dict:
    hq, hkv, d, _ = MODELS[case["model"]]
    gen = _gen(seed)
    b, block = case["batch"], case["block"]
    lens, table, blocks = _tables(_spread(case["lo"], case["hi"], b), block, seed, case["group"], case["prefix"])
    slots = torch.cat([_slots(table, i, n - 1, n, block) for i, n in enumerate(lens)])
    layers = []
    for _ in range(case["layers"]):
        layers.append(dict(kv=_fill_kv(gen, blocks, hkv, d, block, case["kv"]), q=_normal(gen, (b, hq, d)),
                           key=_normal(gen, (b, hkv, d)), value=_normal(gen, (b, hkv, d))))
    dev = _device()
    return dict(lens=lens, table=table.to(dev), slots=slots.to(dev), blocks=blocks, layers=layers,
                seq_lens=torch.tensor(lens, dtype=torch.int32, device=dev))


def _mla_inputs(case: dict, seed: int) -> dict:
    gen = _gen(seed)
    b, h, block = case["batch"], case["heads"], case["block"]
    lens, table, blocks = _tables(_spread(case["lo"], case["hi"], b), block, seed)
    slots = torch.cat([_slots(table, i, n - 1, n, block) for i, n in enumerate(lens)])
    layers = [dict(latent=_normal(gen, (blocks, block, MLA_RANK + MLA_ROPE)), q_nope=_normal(gen, (b, h, MLA_RANK)),
                   q_pe=_normal(gen, (b, h, MLA_ROPE)), kv_c=_normal(gen, (b, MLA_RANK)),
                   k_pe=_normal(gen, (b, MLA_ROPE))) for _ in range(case["layers"])]
    dev = _device()
    return dict(lens=lens, table=table.to(dev), slots=slots.to(dev), blocks=blocks, layers=layers,
                seq_lens=torch.tensor(lens, dtype=torch.int32, device=dev))


def _prefill_inputs(case: dict, seed: int) -> dict:
    hq, hkv, d, _ = MODELS[case["model"]]
    gen = _gen(seed)
    b, block = case["batch"], case["block"]
    new = _spread(case["new_lo"], case["new_hi"], b)
    ctx = _spread(case["ctx_lo"], case["ctx_hi"], b)
    need = [n + c for n, c in zip(new, ctx)]
    lens, table, blocks = _tables(need, block, seed)
    left = list(zip(need, new))  # the shuffled order of the lengths, with their new tokens
    rows = []
    for n in lens:
        k = next(i for i, x in enumerate(left) if x[0] == n)
        rows.append(left.pop(k)[1])
    slots = torch.cat([_slots(table, i, n - m, n, block) for i, (n, m) in enumerate(zip(lens, rows))])
    t = sum(rows)
    dev = _device()
    cu = torch.zeros(b + 1, dtype=torch.int32)
    cu[1:] = torch.cumsum(torch.tensor(rows), 0)
    return dict(lens=lens, rows=rows, table=table.to(dev), slots=slots.to(dev), blocks=blocks, cu=cu.to(dev),
                kv=_fill_kv(gen, blocks, hkv, d, block, case["kv"]), q=_normal(gen, (t, hq, d)),
                key=_normal(gen, (t, hkv, d)), value=_normal(gen, (t, hkv, d)),
                seq_lens=torch.tensor(lens, dtype=torch.int32, device=dev))


def _sample_inputs(case: dict, seed: int) -> dict:
    gen = _gen(seed)
    b, v, dev = case["rows"], case["vocab"], _device()
    # a broad body and, per row, a few likely continuations above it
    logits = _normal(gen, (b, v), torch.float32, 2.0)
    top = torch.randint(0, v, (b, 8), generator=gen, device=dev)
    logits.scatter_add_(1, top, torch.rand((b, 8), generator=gen, device=dev) * 10 + 8)
    logits = logits.to(torch.bfloat16) if case["dtype"] == "bf16" else logits
    full = lambda x, dt=torch.float32: torch.full((b,), x, dtype=dt, device=dev)  # noqa: E731
    p = {"default": {"temperature": full(1.0)},
         "topk_topp": {"temperature": full(0.7), "top_k": full(50, torch.int32), "top_p": full(0.9)},
         "topp": {"temperature": full(1.0), "top_p": full(0.95)},
         "minp": {"temperature": full(1.0), "min_p": full(0.05)},
         "greedy": {"temperature": full(0.0)},
         "penalty": {"temperature": full(0.8), "top_k": full(20, torch.int32), "top_p": full(0.95),
                     "repetition_penalty": full(1.1)}}[case["mode"]]
    seen = None
    if case["mode"] == "penalty":  # about 2% of the vocabulary seen
        words = (v + 31) // 32
        seen = torch.randint(-2 ** 31, 2 ** 31, (5, b, words), generator=gen, device=dev).to(torch.int32)
        seen = seen[0] & seen[1] & seen[2] & seen[3] & seen[4]
    seeds = torch.randint(0, 2 ** 62, (b,), generator=gen, device=dev)
    return dict(logits=logits, params=p, seen=seen, seeds=seeds, step=17)


def _gather_inputs(case: dict, seed: int) -> dict:
    _, hkv, d, _ = MODELS[case["model"]]
    lens, table, blocks = _tables(_spread(case["lo"], case["hi"], case["batch"]), case["block"], seed)
    dev = _device()
    return dict(lens=lens, table=table.to(dev), blocks=blocks, kv=_fill_kv(_gen(seed), blocks, hkv, d, case["block"], case["kv"]),
                seq_lens=torch.tensor(lens, dtype=torch.int32, device=dev))


# --------------------------------------------------------------------------- the library's calls

def _cache(kv, blocks: int, block: int, hkv: int, d: int, kv_dtype: str, shared: bool = False):
    from wavelet_amd import PagedKVCache

    c = PagedKVCache(blocks, block, hkv, d, kv_dtype=kv_dtype, device=_device(), shared_blocks=shared)
    c.k.copy_(kv[0])
    c.v.copy_(kv[1])
    if kv_dtype != "bf16":
        c.k_scale.copy_(kv[2])
        c.v_scale.copy_(kv[3])
    return c


def _cache_outputs(c) -> list:
    return [c.k, c.v] if c.k_scale is None else [c.k, c.v, c.k_scale, c.v_scale]


def prepare(case: dict, seed: int) -> dict:
    kind = case["kind"]
    if kind == "decode":
        from wavelet_amd.plan import DecodeStep, GraphDecodeStep

        hq, hkv, d, _ = MODELS[case["model"]]
        x = _decode_inputs(case, seed)
        caches = []
        for layer in x["layers"]:
            caches.append(_cache(layer.pop("kv"), x["blocks"], case["block"], hkv, d, case["kv"], case["group"] > 0))
        out = torch.zeros((case["layers"], case["batch"], hq, d), dtype=torch.bfloat16, device=_device())
        extra = {}
        if case["group"]:
            n = case["batch"] // case["group"]
            extra = dict(group_size=case["group"], max_prefix_len=case["prefix"],
                         prefix_lens=torch.full((n,), case["prefix"], dtype=torch.int32, device=_device()))
        step = DecodeStep(caches, [y["q"] for y in x["layers"]], [y["key"] for y in x["layers"]],
                          [y["value"] for y in x["layers"]], [out[i] for i in range(case["layers"])], x["table"],
                          x["seq_lens"], x["slots"], d ** -0.5, case["hi"], **extra)
        go = GraphDecodeStep(step).replay if case["graph"] else step.run
        return dict(kind=kind, go=go, keep=(x, step), outputs=[out] + [t for c in caches for t in _cache_outputs(c)])
    if kind == "mla":
        from wavelet_amd import MLALatentCache
        from wavelet_amd.plan import MLADecodeStep

        x = _mla_inputs(case, seed)
        caches = []
        for layer in x["layers"]:
            c = MLALatentCache(x["blocks"], case["block"], MLA_RANK, MLA_ROPE, device=_device())
            c.latent.copy_(layer.pop("latent"))
            caches.append(c)
        out = torch.zeros((case["layers"], case["batch"], case["heads"], MLA_RANK), dtype=torch.bfloat16, device=_device())
        pick = lambda k: [y[k] for y in x["layers"]]  # noqa: E731
        step = MLADecodeStep(caches, pick("q_nope"), pick("q_pe"), pick("kv_c"), pick("k_pe"),
                             [out[i] for i in range(case["layers"])], x["table"], x["seq_lens"], x["slots"],
                             192 ** -0.5, case["hi"])
        return dict(kind=kind, go=step.run, keep=(x, step), outputs=[out] + [c.latent for c in caches])
    if kind == "prefill":
        _, hkv, d, _ = MODELS[case["model"]]
        x = _prefill_inputs(case, seed)
        x["cache"] = _cache(x.pop("kv"), x["blocks"], case["block"], hkv, d, case["kv"])
        return dict(kind=kind, scale=d ** -0.5, longest=max(x["rows"]), context=max(x["lens"]), **x)
    if kind == "sample":
        x = _sample_inputs(case, seed)
        b, words, dev = case["rows"], (case["vocab"] + 31) // 32, _device()
        x["out"] = (torch.empty(b, dtype=torch.int64, device=dev), torch.empty(b, device=dev),
                    torch.empty((b, words), dtype=torch.int32, device=dev), torch.empty(b, dtype=torch.int32, device=dev))
        return dict(kind=kind, **x)
    _, hkv, d, _ = MODELS[case["model"]]
    x = _gather_inputs(case, seed)
    x["cache"] = _cache(x.pop("kv"), x["blocks"], case["block"], hkv, d, case["kv"])
    return dict(kind=kind, total=sum(x["lens"]), dequant=case["dequant"], **x)


def run(s: dict):
    kind = s["kind"]
    if kind in ("decode", "mla"):
        s["go"]()
        return s["outputs"]
    if kind == "prefill":
        from wavelet_amd import prefill_gqa

        out = prefill_gqa(s["q"], s["cache"], s["table"], s["seq_lens"], s["cu"], s["scale"], key=s["key"],
                          value=s["value"], slot_mapping=s["slots"], max_query_len=s["longest"],
                          max_seq_len=s["context"])
        return [out] + _cache_outputs(s["cache"])
    if kind == "sample":
        from wavelet_amd import sample

        return list(sample(s["logits"], seen=s["seen"], seeds=s["seeds"], step=s["step"], return_mask=True,
                           out=s["out"], **s["params"]))
    return list(s["cache"].gather(s["table"], s["seq_lens"], dequant=s["dequant"], total_tokens=s["total"]))


# --------------------------------------------------------------------------- the results in float64

def _tokens64(kv, ids: torch.Tensor, n: int):
    """One sequence's K and V, [n, H, D] in float64, from the blocks `ids` of a layer's cache contents."""
    k, v, ks, vs = kv
    ids = ids.to(torch.int64)
    kk, vv = k[ids], v[ids]
    if ks is not None:
        kk = kk.view(torch.float8_e4m3fn).to(torch.float64) * ks[ids].double()[:, :, None, None, None]
        vv = vv.view(torch.float8_e4m3fn).to(torch.float64) * vs[ids].double()[:, :, None, None]
    kk = kk.double().permute(0, 3, 1, 2, 4).flatten(0, 1).flatten(2)
    vv = vv.double().permute(0, 3, 1, 2).flatten(0, 1)
    return kk[:n], vv[:n]


def _append64(kv, key: torch.Tensor, value: torch.Tensor, slots: torch.Tensor, block: int):
    """The layer's contents after the call's tokens, a block's scale the smallest power of two that holds what it
    held and what it gets (a block begun at its first slot starts afresh)."""
    k, v, ks, vs = kv
    blk, off = slots // block, slots % block
    n, h, d = key.shape
    x = k.shape[-1]
    if ks is None:
        k[blk, :, :, off] = key.view(n, h, d // x, x)
        v[blk, :, :, off] = value
        return k, v, ks, vs
    fresh = torch.unique(blk[off == 0])
    for t, (codes, scale, new) in enumerate(((k, ks, key), (v, vs, value))):
        old = scale.clone()
        old[fresh] = 0
        amax = torch.zeros_like(scale)
        amax.scatter_reduce_(0, blk[:, None].expand(-1, h), new.float().abs().amax(2), "amax")
        want = old.clone()
        touched = torch.unique(blk)
        want[touched] = torch.maximum(old[touched], _pow2_scale(amax[touched]))
        for b0 in touched.split(4096):
            r = (old[b0] / want[b0]).view(-1, h, *([1] * (codes.dim() - 2)))
            codes[b0] = (codes[b0].view(torch.float8_e4m3fn).float() * r).to(torch.float8_e4m3fn).view(torch.uint8)
        c = (new.float() / want[blk][:, :, None]).clamp(-448, 448).to(torch.float8_e4m3fn).view(torch.uint8)
        if t == 0:
            codes[blk, :, :, off] = c.view(n, h, d // x, x)
        else:
            codes[blk, :, :, off] = c
        scale.copy_(want)
    return k, v, ks, vs


def _softmax_av(scores: torch.Tensor, values: torch.Tensor) -> torch.Tensor:
    return torch.softmax(scores, -1) @ values


def exact(case: dict, seed: int):
    kind = case["kind"]
    if kind == "decode":
        hq, hkv, d, _ = MODELS[case["model"]]
        x = _decode_inputs(case, seed)
        out = torch.zeros((case["layers"], case["batch"], hq, d), dtype=torch.float64, device=_device())
        rest = []
        for li, layer in enumerate(x["layers"]):
            kv = _append64(layer["kv"], layer["key"], layer["value"], x["slots"], case["block"])
            for i, n in enumerate(x["lens"]):
                kk, vv = _tokens64(kv, x["table"][i, :-(-n // case["block"])], n)
                q = layer["q"][i].double().view(hkv, hq // hkv, d)
                s = (q @ kk.permute(1, 2, 0).contiguous()) * d ** -0.5
                out[li, i] = _softmax_av(s, vv.transpose(0, 1).contiguous()).reshape(hq, d)
            rest += [None] * (2 if case["kv"] == "bf16" else 4)
            layer.pop("kv")
        return [out] + rest
    if kind == "mla":
        x = _mla_inputs(case, seed)
        out = torch.zeros((case["layers"], case["batch"], case["heads"], MLA_RANK), dtype=torch.float64, device=_device())
        for li, layer in enumerate(x["layers"]):
            rows = layer["latent"].view(-1, MLA_RANK + MLA_ROPE)
            rows[x["slots"]] = torch.cat([layer["kv_c"], layer["k_pe"]], 1)
            for i, n in enumerate(x["lens"]):
                ids = x["table"][i, :-(-n // case["block"])].to(torch.int64)
                c = layer["latent"][ids].flatten(0, 1)[:n].double()
                q = torch.cat([layer["q_nope"][i], layer["q_pe"][i]], 1).double()
                out[li, i] = _softmax_av((q @ c.T.contiguous()) * 192 ** -0.5, c[:, :MLA_RANK].contiguous())
            layer.pop("latent")
        return [out] + [None] * case["layers"]
    if kind == "prefill":
        hq, hkv, d, _ = MODELS[case["model"]]
        x = _prefill_inputs(case, seed)
        kv = _append64(x["kv"], x["key"], x["value"], x["slots"], case["block"])
        out = torch.zeros(x["q"].shape, dtype=torch.float64, device=_device())
        at = 0
        for i, (n, m) in enumerate(zip(x["lens"], x["rows"])):
            kk, vv = _tokens64(kv, x["table"][i, :-(-n // case["block"])], n)
            pos = torch.arange(n - m, n, device=_device())
            hidden = torch.arange(n, device=_device())[None, :] > pos[:, None]
            for h in range(hq):
                g = h // (hq // hkv)
                s = (x["q"][at:at + m, h].double() @ kk[:, g].T.contiguous()) * d ** -0.5
                out[at:at + m, h] = _softmax_av(s.masked_fill_(hidden, -math.inf), vv[:, g].contiguous())
            at += m
        return [out] + [None] * (2 if case["kv"] == "bf16" else 4)
    if kind == "sample":
        x = _sample_inputs(case, seed)
        return [None, _logprobs64(case, x), None, None]
    return None  # bytes


def _shift(z: torch.Tensor, n: int) -> torch.Tensor:
    return (z >> n) & ((1 << (64 - n)) - 1)


def _mix64(z: torch.Tensor) -> torch.Tensor:
    """splitmix64's finaliser on 64-bit words."""
    z = (z ^ _shift(z, 30)) * (0xBF58476D1CE4E5B9 - (1 << 64))
    z = (z ^ _shift(z, 27)) * (0x94D049BB133111EB - (1 << 64))
    return z ^ _shift(z, 31)


def _logprobs64(case: dict, x: dict) -> torch.Tensor:
    """The sampled tokens' log-probabilities over the kept sets: the documented rules and exponential race."""
    out = []
    v, dev, mode, p = case["vocab"], _device(), case["mode"], x["params"]
    golden = 0x9E3779B97F4A7C15
    for b in range(case["rows"]):
        l = x["logits"][b].double()
        if x["seen"] is not None:
            i = torch.arange(v, device=dev)
            seen = ((x["seen"][b][i >> 5] >> (i & 31)) & 1).bool()
            r = float(p["repetition_penalty"][b])
            l = torch.where(seen, torch.where(l > 0, l / r, l * r), l)
        t = float(p["temperature"][b])
        l = l if mode == "greedy" else l / t
        keep = torch.ones(v, dtype=torch.bool, device=dev)
        if "min_p" in p:
            keep &= l >= l.max() + math.log(float(p["min_p"][b]))
        if "top_k" in p:
            keep &= l >= torch.topk(l, int(p["top_k"][b])).values[-1]
        if "top_p" in p:
            w = torch.where(keep, torch.exp(l - l.max()), 0.0)
            s, order = torch.sort(w, descending=True)
            above = torch.cumsum(s, 0) - s
            first = torch.searchsorted(-s, -s)  # the first of each run of equal weights
            keep &= torch.zeros_like(keep).scatter_(0, order, above[first] < float(p["top_p"][b]) * s.sum())
        lp = l - torch.logsumexp(l[keep], 0)
        if mode == "greedy":
            score = l
        else:
            word = (int(x["seeds"][b]) + x["step"] * golden) & ((1 << 64) - 1)
            word = word - (1 << 64) if word >> 63 else word
            stream = _mix64(torch.tensor(word, dtype=torch.int64, device=dev))
            m = _shift(_mix64(stream + torch.arange(v, device=dev)), 32) >> 9
            u = (m.double() + 0.5) * 2.0 ** -23
            score = l - torch.log(-torch.log(u))
        out.append(lp[torch.argmax(torch.where(keep, score, -math.inf))])
    return torch.stack(out)
