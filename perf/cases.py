"""The work that a serving engine has this package do, as cases to time.

One DeepSeek-V4 attention layer calls the package in this order: the q/kv
norms, RoPE and cache inserts before attention (``prep``, ``insert``), the
sparse indexer's logits (``index_prefill``, ``index_decode``), its top-k and
the attention over the selected rows (``attn_prefill``, ``mla_prefill``,
``attn_decode``, ``mla_decode``), and the FP8 output projection (``oproj``).
Sizes are those of this repository's benchmark workloads (``bench.py``,
``flaggems_vllm/testing.py``) or lie between them, odd ones included.

``listed`` gives the cases, ``draw`` more of the same ranges, ``prepare`` the
tensors that the engine holds before the call, ``run`` one call sequence
through the package's public functions, ``exact`` the same outputs in 64 bits
from plain torch.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "flaggems-vllm_amd"))
import flaggems_vllm as fv  # noqa: E402

DEV = "cuda"
HEAD, NOPE, ROPE = 512, 448, 64
PAGE = 64          # tokens per cache page
RATIO = 4          # tokens per compressed key
WINDOW = 128       # sliding-window tokens
EPS = 1e-6
MAX_POS = 65536
SCALE = HEAD ** -0.5
BF16, F32, F64, I32, I64 = torch.bfloat16, torch.float32, torch.float64, torch.int32, torch.int64


# ------------------------------------------------------------------- cases ----

def listed():
    return [
        # a decode step's pre-attention work for a handful of sequences: four short calls, launch-bound
        {"name": "prep_decode_8", "op": "prep", "tokens": 8, "heads": 64, "fp4": False},
        # the same for an odd chunk of a prefill, the wide model and the MXFP4 indexer
        {"name": "prep_prefill_2047", "op": "prep", "tokens": 2047, "heads": 128, "fp4": True},
        # the benchmark's headline call: a full prefill chunk through the fused q-norm / RoPE / cache insert
        {"name": "insert_8192", "op": "insert", "tokens": 8192, "heads": 64},
        # the sparse indexer of a prefill chunk: cached keys gathered, then every query against every visible key
        {"name": "index_prefill_4096x8192", "op": "index_prefill", "queries": 4096, "keys": 8192, "fp4": False},
        # the indexer of a decode step over long contexts, keys read through the page table
        {"name": "index_decode_32x65536", "op": "index_decode", "batch": 32, "next_n": 1, "ctx": 65536, "fp4": False},
        # decode attention of a small ragged batch: top-k of the logits, page slots, attention over window and top-k
        {"name": "attn_decode_24", "op": "attn_decode", "batch": 24, "heads": 64, "keys": 16384, "topk": 512},
        # decode attention of a full batch, window of 128 and 512 selected entries, ragged lengths
        {"name": "mla_decode_512", "op": "mla_decode", "batch": 512, "heads": 64, "extra": 512},
        # prefill attention of three requests: cache rows dequantised and gathered, top-k, index rows, attention
        {"name": "attn_prefill_3001", "op": "attn_prefill", "tokens": 3001, "requests": 3, "ctx": 16384, "heads": 64,
         "topk": 512},
        # prefill attention alone at the reference benchmark's widest heads: the heaviest call here
        {"name": "mla_prefill_v32_4096", "op": "mla_prefill", "tokens": 4096, "kv": 32768, "topk": 2048, "heads": 128,
         "dim": 576, "ragged": False},
        # an odd, ragged chunk at 128 heads and head dim 512
        {"name": "mla_prefill_1021", "op": "mla_prefill", "tokens": 1021, "kv": 65536, "topk": 1024, "heads": 128,
         "dim": 512, "ragged": True},
        # output projection of a decode batch: inverse RoPE, FP8 codes, grouped block-FP8 product (weight streaming)
        {"name": "oproj_decode_96", "op": "oproj", "tokens": 96, "groups": 8, "hpg": 8},
        # the same for a full prefill chunk (matrix-bound)
        {"name": "oproj_prefill_8192", "op": "oproj", "tokens": 8192, "groups": 8, "hpg": 8},
    ]


def _size(rng, lo, hi):
    """An integer of [lo, hi], spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _drawn(rng):
    op = rng.choice(("prep", "insert", "index_prefill", "index_decode", "attn_decode", "mla_decode", "attn_prefill",
                     "mla_prefill", "oproj"))
    if op == "prep":
        return {"op": op, "tokens": _size(rng, 4, 4096), "heads": rng.choice((64, 128)), "fp4": rng.random() < 0.5}
    if op == "insert":
        return {"op": op, "tokens": _size(rng, 256, 8192), "heads": rng.choice((64, 128))}
    if op == "index_prefill":
        return {"op": op, "queries": _size(rng, 16, 4096), "keys": _size(rng, 256, 16384), "fp4": rng.random() < 0.5}
    if op == "index_decode":
        return {"op": op, "batch": _size(rng, 1, 256), "next_n": rng.choice((1, 1, 2)), "ctx": _size(rng, 512, 65536),
                "fp4": rng.random() < 0.3}
    if op == "attn_decode":
        return {"op": op, "batch": _size(rng, 1, 128), "heads": rng.choice((64, 128)), "keys": _size(rng, 600, 65536),
                "topk": rng.choice((512, 1024))}
    if op == "mla_decode":
        return {"op": op, "batch": _size(rng, 1, 512), "heads": rng.choice((64, 128)), "extra": rng.choice((0, 512, 512, 8192))}
    if op == "attn_prefill":
        return {"op": op, "tokens": _size(rng, 64, 4096), "requests": rng.randint(1, 6), "ctx": _size(rng, 4096, 32768),
                "heads": 64, "topk": 512}
    if op == "mla_prefill":
        topk, heads, dim = rng.choice(((512, 64, 512), (1024, 128, 512), (2048, 128, 576)))
        return {"op": op, "tokens": _size(rng, 16, 4096), "kv": _size(rng, 2048, 131072), "topk": topk, "heads": heads,
                "dim": dim, "ragged": rng.random() < 0.5}
    groups, hpg = rng.choice(((8, 8), (16, 8), (16, 14)))
    return {"op": op, "tokens": _size(rng, 1, 8192), "groups": groups, "hpg": hpg}


def _cost(case):
    w = work(case)
    return max(w["bytes"] / 4e12, w["flops"] / 1e15)


def draw(rng):
    most = max(_cost(c) for c in listed())
    while True:
        case = _drawn(rng)
        if _cost(case) <= most:
            return case


# ------------------------------------------------------------------ inputs ----

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(g, *shape, std=1.0):
    x = torch.randn(shape, device=DEV, dtype=BF16, generator=g)
    return x if std == 1.0 else x.mul_(std)


def _cos_sin(max_pos=MAX_POS):
    theta = 10000.0 ** (-torch.arange(0, ROPE, 2, device=DEV, dtype=F64) / ROPE)
    ang = torch.arange(max_pos, device=DEV, dtype=F64)[:, None] * theta
    return torch.cat((ang.cos(), ang.sin()), -1).to(F32)


def _fp8_rows(x):
    """(e4m3fn codes, float32 scale) per row of 128, as the indexer's key cache holds them."""
    sf = x.float().abs().amax(-1).clamp_min(1e-4) / 448.0
    return (x.float() / sf[..., None]).to(torch.float8_e4m3fn), sf


def _mxfp4(x):
    """(packed nibbles [..., 64] uint8, UE8M0 words [...] int32) of x [..., 128]."""
    b = x.float().reshape(*x.shape[:-1], 4, 32)
    e = torch.ceil(torch.log2(b.abs().amax(-1, keepdim=True).clamp_min(1e-30) / 6.0))
    y = (b / torch.exp2(e)).clamp(-6.0, 6.0)
    edges = torch.tensor([0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0], device=DEV)
    code = (torch.bucketize(y.abs(), edges) + 8 * (y < 0)).reshape(x.shape).to(torch.uint8)
    byte = (e.squeeze(-1) + 127).to(I64)
    word = byte[..., 0] | byte[..., 1] << 8 | byte[..., 2] << 16 | byte[..., 3] << 24
    return (code[..., 0::2] | code[..., 1::2] << 4), torch.where(word >= 2 ** 31, word - 2 ** 32, word).to(I32)


def _from_mxfp4(q):
    packed, word = q
    mags = torch.tensor([0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0], device=DEV, dtype=F64)
    code = torch.stack((packed & 15, packed >> 4), -1).reshape(*packed.shape[:-1], 128).to(I64)
    x = mags[code & 7] * (1 - 2 * (code >> 3))
    e = torch.stack([(word >> (8 * i)) & 255 for i in range(4)], -1).to(F64) - 127
    return (x.reshape(*x.shape[:-1], 4, 32) * torch.exp2(e)[..., None]).reshape(x.shape)


def _token_cache(g, pages):
    """[pages, PAGE, 1, 584] uint8: 448 e4m3fn codes and 64 bf16 rope values a token, then 8 scale bytes a token."""
    n = pages * PAGE
    groups = torch.randn(n, 7, 64, device=DEV, generator=g).to(BF16).float()
    e = torch.ceil(torch.log2(groups.abs().amax(-1).clamp_min(1e-4) / 448.0))
    codes = (groups / torch.exp2(e)[..., None]).clamp(-448, 448).reshape(n, NOPE).to(torch.float8_e4m3fn)
    data = torch.cat((codes.view(torch.uint8), _randn(g, n, ROPE).view(torch.uint8).reshape(n, 2 * ROPE)), 1)
    scales = torch.zeros(n, 8, device=DEV, dtype=torch.uint8)
    scales[:, :7] = (e + 127).to(torch.uint8)
    return torch.cat((data.view(pages, -1), scales.view(pages, -1)), 1).view(pages, PAGE, 1, 584)


def _from_token_cache(cache):
    """The cache's rows [pages * page, 512] in 64 bits."""
    pages, page = cache.shape[:2]
    flat = cache.reshape(pages, -1)
    data = flat[:, :page * 576].reshape(-1, 576)
    e = flat[:, page * 576:].reshape(-1, 8)[:, :7].to(F64) - 127
    nope = data[:, :NOPE].contiguous().view(torch.float8_e4m3fn).to(F64).view(-1, 7, 64) * torch.exp2(e)[..., None]
    return torch.cat((nope.view(-1, NOPE), data[:, NOPE:].contiguous().view(BF16).to(F64)), 1)


def _index_cache(g, pages):
    """[pages, PAGE, 132] uint8: PAGE x 128 codes, then PAGE float32 scales."""
    codes, sf = _fp8_rows(_randn(g, pages, PAGE, 128))
    return torch.cat((codes.view(torch.uint8).reshape(pages, -1), sf.view(torch.uint8).reshape(pages, -1)),
                     1).view(pages, PAGE, 132)


def _tables(g, counts):
    """A page table [requests, most pages] of distinct random pages, and the number of pages."""
    need = [-(-c // PAGE) for c in counts]
    pool = torch.randperm(sum(need) + 8, device=DEV, generator=g).to(I32)
    table, at = torch.zeros(len(need), max(need), device=DEV, dtype=I32), 0
    for r, n in enumerate(need):
        table[r, :n] = pool[at:at + n]
        at += n
    return table, pool.numel()


def _lengths(case):
    """Sizes that a ragged case has, made from its own values so that work() knows them: 0.7 to 1.3 of the mean."""
    if case["op"] == "index_decode":
        return [max(1, int(case["ctx"] * (0.7 + 0.6 * ((7 * i + 3) % 10) / 9))) for i in range(case["batch"])]
    if case["op"] == "attn_decode":
        return [max(1, int(case["keys"] * (0.5 + 0.5 * ((7 * i + 3) % 10) / 9))) for i in range(case["batch"])]
    n, r = case["tokens"], case["requests"]  # attn_prefill: (new tokens, context) of each request
    new = [n * (i + 1) // r - n * i // r for i in range(r)]
    return [(t, max(t, int(case["ctx"] * (0.6 + 0.4 * i / max(1, r - 1))))) for i, t in enumerate(new)]


def prepare(case, seed):
    return dict(globals()["_prepare_" + case["op"]](case, _gen(seed)), case=case)


def run(state):
    return globals()["_run_" + state["case"]["op"]](state)


def _prepare_insert(case, g):
    t, pages = case["tokens"], 4 * -(-case["tokens"] // PAGE)
    return {"q": _randn(g, t, case["heads"], HEAD), "kv": _randn(g, t, HEAD),
            "cache": torch.zeros(pages, PAGE * 584, device=DEV, dtype=torch.uint8),
            "slots": torch.randperm(pages * PAGE, device=DEV, generator=g)[:t].contiguous(),
            "pos": torch.randint(0, MAX_POS, (t,), device=DEV, generator=g), "cs": _cos_sin()}


def _run_insert(s):
    fv.fused_deepseek_v4_qnorm_rope_kv_rope_quant_insert(s["q"], s["kv"], s["cache"], s["slots"], s["pos"], s["cs"], EPS,
                                                         PAGE)
    return {"q": s["q"], "cache": s["cache"]}


def _prepare_prep(case, g):
    s, t = _prepare_insert(case, g), case["tokens"]
    s.update(qr=_randn(g, t, 1536), qw=_randn(g, 1536), kw=_randn(g, HEAD), iq=_randn(g, t, 64, 128),
             iw=_randn(g, t, 64), ik=_randn(g, t, 128),
             icache=torch.zeros(s["cache"].shape[0], PAGE, 132, device=DEV, dtype=torch.uint8))
    return s


def _run_prep(s):
    qr, kv = fv.fused_q_kv_rmsnorm(s["qr"], s["kv"], s["qw"], s["kw"], EPS)
    fv.fused_deepseek_v4_qnorm_rope_kv_rope_quant_insert(s["q"], kv, s["cache"], s["slots"], s["pos"], s["cs"], EPS, PAGE)
    iq, iw = fv.fused_indexer_q_rope_quant(s["pos"], s["iq"], s["cs"], s["iw"], 128 ** -0.5, 64 ** -0.5,
                                           use_fp4=s["case"]["fp4"])
    fv.indexer_k_quant_and_cache(s["ik"], s["icache"], s["slots"], 128, "ue8m0")
    return {"qr": qr, "kv": kv, "q": s["q"], "cache": s["cache"], "iq": list(iq) if isinstance(iq, tuple) else iq, "iw": iw,
            "icache": s["icache"]}


def _prepare_index_prefill(case, g):
    m, n = case["queries"], case["keys"]
    table, pages = _tables(g, [n])
    q = _randn(g, m, 64, 128)
    ctx = RATIO * n - m + torch.arange(1, m + 1, device=DEV)
    return {"q": _mxfp4(q) if case["fp4"] else (q.to(torch.float8_e4m3fn), None),
            "w": torch.randn(m, 64, device=DEV, generator=g).abs(), "icache": _index_cache(g, pages), "table": table,
            "cu": torch.tensor([0, n], device=DEV, dtype=I32),
            "k": torch.empty(n, 128, device=DEV, dtype=torch.float8_e4m3fn),
            "ks": torch.empty(n, 4, device=DEV, dtype=torch.uint8),
            "lo": torch.zeros(m, device=DEV, dtype=I32), "hi": (ctx.clamp_min(RATIO) // RATIO).to(I32)}


def _run_index_prefill(s):
    fv.cp_gather_indexer_k_quant_cache(s["icache"], s["k"], s["ks"], s["table"], s["cu"])
    return fv.fp8_fp4_mqa_logits(s["q"], (s["k"], s["ks"].view(F32)), s["w"], s["lo"], s["hi"])


def _max_len(case):
    return -(-int(1.3 * case["ctx"] + 1) // 4096) * 4096


def _prepare_index_decode(case, g):
    lens = _lengths(case)
    table, pages = _tables(g, lens)
    q = _randn(g, case["batch"], case["next_n"], 64, 128)
    return {"q": _mxfp4(q) if case["fp4"] else (q.to(torch.float8_e4m3fn), None),
            "w": torch.randn(case["batch"] * case["next_n"], 64, device=DEV, generator=g),
            "icache": _index_cache(g, pages).unsqueeze(2), "table": table,
            "lens": torch.tensor(lens, device=DEV, dtype=I32)[:, None].repeat(1, case["next_n"])}


def _run_index_decode(s):
    return fv.fp8_fp4_paged_mqa_logits(s["q"], s["icache"], s["w"], s["lens"], s["table"], None, _max_len(s["case"]))


def _prepare_attn_decode(case, g):
    b, lens = case["batch"], _lengths(case)
    table, pages = _tables(g, lens)
    swa = 4 * b
    return {"q": _randn(g, b, 1, case["heads"], HEAD, std=2.0), "cache": _token_cache(g, swa),
            "extra": _token_cache(g, pages), "table": table,
            "logits": torch.randn(b, case["keys"], device=DEV, generator=g),
            "lens": torch.tensor(lens, device=DEV, dtype=I32),
            "swa": torch.randint(0, swa * PAGE, (b, 1, WINDOW), device=DEV, generator=g, dtype=I32),
            "swa_len": torch.full((b,), WINDOW, device=DEV, dtype=I32),
            "sink": torch.randn(case["heads"], device=DEV, generator=g),
            "local": torch.empty(b, case["topk"], device=DEV, dtype=I32),
            "req": torch.arange(b, device=DEV, dtype=I32)}


def _run_attn_decode(s):
    logits, local = s["logits"], s["local"]
    b, topk = local.shape
    fv.top_k_per_row_decode(logits, 1, s["lens"], local, b, logits.stride(0), logits.stride(1), topk)
    slots, count = fv.compute_global_topk_indices_and_lens(local, s["req"], s["table"], PAGE)
    out, lse = fv.flash_mla_with_kvcache(
        s["q"], s["cache"], None, None, HEAD, fv.get_mla_metadata()[0], softmax_scale=SCALE, is_fp8_kvcache=True,
        indices=s["swa"], attn_sink=s["sink"], extra_k_cache=s["extra"], extra_indices_in_kvcache=slots.unsqueeze(1),
        topk_length=s["swa_len"], extra_topk_length=count)
    return {"count": count, "out": out, "lse": lse}


def _prepare_mla_decode(case, g):
    b, pages = case["batch"], 512
    s = {"q": _randn(g, b, 1, case["heads"], HEAD, std=2.0), "cache": _token_cache(g, pages),
         "swa": torch.randint(0, pages * PAGE, (b, 1, WINDOW), device=DEV, generator=g, dtype=I32),
         "swa_len": torch.randint(1, WINDOW + 1, (b,), device=DEV, generator=g, dtype=I32),
         "sink": torch.randn(case["heads"], device=DEV, generator=g), "extra": None, "idx": None, "len": None}
    if case["extra"]:
        n = case["extra"]
        s["extra"] = _token_cache(g, pages)
        s["idx"] = torch.randint(0, pages * PAGE, (b, 1, n), device=DEV, generator=g, dtype=I32)
        s["len"] = torch.randint(1, n + 1, (b,), device=DEV, generator=g, dtype=I32)
    return s


def _run_mla_decode(s):
    out, lse = fv.flash_mla_with_kvcache(
        s["q"], s["cache"], None, None, HEAD, fv.get_mla_metadata()[0], softmax_scale=SCALE, is_fp8_kvcache=True,
        indices=s["swa"], attn_sink=s["sink"], extra_k_cache=s["extra"], extra_indices_in_kvcache=s["idx"],
        topk_length=s["swa_len"], extra_topk_length=s["len"])
    return {"out": out, "lse": lse}


def _prepare_attn_prefill(case, g):
    per = _lengths(case)
    new, ctx = [p[0] for p in per], [p[1] for p in per]
    comp = [c // RATIO for c in ctx]
    swa = [min(c, t + WINDOW - 1) for t, c in per]
    n = max(comp)
    table, pages = _tables(g, comp)
    swa_table, swa_pages = _tables(g, ctx)
    starts, row = [0], []
    for c in comp:
        starts.append(starts[-1] + c)
    lo, hi = [], []
    for r, (t, c) in enumerate(per):
        visible = (torch.arange(c - t + 1, c + 1, device=DEV) // RATIO)
        lo.append(torch.full((t,), starts[r], device=DEV, dtype=I32))
        hi.append((starts[r] + visible).to(I32))
    cum = [0]
    for t in new:
        cum.append(cum[-1] + t)
    ints = lambda v: torch.tensor(v, device=DEV, dtype=I32)  # noqa: E731
    return {"q": _randn(g, case["tokens"], case["heads"], HEAD, std=2.0), "cache": _token_cache(g, pages),
            "swa_cache": _token_cache(g, swa_pages), "table": table, "swa_table": swa_table, "comp": ints(comp),
            "ctx": ints(ctx), "swa": ints(swa), "qsl": ints(cum), "n": n,
            "rows": torch.zeros(len(per), n + max(swa), HEAD, device=DEV, dtype=BF16),
            "logits": torch.randn(case["tokens"], starts[-1], device=DEV, generator=g), "lo": torch.cat(lo),
            "hi": torch.cat(hi), "local": torch.empty(case["tokens"], case["topk"], device=DEV, dtype=I32),
            "sink": torch.randn(case["heads"], device=DEV, generator=g)}


def _run_attn_prefill(s):
    rows, logits, local = s["rows"], s["logits"], s["local"]
    t, topk = local.shape
    fv.dequantize_and_gather_k_cache(rows, s["cache"].view(s["cache"].shape[0], -1), s["comp"], None, s["table"], PAGE)
    fv.dequantize_and_gather_k_cache(rows, s["swa_cache"].view(s["swa_cache"].shape[0], -1), s["ctx"], s["swa"],
                                     s["swa_table"], PAGE, s["n"])
    fv.top_k_per_row_prefill(logits, s["lo"], s["hi"], local, t, logits.stride(0), logits.stride(1), topk)
    idx, count = fv.combine_topk_swa_indices(local, s["qsl"], s["ctx"], s["swa"], WINDOW, RATIO, topk, rows.shape[1],
                                             s["n"])
    out, top, lse = fv.flash_mla_sparse_fwd(s["q"], rows.view(-1, 1, HEAD), idx.unsqueeze(1), SCALE, HEAD, s["sink"], count)
    return {"rows": rows, "count": count, "out": out, "top": top, "lse": lse}


def _prepare_mla_prefill(case, g):
    t, n, topk = case["tokens"], case["kv"], case["topk"]
    step = torch.tensor([p for p in (7919, 104729, 1299709, 15485863, 32452843, 49979687) if math.gcd(p, n) == 1],
                        device=DEV)
    pick = step[torch.randint(0, step.numel(), (t, 1), device=DEV, generator=g)]
    at = torch.randint(0, n, (t, 1), device=DEV, generator=g)
    return {"q": _randn(g, t, case["heads"], case["dim"], std=2.0), "kv": _randn(g, n, 1, case["dim"]),
            "idx": ((at + pick * torch.arange(topk, device=DEV)) % n).to(I32).unsqueeze(1),
            "sink": torch.randn(case["heads"], device=DEV, generator=g),
            "len": torch.randint(1, topk + 1, (t,), device=DEV, generator=g, dtype=I32) if case["ragged"] else None}


def _run_mla_prefill(s):
    out, top, lse = fv.flash_mla_sparse_fwd(s["q"], s["kv"], s["idx"], s["case"]["dim"] ** -0.5, HEAD, s["sink"], s["len"])
    return {"out": out, "top": top, "lse": lse}


def _prepare_oproj(case, g):
    t, h, r = case["tokens"], case["groups"], case["hpg"] * HEAD
    return {"o": _randn(g, t, h * case["hpg"], HEAD), "pos": torch.randint(0, MAX_POS, (t,), device=DEV, generator=g),
            "cs": _cos_sin(), "y": _randn(g, h, 1024, r).to(torch.float8_e4m3fn),
            "ys": torch.rand(h, 8, r // 128, device=DEV, generator=g) * 1e-2 + 1e-3}


def _run_oproj(s):
    codes, scales = fv.fused_inv_rope_fp8_quant(s["o"], s["pos"], s["cs"], s["case"]["groups"], s["case"]["hpg"])
    return {"codes": codes, "scales": scales, "out": fv.fp8_einsum("bhr,hdr->bhd", codes, scales, s["y"], s["ys"])}


# -------------------------------------------------------------------- work ----

def work(case):
    """What a pass cannot do without: every input it needs read once, every output written once."""
    op = case["op"]
    if op in ("prep", "insert"):
        t, h = case["tokens"], case["heads"]
        nbytes = t * (4 * HEAD * h + 2 * HEAD + 584 + 16 + 256)
        if op == "prep":
            nbytes += t * (4 * 1536 + 4 * HEAD) + 4 * (1536 + HEAD)
            nbytes += t * 64 * (256 + (68 if case["fp4"] else 128) + 6) + t * (256 + 132)
        return {"bytes": nbytes, "flops": 0}
    if op == "index_prefill":
        m, n = case["queries"], case["keys"]
        seen = sum(max(1, (RATIO * n - m + i) // RATIO) for i in range(1, m + 1))
        return {"bytes": 132 * 3 * n + m * 64 * (68 if case["fp4"] else 128) + 256 * m + 4 * m * n, "flops": 2 * 64 * 128 * seen}
    if op == "index_decode":
        seen, rows = sum(_lengths(case)), case["batch"] * case["next_n"]
        return {"bytes": 132 * seen + rows * (64 * (68 if case["fp4"] else 128) + 256 + 4 * _max_len(case)),
                "flops": 2 * 64 * 128 * seen * case["next_n"]}
    if op in ("attn_decode", "mla_decode"):
        b, h = case["batch"], case["heads"]
        if op == "attn_decode":
            lens = _lengths(case)
            used = [WINDOW + min(n, case["topk"]) for n in lens]
            rows, nbytes = sum(used), 4 * sum(lens) + 12 * b * case["topk"]
        else:  # uniform lengths: their mean, and a cache row no more often than it is there
            rows = b * ((WINDOW + 1) // 2 + (case["extra"] + 1) // 2)
            nbytes = 4 * rows
        distinct = min(rows, (2 if case["op"] == "mla_decode" and case["extra"] else 1) * 512 * PAGE) \
            if op == "mla_decode" else rows
        return {"bytes": nbytes + 584 * distinct + 4 * HEAD * b * h + 4 * b * h, "flops": 4 * HEAD * h * rows}
    if op == "attn_prefill":
        per, t = _lengths(case), case["tokens"]
        comp = [c // RATIO for _, c in per]
        seen = picked = 0
        for n, c in per:
            for i in range(c - n + 1, c + 1):
                seen += i // RATIO
                picked += min(i // RATIO, case["topk"]) + min(i, WINDOW)
        rows = sum(comp) + sum(min(c, n + WINDOW - 1) for n, c in per)
        return {"bytes": rows * (584 + 1024) + 4 * seen + 4 * t * (2 * case["topk"] + WINDOW) + 4 * HEAD * t * case["heads"],
                "flops": 4 * HEAD * case["heads"] * picked}
    if op == "mla_prefill":
        t, h = case["tokens"], case["heads"]
        rows = t * ((case["topk"] + 1) // 2 if case["ragged"] else case["topk"])
        return {"bytes": 2 * t * h * (case["dim"] + HEAD) + 8 * t * h + 4 * rows + 2 * case["dim"] * min(case["kv"], rows),
                "flops": 2 * (case["dim"] + HEAD) * h * rows}
    t, h, r = case["tokens"], case["groups"], case["hpg"] * HEAD
    return {"bytes": t * h * r * 3 + t * h * r // 32 + h * 1024 * r + 2 * t * h * 1024 + 264 * t,
            "flops": 2 * t * h * 1024 * r}


def tolerance(case):
    """About four times what the path is off its 64-bit value: 1.7e-3 where bf16 outputs are rounded once, 2.2e-3 where
    the probabilities are held in bf16 beside them, 3.5e-3 where the scaled FP8 sums go to bf16, 1.3e-5 for the float32
    logits of FP8 products.  Codes, cache bytes and counts are whole numbers that do not move."""
    op = case["op"]
    if op in ("prep", "insert"):
        return {"rel": 7e-3, "max": 5e-2}
    if op in ("index_prefill", "index_decode"):
        return {"rel": 5e-5, "max": 2e-3}
    return {"rel": 1.4e-2 if op == "oproj" else 9e-3, "max": 1e-1}


# ------------------------------------------------------------------- exact ----

def exact(case, seed):
    s = prepare(case, seed)
    return globals()["_exact_" + case["op"]](case, s)


def _rms(x):
    return x * (x.square().mean(-1, keepdim=True) + EPS).rsqrt()


def _rope(x, cs, pos, inverse=False):
    """x [t, ..., 512] with its last 64 values rotated in pairs."""
    c = cs[pos].to(F64).view(-1, *(1,) * (x.dim() - 2), ROPE)
    cos, sin = c[..., :ROPE // 2], c[..., ROPE // 2:]
    sin = -sin if inverse else sin
    e, o = x[..., NOPE::2], x[..., NOPE + 1::2]
    return torch.cat((x[..., :NOPE], torch.stack((e * cos - o * sin, e * sin + o * cos), -1).flatten(-2)), -1)


def _exact_insert(case, s):
    return {"q": _rope(_rms(s["q"].to(F64)), s["cs"], s["pos"]), "cache": None}


def _exact_prep(case, s):
    qr, kv = _rms(s["qr"].to(F64)) * s["qw"].to(F64), _rms(s["kv"].to(F64)) * s["kw"].to(F64)
    return dict(_exact_insert(case, s), qr=qr, kv=kv, iq=None, iw=None, icache=None)


def _index_logits(q, w, k, sf):
    """q [m, 64, 128], w [m, 64], k [n, 128], sf [n] in 64 bits."""
    out = torch.empty(q.shape[0], k.shape[0], device=DEV, dtype=F64)
    step = max(1, (1 << 27) // (64 * k.shape[0]))
    for i in range(0, q.shape[0], step):
        qi, wi = q[i:i + step], w[i:i + step]
        dots = (qi.reshape(-1, 128) @ k.t()).view(qi.shape[0], 64, -1)
        out[i:i + step] = (dots.clamp_min_(0) * wi[..., None]).sum(1) * sf
    return out


def _index_keys(cache):
    flat = cache.reshape(cache.shape[0], -1)
    codes = flat[:, :PAGE * 128].contiguous().view(torch.float8_e4m3fn).to(F64).view(-1, PAGE, 128)
    return codes, flat[:, PAGE * 128:].contiguous().view(F32).to(F64)


def _index_q(q):
    return q[0].to(F64) if q[1] is None else _from_mxfp4(q)


def _exact_index_prefill(case, s):
    codes, sf = _index_keys(s["icache"])
    pages, n = s["table"][0].long(), case["keys"]
    out = _index_logits(_index_q(s["q"]), s["w"].to(F64), codes[pages].view(-1, 128)[:n], sf[pages].view(-1)[:n])
    return out.masked_fill_(torch.arange(n, device=DEV) >= s["hi"][:, None], -math.inf)


def _exact_index_decode(case, s):
    codes, sf = _index_keys(s["icache"])
    q, w, nn = _index_q(s["q"]).flatten(0, 1), s["w"].to(F64), case["next_n"]
    out = torch.zeros(q.shape[0], _max_len(case), device=DEV, dtype=F64)
    for b, n in enumerate(_lengths(case)):
        pages, rows = s["table"][b, :-(-n // PAGE)].long(), slice(b * nn, (b + 1) * nn)
        out[rows, :n] = _index_logits(q[rows], w[rows], codes[pages].view(-1, 128)[:n], sf[pages].view(-1)[:n])
    return out


def _attend(q, pick, live, scale, sink):
    """q [t, h, d]; pick(i, j): the keys [j - i, k, d] of tokens i to j; live [t, k]."""
    t, h, _ = q.shape
    out = torch.empty(t, h, HEAD, device=DEV, dtype=F64)
    top, lse = torch.empty(t, h, device=DEV, dtype=F64), torch.empty(t, h, device=DEV, dtype=F64)
    step = max(1, (1 << 28) // (live.shape[1] * 1024))
    for i in range(0, t, step):
        j = min(t, i + step)
        k = pick(i, j)
        z = torch.bmm(q[i:j].to(F64), k.transpose(1, 2).contiguous()).mul_(scale)
        z.masked_fill_(~live[i:j, None], -math.inf)
        top[i:j], lse[i:j] = z.amax(-1), torch.logsumexp(z, -1)
        p = torch.exp(z - torch.logaddexp(lse[i:j], sink.to(F64))[..., None])
        out[i:j] = torch.bmm(p, k[..., :HEAD].contiguous())
    return out, top, lse


def _exact_mla_prefill(case, s):
    k, idx = s["kv"][:, 0], s["idx"][:, 0].long()
    live = torch.ones_like(idx, dtype=torch.bool)
    if s["len"] is not None:
        live = torch.arange(idx.shape[1], device=DEV) < s["len"][:, None]
    out, top, lse = _attend(s["q"], lambda i, j: k[idx[i:j]].to(F64), live, case["dim"] ** -0.5, s["sink"])
    return {"out": out, "top": top, "lse": lse}


def _decode(s, extra, idx, live):
    """Attention of one query over the window rows and the rows `idx` of `extra`."""
    rows = torch.cat((_from_token_cache(s["cache"]), extra))
    first = s["cache"].shape[0] * PAGE
    every = torch.cat((s["swa"][:, 0].long(), first + idx), 1)
    ok = torch.cat((torch.arange(WINDOW, device=DEV) < s["swa_len"][:, None], live), 1)
    out, _, lse = _attend(s["q"][:, 0], lambda i, j: rows[every[i:j]], ok, SCALE, s["sink"])
    return out.unsqueeze(1), lse.unsqueeze(2)


def _exact_mla_decode(case, s):
    if s["extra"] is None:
        extra = torch.zeros(0, HEAD, device=DEV, dtype=F64)
        idx = torch.zeros(case["batch"], 0, device=DEV, dtype=I64)
        live = idx > 0
    else:
        extra, idx = _from_token_cache(s["extra"]), s["idx"][:, 0].long()
        live = torch.arange(idx.shape[1], device=DEV) < s["len"][:, None]
    out, lse = _decode(s, extra, idx, live)
    return {"out": out, "lse": lse}


def _exact_attn_decode(case, s):
    z = s["logits"].masked_fill(torch.arange(case["keys"], device=DEV) >= s["lens"][:, None], -math.inf)
    best = z.topk(min(case["topk"], case["keys"]), -1)
    live = best.values > -math.inf
    at = torch.where(live, best.indices, 0)
    idx = s["table"].long().gather(1, at // PAGE) * PAGE + at % PAGE
    out, lse = _decode(s, _from_token_cache(s["extra"]), idx, live)
    return {"count": None, "out": out, "lse": lse}


def _exact_attn_prefill(case, s):
    comp, swa_rows, width = _from_token_cache(s["cache"]), _from_token_cache(s["swa_cache"]), s["rows"].shape[1]
    rows = torch.zeros(s["rows"].shape, device=DEV, dtype=F64)
    base, first = [], []
    for r, (t, c) in enumerate(_lengths(case)):
        n, m = c // RATIO, min(c, t + WINDOW - 1)
        at = torch.arange(n, device=DEV)
        rows[r, :n] = comp[s["table"][r, at // PAGE].long() * PAGE + at % PAGE]
        at = torch.arange(c - m, c, device=DEV)
        rows[r, s["n"]:s["n"] + m] = swa_rows[s["swa_table"][r, at // PAGE].long() * PAGE + at % PAGE]
        pos = torch.arange(c - t, c, device=DEV)
        base.append(torch.full((t,), r * width, device=DEV))
        first.append(torch.stack((pos, torch.full((t,), c - m, device=DEV))))
    base, (pos, start) = torch.cat(base)[:, None], torch.cat(first, 1)
    cols = torch.arange(s["logits"].shape[1], device=DEV)
    z = s["logits"].masked_fill((cols < s["lo"][:, None]) | (cols >= s["hi"][:, None]), -math.inf)
    best = z.topk(min(case["topk"], z.shape[1]), -1)
    live = best.values > -math.inf
    idx = torch.where(live, best.indices - s["lo"][:, None] + base, 0)
    back = pos[:, None] - torch.arange(WINDOW, device=DEV)
    idx = torch.cat((idx, torch.where(back >= 0, base + s["n"] + back - start[:, None], 0)), 1)
    flat = rows.view(-1, HEAD)
    out, top, lse = _attend(s["q"], lambda i, j: flat[idx[i:j]], torch.cat((live, back >= 0), 1), SCALE, s["sink"])
    return {"rows": rows, "count": None, "out": out, "top": top, "lse": lse}


def _exact_oproj(case, s):
    t, h, r = case["tokens"], case["groups"], case["hpg"] * HEAD
    scales = torch.empty(t, h, r // 128, device=DEV, dtype=F64)
    x = torch.empty(t, h, r, device=DEV, dtype=F64)
    for i in range(0, t, 512):
        o = _rope(s["o"][i:i + 512].to(F64), s["cs"], s["pos"][i:i + 512], inverse=True).to(BF16).to(F64)
        blocks = o.view(o.shape[0], h, r // 128, 128)
        sf = blocks.abs().amax(-1).clamp_min(1e-10) / 448.0
        codes = (blocks / sf[..., None]).clamp(-448, 448).to(F32).to(torch.float8_e4m3fn).to(F64)
        scales[i:i + 512] = sf
        x[i:i + 512] = (codes * sf[..., None]).reshape(o.shape[0], h, r)
    y = (s["y"].to(F64).view(h, 8, 128, r // 128, 128) * s["ys"].to(F64)[:, :, None, :, None]).view(h, 1024, r)
    out = torch.stack([x[:, j] @ y[j].t() for j in range(h)], 1)
    return {"codes": None, "scales": scales, "out": out}
