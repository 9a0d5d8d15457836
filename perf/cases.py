"""Cases for timing the paged-KV attention operator through its public entry points.

A case is a dict of sizes and options.  ``kind`` "attend" is one call of
``pagedkv.flash_attn_with_kvcache`` (``pagedkv.decode`` for FP8 caches, whose scales
only that entry takes): decode steps, steps that append their new tokens, speculative
verify steps and prefill chunks over a paged cache.  ``kind`` "append" is one
``pagedkv.reshape_and_cache_flash``: the cache write of a batch of prompts.

Row lengths follow from the case alone (``lens_seed``), so the work of a case is
fixed; values, page placement and slots follow from the seed.
"""
import importlib
import math
import os
import random
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "flashatte-hand_amd"))
pagedkv = importlib.import_module("pagedkv")

LOG_SPREAD = 1.0  # sigma of the "lognormal" row lengths

DEFAULTS = {
    "kind": "attend", "batch": 1, "heads": 32, "kv_heads": 8, "dim": 128, "dtype": "bf16", "kv": "same", "page": 64,
    "len_lo": 1, "len_hi": 4096, "spread": "uniform", "lens_seed": 0,  # cached tokens per row, before the call
    "q": 1,            # query tokens per row
    "new": 0,          # tokens the call appends to each row (0: the caches already hold every token)
    "causal": False, "window": -1, "softcap": 0.0, "alibi": False, "rotary": 0, "lse": False,
}


def _case(**kw):
    return {**DEFAULTS, **kw}


def listed():
    return [
        # The smallest call: one short sequence, a single decode token; latency and launches are all of it.
        _case(name="decode_tiny_f16", heads=8, kv_heads=2, dtype="f16", page=16, len_lo=256, len_hi=256),
        # The evaluator's default shapes (8 query and 8 KV heads of 256 dims, pages of 16 tokens, equal rows):
        # a small interactive batch.
        _case(name="decode_mha256_bf16", batch=4, heads=8, kv_heads=8, dim=256, page=16, len_lo=2048, len_hi=2048),
        # The 8B-class decode step of a serving batch, ragged rows.
        _case(name="decode_8b_bf16", batch=32, len_lo=512, len_hi=4096, lens_seed=1),
        # The same step over an FP8 cache with per-head scales.
        _case(name="decode_8b_fp8", batch=32, len_lo=512, len_hi=4096, lens_seed=1, kv="fp8"),
        # Long contexts, few rows: split-KV over the whole chip.
        _case(name="decode_long_f16", batch=4, dtype="f16", len_lo=32768, len_hi=131072, spread="even"),
        # 70B-class heads, large batch, log-normal rows.
        _case(name="decode_gqa8_bf16", batch=128, heads=64, page=32, len_lo=1, len_hi=16384, spread="lognormal",
              lens_seed=2),
        # One KV head, wide heads, fully scattered small pages, rows from a single token up.
        _case(name="decode_mqa256_f16", batch=256, heads=16, kv_heads=1, dim=256, dtype="f16", page=16, len_lo=1,
              len_hi=8191, lens_seed=3),
        # A decode step as an engine makes it: rotary embedding, cache write and attention in one call.
        _case(name="step_rotary_bf16", batch=32, len_lo=511, len_hi=4095, lens_seed=4, q=1, new=1, rotary=128),
        # Speculative decoding: four drafted tokens per row verified at once.
        _case(name="verify4_bf16", batch=32, len_lo=508, len_hi=4092, lens_seed=5, q=4, new=4, causal=True),
        # Chunked prefill: a chunk of each prompt is appended and attends what came before it.
        _case(name="prefill_chunk_bf16", batch=4, len_lo=0, len_hi=4096, lens_seed=6, q=512, new=512, causal=True),
        # Prefill with a sliding window and capped scores, 256-dim heads, an odd chunk.
        _case(name="prefill_window_f16", batch=3, heads=16, kv_heads=8, dim=256, dtype="f16", page=16, len_lo=100,
              len_hi=6000, lens_seed=7, q=333, new=333, causal=True, window=1023, softcap=50.0),
        # The cache write of a batch of prompts by slot.
        _case(name="append_prompts_bf16", kind="append", batch=32, len_lo=512, len_hi=4096, lens_seed=1),
    ]


def _log_int(rng, lo, hi):
    """An integer spread over the logarithm of [lo, hi], often not a round one."""
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.5))))))


def draw(rng):
    """A case of the listed ones' ranges: decode, appending steps, prefill chunks and cache writes."""
    while True:
        kind = rng.choice(("decode", "decode", "step", "verify", "prefill", "prefill", "append"))
        c = dict(DEFAULTS)
        c["lens_seed"] = rng.randrange(1 << 20)
        c["dtype"] = rng.choice(("bf16", "bf16", "f16"))
        c["dim"] = rng.choice((64, 128, 128, 128, 256))
        c["kv_heads"] = rng.choice((1, 2, 4, 8))
        c["heads"] = c["kv_heads"] * rng.choice((1, 2, 4, 4, 7, 8, 16))
        c["page"] = rng.choice((16, 32, 64, 256))
        c["spread"] = rng.choice(("uniform", "even", "lognormal"))
        c["kv"] = rng.choice(("same", "same", "same", "fp8"))
        c["batch"] = _log_int(rng, 1, 8 if kind == "prefill" else 256)
        c["len_hi"] = _log_int(rng, 16, 131072 if kind == "decode" else 16384)
        c["len_lo"] = rng.choice((1, max(1, c["len_hi"] // 8)))
        if kind == "append":
            c["kind"] = "append"
            c["heads"] = c["kv_heads"]
        elif kind == "decode":
            c["lse"] = rng.random() < 0.25
        elif kind == "step":
            c["new"] = 1
            if rng.random() < 0.5:
                c["rotary"] = c["dim"]
        elif kind == "verify":
            c["q"] = c["new"] = rng.randint(2, 8)
            c["causal"] = True
        else:
            c["q"] = c["new"] = _log_int(rng, 16, 2048)
            c["causal"] = True
            if rng.random() < 0.3:
                c["rotary"] = c["dim"]
        if c["kind"] == "attend":
            extra = rng.choice(("", "", "", "window", "softcap", "alibi"))
            if extra == "window":
                c["window"] = _log_int(rng, 128, 4096)
            elif extra == "softcap":
                c["softcap"] = 30.0
            elif extra == "alibi":
                c["alibi"] = True
        w = work(c)
        if 1 << 16 <= w["bytes"] <= 1.2e9 and w["flops"] <= 6.5e10 and _pool_bytes(c) <= 4e9:
            return c


def _lens(c):
    """Cached tokens of each row before the call."""
    r = random.Random(c["lens_seed"])
    lo, hi, n = c["len_lo"], c["len_hi"], c["batch"]
    if c["spread"] == "even":
        return [lo + (hi - lo) * (i + 1) // n if n > 1 and i + 1 < n else hi for i in range(n)]
    if c["spread"] == "lognormal":
        med = max(1.0, hi / 8)
        return [max(lo, min(hi, round(med * math.exp(LOG_SPREAD * r.gauss(0, 1))))) for _ in range(n)]
    return [r.randint(lo, hi) for _ in range(n)]


def _visible(c, i, total):
    """Keys [lo, hi) that query token i of a row of `total` tokens sees."""
    pos = total - c["q"] + i
    hi = max(0, min(total, pos + 1)) if c["causal"] else total
    lo = max(0, pos - c["window"]) if c["window"] >= 0 else 0
    return min(lo, hi), hi


def _pages(c):
    """Pages each row needs, and the pool's pages."""
    rows = [(n + c["new"] + c["page"] - 1) // c["page"] for n in _lens(c)]
    return rows, sum(rows) + max(1, sum(rows) // 8)


def _elem(c):
    return 1 if c["kv"] == "fp8" else 2


def _pool_bytes(c):
    return 2 * _pages(c)[1] * c["page"] * c["kv_heads"] * c["dim"] * _elem(c)


def work(case):
    c = {**DEFAULTS, **case}
    lens = _lens(c)
    token = 2 * c["kv_heads"] * c["dim"]  # K and V values of one token
    if c["kind"] == "append":
        return {"bytes": sum(lens) * (token * (2 + _elem(c)) + 8), "flops": 0}
    read = pairs = 0
    for n in lens:
        total = n + c["new"]
        first = _visible(c, 0, total)
        last = _visible(c, c["q"] - 1, total)
        read += max(0, min(last[1], n if c["new"] else total) - first[0])  # cached keys some query sees
        # Visible keys grow by a fixed step per token except where they are cut: count them exactly.
        for i in range(c["q"]):
            lo, hi = _visible(c, i, total)
            pairs += hi - lo
    b = read * token * _elem(c)
    b += c["batch"] * c["new"] * token * (2 + _elem(c))
    b += 2 * 2 * c["batch"] * c["q"] * c["heads"] * c["dim"]
    b += 4 * c["batch"] + 4 * sum((n + c["new"] + c["page"] - 1) // c["page"] for n in lens)
    if c["lse"]:
        b += 4 * c["batch"] * c["q"] * c["heads"]
    return {"bytes": b, "flops": 4 * c["heads"] * c["dim"] * pairs}


def _dt(c):
    return torch.bfloat16 if c["dtype"] == "bf16" else torch.float16


def _normal(gen, shape, dt):
    return torch.randn(shape, generator=gen, device="cuda", dtype=dt)


def prepare(case, seed):
    c = {**DEFAULTS, **case}
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed))
    r = random.Random(int(seed))
    dt, D, P, Hk, H, B, M = _dt(c), c["dim"], c["page"], c["kv_heads"], c["heads"], c["batch"], c["q"]
    lens = _lens(c)
    rows, pool = _pages(c)
    order = torch.randperm(pool, generator=torch.Generator().manual_seed(r.getrandbits(40)))
    s = {"case": c, "scales": {}}
    k = _normal(gen, (pool, P, Hk, D), dt)
    v = _normal(gen, (pool, P, Hk, D), dt)
    if c["kv"] == "fp8":
        # One scale per head, as a calibration over the values' range leaves it.
        s["scales"] = {n: (torch.rand((Hk,), generator=gen, device="cuda") * 0.01 + 0.01) for n in ("k_scale", "v_scale")}
        k = _quantise(k, s["scales"]["k_scale"])
        v = _quantise(v, s["scales"]["v_scale"])
    s["k_cache"], s["v_cache"] = k, v
    if c["kind"] == "append":
        n = sum(lens)
        s["key"] = _normal(gen, (n, Hk, D), dt)
        s["value"] = _normal(gen, (n, Hk, D), dt)
        slots, at = [], 0
        for ln, pg in zip(lens, rows):
            pages = order[at:at + pg]
            slots.append((pages[:, None] * P + torch.arange(P)[None, :]).reshape(-1)[:ln])
            at += pg
        s["slots"] = torch.cat(slots).to("cuda")
        return s
    table = torch.zeros((B, max(rows)), dtype=torch.int32)
    at = 0
    for b, pg in enumerate(rows):
        table[b, :pg] = order[at:at + pg].to(torch.int32)
        at += pg
    s["table"] = table.to("cuda")
    s["lens"] = torch.tensor(lens, dtype=torch.int32, device="cuda")
    s["q"] = _normal(gen, (B, M, H, D), dt)
    if c["new"]:
        s["k"] = _normal(gen, (B, c["new"], Hk, D), dt)
        s["v"] = _normal(gen, (B, c["new"], Hk, D), dt)
    if c["rotary"]:
        n = max(rows) * P
        angle = torch.outer(torch.arange(n, dtype=torch.float64),
                            10000.0 ** (-torch.arange(0, c["rotary"], 2, dtype=torch.float64) / c["rotary"]))
        s["cos"], s["sin"] = angle.cos().to(dt).to("cuda"), angle.sin().to(dt).to("cuda")
    if c["alibi"]:
        s["alibi"] = torch.tensor([2.0 ** (-8.0 * (h + 1) / H) for h in range(H)], dtype=torch.float32, device="cuda")
    return s


def run(state):
    s = state
    c = s["case"]
    if c["kind"] == "append":
        pagedkv.reshape_and_cache_flash(s["key"], s["value"], s["k_cache"], s["v_cache"], s["slots"], **s["scales"])
        return {"k_cache": s["k_cache"], "v_cache": s["v_cache"]}
    window = (c["window"], 0) if c["window"] >= 0 else (-1, -1)
    if c["kv"] == "fp8":
        lse = None
        if c["lse"]:
            lse = torch.empty((c["batch"], c["heads"], c["q"]), dtype=torch.float32, device="cuda")
        got = pagedkv.decode(s["q"], s["k_cache"], s["v_cache"], s["table"], s["lens"], k_new=s.get("k"),
                             v_new=s.get("v"), causal=c["causal"], window_size=window, alibi_slopes=s.get("alibi"),
                             softmax_lse=lse, rotary_cos=s.get("cos"), rotary_sin=s.get("sin"),
                             rotary_interleaved=False, softcap=c["softcap"], **s["scales"])
        got = (got, lse) if c["lse"] else got
    else:
        got = pagedkv.flash_attn_with_kvcache(
            s["q"], s["k_cache"], s["v_cache"], k=s.get("k"), v=s.get("v"), rotary_cos=s.get("cos"),
            rotary_sin=s.get("sin"), cache_seqlens=s["lens"], block_table=s["table"], causal=c["causal"],
            window_size=window, softcap=c["softcap"], rotary_interleaved=False, alibi_slopes=s.get("alibi"),
            return_softmax_lse=c["lse"])
    res = {"out": got[0], "lse": got[1]} if c["lse"] else {"out": got}
    if c["new"]:
        res["k_cache"], res["v_cache"] = s["k_cache"], s["v_cache"]
    return res


def tolerance(case):
    # Measured: outputs are 1.6e-3 (bf16) and 2.1e-4 (fp16) off their 64-bit values, the rounding of the output
    # itself; the largest difference over the value is one rounding step (2^-8, 2^-11), and two correct results
    # differ by at most two of them.
    c = {**DEFAULTS, **case}
    if c["kind"] == "append":
        return "exact"
    return {"rel": 6.5e-3, "max": 3e-2} if c["dtype"] == "bf16" else {"rel": 8.5e-4, "max": 4e-3}


# ------------------------------------------------------------------------------------------------ 64-bit results


def _quantise(x, scale):
    """x [..., Hk, D] to e4m3 of x / scale, saturated."""
    return (x.float() * (1.0 / scale)[:, None]).clamp(-448.0, 448.0).to(torch.float8_e4m3fn)


def _rotate(x, cos, sin, first, step):
    """x [B, T, n, D] rotated in halves at positions first[b] + step * t, stored in x's type."""
    R = 2 * cos.shape[1]
    out = x.double().clone()
    for b in range(x.shape[0]):
        pos = first[b] + step * torch.arange(x.shape[1], device=x.device)
        co, si = cos[pos].double()[:, None, :], sin[pos].double()[:, None, :]
        x0, x1 = x[b, ..., :R // 2].double(), x[b, ..., R // 2:R].double()
        out[b, ..., :R // 2] = x0 * co - x1 * si
        out[b, ..., R // 2:R] = x0 * si + x1 * co
    return out.to(x.dtype)


def exact(case, seed):
    s = prepare(case, seed)
    c = s["case"]
    D, P, Hk, H, B, M = c["dim"], c["page"], c["kv_heads"], c["heads"], c["batch"], c["q"]
    fp8 = c["kv"] == "fp8"
    lens = _lens(c)
    kc, vc = s["k_cache"], s["v_cache"]

    def stored(x, name):
        return _quantise(x, s["scales"][name]) if fp8 else x

    if c["kind"] == "append":
        kc.view(-1, Hk, D)[s["slots"]] = stored(s["key"], "k_scale")
        vc.view(-1, Hk, D)[s["slots"]] = stored(s["value"], "v_scale")
        return {"k_cache": kc.double(), "v_cache": vc.double()}
    q = s["q"]
    new_k = s.get("k")
    if c["rotary"]:
        new_k = _rotate(new_k, s["cos"], s["sin"], lens, 1)
        q = _rotate(q, s["cos"], s["sin"], lens, 1 if c["causal"] or c["window"] >= 0 else 0)
    out = torch.empty((B, M, H, D), dtype=torch.float64, device="cuda")
    lse = torch.empty((B, H, M), dtype=torch.float64, device="cuda")
    G = H // Hk
    table = s["table"].long()
    for b in range(B):
        n, total = lens[b], lens[b] + c["new"]
        pos = torch.arange(total, device="cuda")
        slots = table[b, pos // P] * P + pos % P
        if c["new"]:
            kc.view(-1, Hk, D)[slots[n:]] = stored(new_k[b], "k_scale")
            vc.view(-1, Hk, D)[slots[n:]] = stored(s["v"][b], "v_scale")
        k, v = kc.view(-1, Hk, D)[slots].double(), vc.view(-1, Hk, D)[slots].double()
        if fp8:
            k, v = k * s["scales"]["k_scale"].double()[:, None], v * s["scales"]["v_scale"].double()[:, None]
        qpos = (total - M + torch.arange(M, device="cuda")).repeat_interleave(G)[:, None]
        hide = torch.zeros((M * G, total), dtype=torch.bool, device="cuda")
        if c["causal"]:
            hide |= pos[None, :] > qpos
        if c["window"] >= 0:
            hide |= (pos[None, :] < qpos - c["window"]) | (pos[None, :] > qpos)
        for h in range(Hk):
            qh = q[b, :, h * G:(h + 1) * G].double().reshape(M * G, D)
            sc = qh @ k[:, h].t().contiguous() / math.sqrt(D)
            if c["softcap"] > 0:
                sc = c["softcap"] * torch.tanh(sc / c["softcap"])
            if c["alibi"]:
                slope = s["alibi"][h * G:(h + 1) * G].double().repeat(M)[:, None]
                sc -= slope * (qpos - pos[None, :]).abs()
            sc.masked_fill_(hide, -math.inf)
            z = torch.logsumexp(sc, dim=1, keepdim=True)
            o = torch.exp(sc - z) @ v[:, h].contiguous()
            out[b, :, h * G:(h + 1) * G] = o.reshape(M, G, D)
            lse[b, h * G:(h + 1) * G] = z.reshape(M, G).t()
    res = {"out": out}
    if c["lse"]:
        res["lse"] = lse
    if c["new"]:
        res["k_cache"], res["v_cache"] = kc.double(), vc.double()
    return res
