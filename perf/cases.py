"""The decode-path work that a program using this framework has it do, as
timed and checked cases: paged-attention decode, prefix-aware decode, KV
append and the MLP activations, each through its Python entry point.

A case is a dict of plain values.  `kind` names the entry point:
  decode   paged_attention over a ragged batch (heads, kv_heads, head_size,
           block_size, dtype; seqs sequences of len_lo..len_hi tokens)
  cascade  paged_attention_cascade over groups of sequences that share the
           pages of a prefix; `detect` also finds the groups (prefix_groups)
           from the block tables first, as on a new batch composition
  append   paged_kv_append of `tokens` new rows (`form`: "slots", a prefill
           chunk's flat slots, or "tables", one token per sequence)
  act      one MLP activation over [tokens, d] outputs

Sequence lengths are evenly spaced quantiles of the stated distribution
("even" or "log"arithmic between len_lo and len_hi), dealt to the sequences
in a seeded order: every seed has the same work and other inputs.
"""
from __future__ import annotations

import math

import torch

from xllms_amd import activation as ACT
from xllms_amd import paged_attention as PA

DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}
BYTES = {"fp16": 2, "bf16": 2, "fp32": 4}
OPS = {name: (code, ACT.is_gated(code)) for code, name in ACT.OP_NAMES.items()}


def _decode(name, dtype, heads, kv_heads, head_size, seqs, len_lo, len_hi, dist="even",
            block_size=16):
    c = {"kind": "decode", "dtype": dtype, "heads": heads, "kv_heads": kv_heads,
         "head_size": head_size, "block_size": block_size, "seqs": seqs, "len_lo": len_lo,
         "len_hi": len_hi, "dist": dist}
    return {"name": name, **c} if name else c


def _cascade(name, dtype, heads, kv_heads, head_size, seqs, groups, pre_lo, pre_hi, suf_hi, detect,
             block_size=16):
    c = {"kind": "cascade", "dtype": dtype, "heads": heads, "kv_heads": kv_heads,
         "head_size": head_size, "block_size": block_size, "seqs": seqs, "groups": groups,
         "pre_lo": pre_lo, "pre_hi": pre_hi, "suf_hi": suf_hi, "detect": detect}
    return {"name": name, **c} if name else c


def _append(name, dtype, form, tokens, kv_heads, head_size, block_size=16):
    c = {"kind": "append", "dtype": dtype, "form": form, "tokens": tokens, "kv_heads": kv_heads,
         "head_size": head_size, "block_size": block_size}
    return {"name": name, **c} if name else c


def _act(name, op, dtype, tokens, d):
    c = {"kind": "act", "op": op, "dtype": dtype, "tokens": tokens, "d": d}
    return {"name": name, **c} if name else c


def listed():
    return [
        # one user's first tokens on the smallest model (GPT-2-small heads, fp32): pure latency
        _decode("one_short_fp32", "fp32", 12, 12, 64, 1, 96, 96),
        # a handful of users on that model
        _decode("small_batch_fp32", "fp32", 12, 12, 64, 8, 16, 1024),
        # the attention benchmark's own shape: 16 sequences of 1024 tokens, Llama-3-8B heads
        _decode("batch16_ctx1024_fp16", "fp16", 32, 8, 128, 16, 1024, 1024),
        # a full serving batch of an 8B model, ragged lengths
        _decode("serving_batch_fp16", "fp16", 32, 8, 128, 64, 512, 4096),
        # few long documents: the split over one sequence
        _decode("long_context_fp16", "fp16", 32, 8, 128, 4, 8192, 32768),
        # a 70B-shaped batch (GQA 8) in bf16 with a heavy tail of lengths
        _decode("gqa8_batch_bf16", "bf16", 64, 8, 128, 128, 128, 4096, "log"),
        # the fp32 operator on the 8B shape (dtype_size 4)
        _decode("gqa4_batch_fp32", "fp32", 32, 8, 128, 32, 256, 2048),
        # multi-head attention with head_size 80
        _decode("mha80_batch_fp16", "fp16", 32, 32, 80, 24, 100, 2000),
        # wide heads, odd lengths, larger pages
        _decode("wide_heads_bf16", "bf16", 16, 8, 256, 24, 77, 3001, "log", 32),
        # continuous batching with radix-shared system prompts
        _cascade("shared_prefix_fp16", "fp16", 32, 8, 128, 256, 16, 256, 2048, 1024, False),
        # storing the K/V rows of a prefill chunk
        _append("append_prefill_bf16", "bf16", "slots", 8192, 8, 128),
        # the gated MLP activation over a prefill chunk
        _act("silu_and_mul_fp16", "silu_and_mul", "fp16", 2048, 14336),
    ]


# head layouts of the draws: (heads, kv_heads, head_size)
_HEADS = [(12, 12, 64), (32, 8, 128), (32, 8, 128), (64, 8, 128), (64, 4, 128), (32, 32, 128),
          (32, 32, 80), (32, 8, 64), (32, 32, 96), (16, 8, 256), (24, 8, 112), (48, 8, 192)]
_CAP = 600e6  # bytes of one drawn case


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode"] * 7 + ["cascade"] * 2 + ["append", "act"])
    while True:
        if kind == "decode":
            h, k, d = rng.choice(_HEADS)
            hi = _log(rng, 24, 32768)
            c = _decode(None, rng.choice(["fp16", "fp16", "bf16", "fp32"]), h, k, d,
                        _log(rng, 1, 256), max(1, int(hi * rng.uniform(0.02, 1.0))), hi,
                        rng.choice(["even", "log"]), rng.choice([16, 16, 16, 32, 64, 8]))
        elif kind == "cascade":
            h, k, d = rng.choice([(32, 8, 128), (32, 8, 128), (64, 8, 128), (32, 8, 64), (32, 32, 128)])
            groups = _log(rng, 1, 32)
            hi = _log(rng, 64, 4096)
            c = _cascade(None, rng.choice(["fp16", "fp16", "bf16"]), h, k, d,
                         min(320, groups * rng.randint(2, 24) + rng.randint(0, 20)), groups,
                         max(16, int(hi * rng.uniform(0.1, 1.0))), hi, _log(rng, 16, 1024),
                         rng.random() < 0.3)
        elif kind == "append":
            _, k, d = rng.choice(_HEADS)
            form = rng.choice(["slots", "tables"])
            c = _append(None, rng.choice(["fp16", "bf16", "fp32"]), form,
                        _log(rng, 1, 65536 if form == "slots" else 512), k, d)
        else:
            c = _act(None, rng.choice(sorted(OPS)), rng.choice(["fp16", "bf16", "fp32"]),
                     _log(rng, 1, 16384), rng.choice([768, 3072, 11008, 14336, 4099]))
        if work(c)["bytes"] <= _CAP:
            return c


def _lens(case):
    """The batch's lengths, in ascending order (the same for every seed)."""
    n, lo, hi = case["seqs"], case["len_lo"], case["len_hi"]
    u = [(i + 0.5) / n for i in range(n)]
    if case["dist"] == "log":
        return [int(round(lo * (hi / lo) ** x)) for x in u]
    return [int(round(lo + (hi - lo) * x)) for x in u]


def _cascade_lens(case):
    """(prefix length of each group, suffix length of each sequence, group of
    each sequence): one in ten sequences is fresh (one token, no group), the
    others are dealt to the groups in turn."""
    n, ng = case["seqs"], case["groups"]
    fresh = n // 10
    pre = [int(round(case["pre_lo"] + (case["pre_hi"] - case["pre_lo"]) * (i + 0.5) / ng))
           for i in range(ng)]
    group = [-1] * fresh + [i % ng for i in range(n - fresh)]
    # suffixes in an order that is not the groups' (a stride coprime to n)
    step = next(k for k in range(max(1, int(n * 0.618)), 2 * n + 2) if math.gcd(k, n) == 1)
    suf = [1 if group[i] < 0 else
           1 + int((case["suf_hi"] - 1) * (((i * step) % n) + 0.5) / n) for i in range(n)]
    return pre, suf, group


def _randn(shape, dtype, gen):
    return torch.randn(shape, dtype=dtype, device="cuda", generator=gen)


def _tables(lens, bs, gen, pages=None):
    """Block tables [B, widest] of pages dealt from a shuffled pool a quarter
    larger than needed (-1 past each sequence), and the pool's size."""
    need = [-(-n // bs) for n in lens]
    total = sum(need)
    pool = total + total // 4 + 1
    perm = torch.randperm(pool, device="cuda", generator=gen).to(torch.int32)
    n = torch.tensor(need, device="cuda")
    start = torch.cumsum(n, 0) - n
    j = torch.arange(max(need), device="cuda")
    at = (start[:, None] + j[None, :]).clamp(max=pool - 1)
    return torch.where(j[None, :] < n[:, None], perm[at], torch.full_like(perm[at], -1)), pool


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    dt = DTYPES[case["dtype"]]
    kind = case["kind"]
    if kind == "act":
        op, gated = OPS[case["op"]]
        x = _randn((case["tokens"], case["d"] * (2 if gated else 1)), dt, gen) * 2.0
        out = torch.empty((case["tokens"], case["d"]), dtype=dt, device="cuda")
        return {"kind": kind, "op": op, "x": x, "out": out}
    KVH, D, bs = case["kv_heads"], case["head_size"], case["block_size"]
    if kind == "append":
        n = case["tokens"]
        key, value = _randn((n, KVH, D), dt, gen), _randn((n, KVH, D), dt, gen)
        st = {"kind": kind, "key": key, "value": value}
        if case["form"] == "slots":
            # prompts of a few hundred tokens laid end to end over their pages
            lens = [min(389, n - i) for i in range(0, n, 389)]
            tables, pool = _tables(lens, bs, gen)
            slots = []
            for s, L in enumerate(lens):
                t = torch.arange(L, device="cuda")
                slots.append(tables[s][t // bs] * bs + t % bs)
            st["slots"] = torch.cat(slots).to(torch.int32)
        else:
            lens = [1 + (i * 37) % 700 for i in range(n)]
            tables, pool = _tables(lens, bs, gen)
            st["tables"] = tables
            st["positions"] = torch.tensor([L - 1 for L in lens], dtype=torch.int32, device="cuda")
        st["k"] = torch.zeros((pool, KVH, bs, D), dtype=dt, device="cuda")
        st["v"] = torch.zeros((pool, KVH, bs, D), dtype=dt, device="cuda")
        return st

    order = torch.randperm(case["seqs"], device="cuda", generator=gen).tolist()
    st = {"kind": kind, "kv_heads": KVH, "scale": 1.0 / math.sqrt(D)}
    if kind == "decode":
        asc = _lens(case)
        lens = [asc[i] for i in order]
        tables, pool = _tables(lens, bs, gen)
    else:
        pre, suf, group = _cascade_lens(case)
        suf, group = [suf[i] for i in order], [group[i] for i in order]
        shared = [p // bs for p in pre]  # whole pages are shared, the rest is each member's own
        own = [s + (pre[g] - shared[g] * bs if g >= 0 else 0) for s, g in zip(suf, group)]
        lens = [n + (shared[g] * bs if g >= 0 else 0) for n, g in zip(own, group)]
        parts, pool = _tables(own + [max(n, 1) * bs for n in shared], bs, gen)
        width = max(-(-n // bs) for n in lens)
        tables = torch.full((len(lens), width), -1, dtype=torch.int32, device="cuda")
        for s, g in enumerate(group):
            k = shared[g] if g >= 0 else 0
            m = -(-own[s] // bs)
            if k:
                tables[s, :k] = parts[len(own) + g, :k]
            tables[s, k:k + m] = parts[s, :m]
        st["detect"] = case["detect"]
        st["block_size"] = bs
        st["prefix_group"] = torch.tensor([g if g >= 0 and shared[g] > 0 else -1 for g in group],
                                          dtype=torch.int32, device="cuda")
        st["prefix_blocks"] = torch.tensor(shared, dtype=torch.int32, device="cuda")
    st["tables"] = tables.contiguous()
    st["lens"] = torch.tensor(lens, dtype=torch.int32, device="cuda")
    st["q"] = _randn((len(lens), case["heads"], D), dt, gen)
    st["k"] = _randn((pool, KVH, bs, D), dt, gen)
    st["v"] = _randn((pool, KVH, bs, D), dt, gen)
    st["out"] = torch.empty_like(st["q"])
    return st


def run(st):
    kind = st["kind"]
    if kind == "decode":
        PA.paged_attention(st["out"], st["q"], st["k"], st["v"], st["tables"], st["lens"],
                           num_kv_heads=st["kv_heads"], scale=st["scale"])
        return st["out"]
    if kind == "cascade":
        group, blocks = st["prefix_group"], st["prefix_blocks"]
        if st["detect"]:
            group, blocks, _ = PA.prefix_groups(st["tables"], st["lens"],
                                                block_size=st["block_size"])
        PA.paged_attention_cascade(st["out"], st["q"], st["k"], st["v"], st["tables"], st["lens"],
                                   group, blocks, num_kv_heads=st["kv_heads"], scale=st["scale"])
        return st["out"]
    if kind == "append":
        if "slots" in st:
            PA.paged_kv_append(st["k"], st["v"], st["key"], st["value"], slot_mapping=st["slots"])
        else:
            PA.paged_kv_append(st["k"], st["v"], st["key"], st["value"], block_tables=st["tables"],
                               positions=st["positions"])
        return {"k": st["k"], "v": st["v"]}
    ACT.activation(st["op"], st["out"], st["x"])
    return st["out"]


def work(case):
    e = BYTES[case["dtype"]]
    if case["kind"] == "act":
        gated = OPS[case["op"]][1]
        n = case["tokens"] * case["d"]
        return {"bytes": n * e * (3 if gated else 2), "flops": n * 10}
    KVH, D, bs = case["kv_heads"], case["head_size"], case["block_size"]
    if case["kind"] == "append":
        n = case["tokens"]
        return {"bytes": n * KVH * D * e * 4 + n * (4 if case["form"] == "slots" else 8),
                "flops": 0}
    if case["kind"] == "decode":
        lens = _lens(case)
        tokens = distinct = sum(lens)
        entries = sum(-(-n // bs) for n in lens)
    else:
        pre, suf, group = _cascade_lens(case)
        used = sorted({g for g in group if g >= 0})
        shared = sum(pre[g] // bs * bs for g in used)
        own = sum(s + (pre[g] % bs if g >= 0 else 0) for s, g in zip(suf, group))
        distinct = shared + own
        tokens = own + sum(pre[g] // bs * bs for g in group if g >= 0)
        entries = -(-distinct // bs)
    n = case["seqs"]
    return {"bytes": distinct * KVH * D * 2 * e + 2 * n * case["heads"] * D * e + 4 * entries + 4 * n,
            "flops": 4 * tokens * case["heads"] * D}


def tolerance(case):
    if case["kind"] == "append":
        return "exact"  # bytes are copied
    # about four times the relative error against exact() on MI355X: fp16
    # 2.1e-4 (the cascade's fp16 states up to 3.4e-4), bf16 1.7e-3, fp32 2e-7
    # on the listed sizes (sums of up to 32768 terms: 2e-6 allowed)
    return {"fp16": {"rel": 1.2e-3, "max": 1.2e-2}, "bf16": {"rel": 7e-3, "max": 6e-2},
            "fp32": {"rel": 2e-6, "max": 2e-5}}[case["dtype"]]


def exact(case, seed):
    """What run() returns, in 64 bits, from plain torch operations."""
    if case["kind"] == "append":
        return None  # copies, compared bit for bit
    st = prepare(case, seed)
    if case["kind"] == "act":
        x = st["x"].double()
        name, d = case["op"], case["d"]
        g, u = (x[:, :d], x[:, d:]) if OPS[name][1] else (x, None)
        if name == "mul_and_silu":
            g, u = u, g
        if "silu" in name:
            a = g * torch.sigmoid(g)
        elif "tanh" in name:
            a = 0.5 * g * (1 + torch.tanh(math.sqrt(2 / math.pi) * (g + 0.044715 * g ** 3)))
        else:
            a = 0.5 * g * (1 + torch.erf(g / math.sqrt(2)))
        return a if u is None else a * u
    H, KVH, D, bs = case["heads"], case["kv_heads"], case["head_size"], case["block_size"]
    G = H // KVH
    out = torch.empty((case["seqs"], H, D), dtype=torch.float64, device="cuda")
    for s, L in enumerate(st["lens"].tolist()):
        ids = st["tables"][s, :-(-L // bs)].long()
        k = st["k"][ids].double().permute(1, 0, 2, 3).reshape(KVH, -1, D)[:, :L]
        v = st["v"][ids].double().permute(1, 0, 2, 3).reshape(KVH, -1, D)[:, :L]
        q = st["q"][s].double().reshape(KVH, G, D)
        for h in range(KVH):
            p = torch.softmax(q[h] @ k[h].t().contiguous() * st["scale"], dim=-1)
            out[s, h * G:(h + 1) * G] = p @ v[h].contiguous()
    return out
