"""The matrix tile path at the sizes where its lane layout can go wrong: every
head size (V rows in chunks of 2 to 8 dims, one or two groups of chunks, dealt
through LDS or straight from the load registers), one and two row blocks of
query heads, and lengths one token either side of a tile, against the CPU
oracle (rel 1e-5 for fp32, atol 2e-3 + rtol 1e-2 for fp16 / bf16)."""
from __future__ import annotations

import pytest

from oracle import oracle as O
from tests.helpers import assert_close
from xllms_amd import paged_attention as PA
from xllms_amd import workloads as W

pytestmark = pytest.mark.gpu

DT = {"fp16": W.FP16, "bf16": W.BF16, "fp32": W.FP32}


def _check(wl, what, tokens=0, **kw):
    """Against the oracle; tokens: under a table that bounds at least so many
    (the fp32 rule goes by the table)."""
    import torch
    dw = W.upload(wl)
    n, used = dw.block_tables.shape
    bs = dw.key_cache.shape[2]
    tables = torch.full((n, max(used, -(-tokens // bs))), -1, dtype=torch.int32, device="cuda")
    tables[:, :used] = dw.block_tables
    PA.paged_attention(dw.out, dw.query, dw.key_cache, dw.value_cache, tables, dw.seq_lens,
                       num_kv_heads=wl.num_kv_heads, scale=wl.scale, **kw)
    torch.cuda.synchronize()
    assert_close(dw.out.float().cpu().numpy(), O.run_workload(wl, precision="mt"), wl.kv_dtype, what)


@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
@pytest.mark.parametrize("head_size", [32, 64, 80, 96, 112, 128, 192, 256])
@pytest.mark.parametrize("group", [1, 3, 4, 16, 20])
def test_tile_edges(cuda, dtype, head_size, group):
    lens = [1, 2, 3, 4, 5, 15, 16, 17, 31, 32, 33, 0, 255, 1025]
    for bs in (16, 32):
        wl = W.small_case(num_seqs=len(lens), H=2 * group, KVH=2, D=head_size, bs=bs,
                          kv_dtype=DT[dtype], seed=head_size + group + bs, lens=lens)
        print(f"case {dtype} d={head_size} group={group} bs={bs}", flush=True)
        _check(wl, f"{dtype} d={head_size} group={group} bs={bs}")


@pytest.mark.parametrize("head_size", [32, 64, 96, 128])
@pytest.mark.parametrize("group", [5, 8, 16, 17, 32])
def test_fp32_tile_edges(cuda, head_size, group):
    """fp32 automatic plans take the matrix tiles for groups above 4 (at head
    sizes of more than 64 where the table bounds 64 MB): edges of the 16-token
    tile, one and two head tiles, pages of one and two tiles."""
    lens = [1, 2, 3, 4, 5, 15, 16, 17, 31, 32, 33, 0, 255, 1025]
    for bs in (16, 32):
        wl = W.small_case(num_seqs=len(lens), H=2 * group, KVH=2, D=head_size, bs=bs,
                          kv_dtype=W.FP32, seed=head_size + group + bs, lens=lens)
        print(f"case fp32 d={head_size} group={group} bs={bs}", flush=True)
        _check(wl, f"fp32 d={head_size} group={group} bs={bs}", tokens=4096)


@pytest.mark.parametrize("case", [
    # (H, KVH, head_size, sequences, tokens the table bounds, matrix tiles?):
    # either side of the fp32 rule's lines.  Groups of 3 and 4: 512 MB of K/V
    # and 512 tokens at head sizes of more than 64, else 256 MB.  Groups from
    # 5: 64 MB there, 16 MB for at most 112 tokens.  Groups of 1 and 2: never.
    (32, 8, 128, 32, 1952, False), (32, 8, 128, 32, 1968, True),
    (32, 8, 128, 128, 496, False), (32, 8, 128, 128, 512, True),
    (12, 4, 128, 64, 1952, False), (12, 4, 128, 64, 1968, True),
    (32, 8, 96, 32, 2592, False), (32, 8, 96, 32, 2608, True),
    (16, 4, 64, 64, 1952, False), (16, 4, 64, 64, 1968, True),
    (64, 8, 128, 8, 976, False), (64, 8, 128, 8, 992, True),
    (64, 8, 128, 16, 112, False), (64, 8, 128, 32, 64, True), (64, 8, 128, 32, 128, False),
    (64, 4, 128, 16, 976, False), (64, 4, 128, 16, 992, True),
    (16, 8, 128, 64, 4096, False), (32, 32, 128, 64, 4096, False), (12, 12, 64, 64, 8192, False),
])
def test_fp32_tile_path_rule(cuda, case):
    """The tile path on either side of each line, by the number of wavefronts
    of its plan, and the outputs of a batch that fills little of such a
    table."""
    import torch
    H, KVH, D, n, ctx, mfma = case
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    units = n * KVH * (-(-(H // KVH) // 16)) * (ctx // 16 + 2)  # MFMA: 16 tokens, 2 start-up units
    plan = min(cus * (4 if D > 64 else 8), (units // 2 + 3) // 4 * 4)
    waves = PA.auto_waves(n, H, D, KVH, ctx // 16, 16, W.FP32)
    print(f"case {case}: {waves} wavefronts, {plan} on the matrix tiles", flush=True)
    assert (waves == plan) == mfma
    lens = [max(1, min(ctx, 97) - 7 * i % 90) for i in range(n)]
    wl = W.small_case(num_seqs=n, H=H, KVH=KVH, D=D, kv_dtype=W.FP32, seed=n + ctx, lens=lens)
    _check(wl, f"fp32 rule {case}", tokens=ctx)


@pytest.mark.parametrize("n", [2, 31, 33, 130, 1025])
def test_detection_run_lengths(cuda, n):
    """Shared runs one page either side of the 16 pages the detection compares
    at a time, up to the whole table, over batches around its hash table's
    sizes; lengths that end inside a run."""
    import numpy as np
    import torch

    from tests.cascade_cases import detect_prefix_groups
    rng = np.random.default_rng(n)
    width, bs = 50, 16
    tables = rng.permutation(n * width).reshape(n, width).astype(np.int32)
    runs = [1, 15, 16, 17, 31, 32, 33, 49, 50]
    for s in range(1, n):
        if s % 5 != 4:  # shares the first pages of a leader a few rows up
            lead = s - s % 5
            k = runs[s % len(runs)]
            if lead != s:
                tables[s, :k] = tables[lead, :k]
    lens = rng.integers(1, width * bs + 1, size=n).astype(np.int32)
    lens[: min(n, 30)] = width * bs
    group, blocks, count = PA.prefix_groups(torch.from_numpy(tables).cuda(),
                                            torch.from_numpy(lens).cuda(), block_size=bs)
    torch.cuda.synchronize()
    want_group, want_blocks = detect_prefix_groups(tables, lens, bs)
    assert int(count[0]) == len(want_blocks)
    assert np.array_equal(group.cpu().numpy(), want_group)
    assert np.array_equal(blocks.cpu().numpy()[: len(want_blocks)], want_blocks)


@pytest.mark.parametrize("key,scale", [(4e36, 4.0), (3e38, 1.0), (-3e38, 1.0)])
def test_fp32_overflowing_scores(cuda, key, scale):
    """A score that overflows when scaled, or already as a sum (to +inf: NaN
    rows; to -inf: a weight of zero): the matrix tiles (automatic plan) against
    the VALU tiles (explicit plan), NaN for NaN."""
    import torch
    wl = W.small_case(num_seqs=2, H=16, KVH=2, D=64, kv_dtype=W.FP32, seed=7, lens=[40, 33])
    dw = W.upload(wl)
    dw.query.fill_(1.0)
    dw.key_cache.mul_(0.01)
    page = int(dw.block_tables[0, 1])
    dw.key_cache[page, 0, 3] = key  # token 19 of sequence 0, kv head 0

    def run(**kw):
        dw.out.zero_()
        PA.paged_attention(dw.out, dw.query, dw.key_cache, dw.value_cache, dw.block_tables,
                           dw.seq_lens, num_kv_heads=2, scale=scale, **kw)
        torch.cuda.synchronize()
        return dw.out.clone().view(2, 16, 64)
    auto, valu = run(), run(partition_tokens=256)
    print(f"case key={key} scale={scale}", flush=True)
    assert bool(torch.isnan(auto[0, :8]).all()) == (key > 0)
    assert torch.equal(torch.isnan(auto), torch.isnan(valu))
    assert torch.allclose(auto.nan_to_num(), valu.nan_to_num(), rtol=1e-5, atol=1e-6)


@pytest.mark.parametrize("size", [1e5, 1e7, 1e9, 1e12, 1e16, 1e30])
@pytest.mark.parametrize("sign", [1.0, -1.0])
def test_fp32_large_scores(cuda, size, sign):
    """Finite scores so large that the rounding of a scaled score is far above
    1 (log2 units): the largest score of a row still has a weight of 1 and the
    others one of at most 1, as in the VALU tiles (explicit plan), where the
    weights come from the differences of the rounded scores.  The scores are
    size times 1, 1.5 or 2 times a head's factor, exact in fp32 before the
    scale, so every weight is 0 or 1 and both paths average the same rows:
    fp32 sums of at most 40 terms, 40 * 2^-24 < 1e-5."""
    import torch
    wl = W.small_case(num_seqs=2, H=16, KVH=2, D=64, kv_dtype=W.FP32, seed=11, lens=[40, 33])
    dw = W.upload(wl)
    dw.query.zero_()
    dw.query.view(2, 16, 64)[:, :, 5] = torch.arange(1, 17, device="cuda") * float(size) * sign
    tokens = torch.arange(dw.key_cache.shape[0] * 16, device="cuda").view(-1, 1, 16) * 7 % 3
    dw.key_cache.zero_()
    dw.key_cache[:, :, :, 5] = 1.0 + 0.5 * tokens

    def run(**kw):
        dw.out.zero_()
        PA.paged_attention(dw.out, dw.query, dw.key_cache, dw.value_cache, dw.block_tables,
                           dw.seq_lens, num_kv_heads=2, scale=0.125, **kw)
        torch.cuda.synchronize()
        return dw.out.clone()
    auto, valu = run(), run(partition_tokens=256)
    print(f"case size={size} sign={sign}", flush=True)
    assert bool(torch.isfinite(valu).all()) and bool(torch.isfinite(auto).all())
    assert torch.allclose(auto, valu, rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
@pytest.mark.parametrize("head_size", [80, 112])
def test_weights_kept_in_fp32(cuda, dtype, head_size):
    """The weights of automatic plans at head sizes 80 and 112 are fp32 on
    either tile path: the values of three tokens cancel to about 2^-17 (bf16)
    or 2^-20 (fp16) of their size, so a weight of 16 bits shows in the output.
    Against 64 bits: a weight's relative error is below 2^-21 (the roundings
    of the scale, of two scaled scores of up to 3 and of exp2, each 2^-24),
    applied to the three weighted values, and the output's own rounding."""
    import numpy as np
    import torch
    n, L, group, scale = 16, 40, 8, 0.75
    wl = W.small_case(num_seqs=n, H=2 * group, KVH=2, D=head_size, kv_dtype=DT[dtype], seed=3,
                      lens=[L] * n)
    dw = W.upload(wl)
    torch_dt = dw.query.dtype

    def rnd(x):
        return torch.from_numpy(x).to(torch_dt).double().numpy()
    rng = np.random.default_rng(head_size)
    dw.query.zero_()
    dw.query.view(n, 2 * group, head_size)[:, ::group, 0] = 1.0  # the first head of a kv head
    score = rnd(rng.uniform(-2.0, 0.0, (n, L)))
    a, b, c = 1, 18, 37  # in three tiles, the largest score last
    for t, lo in ((a, -1.5), (b, -0.5), (c, 1.0)):
        score[:, t] = rnd(rng.uniform(lo, lo + 0.5, n))
    w = np.exp(scale * (score - score[:, c:c + 1]))
    v = np.zeros((n, L, head_size))
    v[:, a] = rnd(rng.uniform(0.5, 1.0, (n, head_size)))
    v[:, b] = -rnd(v[:, a] * (w[:, a] / w[:, b])[:, None])
    v[:, c] = -rnd(v[:, a] * w[:, a, None] + v[:, b] * w[:, b, None])
    K = np.zeros((n, L, head_size))
    K[:, :, 0] = score
    for cache, rows in ((dw.key_cache, K), (dw.value_cache, v)):
        rows = torch.from_numpy(rows).to(torch_dt).cuda()
        for t in range(L):
            cache[dw.block_tables[:, t // 16].long(), :, t % 16] = rows[:, None, t]
    want = np.einsum("nt,ntd->nd", w, v) / w.sum(1)[:, None]
    size = np.einsum("nt,ntd->nd", w, np.abs(v)) / w.sum(1)[:, None]
    bound = size * 2.0 ** -21 + np.abs(want) * 2.0 ** (-8 if dtype == "bf16" else -11) + \
        (2.0 ** -25 if dtype == "fp16" else 0.0)  # (fp16: the smallest outputs' spacing)
    for part in (0, 256):
        dw.out.zero_()
        PA.paged_attention(dw.out, dw.query, dw.key_cache, dw.value_cache, dw.block_tables,
                           dw.seq_lens, num_kv_heads=2, scale=scale, partition_tokens=part)
        torch.cuda.synchronize()
        got = dw.out.view(n, 2 * group, head_size)[:, ::group].double().cpu().numpy()
        worst = float((np.abs(got - want[:, None]) / bound[:, None]).max())
        print(f"case {dtype} d={head_size} partition={part}: {worst:.3f} of the bound", flush=True)
        assert worst <= 1.0


@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
@pytest.mark.parametrize("head_size", [80, 112])
def test_infinite_values(cuda, dtype, head_size):
    """An infinite value under a weight above 0 makes its output element
    infinite, under the automatic plan as in the VALU tiles (explicit plan):
    no part of a weight is 0."""
    import torch
    wl = W.small_case(num_seqs=2, H=16, KVH=2, D=head_size, kv_dtype=DT[dtype], seed=5,
                      lens=[40, 33])
    dw = W.upload(wl)
    page = int(dw.block_tables[0, 1])
    dw.value_cache[page, 0, 3, 7] = float("inf")      # token 19 of sequence 0, kv head 0
    dw.value_cache[page, 1, 5, 70] = float("-inf")    # token 21, kv head 1

    def run(**kw):
        dw.out.zero_()
        PA.paged_attention(dw.out, dw.query, dw.key_cache, dw.value_cache, dw.block_tables,
                           dw.seq_lens, num_kv_heads=2, scale=0.01, **kw)
        torch.cuda.synchronize()
        return dw.out.clone().view(2, 16, head_size)
    auto, valu = run(), run(partition_tokens=256)
    print(f"case {dtype} d={head_size}", flush=True)
    assert bool((auto[0, :8, 7] == float("inf")).all())
    assert bool((auto[0, 8:, 70] == float("-inf")).all())
    assert int(torch.isfinite(auto).logical_not().sum()) == 16
    assert torch.equal(torch.isfinite(auto), torch.isfinite(valu))


@pytest.mark.parametrize("head_size", [32, 64, 96, 128])
@pytest.mark.parametrize("tokens,seqs", [(16, 256), (40, 256), (300, 64)])
def test_fp32_error_of_the_matrix_tiles(cuda, head_size, tokens, seqs):
    """The matrix tiles (automatic plan) are no further from 64 bits than the
    VALU tiles (explicit plan) in fp32, in the 2-norm over a batch; short
    contexts, whose tiles are mostly one sum, have it hardest.  2% for the
    spread of a batch's error (the norm of some 10^5 independent roundings
    moves by less than 1% with the seed)."""
    import torch
    H, KVH = 16, 2
    wl = W.small_case(num_seqs=seqs, H=H, KVH=KVH, D=head_size, kv_dtype=W.FP32,
                      seed=head_size + tokens, lens=[tokens] * seqs)
    dw = W.upload(wl)
    tables = torch.full((seqs, 512), -1, dtype=torch.int32, device="cuda")  # wide: the fp32 rule
    used = dw.block_tables.shape[1]
    tables[:, :used] = dw.block_tables
    k, v = (c[dw.block_tables.long()].cpu().double().permute(0, 2, 1, 3, 4)
            .reshape(seqs, KVH, -1, head_size)[:, :, :tokens] for c in (dw.key_cache, dw.value_cache))
    q = dw.query.cpu().double().view(seqs, KVH, H // KVH, head_size)
    want = torch.softmax(q @ k.transpose(2, 3).contiguous() * wl.scale, -1) @ v
    err = {}
    for name, part in (("matrix", 0), ("valu", 512)):
        dw.out.zero_()
        PA.paged_attention(dw.out, dw.query, dw.key_cache, dw.value_cache, tables, dw.seq_lens,
                           num_kv_heads=KVH, scale=wl.scale, partition_tokens=part)
        torch.cuda.synchronize()
        err[name] = float((dw.out.cpu().double().view_as(want) - want).norm() / want.norm())
    print(f"case d={head_size} tokens={tokens}: {err}", flush=True)
    assert err["matrix"] <= 1.02 * err["valu"]
