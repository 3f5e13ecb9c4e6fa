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


def _check(wl, what, **kw):
    import torch
    dw = W.upload(wl)
    PA.paged_attention(dw.out, dw.query, dw.key_cache, dw.value_cache, dw.block_tables,
                       dw.seq_lens, num_kv_heads=wl.num_kv_heads, scale=wl.scale, **kw)
    torch.cuda.synchronize()
    assert_close(dw.out.float().cpu().numpy(), O.run_workload(wl, precision="mt"), wl.kv_dtype, what)


@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
@pytest.mark.parametrize("head_size", [32, 64, 96, 128, 192, 256])
@pytest.mark.parametrize("group", [1, 4, 16, 20])
def test_tile_edges(cuda, dtype, head_size, group):
    lens = [1, 2, 3, 4, 5, 15, 16, 17, 31, 32, 33, 0, 255, 1025]
    for bs in (16, 32):
        wl = W.small_case(num_seqs=len(lens), H=2 * group, KVH=2, D=head_size, bs=bs,
                          kv_dtype=DT[dtype], seed=head_size + group + bs, lens=lens)
        print(f"case {dtype} d={head_size} group={group} bs={bs}", flush=True)
        _check(wl, f"{dtype} d={head_size} group={group} bs={bs}")
