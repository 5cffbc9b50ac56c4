"""Small batches whose context chunks all fit the chip at once run on the grid in chunks of 8, 16 or 32
slots of 16 tokens, without the balanced schedule's plan: the rule, and its results at the edges."""
import numpy as np
import pytest
import torch

import kyro_amd
from kyro_amd import workloads as wl
from kyro_amd.attention import describe_attention
from tests import helpers as h

DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32}


def _describe(H, Hkv, D, batch, max_q, blocks, dtype):
    return describe_attention(kyro_amd.PagedAttention(16, H, D, Hkv), batch=batch, total_q=batch * max_q, max_q_len=max_q,
                              max_blocks_per_seq=blocks, num_blocks=batch * blocks, dtype=DTYPES[dtype])


@pytest.mark.parametrize("H,Hkv,D,batch,max_q,blocks,dtype,want", [
    (32, 8, 128, 1, 1, 31, "bf16", "schedule grid, row groups 1, splits 1,"),     # one launch as before
    (32, 8, 128, 1, 1, 32, "bf16", "schedule grid, row groups 1, splits 4,"),     # chunks of 8
    (32, 8, 128, 1, 1, 256, "bf16", "schedule grid, row groups 1, splits 32,"),   # the most of them
    (32, 8, 128, 1, 1, 257, "bf16", "schedule grid, row groups 1, splits 17,"),   # chunks of 16
    (32, 8, 128, 1, 1, 513, "bf16", "schedule balanced"),                         # too few groups for 32
    (8, 8, 128, 1, 1, 750, "bf16", "schedule grid, row groups 1, splits 24,"),    # chunks of 32
    (32, 8, 128, 16, 1, 200, "bf16", "schedule balanced"),                        # more than one a CU
    (32, 8, 128, 1, 1, 9, "f32", "schedule grid, row groups 1, splits 2,"),
    (16, 2, 64, 1, 8, 200, "f32", "schedule grid, row groups 2, splits 13,"),     # at most 16 of them
])
def test_short_chunk_rule(H, Hkv, D, batch, max_q, blocks, dtype, want):
    text = _describe(H, Hkv, D, batch, max_q, blocks, dtype)
    assert want in text, text


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["bf16", "f32"])
@pytest.mark.parametrize("H,Hkv,D,ctx,ql", [
    (32, 8, 128, [1000, 1, 0, 129], [1, 1, 1, 1]),
    (4, 4, 128, [4000, 127, 128, 16], [5, 3, 1, 2]),      # chunks of 16, contexts around a slot
    (32, 8, 128, [3333, 520], [8, 8]),
    (16, 2, 64, [3000, 255, 257], [8, 8, 1]),              # two row groups
])
def test_short_chunks_parity(gpu, dtype, H, Hkv, D, ctx, ql):
    case = wl.make_attention_case(context_lens=ctx, q_lens=ql, num_heads=H, num_kv_heads=Hkv, head_dim=D, dtype=dtype,
                                  seed=sum(ctx))
    attn = kyro_amd.PagedAttention(16, H, D, Hkv)
    text = _describe(H, Hkv, D, len(ctx), int(np.max(ql)), case.block_table.shape[1], dtype)
    assert "schedule grid" in text and "splits 1," not in text, text
    t = h.attention_tensors(case, gpu)
    out = attn.forward(t["query"], t["key_cache"], t["value_cache"], t["block_table"], t["context_lens"],
                       q_start_loc=t["q_start_loc"])
    h.assert_attention_close(out, case, h.oracle_attention(case), h.ATOL_BF16 if dtype == "bf16" else h.ATOL_F32_SUMS)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,H,Hkv,D,ctx,ql", [
    ("bf16", 64, 8, 128, [4000] + [300, 64, 9] * 21, [9] * 64),  # the many-row kernel's list and parts
    ("f32", 32, 8, 64, [300, 17, 0, 260] * 2, [1] * 8),      # short chunks
    ("f32", 32, 8, 128, [300, 17, 0, 260], [1] * 4),
    ("bf16", 8, 8, 256, [300, 17, 0, 260], [1] * 4),
])
def test_capture_without_a_reserve_takes_a_form_without_scratch(gpu, dtype, H, Hkv, D, ctx, ql):
    """Forms chosen for speed alone need scratch at these shapes. A graph captured on a context whose arena
    is empty takes the form that needs none."""
    from kyro_amd import _lib

    case = wl.make_attention_case(context_lens=ctx, q_lens=ql, num_heads=H, num_kv_heads=Hkv, head_dim=D, dtype=dtype,
                                  seed=D + len(ctx))
    t = h.attention_tensors(case, gpu)
    attn = kyro_amd.PagedAttention(16, H, D, Hkv)
    args = (t["query"], t["key_cache"], t["value_cache"], t["block_table"], t["context_lens"])
    context = _lib.Context(gpu.index or 0)
    kw = dict(q_start_loc=t["q_start_loc"], max_q_len=max(ql), context=context)
    s = torch.cuda.Stream(gpu)
    with torch.cuda.stream(s):  # binds the context to s; one split takes no scratch
        out = attn.forward_async(*args, num_splits=1, schedule="grid", **kw)
    context.sync()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        attn.forward_async(*args, out=out, **kw)
    for _ in range(3):
        out.zero_()
        g.replay()
        torch.cuda.synchronize()
        h.assert_attention_close(out, case, h.oracle_attention(case), h.ATOL_BF16 if dtype == "bf16" else h.ATOL_F32_SUMS)
    del g
    context.sync()
