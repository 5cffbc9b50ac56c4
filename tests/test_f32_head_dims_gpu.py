"""The f32 MFMA attention kernel at head dims 64, 80, 96 and 112 against the oracle: one and two row
tiles, one and two kv heads a workgroup, the grid with and without splits and the balanced schedule."""
import pytest
import torch

import kyro_amd
from kyro_amd import workloads as wl
from kyro_amd.attention import describe_attention
from tests import helpers as h

pytestmark = pytest.mark.gpu

# (heads, kv heads, context lengths, query rows, num_splits)
SHAPES = {
    "mha_decode": ((4, 4), [1, 15, 16, 17, 33, 0, 500], [1] * 7, 0),
    "pairs_two_tiles": ((16, 4), [300, 31, 64, 7], [5, 8, 1, 7], 0),  # up to 32 rows a kv head
    "odd_heads_three_groups": ((24, 3), [129, 700], [9, 4], 0),       # 72 rows: three 32-row groups
    "grid_splits": ((8, 2), [900, 41, 257], [2, 3, 1], 3),
    "balanced": ((8, 2), [6000, 60, 900, 3000, 5], [3, 1, 4, 2, 4], 0),  # a table wider than 4096 tokens
}


@pytest.mark.parametrize("D", [64, 80, 96, 112])
@pytest.mark.parametrize("name", sorted(SHAPES))
def test_f32_head_dims_parity(gpu, name, D):
    (H, Hkv), ctx, ql, splits = SHAPES[name]
    block = 32 if D == 80 else 16
    case = wl.make_attention_case(context_lens=ctx, q_lens=ql, num_heads=H, num_kv_heads=Hkv, head_dim=D,
                                  block_size=block, dtype="f32", seed=D)
    attn = kyro_amd.PagedAttention(block, H, D, Hkv)
    text = describe_attention(attn, batch=len(ctx), total_q=sum(ql), max_q_len=max(ql),
                              max_blocks_per_seq=case.block_table.shape[1], num_blocks=case.key_cache.shape[0],
                              dtype=torch.float32, num_splits=splits)
    assert text.startswith("attn_mfma_f32_kernel"), text
    t = h.attention_tensors(case, gpu)
    for x in ("key_cache", "value_cache"):  # slots past a context hold NaN
        for b, n in enumerate(ctx):
            if n % block:
                t[x][int(case.block_table[b, n // block]), :, n % block:, :] = float("nan")
    out = attn.forward(t["query"], t["key_cache"], t["value_cache"], t["block_table"], t["context_lens"],
                       q_start_loc=t["q_start_loc"], num_splits=splits)
    h.assert_attention_close(out, case, h.oracle_attention(case), h.ATOL_F32_SUMS)


def test_f32_head_dims_stay_refused_by_name(gpu):
    case = wl.make_attention_case(context_lens=[40], q_lens=[1], num_heads=4, num_kv_heads=2, head_dim=64, dtype="f32")
    t = h.attention_tensors(case, gpu)
    attn = kyro_amd.PagedAttention(16, 4, 64, 2)
    for kw in ({"path": "mfma"}, {"schedule": "balanced"}):
        with pytest.raises(kyro_amd.KyroError):
            attn.forward(t["query"], t["key_cache"], t["value_cache"], t["block_table"], t["context_lens"],
                         q_start_loc=t["q_start_loc"], **kw)


# (heads, kv heads, sequences, query rows, context): contexts short enough that rounding of the scores
# and of the first sums shows, one and two row tiles, and prompts (the many-row kernel).
PRECISION = {
    "decode": (32, 8, 48, 1, 16),
    "mha": (16, 16, 48, 1, 64),
    "verify": (32, 8, 16, 5, 33),
    "prompt": (16, 4, 4, 64, 64),
    "long_prompt": (16, 4, 2, 200, 200),
    "chunk": (16, 4, 2, 64, 500),
}


@pytest.mark.parametrize("D", [64, 80, 96, 112])
@pytest.mark.parametrize("name", sorted(PRECISION))
def test_f32_error_against_64_bits_is_the_vector_kernels(gpu, name, D):
    """Automatic choice must not cost precision over the vector kernel's tree sums: the same 32-bit
    operations in chains no deeper give the same error up to sampling. The ratio of two error norms over
    50 thousand values or more scatters by about 1%, and a few operations more or fewer in either kernel
    move it by another 2%; chains twice as long make it 1.08 or more at every shape but "chunk"."""
    H, Hkv, B, q, ctx = PRECISION[name]
    case = wl.make_attention_case(context_lens=[ctx] * B, q_lens=[q] * B, num_heads=H, num_kv_heads=Hkv, head_dim=D,
                                  dtype="f32", seed=D + ctx)
    t = h.attention_tensors(case, gpu)
    attn = kyro_amd.PagedAttention(case.block_size, H, D, Hkv)
    exact = h.attention_float64(case)
    err = {}
    for path in ("auto", "vector"):
        out = attn.forward(t["query"], t["key_cache"], t["value_cache"], t["block_table"], t["context_lens"],
                           q_start_loc=t["q_start_loc"], path=path)
        err[path] = float((out.cpu().double() - exact).norm() / exact.norm())
    assert err["auto"] <= 1.05 * err["vector"], err


@pytest.mark.parametrize("D", [64, 112])
def test_f32_context_of_one_token_is_its_value(gpu, D):
    case = wl.make_attention_case(context_lens=[1] * 8, q_lens=[1] * 8, num_heads=8, num_kv_heads=2, head_dim=D,
                                  dtype="f32", seed=D)
    t = h.attention_tensors(case, gpu)
    out = kyro_amd.PagedAttention(16, 8, D, 2).forward(t["query"], t["key_cache"], t["value_cache"], t["block_table"],
                                                       t["context_lens"], q_start_loc=t["q_start_loc"])
    v = t["value_cache"][t["block_table"][:, 0], :, 0, :]
    assert torch.equal(out, v.repeat_interleave(4, dim=1))
