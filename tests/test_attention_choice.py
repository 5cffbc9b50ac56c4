"""Which kernel, schedule and parts an attention call takes, as the library describes its own choice (host
only; 256 CUs)."""
import ctypes

import pytest
import torch

import kyro_amd
from kyro_amd import _lib
from kyro_amd.attention import describe_attention

DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32}


def describe(H, Hkv, D, batch, max_q, blocks, dtype="bf16", total_q=None, **kw):
    return describe_attention(kyro_amd.PagedAttention(16, H, D, Hkv), batch=batch, total_q=total_q or batch * max_q,
                              max_q_len=max_q, max_blocks_per_seq=blocks, num_blocks=batch * blocks, dtype=DTYPES[dtype],
                              **kw)


@pytest.mark.parametrize("H,Hkv,D,batch,max_q,blocks,dtype", [
    (32, 8, 128, 2, 4, 63, "bf16"), (8, 2, 128, 1, 1, 19, "bf16"), (32, 8, 64, 4, 1, 19, "bf16"),
    (32, 8, 128, 2, 8, 256, "f32"), (28, 4, 80, 4, 1, 256, "f32"),
])
def test_padding_rows_do_not_choose_the_kernel(H, Hkv, D, batch, max_q, blocks, dtype):
    """q may have rows that belong to no sequence (a batch padded to a captured size): the call takes the
    kernel of the rows its sequences can bring, not the one for many rows."""
    text = describe(H, Hkv, D, batch, max_q, blocks, dtype, total_q=512)
    assert text == describe(H, Hkv, D, batch, max_q, blocks, dtype)
    assert "attn_mfma" in text, text


def part_tiles(H, Hkv, D, batch, max_q, blocks, dtype, ctx, total_q=None):
    """(tiles of a part, most parts) of a sequence of ctx tokens in the many-row kernel; (0, 0) if listed."""
    p = _lib.PagedAttentionParams(16, H, D, Hkv, batch, total_q or batch * max_q, blocks, batch * blocks,
                                  _lib.KYRO_BF16 if dtype == "bf16" else _lib.KYRO_F32, _lib.KYRO_BF16, 1, 0.0, 0, 0, max_q, 0, 0)
    splits = ctypes.c_int()
    n = _lib.lib().kyro_testing_prefill_part_tiles(ctypes.byref(p), 1, ctx, ctypes.byref(splits))
    assert n >= 0
    return n, splits.value


@pytest.mark.parametrize("H,Hkv,D,max_q,dtype", [(32, 8, 128, 64, "bf16"), (16, 1, 128, 128, "bf16"), (16, 1, 192, 24, "bf16"),
                                                 (32, 8, 64, 64, "f32"), (8, 8, 128, 512, "f32")])
def test_parts_follow_the_context_not_the_table(H, Hkv, D, max_q, dtype):
    """One sequence of 4096 tokens in tables of 1 to 64 times that width."""
    tile = 64 if dtype == "bf16" and D <= 128 else 32
    T = 4096 // tile
    tight, most = part_tiles(H, Hkv, D, 1, max_q, 256, dtype, 4096)
    for width in (512, 2048, 16384):
        n, splits = part_tiles(H, Hkv, D, 1, max_q, width, dtype, 4096)
        assert n <= tight and -(-T // n) <= splits
        assert -(-T // n) <= 2 * -(-T // tight)  # nor more parts to merge than twice those of the tight table


@pytest.mark.parametrize("blocks", [64, 300, 4096, 60000])
@pytest.mark.parametrize("dtype", ["bf16", "f32"])
def test_parts_cover_every_length(blocks, dtype):
    tile = 64 if dtype == "bf16" else 32
    for ctx in [0, 1, 2, tile - 1, tile, tile + 1] + [blocks * 16 * i // 97 for i in range(98)]:
        n, splits = part_tiles(32, 8, 64, 1, 128, blocks, dtype, ctx)
        T = -(-ctx // tile)
        assert (n >= 1 or T == 0) and n * splits >= T


def test_sequences_that_may_differ_have_short_parts_or_a_list():
    """Without a list no part of several sequences may pass 1024 tokens (f32: 256) whatever their lengths, or
    twice that where they bring about the same rows."""
    # one row on up to 8192 tokens beside 64-token prompts: listed; on up to 2000 beside 128-token ones: parts
    assert part_tiles(32, 8, 128, 12, 64, 512, "bf16", 8192, total_q=8 * 64 + 4) == (0, 0)
    n, splits = part_tiles(8, 2, 128, 24, 128, 125, "bf16", 2000, total_q=16 + 8 * 128)
    assert splits > 1 and n * 64 <= 1024
    assert part_tiles(16, 1, 128, 2, 128, 8192, "bf16", 4096) == (0, 0)
    assert part_tiles(32, 8, 64, 4, 32, 4096, "f32", 4096) == (0, 0)
    n, splits = part_tiles(32, 8, 128, 2, 64, 256, "bf16", 4096)
    assert splits > 1 and n * 64 <= 1024
    assert part_tiles(32, 8, 128, 16, 128, 64, "bf16", 1024)[1] == 1


@pytest.mark.parametrize("H,Hkv,D,batch,max_q,blocks,dtype,want", [
    # the splits and row groups of a unit group share an XCD: few unit groups do not fill the chip
    (16, 1, 128, 1, 24, 125, "f32", "schedule balanced"),
    (16, 1, 192, 1, 8, 256, "bf16", "schedule balanced"),
    (8, 2, 224, 2, 32, 256, "bf16", "schedule balanced"),
    (28, 4, 128, 1, 24, 125, "f32", "schedule balanced"),
    (16, 1, 96, 1, 1, 256, "bf16", "schedule grid, row groups 1, splits 32,"),
    # one launch takes these whole; two chunks cost more than they save
    (16, 1, 160, 1, 1, 16, "bf16", "schedule grid, row groups 1, splits 1,"),
    (28, 4, 160, 32, 4, 19, "bf16", "schedule grid, row groups 2, splits 1,"),
    (32, 32, 64, 4, 1, 19, "f32", "schedule grid, row groups 1, splits 1,"),
    (4, 4, 64, 1, 8, 16, "f32", "schedule grid, row groups 1, splits 1,"),
    (32, 8, 160, 1, 1, 19, "bf16", "schedule grid, row groups 1, splits 3,"),
    (32, 8, 128, 1, 1, 9, "f32", "schedule grid, row groups 1, splits 2,"),
    (4, 4, 160, 1, 1, 25, "bf16", "schedule grid, row groups 1, splits 4,"),
])
def test_short_chunks_where_they_fit_and_pay(H, Hkv, D, batch, max_q, blocks, dtype, want):
    text = describe(H, Hkv, D, batch, max_q, blocks, dtype)
    assert want in text, text


@pytest.mark.parametrize("H,Hkv,D,batch,max_q,blocks,dtype,many", [
    # short contexts in one round of workgroups stay with the kernels that stream K/V per wave
    (8, 8, 256, 2, 256, 16, "bf16", False),
    (8, 8, 224, 1, 512, 32, "bf16", False),
    (4, 4, 192, 2, 300, 32, "bf16", True),    # fewer workgroups than CUs: split, so scheduled on the device
    (8, 8, 256, 4, 256, 16, "bf16", True),    # two rounds
    (32, 8, 256, 1, 64, 16, "bf16", True),    # two waves a head
    (8, 8, 128, 2, 256, 16, "bf16", True),
    (28, 4, 128, 4, 128, 8, "f32", False),
    (28, 4, 128, 4, 128, 19, "f32", True),
    (8, 1, 128, 1, 256, 19, "f32", True),     # one kv head: its row groups queue on one XCD
    (8, 1, 128, 8, 64, 19, "f32", False),
    (8, 2, 112, 1, 64, 4, "f32", False),
    (8, 2, 112, 1, 64, 9, "f32", True),
])
def test_one_round_of_short_contexts_keeps_its_kernel(H, Hkv, D, batch, max_q, blocks, dtype, many):
    text = describe(H, Hkv, D, batch, max_q, blocks, dtype)
    assert ("attn_prefill_kernel" in text) == many, text


def test_even_sequences_make_no_more_parts_than_they_need():
    assert part_tiles(64, 8, 128, 32, 8, 256, "bf16", 4096) == (32, 2)


def test_describe_names_what_the_many_row_kernel_launches():
    """The plan kernel only where the work is listed, the merge only where there may be parts."""
    listed = describe(32, 8, 64, 6, 512, 500)
    assert "listed by attn_prefill_plan_kernel" in listed and "+ attn_prefill_combine_kernel" in listed
    parts = describe(32, 8, 128, 1, 64, 256)
    assert "attn_prefill_plan_kernel" not in parts and "parts per row group up to 13" in parts
    assert "+ attn_prefill_combine_kernel" in parts
    whole = describe(32, 8, 128, 16, 128, 64)
    assert "parts per row group up to 1," in whole
    assert "plan" not in whole and "combine" not in whole and "16-byte" in whole


@pytest.mark.parametrize("D,dtype", [(64, "bf16"), (128, "bf16"), (256, "bf16"), (64, "f32"), (128, "f32")])
def test_many_row_kernel_follows_the_reuse_hint(D, dtype):
    for reuse, want in (("stream", "stream"), ("shared", "cached"), ("auto", "cached")):
        assert f"attn_prefill_kernel<{dtype}, head_dim {D}, K/V loads {want}>" in describe(32, 8, D, 2, 512, 64, dtype,
                                                                                       kv_reuse=reuse)
    assert "K/V loads stream" in describe(64, 8, 128, 64, 9, 256)  # each slab read once
