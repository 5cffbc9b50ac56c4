"""Attention with many query rows per kv head (prompts and chunks of prompts): the many-row kernel
against the oracle where its tiles, row groups, parts and schedules have their edges."""
import numpy as np
import pytest
import torch

import kyro_amd
from kyro_amd import workloads as wl
from kyro_amd.attention import describe_attention
from tests import helpers as h

pytestmark = pytest.mark.gpu

# (heads, kv heads, context lengths, query rows). Row groups are 128 rows (token x head of the
# group), waves 32, K/V tiles 64 or 32 tokens.
EDGES = {
    # four heads a kv head: 124, 128, 132, 256, 260, .. rows; contexts around a tile, one token, none
    "edges": ((8, 2), [31, 32, 33, 70, 65, 1, 0, 300], [31, 32, 33, 64, 65, 1, 3, 200]),
    # rows that see nothing (context shorter than the new rows), a group of 7
    "gqa7": ((14, 2), [40, 700, 33], [60, 100, 33]),
    # few row groups over a long context: split into parts by the host alone
    "parts": ((8, 1), [5000, 4990], [64, 40]),
    # lengths far apart: the listed schedule, with and without split row groups
    "ragged": ((8, 2), [3000, 90, 700, 17, 1500], [40, 80, 512, 17, 200]),
}
# a verify step of 72 rows per kv head: one row group a unit, streaming loads
EDGES["verify72"] = ((64, 8), [700, 9, 64, 65, 300, 1, 0, 1300] * 2, [9] * 16)
DIMS = [("bf16", D) for D in (64, 80, 96, 112, 128, 160, 192, 224, 256)] + [("f32", D) for D in (64, 80, 96, 112, 128)]


def _case(name, dtype, D, block=16, seed=0):
    (H, Hkv), ctx, ql = EDGES[name]
    if dtype == "f32" and D == 128:  # this path takes f32 from 512 rows a sequence on
        H *= 4
    return wl.make_attention_case(context_lens=ctx, q_lens=ql, num_heads=H, num_kv_heads=Hkv, head_dim=D,
                                  block_size=block, dtype=dtype, seed=seed + D)


def _attention(case):
    return kyro_amd.PagedAttention(case.block_size, case.num_heads, case.head_dim, case.num_kv_heads)


def _args(t):
    return t["query"], t["key_cache"], t["value_cache"], t["block_table"], t["context_lens"]


def _takes_many_rows(case):
    q = np.diff(case.q_start_loc)
    dtype = torch.bfloat16 if case.dtype == "bf16" else torch.float32
    return "attn_prefill_kernel" in describe_attention(
        _attention(case), batch=case.batch, total_q=int(q.sum()), max_q_len=int(q.max()),
        max_blocks_per_seq=case.block_table.shape[1], num_blocks=case.key_cache.shape[0], dtype=dtype)


# 72 rows per kv head take this kernel in bf16 at head dim 128 alone.
@pytest.mark.parametrize("name,dtype,D", [(name, dtype, D) for name in sorted(EDGES) for dtype, D in DIMS
                                          if name != "verify72" or (dtype, D) == ("bf16", 128)], ids=lambda x: str(x))
def test_many_rows_parity(gpu, name, dtype, D):
    case = _case(name, dtype, D, block=32 if D % 96 == 0 else 16)
    t = h.attention_tensors(case, gpu)
    exp = h.oracle_attention(case)
    out = _attention(case).forward(*_args(t), q_start_loc=t["q_start_loc"])
    h.assert_attention_close(out, case, exp, h.ATOL_BF16 if dtype == "bf16" else h.ATOL_F32_SUMS)


def test_the_edges_reach_the_many_row_kernel():
    taken = [name for name in sorted(EDGES) for dtype, D in (("bf16", 128), ("f32", 64)) if _takes_many_rows(_case(name, dtype, D))]
    assert taken == [name for name in sorted(EDGES) for _ in range(1 if name == "verify72" else 2)]


@pytest.mark.parametrize("dtype,D,block", [("bf16", 128, 16), ("bf16", 80, 64), ("f32", 64, 32)])
def test_many_rows_block_sizes_noncausal_and_nan_past_the_context(gpu, dtype, D, block):
    """Every cache slot past a context holds NaN, and so does every block no table names."""
    case = _case("ragged", dtype, D, block=block, seed=3)
    assert _takes_many_rows(case)
    t = h.attention_tensors(case, gpu)
    used = torch.zeros(case.key_cache.shape[0], block, dtype=torch.bool)
    for b in range(case.batch):
        for i in range(int(case.context_lens[b])):
            used[int(case.block_table[b, i // block]), i % block] = True
    hole = (~used).to(gpu)[:, None, :, None]
    for x in ("key_cache", "value_cache"):
        t[x] = t[x].masked_fill(hole, float("nan"))
    for causal in (True, False):
        out = _attention(case).forward(*_args(t), q_start_loc=t["q_start_loc"], causal=causal, out_dtype=torch.bfloat16)
        assert out.dtype == torch.bfloat16
        h.assert_attention_close(out, case, h.oracle_attention(case, causal=causal),
                                 h.ATOL_BF16 if dtype == "bf16" else h.ATOL_BF16 / 2)


def test_many_rows_after_a_much_larger_score(gpu):
    """One early token with a score hundreds above the rest: the running reference must not let the
    accumulator overflow while later tiles' maxima are far below it."""
    case = _case("ragged", "bf16", 128, seed=5)
    t = h.attention_tensors(case, gpu)
    first = t["block_table"][:, 0]
    t["key_cache"][first, :, 0, :] = 40.0 * torch.sign(t["key_cache"][first, :, 0, :].float()).to(torch.bfloat16)
    case.key_cache = t["key_cache"].view(torch.int16).cpu().numpy().view(np.uint16)
    out = _attention(case).forward(*_args(t), q_start_loc=t["q_start_loc"])
    h.assert_attention_close(out, case, h.oracle_attention(case), 4 * h.ATOL_BF16)  # values up to 4


@pytest.mark.parametrize("dtype,D", [("bf16", 128), ("bf16", 64), ("f32", 64), ("f32", 128)])
def test_many_rows_large_values_after_a_much_larger_score(gpu, dtype, D):
    """The same with values of 1e30: every weighted sum is far below the type's largest value, and so must
    be whatever the kernel holds on the way. (bf16: three roundings of 2^-9; sums of like sign aside, the
    error of an output is bounded by 4 * 2^-9 of the largest value.)"""
    case = _case("ragged", dtype, D, seed=6)
    t = h.attention_tensors(case, gpu)
    first = t["block_table"][:, 0]
    t["key_cache"][first, :, 0, :] = 40.0 * torch.sign(t["key_cache"][first, :, 0, :])
    t["value_cache"] *= 1e30
    for x in ("key_cache", "value_cache"):
        host = t[x].cpu()
        setattr(case, x, host.view(torch.int16).numpy().view(np.uint16) if dtype == "bf16" else host.numpy())
    out = _attention(case).forward(*_args(t), q_start_loc=t["q_start_loc"]).cpu().double()
    assert torch.isfinite(out).all()
    exact = h.attention_float64(case)
    assert float((out - exact).abs().max()) <= (4 * 2.0 ** -9 if dtype == "bf16" else 1e-4) * float(t["value_cache"].abs().max())


@pytest.mark.parametrize("dtype,D", [("bf16", 128), ("bf16", 256), ("f32", 64)])
@pytest.mark.parametrize("heads,ctx,ql", [((8, 1), [5000], [64]), ((8, 2), [700], [512]), ((8, 1), [64], [64]),
                                          ((16, 1), [3000, 40, 0, 900], [32, 40, 3, 32]), ((8, 2), [0], [200])])
def test_many_rows_wide_table(gpu, dtype, D, heads, ctx, ql):
    """Tables of 32768 tokens, as a server that sizes them for its longest context passes: parts by the
    context of one sequence, a list for several."""
    case = wl.make_attention_case(context_lens=ctx, q_lens=ql, num_heads=heads[0], num_kv_heads=heads[1], head_dim=D,
                                  dtype=dtype, seed=D + len(ctx))
    table = np.zeros((case.batch, 2048), np.int64)
    table[:, :case.block_table.shape[1]] = case.block_table
    case.block_table = table
    assert _takes_many_rows(case)
    t = h.attention_tensors(case, gpu)
    out = _attention(case).forward(*_args(t), q_start_loc=t["q_start_loc"])
    h.assert_attention_close(out, case, h.oracle_attention(case), h.ATOL_BF16 if dtype == "bf16" else h.ATOL_F32_SUMS)


@pytest.mark.parametrize("dtype,D", DIMS, ids=lambda x: str(x))
def test_many_rows_reuse_hint_never_changes_the_result(gpu, dtype, D):
    case = _case("ragged", dtype, D, seed=13)
    assert _takes_many_rows(case)
    t = h.attention_tensors(case, gpu)
    outs = [_attention(case).forward(*_args(t), q_start_loc=t["q_start_loc"], kv_reuse=r) for r in ("auto", "shared", "stream")]
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])


def test_many_rows_errors_latch(gpu):
    """A bad block id, a context longer than its table and rows out of order are reported; the
    sequences without a fault are computed as before."""
    case = _case("ragged", "bf16", 128, seed=7)
    exp = h.oracle_attention(case)
    attn = _attention(case)
    for fault in ("block", "context", "rows"):
        t = h.attention_tensors(case, gpu)
        hurt = {2}
        if fault == "block":
            t["block_table"][2, 3] = case.key_cache.shape[0]
        elif fault == "context":
            t["context_lens"][2] = case.block_table.shape[1] * 16 + 1
        else:
            t["q_start_loc"][3] = t["q_start_loc"][2] - 1
            hurt = {2, 3}  # both have the entry as a bound
        out = torch.zeros_like(t["query"], dtype=torch.float32)
        with pytest.raises(kyro_amd.KyroError):
            attn.forward(*_args(t), q_start_loc=t["q_start_loc"], max_q_len=512, out=out)
        h.assert_attention_close(out, case, {b: e for b, e in exp.items() if b not in hurt}, h.ATOL_BF16)


@pytest.mark.parametrize("name", ["parts", "ragged"])
def test_many_rows_replay_from_a_graph(gpu, name):
    case = _case(name, "bf16", 128, seed=9)
    t = h.attention_tensors(case, gpu)
    attn = _attention(case)
    kw = dict(q_start_loc=t["q_start_loc"], max_q_len=int(np.diff(case.q_start_loc).max()))
    eager = attn.forward(*_args(t), **kw)
    out = torch.zeros_like(eager)
    s = torch.cuda.Stream(gpu)
    s.wait_stream(torch.cuda.current_stream(gpu))
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        attn.forward_async(*_args(t), out=out, **kw)
    for _ in range(3):
        out.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager)
        assert torch.equal(attn.forward(*_args(t), **kw), eager)


def test_many_rows_misaligned_cache_takes_another_kernel(gpu):
    """Caches that start 8 bytes off a 16-byte boundary run on the kernels that stream K/V per wave: bit for
    bit what the grid schedule by name gives, and not what the many-row kernel gives."""
    case = _case("edges", "bf16", 128, seed=11)
    assert _takes_many_rows(case)
    t = h.attention_tensors(case, gpu)
    kw = dict(q_start_loc=t["q_start_loc"])
    many = _attention(case).forward(*_args(t), **kw)
    grid = _attention(case).forward(*_args(t), schedule="grid", **kw)
    for x in ("key_cache", "value_cache"):
        flat = torch.zeros(t[x].numel() + 8, dtype=torch.bfloat16, device=gpu)
        flat[4:4 + t[x].numel()] = t[x].flatten()
        t[x] = flat[4:4 + t[x].numel()].view(t[x].shape)
        assert t[x].data_ptr() % 16 == 8
    out = _attention(case).forward(*_args(t), **kw)
    h.assert_attention_close(out, case, h.oracle_attention(case), h.ATOL_BF16)
    assert torch.equal(out, grid) and not torch.equal(out, many)
